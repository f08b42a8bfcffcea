// What the prefill grouped GEMMs share: kernel arguments, an item's metadata, and the order in
// which the workgroups walk the tile list.
//
// Two things bound a prefill GEMM, and a chunk whose routing is skewed has both. A tile alone with
// its expert is bound by its weights' read: 256 columns x 2560 deep are 655 KB, which a CU takes
// from HBM at 25-50 KB/us (its vector L1 keeps at most its 32 KB in flight) and which nobody
// else needs. The tiles of an expert that has several share their weights in an XCD's L2 and
// are bound by the matrix cores and the LDS. Walked in list order the CUs of an XCD meet the two
// kinds in phases, and the phases add up: at 4096 tokens of Zipf(1.1) routing over 512 experts
// (701 tiles, 240 of them of shared experts) gate_up took 580-600 us, the shared tiles alone 240
// and the others alone 300. So each XCD's workgroups are split between the two kinds in
// proportion to their cost, and both run all the time (below, Sched).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemm_common.h"
#include "prefill.h"
#include "wave.h"

namespace rlu {
namespace pf {

constexpr int TB = 8;           // 16-row blocks per tile: the tile list's tile size
constexpr int NXCD = 8;
constexpr int NWAVE = 8;        // waves per workgroup
constexpr int BUF_WORD3 = 0x00020000;   // raw buffer descriptor word 3 on gfx9 (no format)
// Buffer cache policies of the weight loads. Weights read once stream (7.0 against 6.0-6.3 TB/s
// over 256 CUs); those several tiles read must stay in the L2 (a region all CUs of an XCD read
// in step: 29 TB/s plain, 17-20 streaming).
constexpr int POL_STREAM = 2, POL_SHARED = 0;

struct Args {
  const uint8_t* qx;
  const float* xs;
  const uint8_t* wq;
  const float* ws;
  const int* sorted_ids;
  const int* eids;
  const uint8_t* wq1;            // the second set (tiles with set bit 1); the first when unused
  const float* ws1;
  const int* sorted_ids1;
  const int* eids1;
  bool two;                      // a two-set tile list
  bool far;                      // ... of which the second set is in host memory
  const int* tiles;
  const int* ntiles;
  uint16_t* y;
  const float* tw;
  uint8_t* q2;
  float* s2;
  int mtk;
  int top_k;
  int K;
  int N;
};

struct Item {
  int b0, nbk, e, n0, set;
};

typedef unsigned v2u __attribute__((ext_vector_type(2)));

// The gate_up-shaped kernel of prefill_roll.hip; launched for K % 128 == 0, K >= 512.
void launch_roll(const Args& a, int max_tiles, hipStream_t stream);

constexpr int ORD_MAX = 2048;   // tiles of one XCD's share that the LDS order holds
constexpr int SORT_MAX = 16384; // tiles the scheduler takes
constexpr int ORD_BYTES = ORD_MAX * 2;
constexpr int SCRATCH_BYTES = SORT_MAX + 64 + 2 * (SORT_MAX / WAVE) * 4;

// The list of tiles a workgroup walks and its place in it: its items are first + m * step of the
// n * (column groups) items of the list, tile k of which is `tile(k)`.
struct Sched {
  int n, first, step;
  int base, dir;                // LDS index of tile 0 and direction; dir 0: tile base + k
  bool shared;                  // the tiles of experts with several

  __device__ __forceinline__ int tile(const unsigned char* ord, int k) const {
    if (dir == 0) return base + k;
    return uniform((int)reinterpret_cast<const uint16_t*>(ord)[base + dir * k]);
  }
};

// Cost of a tile of k blocks in units of about 2.2 us per 256 x 2560 item: 15 + 2.3 k us from a
// hot L2. With 7 + k for both kinds gate_up at 4096 / 8192 tokens takes 505 / 720 us; dearer or
// cheaper unshared tiles (10 + k, 5 + k) 541 / 769 and 533 / 777.
__device__ __forceinline__ int tile_cost(int k) { return 7 + k; }

// Rows per tile below which the list order is kept: most tiles are then alone with their expert
// and a split gains nothing (2048 tokens over 512 experts, 35 rows per tile: gate_up + down 698 ->
// 650 us with the split; 1200 tokens, 22 rows: 610 -> 633).
constexpr int SPLIT_ROWS = 24;

// Every workgroup computes the same split from the tile list, in LDS (2-4 us): shared tiles go to
// the XCDs in contiguous runs of equal cost (an expert's tiles then run in one L2), the others
// round-robin; each XCD's workgroups (b % 8 is the XCD of workgroup b) are divided between its
// two lists by cost (ncg: column groups, items per tile). scratch: SCRATCH_BYTES of LDS that the
// kernel does not use yet; ord: ORD_BYTES that it keeps. List order, an equal share of the tiles
// per XCD, where there is nothing to split.
// far: a two-set list's second set is in host memory. Its tiles wait for the host link, for fifty times
// as long as all the others together, and they stand behind the first set's, so in list order each
// XCD leaves the link idle until its unshared tiles of the first set are done: the unshared tiles
// are then walked from the end. 512 experts, 257 of them resident, 2048 / 4096 tokens: 28.2 ->
// 27.2 / 27.5 ms (unsplit, 27.6 / 27.5); 128 experts, 65 resident, 617 / 4096 tokens: 6.59 -> 5.51 /
// 5.71 -> 5.45 ms (unsplit 6.45 / 6.78). From both ends in turn: 28.0 / 27.8, 6.15 / 5.71. With both
// sets in HBM the reverse order costs 1-3% (2048 tokens 686 -> 704 us): the resident experts'
// larger tiles then come last.
template <bool TWO>
__device__ __forceinline__ Sched make_sched(unsigned char* scratch, unsigned char* ord,
                                            const int* __restrict__ tiles, int nt, int mtk, int ncg,
                                            const int* __restrict__ eids,
                                            const int* __restrict__ eids1, bool far) {
  const int nx = gridDim.x % NXCD == 0 ? NXCD : 1;
  const int x = (int)blockIdx.x % nx, j = (int)blockIdx.x / nx, per = (int)gridDim.x / nx;
  Sched s;
  s.first = j;
  s.step = per;
  s.base = (int)((long long)nt * x / nx);
  s.n = (int)((long long)nt * (x + 1) / nx) - s.base;
  s.dir = 0;
  s.shared = false;
  if (nt > SORT_MAX || per < 2 || per > 1023 || mtk < (long long)SPLIT_ROWS * nt) return s;
  constexpr int MAXCH = SORT_MAX / WAVE;
  const int lane = lane_id(), w = uniform((int)threadIdx.x / WAVE);
  uint8_t* nb = scratch;                            // block count | shared << 4, per tile
  int* sum = reinterpret_cast<int*>(scratch + SORT_MAX);
  int* cost = sum + 16;                             // per 64-tile chunk: cost of the shared tiles
  int* alone = cost + MAXCH;                        // ... and number of the others, then their
                                                    // sums over the chunks before
  const int nch = (nt + WAVE - 1) / WAVE;
  // a tile is shared when a neighbour of the list is of the same expert (only a full tile has a
  // successor of its own expert)
  for (int c = w; c < nch; c += NWAVE) {
    const int i = c * WAVE + lane;
    const bool in = i < nt;
    auto expert = [&](int q, int wd) __attribute__((always_inline)) {
      return (TWO && (wd >> 16) ? eids1 : eids)[tiles[2 * q]];
    };
    const int wd = in ? tiles[2 * i + 1] : 0, k = wd & 0xffff;
    const int wp = in && i > 0 ? tiles[2 * i - 1] : 0;
    const int wn = in && i + 1 < nt ? tiles[2 * i + 3] : 0;
    bool shared = false;
    if (k == TB || (wp & 0xffff) == TB) {
      const int e = expert(i, wd);
      shared = (k == TB && wn && (wn >> 16) == (wd >> 16) && expert(i + 1, wn) == e) ||
               ((wp & 0xffff) == TB && (wp >> 16) == (wd >> 16) && expert(i - 1, wp) == e);
    }
    if (in) nb[i] = (uint8_t)(k | (shared ? 16 : 0));
    const int cs = wave_sum(in && shared ? tile_cost(k) : 0);
    const int na = __popcll(__ballot(in && !shared));
    if (lane == 0) {
      cost[c] = cs;
      alone[c] = na;
    }
  }
  __syncthreads();
  if (w == 0) {
    int rc = 0, ra = 0;
    for (int c0 = 0; c0 < nch; c0 += WAVE) {
      const int c = c0 + lane;
      const int vc = c < nch ? cost[c] : 0, va = c < nch ? alone[c] : 0;
      const int ic = wave_incl_scan(vc), ia = wave_incl_scan(va);
      if (c < nch) {
        cost[c] = rc + ic - vc;
        alone[c] = ra + ia - va;
      }
      rc += readlane(ic, WAVE - 1);
      ra += readlane(ia, WAVE - 1);
    }
    if (lane < 5) sum[lane] = lane == 0 ? rc : lane == 1 ? ra : 0;
  }
  __syncthreads();
  const int total = uniform(sum[0]), nalone = uniform(sum[1]);
  // nothing shared; or, the same answer on every XCD, more tiles than an XCD's order surely holds
  // (the midpoints of shared tiles are at least tile_cost(1) apart)
  if (total == 0 || total / (nx * tile_cost(1)) + nalone / nx + 2 > ORD_MAX) {
    __syncthreads();                                // every wave has read the sums
    return s;
  }
  uint16_t* o = reinterpret_cast<uint16_t*>(ord);
  // shared tile at cost [p, p + c) of the total: XCD floor(nx * its midpoint / total)
  auto mine = [&](int p, int c) __attribute__((always_inline)) {
    return (int)((long long)(2 * p + c) * nx / (2LL * total)) == x;
  };
  // this XCD's others, from the back of the order; its shared tiles' number and cost
  const int na = nalone > x ? (nalone - x + nx - 1) / nx : 0;
  int ns = 0, cs = 0, ca = 0;
  for (int c = w; c < nch; c += NWAVE) {
    const int i = c * WAVE + lane;
    const int v = i < nt ? nb[i] : 0, k = v & 15;
    const bool shd = (v & 16) != 0, oth = v != 0 && !shd;
    const int tc = shd ? tile_cost(k) : 0;
    const int p = cost[c] + wave_incl_scan(tc) - tc;
    const int q = alone[c] + mbcnt(__ballot(oth));
    if (oth && q % nx == x) {
      o[ORD_MAX - 1 - (TWO && far ? na - 1 - q / nx : q / nx)] = (uint16_t)i;
      ca += tile_cost(k);
    }
    if (shd && mine(p, tc)) {
      ++ns;
      cs += tc;
    }
  }
  ns = wave_sum(ns);
  cs = wave_sum(cs);
  ca = wave_sum(ca);
  if (lane == 0) {
    atomicAdd(&sum[2], ns);
    atomicAdd(&sum[3], cs);
    atomicAdd(&sum[4], ca);
  }
  __syncthreads();
  const int nshared = uniform(sum[2]);
  cs = uniform(sum[3]);
  ca = uniform(sum[4]);
  if (w == 0) {                                     // its shared tiles, in list order
    int n = 0;
    for (int c = 0; c < nch && n < nshared; ++c) {
      const int i = c * WAVE + lane;
      const int v = i < nt ? nb[i] : 0;
      const bool shd = (v & 16) != 0;
      const int tc = shd ? tile_cost(v & 15) : 0;
      const int p = cost[c] + wave_incl_scan(tc) - tc;   // (a scan: every lane takes part)
      const bool me = shd && mine(p, tc);
      const uint64_t m = __ballot(me);
      if (me) o[n + mbcnt(m)] = (uint16_t)i;
      n += __popcll(m);
    }
  }
  __syncthreads();                                  // the order is written, the scratch is read
  // Workgroups of the shared list: the number whose slower list is done first, in whole items at
  // the list's mean cost (a share rounded to whole workgroups leaves a list of one or two
  // workgroups up to half as long again: down of 128 experts at 4096 tokens, 320 tiles, 147
  // against 135 us).
  int js = na == 0 ? per : 0;
  if (nshared && na) {
    const int ia = nshared * ncg, ib = na * ncg;
    const float ta = (float)cs / nshared, tb = (float)ca / na;
    uint32_t best = ~0u, worst = 0;
    for (int q = 1 + lane; q < per; q += WAVE) {
      const float t = fmaxf((float)((ia + q - 1) / q) * ta,
                            (float)((ib + per - q - 1) / (per - q)) * tb);
      best = min(best, (uint32_t)fminf(16.f * t, 4194303.f) << 10 | (uint32_t)q);
    }
    wave_minmax_u32(best, worst);
    js = (int)(best & 1023);
  }
  s.shared = j < js;
  s.n = s.shared ? nshared : na;
  s.first = s.shared ? j : j - js;
  s.step = s.shared ? js : per - js;
  s.base = s.shared ? 0 : ORD_MAX - 1;
  s.dir = s.shared ? 1 : -1;
  return s;
}

}  // namespace pf
}  // namespace rlu
