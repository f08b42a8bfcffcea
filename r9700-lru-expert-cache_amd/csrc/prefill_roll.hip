// The rolled prefill GEMM: same items, operands, tile list and numerics as the unrolled kernel of
// prefill.hip (equal bit for bit), for K a run-time multiple of 128 from 512 on, with the K loop a
// loop and each step software-pipelined. It runs gate_up of the 2560-wide model, alone or
// with SiLU-mul-quant in its epilogue, and both GEMMs of shapes with such a K: at 2048 / 8192
// tokens over 128 experts gate_up (K 2048, N 1536) takes 143 / 400 us, tiled_k 190 / 565; over 64
// experts down (K 1024, N 2048) 94 / 252 us, tiled_k 117 / 426. At one or two blocks per tile the
// two kinds differ less (64 tokens: 68 against 79 us, and 37 against 39).
//
// Bound: with few rows per tile the weight read (all 512 experts of gate_up, 2.01 GB, in 330-345
// us = 5.9-6.1 TB/s; a bare read in this pattern, 7.0); with full tiles, at 1.2-1.3 PFLOP/s with the
// weights in the L2, three units that overlap only in part: a step of 8 blocks is 32 cycles for each of
// a SIMD's 32 MFMAs, 128 KB of LDS reads (each fragment feeds two MFMAs), about as long, and the
// scaling of every product. Counted over 32 experts' full tiles with the activation: MFMA busy
// 23% of the cycles, LDS 21% (1% conflicts), vector instructions 40%, at 2.2 GHz.
//
//   * An item is (tile of <= 8 16-row blocks of one expert, 256 columns); wave w of 8 owns 2
//     16-column weight strips and streams them through a ring of KC = 4 register steps that runs
//     on across chunks and items. Rows go to LDS in chunks of KC steps, double-buffered, loaded
//     into registers one chunk ahead; one barrier per chunk.
//   * The unrolled form (40 steps of code, 90 KB, past the 64 KB instruction cache) issued each
//     block's LDS read, MFMA and scaling one after another. Here the step's code is a 12 KB
//     loop body in which a block's operands are read two blocks ahead and its products scaled
//     one block later, and the activation x weight scale is multiplied once per row when the
//     chunk is staged instead of in every wave. Full tiles of 32 experts (320 tiles): 277-306 ->
//     252-264 us; in cycles 884k -> 679k, of which the lower clock gives back a part.
//   * A wave whose block the tile does not have loads and stages nothing.
//   * Item metadata comes through vector loads, a stage per chunk, two items ahead.
//   * The order of the items is Sched's (prefill_sched.h); the workgroups of the shared list load
//     weights with the plain cache policy, the others streaming.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemm_common.h"
#include "numerics.h"
#include "prefill_sched.h"
#include "quant_row.h"
#include "rlu.h"
#include "wave.h"

namespace rlu {
namespace pf {
namespace roll {

constexpr int S = 2;                   // 16-column weight strips per wave
constexpr int C = 16 * S * NWAVE;      // columns per item
constexpr int KC = 4;                  // K steps per activation chunk, and depth of the weight ring

// LDS: the small arrays, the two activation buffers (at most 64 KB each, so that every constant
// offset into one fits the 16-bit offset of a ds instruction), each wave's epilogue staging (one
// block's [16 rows][S 16 columns] bf16) and the order
constexpr int SX = 2 * 2 * KC * TB * 16;                   // float [buf][col block][ks][row]
constexpr int RW = 2 * TB * 16;                            // int / float [par][row]
constexpr int A_OFF = (SX + 2 * RW) * 4;
constexpr int A_BUF = TB * KC * 2 * 1024;                  // [blk][ks][h][lane] x 16 B
static_assert(A_BUF <= 65536, "an activation buffer must fit one ds offset range");
constexpr int EPI_W = 16 * S * 16 * 2;
constexpr int EPI_OFF = A_OFF + 2 * A_BUF;
constexpr int ORD_OFF = EPI_OFF + NWAVE * EPI_W;
constexpr size_t LDS = (size_t)ORD_OFF + ORD_BYTES;
static_assert(SCRATCH_BYTES <= ORD_OFF, "the scheduler's scratch lies below the order");
// blocks of bf16 outputs ([16 rows][C]) one activation buffer holds in the ACT epilogue
constexpr int BP = A_BUF / (16 * C * 2);
static_assert(BP >= 1 && TB % BP == 0, "an epilogue pass holds whole blocks");

// the value of lane I of this lane's quad
template <int I>
__device__ __forceinline__ float quad(float x) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), I * 0x55, 0xf, 0xf, true));
}

// Chunks of an item of nk steps. TAIL: the last chunk has what KC leaves of them, nothing where they
// are one chunk alone (the metadata pipeline takes two). (max and no branch: on one, the compiler
// copies the loop for two chunks and spills 155-202 registers.)
template <bool TAIL>
__host__ __device__ __forceinline__ int chunks(int nk) {
  return TAIL ? max(2, (nk + KC - 1) / KC) : nk / KC;
}
inline bool has_tail(int K) { return K % (KC * 128) != 0 || K < 2 * KC * 128; }

// Chunk c's loads of one lane's row, byte va of qbytes bytes of activations on: ld(ks, h, bytes,
// voffset, soffset) reads 16 bytes through a buffer of `bytes`, zeros where voffset is past it. Only
// the vector offset is sure to count in a buffer's range check, so a step that K does not have
// (TAIL) and every step of a block that the tile does not have take an empty buffer, instead of
// reading on: into the next row, and behind the last one past the tensor.
template <bool TAIL, class LD>
__host__ __device__ __forceinline__ void row_loads(int qbytes, int nk, int va, int c, bool live,
                                                   const LD& ld) {
#pragma unroll
  for (int ks = 0; ks < KC; ++ks) {
    const int bytes = live && (!TAIL || c * KC + ks < nk) ? qbytes : 0;
    ld(ks, 0, bytes, va + ks * 128, c * KC * 128);
    ld(ks, 1, bytes, va + ks * 128 + 64, c * KC * 128);
  }
}

// The weight steps that chunk c's walk loads ahead: the next chunk's, of this item or (last) of the next.
// After a workgroup's last item (!more) none: its first KC steps again would be 33 MB over 256
// workgroups, 0.55 ms where the weights come over the host link (gate_up over 256 experts, half of
// them in host memory, 195 tokens: layer step 4.68 -> 4.09 ms).
template <bool TAIL>
__host__ __device__ __forceinline__ int steps_ahead(int nk, int c, bool last, bool more) {
  if (last) return more ? KC : 0;
  return TAIL ? nk - (c + 1) * KC : KC;
}

// ACT: SiLU-mul-quant in the epilogue. N = 2 I (gate | up); item g covers gate columns [128 g,
// 128 g + 128) (waves 0 .. 3) and the matching up columns [I + 128 g, ...) (waves 4 .. 7), so
// each output row's 128-column activation group is whole in one item. The epilogue writes q2
// [mtk, I] e4m3 and s2 [mtk, I / 128] instead of y, computed from the bf16-rounded GEMM outputs
// exactly as silu_mul_quant_k computes them from y (same silu, product and amax reduction, same
// rounding). TWT: routed weights. TWO: the tile list covers two aligns (bit 16 of a tile's block
// count picks the set). POL: the weight loads' cache policy.
template <int POL, bool TWT, bool ACT, bool TWO, bool WIDE, bool TAIL>
__device__ __forceinline__ void items(
    const Sched& sc, const uint8_t* __restrict__ qx, const float* __restrict__ xs,
    const uint8_t* __restrict__ wq, const float* __restrict__ ws,
    const int* __restrict__ sorted_ids, const int* __restrict__ eids,
    const uint8_t* __restrict__ wq1, const float* __restrict__ ws1,
    const int* __restrict__ sorted_ids1, const int* __restrict__ eids1,
    const int* __restrict__ tiles, uint16_t* __restrict__ y, const float* __restrict__ tw,
    uint8_t* __restrict__ q2, float* __restrict__ s2, int mtk, int top_k, int K, int N,
    int qbytes) {
  static_assert(!ACT || !TWT, "gate_up takes no routed weights");
  extern __shared__ __align__(16) unsigned char smem[];
  float* sx = reinterpret_cast<float*>(smem);
  int* rows = reinterpret_cast<int*>(sx + SX);
  float* twl = reinterpret_cast<float*>(rows + RW);

  const int lane = lane_id();
  const int w = uniform((int)(threadIdx.x / WAVE));
  const int r16 = lane & 15, c4 = lane >> 4;
  const int cb = w / (NWAVE / 2);                       // this wave's 128-column scale block
  const int nk = K / 128;
  const int nch = chunks<TAIL>(nk);
  const int ncg = N / C;
  // first output column of scale block h of an item starting at column n0
  auto bcol = [&](int n0, int h) __attribute__((always_inline)) -> int {
    return ACT ? n0 / 2 + h * (N / 2) : n0 + h * 128;
  };
  const int wcol = (w - cb * (NWAVE / 2)) * S * 16;     // this wave's columns inside its block
  const int cnt = (sc.n * ncg - sc.first + sc.step - 1) / sc.step;   // this workgroup's items

  // An item's place in the order: its tile and its first column. Its metadata is read through
  // vector loads issued chunks ahead (tile words during one chunk, expert id and row ids during
  // a later one): they retire in order with the weights, where scalar loads would make every LDS
  // wait behind them wait for the memory.
  int vz;                                           // a zero the compiler takes for per-lane
  asm volatile("v_mov_b32 %0, 0" : "=v"(vz));
  struct Place {
    int ti, n0;
  };
  auto place = [&](int m) __attribute__((always_inline)) {
    const int it = sc.first + (m < cnt ? m : cnt - 1) * sc.step;
    const int k = it / ncg;
    return Place{sc.tile(smem + ORD_OFF, k), (it - k * ncg) * C};
  };
  auto load_tile = [&](const Place& p) __attribute__((always_inline)) -> v2u {
    return *reinterpret_cast<const v2u*>(tiles + 2 * p.ti + vz);
  };
  auto take_tile = [&](v2u t, Item& r) __attribute__((always_inline)) {
    const int nw = uniform((int)t.y);              // block count | set << 16 (TWO)
    r.b0 = uniform((int)t.x);
    r.nbk = TWO ? nw & 0xffff : nw;
    r.set = TWO ? nw >> 16 : 0;
  };
  auto load_eid = [&](const Item& r) __attribute__((always_inline)) -> int {
    return (r.set ? eids1 : eids)[r.b0 + vz];
  };
  // the sorted id of row r16 of this wave's block of an item (any id where it has no such block)
  auto load_id = [&](const Item& r) __attribute__((always_inline)) -> int {
    return (r.set ? sorted_ids1 : sorted_ids)[(r.b0 + (w < r.nbk ? w : 0)) * 16 + r16];
  };
  // this wave's strips of an item, as a buffer: strip s, step k, half h at s 16 K + k 2048 +
  // h 1024 + lane 16 (the base and the step offset stay in scalar registers)
  // steps: 0 for a buffer whose loads touch no memory
  auto wbuf = [&](const uint8_t* p, bool any) __attribute__((always_inline)) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, any ? S * 16 * K : 0, BUF_WORD3);
  };
  auto wptr = [&](const Item& it) __attribute__((always_inline)) {
    return (it.set ? wq1 : wq) + ((size_t)it.e * N + bcol(it.n0, cb) + wcol) * K;
  };

  // ---- registers ----
  v4u rb[KC][S][2];                    // weight ring
  v4u ra[KC][2];                      // next chunk's activation rows (this wave's block)
  float rx, rw0, rw1, rt;             // ... their scales, the item's block scales, routed weight
  v4f acc[TB][S];

  const int voff = lane * 16;
  auto issue_b = [&](int j, __amdgpu_buffer_rsrc_t base, int off) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      rb[j][s][0] = __builtin_bit_cast(
          v4u, __builtin_amdgcn_raw_buffer_load_b128(base, voff, s * 16 * K + off, POL));
      rb[j][s][1] = __builtin_bit_cast(
          v4u, __builtin_amdgcn_raw_buffer_load_b128(base, voff + 1024, s * 16 * K + off, POL));
    }
  };
  // what the staging of an item's chunks needs: this lane's row (r16 of this wave's block) in
  // the activation rows and their scales, and the item's weight scales
  struct Rows {
    int va;                           // byte offset of the row, + 16 c4 (WIDE: the row)
    int vx;                           // index of the row's scales
    const float* w0;                  // weight scales of the first column block (scalar)
    int so;                           // sorted id (mtk: no row)
    bool live;                        // the item has this wave's block (wave-uniform)
  };
  const int ksl = c4 < KC ? c4 : KC - 1;
  const int wrow = (ACT ? N / 256 : 1) * nk;        // to the second column block's scales
  auto rows_of = [&](const Item& it, int id) __attribute__((always_inline)) {
    Rows r;
    r.so = w < it.nbk ? id : mtk;
    const int arow = r.so < mtk ? r.so / top_k : 0;
    r.va = WIDE ? arow : arow * K + 16 * c4;
    r.vx = arow * nk;
    r.w0 = (it.set ? ws1 : ws) + ((size_t)it.e * (N / 128) + bcol(it.n0, 0) / 128) * nk;
    r.live = w < it.nbk;
    return r;
  };
  // Chunk c of an item's rows and scales. Without its block a wave reads through empty buffers
  // (row_loads): at one block per tile the rows of the other seven waves cost 2-4 us of 28 per
  // item. WIDE: activations past 2 GB take 64-bit addresses, not a buffer.
  auto stage_a = [&](const Rows& r, int c) __attribute__((always_inline)) {
    if constexpr (WIDE) {
      const uint8_t* p = qx + (size_t)r.va * K + c * KC * 128 + 16 * c4;
#pragma unroll
      for (int ks = 0; ks < KC; ++ks) {
        const int o = TAIL && c * KC + ks >= nk ? -c * KC * 128 : ks * 128;
        ra[ks][0] = *reinterpret_cast<const v4u*>(p + o);
        ra[ks][1] = *reinterpret_cast<const v4u*>(p + o + 64);
      }
    } else {
      row_loads<TAIL>(qbytes, nk, r.va, c, r.live,
                      [&](int ks, int h, int bytes, int voffset, int soffset)
                          __attribute__((always_inline)) {
        ra[ks][h] = __builtin_bit_cast(
            v4u, __builtin_amdgcn_raw_buffer_load_b128(
                     __builtin_amdgcn_make_buffer_rsrc((void*)qx, 0, bytes, BUF_WORD3), voffset,
                     soffset, 0));
      });
    }
    const int k = TAIL ? min(c * KC + ksl, nk - 1) : c * KC + ksl;
    rx = xs[r.vx + k];
    rw0 = r.w0[k];
    rw1 = r.w0[k + wrow];
    if (TWT) rt = tw[r.so < mtk ? r.so : 0];
  };
  unsigned abase[2], sbase[2];        // LDS byte addresses: [0] read, [1] written
  abase[0] = A_OFF;
  abase[1] = abase[0] + A_BUF;
  sbase[0] = 0;
  sbase[1] = 2 * KC * TB * 16 * 4;
  auto write_a = [&](const Rows& r) __attribute__((always_inline)) {
    if (r.live) {
      unsigned char* pa = smem + abase[1] + w * KC * 2048 + lane * 16;
#pragma unroll
      for (int ks = 0; ks < KC; ++ks)
#pragma unroll
        for (int h = 0; h < 2; ++h) *reinterpret_cast<v4u*>(pa + (ks * 2 + h) * 1024) = ra[ks][h];
      if (c4 < KC) {
        float* ps = reinterpret_cast<float*>(smem + sbase[1]) + c4 * TB * 16 + w * 16 + r16;
        const float v = r.so < mtk ? rx : 0.f;
        ps[0] = v * rw0;
        ps[KC * TB * 16] = v * rw1;
      }
    }
  };
  auto write_rows = [&](const Rows& r, int par) __attribute__((always_inline)) {
    if (c4 == 0) {
      rows[par * TB * 16 + w * 16 + r16] = r.so;
      twl[par * TB * 16 + w * 16 + r16] = TWT ? rt : 1.f;
    }
  };
  auto swap = [&]() __attribute__((always_inline)) {
    unsigned t = abase[0];
    abase[0] = abase[1], abase[1] = t;
    t = sbase[0], sbase[0] = sbase[1], sbase[1] = t;
  };

  // ---- prologue: items 0 and 1, item 0's first chunk and its first D weight steps ----
  Item mA, mB, mC;
  Rows rA, rB;
  {
    const Place p0 = place(0), p1 = place(1);
    const v2u t0 = load_tile(p0), t1 = load_tile(p1);
    take_tile(t0, mA);
    take_tile(t1, mB);
    const int e0 = load_eid(mA), e1 = load_eid(mB);
    const int i0 = load_id(mA), i1 = load_id(mB);
    mA.e = uniform(e0), mA.n0 = p0.n0;
    mB.e = uniform(e1), mB.n0 = p1.n0;
    rA = rows_of(mA, i0);
    rB = rows_of(mB, i1);
  }
  const uint8_t* bcur = wptr(mA);
  const uint8_t* bnext = wptr(mB);
#pragma unroll
  for (int j = 0; j < KC; ++j) issue_b(j, wbuf(bcur, true), j * 2048);
  stage_a(rA, 0);
  write_a(rA);
  write_rows(rA, 0);
  mC = mB;
  swap();
  __syncthreads();

  for (int m = 0; m < cnt; ++m) {
    const int par = m & 1;
    const Place pC = place(m + 2);
    int eC = 0, idC = 0;
#pragma unroll
    for (int bk = 0; bk < TB; ++bk)
#pragma unroll
      for (int s = 0; s < S; ++s) acc[bk][s] = v4f{0.f, 0.f, 0.f, 0.f};
    for (int c = 0; c < nch; ++c) {
      const bool last = c + 1 == nch;
      const uint8_t* bld = last ? bnext : bcur;
      const int woff = last ? 0 : (c + 1) * KC * 2048;
      const int ahead = steps_ahead<TAIL>(nk, c, last, m + 1 < cnt);   // steps of the next chunk
      const int here = TAIL && last ? nk - c * KC : KC;           // ... of this one
      // the next chunk: this item's, or the next item's first
      Rows st = rA;
      if (last) st = rB;
      stage_a(st, last ? 0 : c + 1);
      // item m + 2, a step further each chunk: its tile words, then its expert and row ids
      const v2u tC = load_tile(pC);
      eC = load_eid(mC);
      idC = load_id(mC);
      // One step over the tile's blocks in pairs, the last first: 7 and 6, 5 and 4, 3 and 2 when
      // the tile has them, then 1 and 0 (a block past the tile's computes on stale rows that
      // are never stored). A unit is one block: its MFMAs, the LDS reads of the block two
      // further on into the operand registers just read, and the scaling of the block before
      // it. The empty asm statements keep the compiler from sinking MFMAs and scalings out of
      // their unit.
      const bool r6 = mA.nbk > 6, r4 = mA.nbk > 4, r2 = mA.nbk > 2;
      const unsigned ab = abase[0] + lane * 16;
      const unsigned sb = sbase[0] + (cb * KC * TB * 16 + 4 * c4 + (r16 & 3)) * 4;
      const int top = r6 ? 6 : r4 ? 4 : r2 ? 2 : 0;   // blocks above block 1 that run
      const unsigned abt = ab + top * KC * 2048, sbt = sb + top * 64;
      v4u af[2][2];
      float fs[2], fp;
      v4f d[2][S];
      auto rd = [&](int ks, int bk, unsigned xa, unsigned xs) __attribute__((always_inline)) {
        af[bk & 1][0] = *reinterpret_cast<const v4u*>(smem + xa + (bk * KC + ks) * 2048);
        af[bk & 1][1] = *reinterpret_cast<const v4u*>(smem + xa + (bk * KC + ks) * 2048 + 1024);
        fs[bk & 1] = *reinterpret_cast<const float*>(smem + xs + (ks * TB + bk) * 64);
      };
      auto scale = [&](int bk) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
          const v4f p = d[bk & 1][s];
          acc[bk][s][0] = fmaf(quad<0>(fp), p[0], acc[bk][s][0]);
          acc[bk][s][1] = fmaf(quad<1>(fp), p[1], acc[bk][s][1]);
          acc[bk][s][2] = fmaf(quad<2>(fp), p[2], acc[bk][s][2]);
          acc[bk][s][3] = fmaf(quad<3>(fp), p[3], acc[bk][s][3]);
          asm volatile("" : "+v"(acc[bk][s]));
        }
      };
      auto unit = [&](int ks, int bk, bool first) __attribute__((always_inline)) {
        const v8i a = pack8(af[bk & 1][0], af[bk & 1][1]);
#pragma unroll
        for (int s = 0; s < S; ++s) {
          d[bk & 1][s] = mfma_f8(a, pack8(rb[ks][s][0], rb[ks][s][1]));
          asm volatile("" : "+v"(d[bk & 1][s]));
        }
        const float fn = fs[bk & 1];
        if (bk >= 2)
          rd(ks, bk - 2, ab, sb);
        else if (ks + 1 < KC)
          rd(ks + 1, bk, abt, sbt);                 // the next step's first two blocks
        if (!first) scale(bk + 1);
        fp = fn;
        __builtin_amdgcn_sched_barrier(0);
      };
      rd(0, 1, abt, sbt);
      rd(0, 0, abt, sbt);
#pragma unroll
      for (int ks = 0; ks < KC; ++ks) {
        if (TAIL && ks >= here) {                   // (uniform) the ring runs on
          issue_b(ks, wbuf(bld, TAIL ? ks < ahead : ahead > 0), woff + ks * 2048);
          continue;
        }
        if (r6) {
          unit(ks, 7, true);
          unit(ks, 6, false);
          scale(6);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (r4) {
          unit(ks, 5, true);
          unit(ks, 4, false);
          scale(4);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (r2) {
          unit(ks, 3, true);
          unit(ks, 2, false);
          scale(2);
          __builtin_amdgcn_sched_barrier(0);
        }
        unit(ks, 1, true);
        unit(ks, 0, false);
        issue_b(ks, wbuf(bld, TAIL ? ks < ahead : ahead > 0), woff + ks * 2048);
        scale(0);
        __builtin_amdgcn_sched_barrier(0);
      }
      write_a(st);
      if (last) write_rows(st, par ^ 1);
      take_tile(tC, mC);
      swap();
      __syncthreads();
    }
    // epilogue, plain GEMM: each wave writes its own S 16 columns, block by block, through
    // its own LDS staging area -- the bf16 outputs (x routed weight) of one block as [16
    // rows][S 16], read back as 16-byte row pieces, four consecutive lanes to a row -- with
    // nontemporal stores (the rows are scattered and not re-read here; kept out of L2 they
    // leave it to the weight stream). No workgroup barrier: a wave that finishes its strips
    // goes on to the next item, whose weights its ring already holds, while the others
    // still store. The row ids and routed weights read here were written before the
    // chunk-end barrier that closed the previous item, and are rewritten only after the
    // next item's first one.
    if constexpr (!ACT) {
      uint16_t* st = reinterpret_cast<uint16_t*>(smem + EPI_OFF + w * EPI_W);
      const int cw = bcol(mA.n0, cb) + wcol;
      constexpr int RC = S * 2;                         // 16-byte pieces per staged row
#pragma unroll
      for (int bk = 0; bk < TB; ++bk) {
        if (bk < mA.nbk) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float wt = twl[par * TB * 16 + bk * 16 + 4 * c4 + i];
#pragma unroll
            for (int s = 0; s < S; ++s)
              st[(4 * c4 + i) * S * 16 + s * 16 + r16] = f32_to_bf16(acc[bk][s][i] * wt);
          }
          wave_lds_sync();
#pragma unroll
          for (int u0 = 0; u0 < 16 * RC; u0 += WAVE) {
            const int u = u0 + lane;
            if (16 * RC % WAVE == 0 || u < 16 * RC) {
              const int rr = u / RC, ch = u - rr * RC;
              const int so = rows[par * TB * 16 + bk * 16 + rr];
              const v4u v = *reinterpret_cast<const v4u*>(st + rr * S * 16 + ch * 8);
              if (so < mtk)
                __builtin_nontemporal_store(
                    v, reinterpret_cast<v4u*>(y + (size_t)so * N + cw + ch * 8));
            }
          }
          wave_lds_sync();
        }
      }
    } else {
      // epilogue, SiLU-mul-quant: through the activation buffer this item's last chunk used
      // (free after the chunk-end barrier) each wave puts its bf16 outputs into a [rows][C]
      // tile; then 16-lane groups take whole rows (128 gate + 128 up columns), one row each.
      // Blocks go BP at a time when the tile does not fit.
      uint16_t* ot = reinterpret_cast<uint16_t*>(smem + abase[1]);
#pragma unroll
      for (int p0 = 0; p0 < TB; p0 += BP) {
        if (p0 < mA.nbk) {
#pragma unroll
          for (int t = 0; t < BP; ++t) {
            const int bk = p0 + t;
            if (bk < TB && bk < mA.nbk) {
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const int rr = t * 16 + 4 * c4 + i;
#pragma unroll
                for (int s = 0; s < S; ++s)
                  ot[rr * C + (w * S + s) * 16 + r16] = f32_to_bf16_hw(acc[bk][s][i]);
              }
            }
          }
          __syncthreads();
          const int nr = ((mA.nbk < p0 + BP ? mA.nbk : p0 + BP) - p0) * 16;
          // one 16-lane row group per output row, lane l on columns [8 l, 8 l + 8) of the
          // item's 128-column group (nr is a multiple of 16, so every wave's four groups
          // run the same trip count and the DPP reduction sees whole groups)
          const int I = N / 2, g = mA.n0 / C, l16 = lane & 15;
          for (int rr = (int)threadIdx.x / 16; rr < nr; rr += NWAVE * 4) {
            float gv[8], uv[8], a[8];
            unpack8_bf16(*reinterpret_cast<const uint4*>(ot + rr * C + 8 * l16), gv);
            unpack8_bf16(*reinterpret_cast<const uint4*>(ot + rr * C + 128 + 8 * l16), uv);
            uint32_t mx = 0;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
              a[j] = bf16_to_f32(f32_to_bf16_hw(__fmul_rn(silu_of_bf16(gv[j]), uv[j])));
              mx = max(mx, abs_bits(a[j]));
            }
            const float sc = scale_of(row_max_u32(mx));
            const uint2 qv = quant8(a, sc);
            const int so = rows[par * TB * 16 + p0 * 16 + rr];
            if (so < mtk) {
              __builtin_nontemporal_store(
                  v2u{qv.x, qv.y},
                  reinterpret_cast<v2u*>(q2 + (size_t)so * I + g * 128 + 8 * l16));
              if (l16 == 0) __builtin_nontemporal_store(sc, s2 + (size_t)so * (I / 128) + g);
            }
          }
          __syncthreads();
        }
      }
    }
    // advance: the next item becomes current
    mC.e = uniform(eC);
    mC.n0 = pC.n0;
    mA = mB;
    mB = mC;
    rA = rB;
    rB = rows_of(mB, idC);
    bcur = bnext;
    bnext = wptr(mB);
  }
}

template <bool TWT, bool ACT, bool TWO, bool WIDE, bool TAIL>
__global__ __launch_bounds__(NWAVE * WAVE, 2) void roll_k(
    const uint8_t* __restrict__ qx, const float* __restrict__ xs, const uint8_t* __restrict__ wq,
    const float* __restrict__ ws, const int* __restrict__ sorted_ids,
    const int* __restrict__ eids, const uint8_t* __restrict__ wq1, const float* __restrict__ ws1,
    const int* __restrict__ sorted_ids1, const int* __restrict__ eids1,
    const int* __restrict__ tiles, const int* __restrict__ ntiles, uint16_t* __restrict__ y,
    const float* __restrict__ tw, uint8_t* __restrict__ q2, float* __restrict__ s2, int mtk,
    int top_k, int K, int N, int qbytes, bool far) {
  extern __shared__ __align__(16) unsigned char smem[];
  const Sched sc = make_sched<TWO>(smem, smem + ORD_OFF, tiles, ntiles[0], mtk, N / C, eids,
                                  eids1, far);
  if (sc.first >= sc.n * (N / C)) return;
  // two copies of the body: the policy is part of the load instructions, and a branch on it in
  // every step cost 2-5%
  if (sc.shared)
    items<POL_SHARED, TWT, ACT, TWO, WIDE, TAIL>(sc, qx, xs, wq, ws, sorted_ids, eids, wq1, ws1,
                                           sorted_ids1, eids1, tiles, y, tw, q2, s2, mtk, top_k,
                                           K, N, qbytes);
  else
    items<POL_STREAM, TWT, ACT, TWO, WIDE, TAIL>(sc, qx, xs, wq, ws, sorted_ids, eids, wq1, ws1,
                                           sorted_ids1, eids1, tiles, y, tw, q2, s2, mtk, top_k,
                                           K, N, qbytes);
}

// row_loads' 16-byte loads, over the first and the last of `rows` rows of K bytes, that reach bytes
// outside of their own row
template <bool TAIL>
static int loads_outside(int rows, int K) {
  int bad = 0;
  for (int row : {0, rows - 1})
    for (int c4 = 0; c4 < 4; ++c4)
      for (int live = 0; live < 2; ++live)
        for (int c = 0; c < chunks<TAIL>(K / 128); ++c)
          row_loads<TAIL>(rows * K, K / 128, row * K + 16 * c4, c, live != 0,
                          [&](int, int, int bytes, int voffset, int soffset) {
            const long long at = (long long)voffset + soffset - (long long)row * K;
            if (voffset < bytes && (!live || at < 0 || at + 16 > K)) ++bad;
          });
  return bad;
}

// the weight steps a workgroup of `items` items loads, the ring's first fill and what follows
template <bool TAIL>
static long long steps_loaded(int items, int nk) {
  long long steps = KC;
  for (int m = 0; m < items; ++m)
    for (int c = 0; c < chunks<TAIL>(nk); ++c)
      steps += max(0, min(KC, steps_ahead<TAIL>(nk, c, c + 1 == chunks<TAIL>(nk), m + 1 < items)));
  return steps;
}

}  // namespace roll

void launch_roll(const Args& a, int max_tiles, hipStream_t stream) {
  using namespace roll;
  const long long items = (long long)max_tiles * (a.N / C);
  int grid = device_cus();
  if (grid > items) grid = (int)items;
  if (grid >= NXCD) grid -= grid % NXCD;
  // bytes of the activation rows any id below mtk names; 32-bit offsets reach 2 GB of them
  const long long qbytes = (long long)((a.mtk + (long long)a.top_k - 1) / a.top_k) * a.K;
  const bool wide = qbytes > 0x7fffffff;
  const bool tail = has_tail(a.K);
#define RLU_PF1(T, A, TW, WD, TL)                                                             \
  hipLaunchKernelGGL((roll_k<T, A, TW, WD, TL>), dim3(grid), dim3(NWAVE * WAVE), LDS, stream,  \
                     a.qx, a.xs, a.wq, a.ws, a.sorted_ids, a.eids, a.wq1, a.ws1,               \
                     a.sorted_ids1, a.eids1, a.tiles, a.ntiles, a.y, a.tw, a.q2, a.s2, a.mtk,  \
                     a.top_k, a.K, a.N, wide ? 0 : (int)qbytes, a.far)
#define RLU_PF2(T, A, TW)                                                                     \
  do {                                                                                        \
    if (wide)                                       /* (the tail's code takes any K) */       \
      RLU_PF1(T, A, TW, true, true);                                                          \
    else if (tail)                                                                            \
      RLU_PF1(T, A, TW, false, true);                                                         \
    else                                                                                      \
      RLU_PF1(T, A, TW, false, false);                                                        \
  } while (0)
#define RLU_PF(T, A)                                                                          \
  do {                                                                                        \
    if (a.two)                                                                                \
      RLU_PF2(T, A, true);                                                                    \
    else                                                                                      \
      RLU_PF2(T, A, false);                                                                   \
  } while (0)
  if (a.q2)
    RLU_PF(false, true);
  else if (a.tw)
    RLU_PF(true, false);
  else
    RLU_PF(false, false);
#undef RLU_PF
#undef RLU_PF2
#undef RLU_PF1
}

}  // namespace pf
}  // namespace rlu

// Host only: counts into *bad the loads of activation rows by which the rolled kernel would touch
// bytes outside of its row, over the first and the last of `rows` rows of K, with only the vector
// offset in the buffers' range check. Returns -1 (bad sizes or NULL), -2 (K % 128, K < 512, or
// activations past 2 GB, which take 64-bit addresses).
extern "C" int rlu_selftest_prefill_rows(int rows, int K, unsigned long long* bad) {
  using namespace rlu::pf::roll;
  if (rows < 1 || K < 1 || !bad) return -1;
  if (K % 128 || K < 512 || (long long)rows * K > 0x7fffffff) return -2;
  *bad = has_tail(K) ? loads_outside<true>(rows, K) : loads_outside<false>(rows, K);
  return 0;
}

// Host only: the weight steps (of 128 deep, 32 KB) that a workgroup of the rolled kernel loads for `items`
// items of K. Returns -1 (bad sizes or NULL), -2 (K % 128 or K < 512).
extern "C" int rlu_selftest_prefill_steps(int items, int K, unsigned long long* steps) {
  using namespace rlu::pf::roll;
  if (items < 1 || K < 1 || !steps) return -1;
  if (K % 128 || K < 512) return -2;
  *steps = has_tail(K) ? steps_loaded<true>(items, K / 128) : steps_loaded<false>(items, K / 128);
  return 0;
}
