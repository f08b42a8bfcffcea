// The grouped fp8 GEMM of a prefill chunk (tens of rows per expert), streamed: same operands,
// row contract, tile list and numerics as tiled_k (gemm_tiled.hip) and moe_gemm_k (gemm.hip),
// bit for bit, for K = 768 (down of the 2560-wide model). Other K run the rolled form
// (prefill_roll.hip, roll_takes) or tiled_k.
//
// The unrolled form stays here because an item of 6 steps is short: the ring holds a whole item
// ahead, and the rolled form's per-chunk work costs 5% at one block per tile (193 against 203 us).
//
// Why a second kernel: at 80 rows per expert the work is weight streaming (about 160 FLOP per
// weight byte, under the fp8 ridge of ~625), so what matters is how many weight bytes each CU
// keeps in flight. tiled_k stages both operands through LDS one K step ahead, so a CU has one
// step (~48 KB) in flight and restarts its pipeline at every tile. Here:
//
//   * An item is (tile of <= 8 16-row blocks of one expert, 16 S W output columns). Each of the
//     W waves owns S 16-column weight strips and computes every block of the tile for them, so
//     a weight fragment is used from registers by all the tile's blocks and never goes through
//     LDS. Each wave streams its strips through a ring of D register stages (buffer loads,
//     streaming, or with the plain cache policy where an expert has several tiles) with no
//     barrier on them, and the ring runs on across item boundaries: the last D steps of an item
//     issue the first D steps of the next one. Up to D x 32 KB = 192 KB of weights are in flight
//     per CU.
//   * The tile's activation rows (gathered through sorted_ids) go to LDS in chunks of KC K
//     steps, double-buffered, loaded into registers one whole chunk ahead -- the next item's
//     first chunk during this item's last one -- and written at the chunk's end, so waiting
//     for them only waits for weight loads issued before them, which the ring needs by then
//     anyway (the vector-memory counter retires in order). One barrier per chunk.
//   * The activation scales of the chunk ride with it (LDS), the weight-block scales of an
//     item come through scalar loads, and the routed weights and row ids of the next item are
//     staged with its first chunk, so the epilogue reads LDS only. In the epilogue each wave
//     turns its own strips' bf16 outputs into 16-byte row pieces through a small LDS area of
//     its own and stores them nontemporally (the rows are scattered and not re-read here;
//     kept out of L2 they leave it to the weight stream), with no workgroup barrier, so a
//     wave that finishes early starts the next item, whose weights are already in flight.
//   * Item metadata (tile, expert) is read through scalar loads two items ahead, the next
//     tile's sorted ids one item ahead.
//   * The order of the items is Sched's (prefill_sched.h): the column groups of a tile run at the
//     same time on CUs sharing one L2, which holds the tile's rows once; tiles of experts with
//     several run on some of an XCD's workgroups, with plain weight loads, the others on the
//     rest, streaming. At 4096 / 8192 tokens of Zipf(1.1) routing over 512 experts down takes
//     262 / 420 us (318 / 445 in list order, all streaming).
//   * One launch can cover two aligns over two weight sets (a layer's resident slots and the
//     full tensor it reads non-resident experts from): the tile list then names the set of
//     each tile (bit 16 of its block count), and an item takes its expert ids, sorted ids,
//     weights and scales from that set. Both aligns index the same activation rows and write
//     the same output.
// Per step, acc = fma(mfma(a, b), xs * ws, acc) in ascending k from zero: the same sequence of
// operations as moe_gemm_k with sk = 1, so the outputs are equal bit for bit.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemm_common.h"
#include "numerics.h"
#include "prefill.h"
#include "prefill_sched.h"
#include "wave.h"

namespace rlu {
namespace pf {
namespace k768 {

constexpr int W = NWAVE;               // waves per workgroup
constexpr int S = 2;                   // 16-column weight strips per wave
constexpr int NK = 6;                  // K / 128
constexpr int K = NK * 128;
constexpr int KC = 3;                  // K steps per activation chunk
constexpr int D = 6;                   // depth of the weight ring in steps
constexpr int NCH = NK / KC;           // chunks per item
constexpr int C = 16 * S * W;          // columns per item
static_assert(NK % KC == 0 && TB == W && (2 * NK) % D == 0, "config");
// two chunks at least: a chunk-end barrier then separates an item's epilogue (LDS reads of its
// row ids) from the writes of the row ids two items on
static_assert(NCH >= 2, "at least two chunks per item");
// LDS: the small arrays first, then the two activation buffers, each under 64 KB so that every
// constant offset into it fits the 16-bit offset of a ds instruction
constexpr int SX = 2 * KC * TB * 16;                       // float [buf][ks][row]
constexpr int RW = 2 * TB * 16;                            // int / float [par][row]
constexpr int A_OFF = (SX + 2 * RW) * 4;
constexpr int A_BUF = TB * KC * 2 * 1024;                  // [blk][ks][h][lane] x 16 B
static_assert(A_BUF <= 65536, "an activation buffer must fit one ds offset range");
// each wave's own epilogue staging: one block's [16 rows][S 16 columns] bf16
constexpr int EPI_W = 16 * S * 16 * 2;
constexpr int EPI_OFF = A_OFF + 2 * A_BUF;
constexpr int ORD_OFF = EPI_OFF + W * EPI_W;
constexpr size_t LDS = (size_t)ORD_OFF + ORD_BYTES;
static_assert(SCRATCH_BYTES <= ORD_OFF, "the scheduler's scratch lies below the order");

// TWT: routed weights. TWO: the tile list covers two aligns (bit 16 of a tile's block count picks
// the set); the one-set kernels take no second set, whose pointers would otherwise hold scalar
// registers for the whole launch. POL: the weight loads' cache policy.
template <int POL, bool TWT, bool TWO>
__device__ __forceinline__ void items(
    const Sched& sc, const uint8_t* __restrict__ qx, const float* __restrict__ xs,
    const uint8_t* __restrict__ wq, const float* __restrict__ ws,
    const int* __restrict__ sorted_ids, const int* __restrict__ eids,
    const uint8_t* __restrict__ wq1, const float* __restrict__ ws1,
    const int* __restrict__ sorted_ids1, const int* __restrict__ eids1,
    const int* __restrict__ tiles, uint16_t* __restrict__ y, const float* __restrict__ tw,
    int mtk, int top_k, int N) {
  extern __shared__ __align__(16) unsigned char smem[];
  float* sx = reinterpret_cast<float*>(smem);
  int* rows = reinterpret_cast<int*>(sx + SX);
  float* twl = reinterpret_cast<float*>(rows + RW);

  const int lane = lane_id();
  const int w = uniform((int)(threadIdx.x / WAVE));
  const int r16 = lane & 15, c4 = lane >> 4;
  // this lane's byte address in each activation buffer, opaque to the compiler so that the
  // constant part of every fragment address stays in the instruction's offset field
  unsigned abase[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    abase[q] = A_OFF + q * A_BUF + lane * 16;
    asm volatile("" : "+v"(abase[q]));
  }
  auto afrag = [&](int q, int off) __attribute__((always_inline)) -> v4u {
    return *reinterpret_cast<const v4u*>(smem + abase[q] + off);
  };
  const int ncg = N / C;
  // first output column of this wave's strips in an item starting at column n0
  auto col0 = [&](int n0) __attribute__((always_inline)) -> int { return n0 + w * S * 16; };
  const int cnt = (sc.n * ncg - sc.first + sc.step - 1) / sc.step;   // this workgroup's items

  auto meta = [&](int m) __attribute__((always_inline)) {
    const int it = sc.first + (m < cnt ? m : cnt - 1) * sc.step;
    const int k = it / ncg;
    const int ti = sc.tile(smem + ORD_OFF, k);
    Item r;
    r.b0 = tiles[2 * ti];
    const int nw = tiles[2 * ti + 1];              // block count | set << 16 (TWO)
    r.nbk = TWO ? nw & 0xffff : nw;
    r.set = TWO ? nw >> 16 : 0;
    r.e = (r.set ? eids1 : eids)[r.b0];
    r.n0 = (it - k * ncg) * C;
    return r;
  };
  // this wave's strips of an item, as a buffer: strip s, step k, half h at s 16 K + k 2048 +
  // h 1024 + lane 16 (the base and the step offset stay in scalar registers)
  auto wbase = [&](const Item& it) __attribute__((always_inline)) {
    return __builtin_amdgcn_make_buffer_rsrc(
        (void*)((it.set ? wq1 : wq) + ((size_t)it.e * N + col0(it.n0)) * K), 0, S * 16 * K,
        BUF_WORD3);
  };
  // the sorted id of row r16 of block blk of an item (mtk past the tile): one vector load,
  // issued at an item's start and used at its last chunk, so waiting for it costs nothing
  auto load_id = [&](const Item& it, int blk) __attribute__((always_inline)) {
    const bool in = blk < it.nbk;
    const int v = (it.set ? sorted_ids1 : sorted_ids)[(it.b0 + (in ? blk : 0)) * 16 + r16];
    return in ? v : mtk;
  };

  // ---- registers ----
  v4u rb[D][S][2];                    // weight ring
  v4u ra[KC][2];                      // next chunk's activation rows (this wave's block)
  float rx;                           // ... and their scales
  float rt;                           // next item's routed weight of row r16
  int son;                            // next item's sorted id of row r16
  int arow_c, arow_n;                 // activation row of row r16 (current / next item)
  bool val_c, val_n;
  int id_n;                           // next item's sorted id of row r16
  v4f acc[TB][S];

  const int voff = lane * 16;
  auto issue_b = [&](int j, __amdgpu_buffer_rsrc_t base, int k) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      rb[j][s][0] = __builtin_bit_cast(
          v4u, __builtin_amdgcn_raw_buffer_load_b128(base, voff, s * 16 * K + k * 2048, POL));
      rb[j][s][1] = __builtin_bit_cast(
          v4u, __builtin_amdgcn_raw_buffer_load_b128(base, voff + 1024, s * 16 * K + k * 2048,
                                                     POL));
    }
  };
  // the row of an item from its id: activation row and validity of row r16 of this wave's block
  auto row_of = [&](int id, int& arow, bool& val) __attribute__((always_inline)) {
    son = id;
    val = id < mtk;
    arow = val ? id / top_k : 0;
  };
  // chunk c of an item's activation rows and scales, into ra / rx; with first_chunk, also the
  // item's routed weights (rt)
  auto stage_a = [&](int arow, bool val, int c, bool first_chunk) __attribute__((always_inline)) {
    const uint8_t* p = qx + (size_t)arow * K + c * KC * 128 + 16 * c4;
#pragma unroll
    for (int ks = 0; ks < KC; ++ks) {
      ra[ks][0] = *reinterpret_cast<const v4u*>(p + ks * 128);
      ra[ks][1] = *reinterpret_cast<const v4u*>(p + ks * 128 + 64);
    }
    const float v = xs[(size_t)arow * NK + c * KC + (c4 < KC ? c4 : KC - 1)];
    rx = val ? v : 0.f;
    if (TWT && first_chunk) rt = tw[val ? son : 0];
  };
  auto write_a = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < KC; ++ks)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        *reinterpret_cast<v4u*>(smem + abase[buf] + w * KC * 2048 + (ks * 2 + h) * 1024) =
            ra[ks][h];
    if (c4 < KC) sx[(buf * KC + c4) * TB * 16 + w * 16 + r16] = rx;
  };
  auto write_rows = [&](int par) __attribute__((always_inline)) {
    if (c4 == 0) {
      rows[par * TB * 16 + w * 16 + r16] = son;
      twl[par * TB * 16 + w * 16 + r16] = TWT ? rt : 1.f;
    }
  };

  // ---- prologue: item 0's first chunk, rows, scales; its first D weight steps ----
  Item mA = meta(0), mB = meta(1);
  __amdgpu_buffer_rsrc_t bcur = wbase(mA);
  __amdgpu_buffer_rsrc_t bnext = wbase(mB);
  {
    const int id0 = load_id(mA, w);
    row_of(id0, arow_c, val_c);
#pragma unroll
    for (int j = 0; j < D; ++j) issue_b(j, bcur, j);
    stage_a(arow_c, val_c, 0, true);
    write_a(0);
    write_rows(0);
    id_n = load_id(mB, w);
  }
  __syncthreads();

  for (int m = 0; m < cnt; m += 2) {
#pragma unroll
    for (int par = 0; par < 2; ++par) {
      if (par == 1 && m + 1 >= cnt) break;
      const Item mC = meta(m + par + 2);
#pragma unroll
      for (int bk = 0; bk < TB; ++bk)
#pragma unroll
        for (int s = 0; s < S; ++s) acc[bk][s] = v4f{0.f, 0.f, 0.f, 0.f};
      // the weight-block scales of this wave's strips, one per step: scalar loads (they never
      // enter the vector-memory counter the weight ring waits on)
      const float* wsrow =
          (mA.set ? ws1 : ws) + ((size_t)mA.e * (N / 128) + col0(mA.n0) / 128) * NK;
      float wsr[NK];
#pragma unroll
      for (int k = 0; k < NK; ++k) wsr[k] = wsrow[k];
#pragma unroll
      for (int c = 0; c < NCH; ++c) {
        const int qb = (par * NCH + c) & 1;
        if (c + 1 < NCH) {
          stage_a(arow_c, val_c, c + 1, false);
        } else {                                    // the next item's first chunk
          row_of(id_n, arow_n, val_n);
          stage_a(arow_n, val_n, 0, true);
        }
#pragma unroll
        for (int ks = 0; ks < KC; ++ks) {
          const int k = c * KC + ks;
          const int j = (par * NK + k) % D;
          const float wsk = wsr[k];
          v8i bf[S];
#pragma unroll
          for (int s = 0; s < S; ++s) bf[s] = pack8(rb[j][s][0], rb[j][s][1]);
          // a branch per block on the tile's block count; scheduling fenced every two
#pragma unroll
          for (int bk = 0; bk < TB; ++bk) {
            if (bk < mA.nbk) {
              const int off = (bk * KC + ks) * 2048;
              const v8i af = pack8(afrag(qb, off), afrag(qb, off + 1024));
              const v4f xr = *reinterpret_cast<const v4f*>(
                  &sx[(qb * KC + ks) * TB * 16 + bk * 16 + 4 * c4]);
              v4f f;
#pragma unroll
              for (int i = 0; i < 4; ++i) f[i] = xr[i] * wsk;
#pragma unroll
              for (int s = 0; s < S; ++s) {
                const v4f d = mfma_f8(af, bf[s]);
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[bk][s][i] = fmaf(d[i], f[i], acc[bk][s][i]);
              }
              if (bk % 2 == 1) __builtin_amdgcn_sched_barrier(0);
            }
          }
          if (k + D < NK)
            issue_b(j, bcur, k + D);
          else
            issue_b(j, bnext, k + D - NK);
          // keep each step's LDS reads and MFMAs in their step (hoisting the reads of later
          // steps ahead would hold a chunk of A fragments in registers)
          __builtin_amdgcn_sched_barrier(0);
        }
        write_a(qb ^ 1);
        if (c + 1 == NCH) write_rows(par ^ 1);
        __syncthreads();
      }
      // epilogue: each wave writes its own S 16 columns, block by block, through
      // its own LDS staging area -- the bf16 outputs (x routed weight) of one block as [16
      // rows][S 16], read back as 16-byte row pieces, four consecutive lanes to a row -- with
      // nontemporal stores (the rows are scattered and not re-read here; kept out of L2 they
      // leave it to the weight stream). No workgroup barrier: a wave that finishes its strips
      // goes on to the next item, whose weights its ring already holds, while the others
      // still store. The row ids and routed weights read here were written before the
      // chunk-end barrier that closed the previous item, and are rewritten only after the
      // next item's first one.
      uint16_t* st = reinterpret_cast<uint16_t*>(smem + EPI_OFF + w * EPI_W);
      const int cw = col0(mA.n0);
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
      // advance: the next item becomes current
      arow_c = arow_n;
      val_c = val_n;
      mA = mB;
      mB = mC;
      bcur = bnext;
      bnext = wbase(mB);
      id_n = load_id(mB, w);
    }
  }
}

template <bool TWT, bool TWO>
__global__ __launch_bounds__(W * WAVE, 2) void stream_k(
    const uint8_t* __restrict__ qx, const float* __restrict__ xs, const uint8_t* __restrict__ wq,
    const float* __restrict__ ws, const int* __restrict__ sorted_ids,
    const int* __restrict__ eids, const uint8_t* __restrict__ wq1, const float* __restrict__ ws1,
    const int* __restrict__ sorted_ids1, const int* __restrict__ eids1,
    const int* __restrict__ tiles, const int* __restrict__ ntiles, uint16_t* __restrict__ y,
    const float* __restrict__ tw, int mtk, int top_k, int N, bool far) {
  extern __shared__ __align__(16) unsigned char smem[];
  const Sched sc = make_sched<TWO>(smem, smem + ORD_OFF, tiles, ntiles[0], mtk, N / C, eids,
                                  eids1, far);
  if (sc.first >= sc.n * (N / C)) return;
  if (sc.shared)                                    // two copies: the policy is in the loads
    items<POL_SHARED, TWT, TWO>(sc, qx, xs, wq, ws, sorted_ids, eids, wq1, ws1, sorted_ids1,
                                eids1, tiles, y, tw, mtk, top_k, N);
  else
    items<POL_STREAM, TWT, TWO>(sc, qx, xs, wq, ws, sorted_ids, eids, wq1, ws1, sorted_ids1,
                                eids1, tiles, y, tw, mtk, top_k, N);
}

}  // namespace k768

static void launch_k768(const Args& a, int max_tiles, hipStream_t stream) {
  using namespace k768;
  const long long items = (long long)max_tiles * (a.N / C);
  int grid = device_cus();
  if (grid > items) grid = (int)items;
  if (grid >= NXCD) grid -= grid % NXCD;
#define RLU_PF(T, TW)                                                                         \
  hipLaunchKernelGGL((stream_k<T, TW>), dim3(grid), dim3(W * WAVE), LDS, stream, a.qx, a.xs,  \
                     a.wq, a.ws, a.sorted_ids, a.eids, a.wq1, a.ws1, a.sorted_ids1, a.eids1,  \
                     a.tiles, a.ntiles, a.y, a.tw, a.mtk, a.top_k, a.N, a.far)
  if (a.tw && a.two)
    RLU_PF(true, true);
  else if (a.tw)
    RLU_PF(true, false);
  else if (a.two)
    RLU_PF(false, true);
  else
    RLU_PF(false, false);
#undef RLU_PF
}

}  // namespace pf

// Whether p is the device address of pinned host memory (no: memory the runtime does not know)
static bool in_host_memory(const void* p) {
  hipPointerAttribute_t at;
  if (hipPointerGetAttributes(&at, p) == hipSuccess) return at.type == hipMemoryTypeHost;
  (void)hipGetLastError();                          // the entry points return the launch's status
  return false;
}

// the kernel arguments; without a second set, set 1 repeats set 0 (no tile names it)
static pf::Args make_args(const void* qx, const float* xs, const void* wq, const float* ws,
                          const int* sorted_ids, const int* expert_ids, const PfSecond* second,
                          const int* tiles, const int* ntiles, const float* topk_weights,
                          void* y, void* q2, float* s2, int mtk, int top_k, int K, int N) {
  const PfSecond one{wq, ws, sorted_ids, expert_ids};
  const PfSecond& b = second ? *second : one;
  return pf::Args{(const uint8_t*)qx, xs, (const uint8_t*)wq, ws, sorted_ids, expert_ids,
                  (const uint8_t*)b.wq, b.ws, b.sorted_ids, b.expert_ids, second != nullptr,
                  second && in_host_memory(b.wq), tiles, ntiles,
                  (uint16_t*)y, topk_weights, (uint8_t*)q2, s2, mtk, top_k, K, N};
}

bool prefill_stream_built(int K, int N) { return (K == 2560 || K == 768) && N % 256 == 0; }

// The rolled kernel's K: a multiple of its chunk of 4 steps from two chunks on; any other K from one
// chunk on once the rows alone make two items per CU (64 experts, 8192 tokens, down of K = 1408
// 533 -> 401 us, 2048 tokens 152 -> 149; 32 experts, 2048 tokens, K = 896 103 -> 86). Below, its one
// workgroup per CU leaves a part of the CUs idle in the last round, and a short or broken K makes
// up for less of that (32 experts, 512 tokens, K = 896: 52 against 46 us of tiled_k; 256 experts, 64
// tokens, K = 512: 45 against 39).
static bool roll_takes(int mtk, int K, int N) {
  if (K % 128 || K < 512 || N % 256) return false;
  return (K % 512 == 0 && K >= 1024) ||
         (long long)mtk * N >= 2LL * 16 * pf::TB * 256 * device_cus();
}

int launch_prefill_stream(const void* qx, const float* xs, const void* wq, const float* ws,
                          const int* sorted_ids, const int* expert_ids, const PfSecond* second,
                          const int* tiles, const int* ntiles, int max_tiles,
                          const float* topk_weights, void* y, int mtk, int top_k, int K, int N,
                          hipStream_t stream) {
  if (N % 256) return -1;
  const pf::Args a = make_args(qx, xs, wq, ws, sorted_ids, expert_ids, second, tiles, ntiles,
                               topk_weights, y, nullptr, nullptr, mtk, top_k, K, N);
  if (K == 768)
    pf::launch_k768(a, max_tiles, stream);
  else if (roll_takes(mtk, K, N))
    pf::launch_roll(a, max_tiles, stream);
  else
    return -1;
  return 0;
}

bool prefill_stream_act_built(int K, int N) { return K == 2560 && N % 256 == 0; }

bool prefill_stream_takes(int mtk, int K, int N, bool act) {
  return (!act && K == 768 && N % 256 == 0) || roll_takes(mtk, K, N);
}

int launch_prefill_stream_act(const void* qx, const float* xs, const void* wq, const float* ws,
                              const int* sorted_ids, const int* expert_ids,
                              const PfSecond* second, const int* tiles, const int* ntiles,
                              int max_tiles, void* q2, float* s2, int mtk, int top_k, int K,
                              int N, hipStream_t stream) {
  if (!roll_takes(mtk, K, N)) return -1;
  const pf::Args a = make_args(qx, xs, wq, ws, sorted_ids, expert_ids, second, tiles, ntiles,
                               nullptr, nullptr, q2, s2, mtk, top_k, K, N);
  pf::launch_roll(a, max_tiles, stream);
  return 0;
}

}  // namespace rlu
