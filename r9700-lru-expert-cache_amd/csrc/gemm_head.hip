// The dense fp8 block-scaled GEMM of the target lm_head for up to 64 rows at once: y[M, N] = A[M,
// K] W[N, K]^T, each row equal bit for bit to rlu_gemm_fp8blk_m16's (gemm.hip): the same steps,
// the same split of K and the same order of its partial sums.
//
// Bound: the weights' read, 389 MB at vocab 151936 x 2560. In launches of 16 rows 64 rows read
// them four times (275 us, 20 rows 135, 16 rows 73); here one launch reads them once and uses each
// fragment for all of the MB 16-row blocks: 100 us at 64 rows, 66 at 20, 64 at 16, 61 at 8 (5.9 -
// 6.4 TB/s at up to 20 rows). What more rows cost is the activations, which each wave takes from
// the L2 again: at 64 rows as many bytes as weights, through the same vector L1, which holds at
// most its 32 KB in flight.
//
//   * An item is 64 columns (4 strips of 16), K split over SK = 4 waves where K / 128 allows, as in
//     moe_gemm_k. A step (128 deep) is in flight per wave, three with one block: more (or
//     one wave per SIMD with 128 columns) measured slower (64 rows with two steps 123 us,
//     with 128 columns 106, one block with four steps 66).
//   * Loads go through buffers of zero size past the wave's last step, so the ring's padding steps
//     touch no memory; moe_gemm_k re-reads its last step there.
//   * Each wave finishes the strips s with s / OWN == ks, so the waves share the sums and stores.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemm_common.h"
#include "gemm_item.h"
#include "numerics.h"
#include "rlu.h"
#include "wave.h"

namespace rlu {
namespace head {

constexpr int NW = 4;                   // waves per workgroup
constexpr int NPW = 4;                  // 16-column strips per item
constexpr int BUF_WORD3 = 0x00020000;  // raw buffer descriptor word 3 on gfx9 (no format)
__host__ __device__ constexpr int ring(int mb) { return mb == 1 ? 3 : 1; }   // steps in flight
// blocks per exchange of partial sums (32 KB of LDS)
__host__ __device__ constexpr int exchange(int mb) { return mb == 1 ? 1 : 2; }

template <int MB, int SK>
__global__ __launch_bounds__(NW * WAVE, 2) void head_k(const uint8_t* __restrict__ qx,
                                                    const float* __restrict__ xs,
                                                    const uint8_t* __restrict__ wq,
                                                    const float* __restrict__ ws,
                                                    uint16_t* __restrict__ y, int M, int K,
                                                    int N) {
  constexpr int D = ring(MB);
  constexpr int IPG = NW / SK;                      // items per workgroup
  static_assert(NPW % SK == 0 && NW % SK == 0, "strips divide over the K splits");
  constexpr int BP = exchange(MB);
  constexpr int OWN = NPW / SK;                     // strips a wave finishes
  extern __shared__ float lds[];                    // scales [NW][nsteps][MB 16], then partials
  const int lane = lane_id();
  const int w = uniform((int)threadIdx.x / WAVE);
  const int sub = w / SK, ks = w % SK;
  const int r16 = lane & 15, c4 = lane >> 4;
  const int nkg = K / 128, kpw = nkg / SK, kg0 = ks * kpw;
  const int nsteps = (kpw + D - 1) / D * D;
  const int item = (int)blockIdx.x * IPG + sub;
  const bool live = item < N / (16 * NPW);
  const int n0 = (live ? item : 0) * 16 * NPW;
  float* sx = lds + w * nsteps * MB * 16;

  // scales of step k = 4 m + c4 of row r16 of each block, ahead of the weights
  float xv[MB][XM], wv[XM];
#pragma unroll
  for (int m = 0; m < XM; ++m) {
    if (4 * m < nsteps) {
      const int k = kg0 + min(4 * m + c4, kpw - 1);
      wv[m] = ws[(size_t)(n0 / 128) * nkg + k];
#pragma unroll
      for (int b = 0; b < MB; ++b) xv[b][m] = xs[(size_t)min(16 * b + r16, M - 1) * nkg + k];
    }
  }
  v4u ra[D][MB][2], rb[D][NPW][2];
  const int va = r16 * K + kg0 * 128 + 16 * c4;
  auto issue = [&](int j, int k) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t a =
        __builtin_amdgcn_make_buffer_rsrc((void*)qx, 0, k < kpw ? M * K : 0, BUF_WORD3);
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      ra[j][b][0] = __builtin_bit_cast(
          v4u, __builtin_amdgcn_raw_buffer_load_b128(a, va + b * 16 * K + k * 128, 0, 0));
      ra[j][b][1] = __builtin_bit_cast(
          v4u, __builtin_amdgcn_raw_buffer_load_b128(a, va + b * 16 * K + k * 128 + 64, 0, 0));
    }
    const __amdgpu_buffer_rsrc_t q = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(wq + (size_t)n0 * K + (size_t)kg0 * 2048), 0, k < kpw ? 16 * NPW * K : 0,
        BUF_WORD3);
#pragma unroll
    for (int s = 0; s < NPW; ++s) {
      rb[j][s][0] = __builtin_bit_cast(
          v4u, __builtin_amdgcn_raw_buffer_load_b128(q, lane * 16, s * 16 * K + k * 2048, 2));
      rb[j][s][1] = __builtin_bit_cast(
          v4u,
          __builtin_amdgcn_raw_buffer_load_b128(q, lane * 16 + 1024, s * 16 * K + k * 2048, 2));
    }
  };
  v4f acc[MB][NPW];
#pragma unroll
  for (int b = 0; b < MB; ++b)
#pragma unroll
    for (int s = 0; s < NPW; ++s) acc[b][s] = v4f{0.f, 0.f, 0.f, 0.f};
  auto step = [&](int j, int k) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      const v4f f = *reinterpret_cast<const v4f*>(sx + (k * MB + b) * 16 + 4 * c4);
      const v8i av = pack8(ra[j][b][0], ra[j][b][1]);
#pragma unroll
      for (int s = 0; s < NPW; ++s) {
        const v4f d = mfma_f8(av, pack8(rb[j][s][0], rb[j][s][1]));
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[b][s][i] = fmaf(d[i], f[i], acc[b][s][i]);
      }
    }
  };
#pragma unroll
  for (int j = 0; j < D; ++j) issue(j, j);
#pragma unroll
  for (int m = 0; m < XM; ++m) {
    const int k = 4 * m + c4;
    if (4 * m < nsteps && k < nsteps)
#pragma unroll
      for (int b = 0; b < MB; ++b) sx[(k * MB + b) * 16 + r16] = k < kpw ? xv[b][m] * wv[m] : 0.f;
  }
  wave_lds_sync();
  int c0 = 0;
  for (; c0 + D < nsteps; c0 += D) {
#pragma unroll
    for (int j = 0; j < D; ++j) {
      step(j, c0 + j);
      issue(j, c0 + j + D);
    }
  }
#pragma unroll
  for (int j = 0; j < D; ++j) step(j, c0 + j);

  // split-K: wave ks finishes the strips OWN ks ..; partials of the others through LDS, added in
  // split order, BP blocks at a time
  float* red = lds + NW * nsteps * MB * 16;         // [wave][strip][BP][64][4]
#pragma unroll
  for (int b0 = 0; b0 < MB; b0 += BP) {
    if (SK > 1) {
      if (b0) __syncthreads();
#pragma unroll
      for (int s = 0; s < NPW; ++s)
        if (s / OWN != ks)
#pragma unroll
          for (int b = b0; b < b0 + BP && b < MB; ++b)
            *reinterpret_cast<v4f*>(red + (((w * NPW + s) * BP + b - b0) * WAVE + lane) * 4) =
                acc[b][s];
      __syncthreads();
    }
#pragma unroll
    for (int s = 0; s < NPW; ++s) {
      if (s / OWN != ks) continue;                  // (uniform)
#pragma unroll
      for (int b = b0; b < b0 + BP && b < MB; ++b) {
        v4f t;
#pragma unroll
        for (int x = 0; x < SK; ++x) {
          v4f p = acc[b][s];
          if (x != ks)
            p = *reinterpret_cast<const v4f*>(
                red + ((((sub * SK + x) * NPW + s) * BP + b - b0) * WAVE + lane) * 4);
#pragma unroll
          for (int i = 0; i < 4; ++i) t[i] = x ? t[i] + p[i] : p[i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = 16 * b + 4 * c4 + i;
          if (live && row < M) y[(size_t)row * N + n0 + s * 16 + r16] = f32_to_bf16(t[i]);
        }
      }
    }
  }
}

template <int MB>
static int launch(int sk, hipStream_t st, const uint8_t* qx, const float* xs, const uint8_t* wq,
                  const float* ws, uint16_t* y, int M, int K, int N) {
  constexpr int D = ring(MB);
  const int nsteps = (K / 128 / sk + D - 1) / D * D;
  const int items = N / (16 * NPW), ipg = NW / sk;
  const size_t lds = (size_t)NW * nsteps * MB * 64 + (sk > 1 ? NW * NPW * exchange(MB) * 1024 : 0);
#define RLU_H(SK)                                                                            \
  hipLaunchKernelGGL((head_k<MB, SK>), dim3((items + ipg - 1) / ipg), dim3(NW * WAVE), lds, \
                     st, qx, xs, wq, ws, y, M, K, N)
  if (sk == 4) RLU_H(4);
  else if (sk == 2) RLU_H(2);
  else RLU_H(1);
#undef RLU_H
  return (int)hipGetLastError();
}

}  // namespace head
}  // namespace rlu

extern "C" int rlu_gemm_fp8blk_m64(const void* qx, const float* xs, const void* w,
                                   const float* ws, void* y, int M, int N, int K,
                                   hipStream_t stream) {
  using namespace rlu;
  if (M < 1 || M > 64 || K <= 0 || N <= 0) return -1;
  if (K % 128 || N % 128) return -2;
  const int nkg = K / 128, sk = nkg % 4 == 0 ? 4 : nkg % 2 == 0 ? 2 : 1;
  if (nkg / sk > MAXKPW) return -4;
  if (!qx || !xs || !w || !ws || !y) return -1;
  const auto* q = (const uint8_t*)qx;
  const auto* p = (const uint8_t*)w;
  auto* o = (uint16_t*)y;
  if (M <= 16) return head::launch<1>(sk, stream, q, xs, p, ws, o, M, K, N);
  if (M <= 32) return head::launch<2>(sk, stream, q, xs, p, ws, o, M, K, N);
  if (M <= 48) return head::launch<3>(sk, stream, q, xs, p, ws, o, M, K, N);
  return head::launch<4>(sk, stream, q, xs, p, ws, o, M, K, N);
}
