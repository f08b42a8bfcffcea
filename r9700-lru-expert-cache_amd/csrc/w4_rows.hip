// The W4 lm_head for 17 .. 64 rows in one weight read (w4.hip holds the format and the kernel for up
// to 16, whose x fits in LDS whole).
//
// Bound: the codes and scales are 207 MB at vocab 151936 x 2560, and launches of 16 rows (40-43 us
// each) read and dequantize them again for every 16 rows: 20 rows 85 us, 64 rows 165. One read
// for all takes 49 us at 17-32 rows, 59 at 48 and 73 at 64, where the matrix cores, the
// dequantization and the LDS reads of x, 5, 8 and 4 us per 16 rows alone, overlap only in part.
//
//   * x of 64 rows (328 KB at K = 2560) does not fit in LDS, so here K is the outer loop: each of 8 x
//     CUs waves owns up to PMAX 16-row strips of W for the whole K (37.1 strips per CU at that
//     vocab, in waves of 4 or 5) with their f32 accumulators in registers, and the workgroup
//     stages x in chunks of CG 128-deep groups, double-buffered, loaded one chunk ahead, one
//     barrier per chunk. Past PMAX strips per wave the launch makes equal passes over W.
//   * A wave's codes and scale words run in a ring of registers a chunk (more for few strips)
//     ahead, through buffers of zero size past K and past the wave's strips.
//   * Strips go SB at a time: dequantized once, then the blocks of x in turn. The next block's
//     fragments are read into the registers the MFMAs just read, and a block is scaled behind
//     the next one's MFMAs (the empty asm statements keep that order). Against reading and
//     scaling each block in turn: 64 rows 79 -> 73 us, 48 rows 65 -> 59. SB 3 has too few
//     registers at 4 blocks (79 us), SB 1 rereads x (75).
//   * Offset and zero: the wave that stages a block's group also sums its rows with MFMAs of ones; a
//     group's product is then scale * (d - (128 + zero) * sum), in f32.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemm_common.h"
#include "numerics.h"
#include "rlu.h"
#include "w4_dequant.h"
#include "wave.h"

namespace rlu {
namespace w4 {

constexpr int RW = 8;          // waves per workgroup
constexpr int CG = 2;          // 128-deep groups per activation chunk
constexpr int PMAX = 5;        // strips per wave

// groups of weights in flight per wave of p strips
__host__ __device__ constexpr int rows_ring(int p) { return p == 1 ? 8 : p == 2 ? 4 : 2; }

template <int MB, int P>
__global__ __launch_bounds__(RW * WAVE, 2) void rows_k(const uint16_t* __restrict__ x, int M,
                                                       int K, const v4u* __restrict__ wq,
                                                       const unsigned* __restrict__ sz,
                                                       uint16_t* __restrict__ y, int N,
                                                       int passes) {
  constexpr int D = rows_ring(P), DC = D / CG;
  constexpr int SB = MB < 4 ? 3 : 2;                // strips dequantized at a time
  static_assert(D % CG == 0 && CG * MB <= RW, "whole chunks; a wave stages one block of a group");
  __shared__ v4u xa[2][CG][MB][4][WAVE];
  __shared__ __align__(16) float xsl[2][CG][MB * 16];   // minus the rows' sums over the group
  const int lane = lane_id();
  const int w = uniform((int)threadIdx.x / WAVE);
  const int r16 = lane & 15, c4 = lane >> 4;
  const int G = K / 128, NS = N / 16, NCH = (G + CG - 1) / CG;
  const unsigned mask = uniform(0x000F000F), magic = 0x43004300u;
  const int slots = passes * (int)gridDim.x * RW;
  const int ga = w / MB, ba = w - ga * MB;          // the group and block this wave stages
  const bool stages = w < CG * MB;

  v4u ra[4];
  auto stage = [&](int c) __attribute__((always_inline)) {
    const int g = c * CG + ga;
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        (void*)x, 0, stages && g < G ? M * K * 2 : 0, BUF_WORD3);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      ra[i] = __builtin_bit_cast(
          v4u, __builtin_amdgcn_raw_buffer_load_b128(
                   rx, (16 * ba + r16) * K * 2 + c4 * 16 + i * 64, g * 256, 0));
  };
  auto write_a = [&](int buf) __attribute__((always_inline)) {
    if (stages) {
      const v4u ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
      v4f d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        xa[buf][ga][ba][i][lane] = ra[i];
        d = mfma_bf16(ones, ra[i], d);
      }
      if (c4 == 0) xsl[buf][ga][ba * 16 + r16] = -d[0];
    }
  };

  for (int p = 0; p < passes; ++p) {
    const long long q = (long long)p * gridDim.x * RW + (int)blockIdx.x * RW + w;
    const int s0 = (int)(NS * q / slots), cnt = (int)(NS * (q + 1) / slots) - s0;
    v4u rw[D][P];
    unsigned rs[D][P];
    auto load = [&](int j, int g) __attribute__((always_inline)) {
      const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(wq + (size_t)s0 * G * 64), 0, g < G ? cnt * G * 1024 : 0, BUF_WORD3);
      const __amdgpu_buffer_rsrc_t rz = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(sz + (size_t)s0 * G * 16), 0, g < G ? cnt * G * 64 : 0, BUF_WORD3);
#pragma unroll
      for (int s = 0; s < P; ++s) {
        rw[j][s] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(
                                               rq, lane * 16, (s * G + g) * 1024, SLC));
        rs[j][s] = __builtin_amdgcn_raw_buffer_load_b32(rz, r16 * 4, (s * G + g) * 64, 0);
      }
    };
    v4f acc[MB][P];
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
      for (int s = 0; s < P; ++s) acc[b][s] = v4f{0.f, 0.f, 0.f, 0.f};
    stage(0);
#pragma unroll
    for (int j = 0; j < D; ++j) load(j, j);
    write_a(0);
    lds_barrier();
    for (int c0 = 0; c0 < NCH; c0 += DC) {
#pragma unroll
      for (int jc = 0; jc < DC; ++jc) {
        const int c = c0 + jc, buf = c & 1;
        stage(c + 1);
        v4u a[4];
        v4f nx[2], d[2][SB];
        auto rda = [&](int gi, int bk, int i) __attribute__((always_inline)) {
          a[i] = xa[buf][gi][bk][i][lane];
        };
        auto rdn = [&](int gi, int bk) __attribute__((always_inline)) {
          nx[bk & 1] = *reinterpret_cast<const v4f*>(&xsl[buf][gi][bk * 16 + 4 * c4]);
        };
#pragma unroll
        for (int i = 0; i < 4; ++i) rda(0, 0, i);
#pragma unroll
        for (int gi = 0; gi < CG; ++gi) {
          const int j = jc * CG + gi;
#pragma unroll
          for (int sb = 0; sb < P; sb += SB) {
            v4u b[SB][4];
            float sc[SB], zz[SB];
            rdn(gi, 0);
#pragma unroll
            for (int t = 0; t < SB && sb + t < P; ++t) {
              const unsigned sv = rs[j][sb + t];
              dequant(rw[j][sb + t], mask, magic, b[t]);
              sc[t] = __uint_as_float(sv << 16);
              zz[t] = 128.0f + (float)(short)(sv >> 16);
            }
            if (sb + SB >= P) load(j, c * CG + gi + D);
            auto scale = [&](int bk) __attribute__((always_inline)) {
#pragma unroll
              for (int t = 0; t < SB && sb + t < P; ++t) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                  acc[bk][sb + t][i] = fmaf(sc[t], fmaf(nx[bk & 1][i], zz[t], d[bk & 1][t][i]),
                                            acc[bk][sb + t][i]);
                asm volatile("" : "+v"(acc[bk][sb + t]));
              }
            };
#pragma unroll
            for (int bk = 0; bk < MB; ++bk) {
              const bool lastb = bk + 1 == MB, lastu = lastb && sb + SB >= P;
              const int ng = lastu ? gi + 1 : gi, nb = lastb ? 0 : bk + 1;   // the next unit
#pragma unroll
              for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int t = 0; t < SB && sb + t < P; ++t) {
                  d[bk & 1][t] =
                      mfma_bf16(a[i], b[t][i], i ? d[bk & 1][t] : v4f{0.f, 0.f, 0.f, 0.f});
                  asm volatile("" : "+v"(d[bk & 1][t]));
                }
                if (ng < CG) rda(ng, nb, i);
              }
              if (bk > 0) scale(bk - 1);
              if (!lastb) rdn(gi, bk + 1);
              __builtin_amdgcn_sched_barrier(0);
            }
            scale(MB - 1);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        write_a(buf ^ 1);
        lds_barrier();
      }
    }
#pragma unroll
    for (int s = 0; s < P; ++s)
      if (s < cnt)
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int row = 16 * b + 4 * c4 + i;
            if (row < M) y[(size_t)row * N + (s0 + s) * 16 + r16] = f32_to_bf16(acc[b][s][i]);
          }
  }
}

template <int MB>
static int launch_rows(const uint16_t* x, int M, int K, const v4u* wq, const unsigned* sz,
                       uint16_t* y, int N, hipStream_t st) {
  const int NS = N / 16;
  int grid = device_cus();
  if (grid > (NS + RW - 1) / RW) grid = (NS + RW - 1) / RW;
  const int per = (NS + grid * RW - 1) / (grid * RW);          // strips per wave
  const int passes = (per + PMAX - 1) / PMAX;
  const int p = (NS + grid * RW * passes - 1) / (grid * RW * passes);
#define RLU_R(P)                                                                            \
  hipLaunchKernelGGL((rows_k<MB, P>), dim3(grid), dim3(RW * WAVE), 0, st, x, M, K, wq, sz, \
                     y, N, passes)
  switch (p) {
    case 1: RLU_R(1); break;
    case 2: RLU_R(2); break;
    case 3: RLU_R(3); break;
    case 4: RLU_R(4); break;
    default: RLU_R(5); break;
  }
#undef RLU_R
  return (int)hipGetLastError();
}

}  // namespace w4
}  // namespace rlu

extern "C" int rlu_gemm_w4_m64(const void* x, int M, int K, const void* wq, const unsigned* sz,
                               void* y, int N, hipStream_t stream) {
  using namespace rlu::w4;
  if (M < 17 || M > 64 || K <= 0 || N <= 0) return -1;
  if (K % 128 || N % 32 || K > MAXK) return -2;
  const int G = K / 128;                            // (the 16-row kernel's K)
  if (G / (G % 4 == 0 ? 4 : G % 2 == 0 ? 2 : 1) > MAXGQ) return -2;
  if ((long long)N * K / 2 >= (1LL << 31)) return -2;
  if (!x || !wq || !sz || !y) return -1;
  const auto* a = (const uint16_t*)x;
  const auto* q = (const rlu::v4u*)wq;
  auto* o = (uint16_t*)y;
  if (M <= 32) return launch_rows<2>(a, M, K, q, sz, o, N, stream);
  if (M <= 48) return launch_rows<3>(a, M, K, q, sz, o, N, stream);
  return launch_rows<4>(a, M, K, q, sz, o, N, stream);
}
