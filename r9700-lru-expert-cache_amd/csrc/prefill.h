// The streamed prefill grouped GEMMs (prefill.hip, prefill_roll.hip), launched by the tiled entry
// points of gemm_tiled.hip for the K they take.
#pragma once
#include <hip/hip_runtime.h>

namespace rlu {

// The second weight set and align of a two-set launch: the tiles whose block count carries
// bit 16 take their expert ids, sorted ids, weights and block scales from here.
struct PfSecond {
  const void* wq;
  const float* ws;
  const int* sorted_ids;
  const int* expert_ids;
};

// K and N of the two-set entry points of gemm_tiled.hip (rlu_moe_gemm_prefill's are
// prefill_stream_takes).
bool prefill_stream_built(int K, int N);

// Whether the launches below take mtk rows of this shape (act: the one with the activation).
bool prefill_stream_takes(int mtk, int K, int N, bool act);

// Launches a streamed kernel over a tile list (tiles of <= 8 blocks) when one takes K and N (K =
// 768, or what roll_takes says, N % 256 == 0), and returns 0; returns -1 (nothing
// launched) otherwise. second: null for a one-set tile list.
int launch_prefill_stream(const void* qx, const float* xs, const void* wq, const float* ws,
                          const int* sorted_ids, const int* expert_ids, const PfSecond* second,
                          const int* tiles, const int* ntiles, int max_tiles,
                          const float* topk_weights, void* y, int mtk, int top_k, int K, int N,
                          hipStream_t stream);

// The same kernel for gate_up with SiLU-mul-quant in its epilogue: writes q2 [mtk, N / 2] e4m3
// and s2 [mtk, N / 256] (group-128 scales) instead of the bf16 output. Returns -1 (nothing
// launched) where roll_takes says no; prefill_stream_act_built: the K and N of the _silu_quant entry points.
bool prefill_stream_act_built(int K, int N);
int launch_prefill_stream_act(const void* qx, const float* xs, const void* wq, const float* ws,
                              const int* sorted_ids, const int* expert_ids,
                              const PfSecond* second, const int* tiles, const int* ntiles,
                              int max_tiles, void* q2, float* s2, int mtk, int top_k, int K,
                              int N, hipStream_t stream);

}  // namespace rlu
