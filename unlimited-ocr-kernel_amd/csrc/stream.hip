// Launches of the weight-streaming grouped GEMM (stream.hpp).
#include "stream.hpp"

namespace uocr {

namespace {

template <int KR, int KSH, bool SPLIT, bool GATEUP, bool Q8>
__global__ __launch_bounds__(kStreamThreads, 4) void stream_kernel(DeviceLayer L, Scratch S,
                                                                   MfmaPlanes P, int T, int lists) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  stream_work<KR, KSH, SPLIT, GATEUP, Q8>(L, S, P, T, lists, (int)blockIdx.x, lds);
}

template <bool GATEUP>
void launch_stream(const DeviceLayer& L, const Scratch& S, const MfmaPlanes& P, int T,
                   int tiles_bound, bool bf16_only, int lists, hipStream_t s) {
  stream_select<GATEUP>(L, T, tiles_bound, bf16_only, lists,
                        [&](auto kr, auto ksh, auto split, auto q8, unsigned blocks, size_t lds) {
                          stream_kernel<kr(), ksh(), split(), GATEUP, q8()>
                              <<<dim3(blocks), dim3(kStreamThreads), lds, s>>>(L, S, P, T, lists);
                        });
}

}  // namespace

// Where this engine is the faster one (one layer, one box, us a layer against
// gemm.hip's tiles with the shared expert on a second stream). INT8 weights:
// everywhere (even routing: 17 tokens 120 -> 64, 273 134 -> 93, 512 145 ->
// 112, 1024 239 -> 190, 2048 386 -> 308). BF16 weights: up to the batch where
// 256 x 256 tiles fill. FP32 class, even / Zipf / hot routing: 512 tokens 173
// -> 141 / 186 -> 153 / 190 -> 149, 896 189 -> 188 / 202 -> 189 / 220 -> 184,
// but 1024 192 -> 199 / 207 -> 211 / 224 -> 199 and 2048 300 -> 312 / 314 ->
// 328 / 305 -> 333. BF16 activations: 512 137 -> 124 / 150 -> 137 / 148 -> 136,
// 640 140 -> 140 / 153 -> 146 / 155 -> 143, but 768 143 -> 151 / 153 -> 150 /
// 159 -> 155.
bool stream_preferred(const DeviceLayer& L, int T, bool bf16_only) {
  return L.quant_mode != kQuantNone || T <= (bf16_only ? 640 : 896);
}

void launch_stream_gateup(const DeviceLayer& L, const Scratch& S, const MfmaPlanes& P, int T,
                          int tiles_bound, bool bf16_only, int lists, hipStream_t s) {
  launch_stream<true>(L, S, P, T, tiles_bound, bf16_only, lists, s);
}

void launch_stream_down(const DeviceLayer& L, const Scratch& S, const MfmaPlanes& P, int T,
                        int tiles_bound, bool bf16_only, int lists, hipStream_t s) {
  launch_stream<false>(L, S, P, T, tiles_bound, bf16_only, lists, s);
}

}  // namespace uocr
