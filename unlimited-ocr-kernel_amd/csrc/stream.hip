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

// Where this engine is the faster one (us a layer, against gemm.hip's tiles
// with the shared expert on a second stream; layers in rotation, so that the
// weights come from memory, except where one layer is said).
//
// INT8 weights: everywhere. Model shape, even / Zipf / hot routing: 17 tokens
// 124 -> 69 / 57 / 50, 512 146 -> 117 / 169 -> 130 / 174 -> 137, 1024 223 ->
// 183 / 222 -> 186 / 229 -> 190, 4096 657 -> 569 / 655 -> 569 / 657 -> 570.
// Slower in one place of thirteen other shapes: 640 to 896 tokens in the FP32
// class on 8 or 16 wide experts, by up to 5% (16 experts, hidden 4096, inner
// 1024: 768 tokens 391 -> 407, but 512 376 -> 356 and 1024 552 -> 484).
//
// BF16 weights: up to the batch where 256 x 256 tiles fill. Model shape, FP32
// class, even / Zipf / hot routing: 512 tokens 165 -> 137 / 176 -> 151 / 183 ->
// 148, 768 173 -> 174 / 187 -> 176 / 198 -> 172, 896 178 -> 185 / 195 -> 189 /
// 214 -> 185, but (one layer) 1024 192 -> 199 / 207 -> 211 / 224 -> 199 and 2048
// 300 -> 312 / 314 -> 328 / 305 -> 333. BF16 activations: 512 133 -> 122 / 146
// -> 134 / 143 -> 134, 640 134 -> 141 / 147 -> 143 / 148 -> 140, but (one layer)
// 768 143 -> 151 / 153 -> 150 / 159 -> 155.
//
// That batch is smaller in wider layers: the tiles' time is mostly the depth
// of a round or two of items, this engine's grows with the operations. It
// fell behind at 6.5 to 13 G multiply-adds a pass, hence the second limit, the
// operations of the model shape's 896 (640) tokens. FP32 class, even routing:
// hidden 2048, inner 1408, 64 experts top-6: 350 tokens 283 -> 271, 640 312 ->
// 347; hidden 4096, inner 4096, 8 experts top-2: 128 tokens 419 -> 360, 512 457
// -> 605; hidden 2880, inner 2880, 32 experts top-4: 128 tokens 513 -> 500, 512
// 542 -> 642. Below it the tiles stay ahead in one shape found, where they fill
// one round and most groups just pass one row tile of this engine: hidden 2048,
// inner 768, 64 experts top-8, 576 tokens 195 -> 221 (but Zipf 265 -> 214).
bool stream_preferred(const DeviceLayer& L, int T, bool bf16_only) {
  if (L.quant_mode != kQuantNone) return true;
  const double macs = (double)T * L.H * ((double)L.K * L.I + L.S);
  return T <= (bf16_only ? 640 : 896) && macs <= (bf16_only ? 5.9e9 : 8.25e9);
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
