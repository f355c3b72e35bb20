// Weight-streaming grouped GEMM for batches whose expert groups are small:
// every weight is used by a few dozen token rows at most, so the launch is
// bound by reading the weights from HBM and the matrix cores only have to
// keep up.
//
// Reference roles: the per-expert GEMMs of Decoder::experts / feed_forward
// (src/decoder/mod.rs:114-122, 197-218), as gemm.hip.
//
// A workgroup of 8 waves computes up to 64 token rows x 256 output features
// of one group with v_mfma_f32_32x32x16_bf16, activations the first operand;
// a wave owns 32 features (for gate/up 16 gate rows and the 16 up rows beside
// them). The weights go from the k-blocked panels straight to the registers
// of the one wave that uses them, two 64-deep chunks ahead, and never through
// LDS; only the activation planes, which all waves read, are staged there
// (double buffered, one barrier per chunk). Two workgroups share a CU, four
// waves a SIMD, so one's waits, conversions and epilogue are covered by the
// others' loads and products (4-wave workgroups of 64 features a wave, two or
// three a CU: 512-token INT8 layer 151 against 125 us). The routed and the
// shared expert's items run in one launch. Gate/up of 61 tokens, BF16: 302 MB
// in 59 us, 5.1 TB/s (88 us before, and 122 us of the shared expert's on a
// second stream); 512 tokens, INT8: 73 us, where the last round of workgroups
// and the widening and scaling VALU work add to the reads.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "mfma.hpp"
#include "moe_kernels.hpp"

namespace uocr {

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 512;
constexpr int kItemN = 256;

__device__ __forceinline__ uint4 load16(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t soff) {
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, 0);
  return make_uint4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t load_rsrc(const void* base, uint32_t bytes) {
  return store_rsrc(const_cast<void*>(base), bytes);
}

// Workgroup barrier that orders LDS only: outstanding global loads stay in
// flight across it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// One 32-deep stage of a wave's 32 weight rows, as the lane holds it: row
// lane % 32, k = 16 (lane / 32) .. +15 of the block (MFMA step s takes the
// eight from 8 s on; the activation fragments follow that order).
template <bool Q8>
struct WeightStage {
  uint4 w[Q8 ? 1 : 2];  // Q8: both steps; BF16: [s]
  float scale;          // Q8: the row's block scale
};

// Rows r0 .. of group g (at most 32 MT), features n0 .. n0 + 256 / KS - 1.
// KS = 2: two sets of four waves take half of K each; the first adds the
// second's sums.
template <int MT, int KS, bool SPLIT, bool GATEUP, bool Q8>
__device__ __forceinline__ void stream_item(const DeviceLayer& L, const Scratch& S,
                                            const MfmaPlanes& P, int T, int g, int r0, int n0,
                                            int base, int mrows, char* lds) {
  static_assert(!GATEUP || KS == 1, "gate and up sums stay whole");
  constexpr int kAP = SPLIT ? 2 : 1;
  constexpr int kRows = 32 * MT;
  constexpr uint32_t kPlane = kRows * 64;      // one plane of one 32-block
  constexpr uint32_t kBuf = 2 * kAP * kPlane;  // a 64-deep chunk
  constexpr int kSetThreads = kThreads / KS;   // threads that share a chunk
  constexpr int kPiecesAll = (int)(kBuf / 16);
  constexpr int kPieces = kPiecesAll >= kSetThreads ? kPiecesAll / kSetThreads : 1;
  const bool routed = g < L.E;
  const int W = L.width(g);
  const int N = GATEUP ? 2 * W : L.H;
  const int K = GATEUP ? L.H : W;
  const int nc = K / 64 / KS;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int set = wave / (8 / KS), wn = wave % (8 / KS);
  const int fr = lane & 31, fc = lane >> 5;
  // A wave past the last column (N is a multiple of 64) multiplies zeros.
  const bool live = n0 + 32 * wn < N;
  char* ring = lds + set * 2 * kBuf;
  const int blk0 = set * nc * 2;  // the set's first 32-block of K

  // ---- activations: thread tid brings 16-byte chunk tid % 4 of a row, for
  // kPieces of the chunk's (block, plane) panels. Rows past the group read
  // as zeros (offset outside the resource). LDS: [block][plane][row][64 B],
  // chunk c of row r at position c ^ ((r >> 2) & 3), which spreads the
  // fragment reads of 16 consecutive rows over all banks.
  const uint16_t* hi = GATEUP ? P.x_hi : routed ? P.h_hi : P.hs_hi;
  const uint16_t* lo = GATEUP ? P.x_lo : routed ? P.h_lo : P.hs_lo;
  const uint32_t a_rows = GATEUP || !routed ? (uint32_t)T : (uint32_t)T * L.K;
  const int stid = tid % kSetThreads;
  const int arow = (stid >> 2) % kRows;
  int src = -1;
  if (arow < mrows) src = GATEUP && routed ? S.perm_rows[base + r0 + arow] : base + r0 + arow;
  const uint32_t a_off = src >= 0 ? (uint32_t)src * 64u + 16u * (tid & 3) : kDmaOut;
  const uint32_t a_lds = (uint32_t)arow * 64u + 16u * ((tid & 3) ^ ((arow >> 2) & 3));
  // Panel (block * kAP + plane) of piece i; wave-uniform. A chunk of fewer
  // pieces than threads is loaded by the first of them only.
  constexpr int kWavesPerPanel = kRows * 4 / 64;
  auto panel = [&](int i) { return (wave % (8 / KS) + 8 / KS * i) / kWavesPerPanel; };
  const bool loads_a = kPiecesAll >= kSetThreads || panel(0) < 2 * kAP;
  uint4 areg[kPieces];
  auto load_a = [&](int c) {
    if (!loads_a) return;
#pragma unroll
    for (int i = 0; i < kPieces; i++) {
      const int bp = panel(i);
      const int blk = blk0 + 2 * c + bp / kAP;
      // No record is in range past the set's last chunk.
      const __amdgpu_buffer_rsrc_t rs =
          load_rsrc(SPLIT && bp % kAP ? lo : hi, c < nc ? a_rows * (uint32_t)K * 2u : 0u);
      areg[i] = load16(rs, a_off, (uint32_t)blk * a_rows * 64u);
    }
  };
  auto store_a = [&](int buf) {
    if (!loads_a) return;
#pragma unroll
    for (int i = 0; i < kPieces; i++)
      *reinterpret_cast<uint4*>(ring + buf * kBuf + panel(i) * kPlane + a_lds) = areg[i];
  };

  // ---- weights, from the panels ([K/32][N][32]) and the block-major scales.
  // Gate/up: lanes 0..15 of a half hold gate rows, lanes 16..31 the up rows
  // of the same hidden columns (gate and up rows alternate in blocks of 32).
  const void* wmat;
  const float* wscale = nullptr;
  if constexpr (Q8) {
    wmat = GATEUP ? (const void*)(L.q13k + L.w13_offset(g)) : (const void*)(L.q2k + L.w2_offset(g));
    wscale = GATEUP ? L.s13k + L.s13_offset(g) : L.s2k + L.s2_offset(g);
  } else {
    wmat = GATEUP ? (const void*)(L.w13k + L.w13_offset(g)) : (const void*)(L.w2k + L.w2_offset(g));
  }
  constexpr uint32_t kRowB = Q8 ? 32 : 64;  // bytes of a row in one block
  const int wrow = GATEUP ? n0 + 64 * (wn >> 1) + 2 * (fr & 16) + 16 * (wn & 1) + (fr & 15)
                          : n0 + 32 * wn + fr;
  const uint32_t w_off = live ? (uint32_t)wrow * kRowB + (kRowB / 2) * fc : kDmaOut;
  const uint32_t s_off = live ? (uint32_t)wrow * 4u : kDmaOut;
  WeightStage<Q8> ws[2][2];  // [chunk parity][block of the chunk]
  auto load_w = [&](WeightStage<Q8>& st, int c, int b) {
    const uint32_t blk = (uint32_t)(blk0 + 2 * c + b);
    const __amdgpu_buffer_rsrc_t rs =
        load_rsrc(wmat, c < nc ? (uint32_t)N * K * (Q8 ? 1u : 2u) : 0u);
    st.w[0] = load16(rs, w_off, blk * N * kRowB);
    if constexpr (Q8) {
      const __amdgpu_buffer_rsrc_t rs_s =
          load_rsrc(wscale, c < nc ? (uint32_t)N * (K / kQBlock) * 4u : 0u);
      st.scale = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs_s, s_off, blk * N * 4u, 0));
    } else {
      st.w[1] = load16(rs, w_off + 16, blk * N * kRowB);
    }
  };

  floatx16 acc[MT];
#pragma unroll
  for (int mi = 0; mi < MT; mi++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[mi][r] = 0.0f;

  auto mma = [](const bf16x8& a, const bf16x8& b, const floatx16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  };
  // One 32-deep block: BF16 weights accumulate across blocks; an INT8
  // block's exact products go into a partial tile that its block scale folds
  // into the accumulator with one FMA per element.
  auto compute = [&](const WeightStage<Q8>& st, const char* a) {
    bf16x8 fb[2];
    if constexpr (Q8) {
      // (Opaque here, or the compiler keeps the widened bytes, not the
      // words, across iterations.)
      uint4 q = st.w[0];
      asm volatile("" : "+v"(q.x), "+v"(q.y), "+v"(q.z), "+v"(q.w));
      fb[0] = widen_int8x8(q.x, q.y);
      fb[1] = widen_int8x8(q.z, q.w);
    } else {
      fb[0] = as_bf16x8(st.w[0]);
      fb[1] = as_bf16x8(st.w[1]);
    }
#pragma unroll
    for (int mi = 0; mi < MT; mi++) {
      const int row = 32 * mi + fr;
      auto frag = [&](int p, int s) {
        return as_bf16x8(*reinterpret_cast<const uint4*>(
            a + p * kPlane + row * 64 + 16 * ((2 * fc + s) ^ ((row >> 2) & 3))));
      };
      floatx16 part = {};
      floatx16& sum = Q8 ? part : acc[mi];
#pragma unroll
      for (int s = 0; s < 2; s++)
#pragma unroll
        for (int p = 0; p < kAP; p++) sum = mma(frag(p, s), fb[s], sum);
      if constexpr (Q8)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[mi][r] = __builtin_fmaf(part[r], st.scale, acc[mi][r]);
    }
  };

  // ---- chunk c multiplies from LDS buffer c % 2 and weight set c % 2 (each
  // stage of which is reloaded for chunk c + 2 as soon as it is used), while
  // the activations of chunk c + 1 wait in registers for the other buffer.
  // That buffer's last readers (chunk c - 1) passed the barrier that ended it.
  auto chunk = [&](auto par, int c) {
    constexpr int kPar = decltype(par)::value;
#pragma unroll
    for (int b = 0; b < 2; b++) {
      compute(ws[kPar][b], ring + kPar * kBuf + b * kAP * kPlane);
      __builtin_amdgcn_sched_barrier(0);
      load_w(ws[kPar][b], c + 2, b);
    }
    store_a(kPar ^ 1);
    load_a(c + 2);
    lds_barrier();
  };
  load_a(0);
#pragma unroll
  for (int i = 0; i < 4; i++) load_w(ws[i / 2][i % 2], i / 2, i % 2);
  store_a(0);
  load_a(1);
  lds_barrier();
  for (int c = 0; c + 1 < nc; c += 2) {
    chunk(std::integral_constant<int, 0>{}, c);
    chunk(std::integral_constant<int, 1>{}, c + 1);
  }
  if (nc & 1) chunk(std::integral_constant<int, 0>{}, nc - 1);

  if constexpr (KS == 2) {
    // The rings are free (every wave is past the last chunk's barrier).
    float* sums = reinterpret_cast<float*>(lds) + wn * (MT * 16 * 64) + lane;
    if (set) {
#pragma unroll
      for (int i = 0; i < MT * 16; i++) sums[i * 64] = acc[i / 16][i % 16];
    }
    lds_barrier();
    if (set) return;
#pragma unroll
    for (int i = 0; i < MT * 16; i++) acc[i / 16][i % 16] += sums[i * 64];
  }
  if (!live) return;

  // Element (mi, r) of this lane: token row 32 mi + 8 (r/4) + 4 fc + r%4, the
  // lane's weight row. Stores go through a resource over exactly the item's
  // rows (rows >= mrows fall past it and are dropped).
  if constexpr (GATEUP) {
    // Lanes fr < 16 hold gate values and lanes fr + 16 the up values of the
    // same elements: the former take elements 0..7, the latter 8..15. The
    // item's rows of one 32-column block of the h planes are one contiguous
    // run of mrows x 64 bytes.
    uint16_t* h_hi = routed ? P.h_hi : P.hs_hi;
    uint16_t* h_lo = routed ? P.h_lo : P.hs_lo;
    const size_t hrows = routed ? (size_t)T * L.K : (size_t)T;
    const size_t run = ((size_t)(n0 / 64 + (wn >> 1)) * hrows + base + r0) * 32;
    const __amdgpu_buffer_rsrc_t rs_hi = store_rsrc(h_hi + run, (uint32_t)mrows * 64u);
    const __amdgpu_buffer_rsrc_t rs_lo = store_rsrc(h_lo + run, (uint32_t)mrows * 64u);
    const bool up = fr & 16;
    const int voff = (4 * fc + (up ? 16 : 0)) * 64 + 2 * (16 * (wn & 1) + (fr & 15));
#pragma unroll
    for (int mi = 0; mi < MT; mi++)
#pragma unroll
      for (int r = 0; r < 8; r++) {
        const float other = __shfl_xor(up ? acc[mi][r] : acc[mi][r + 8], 16);
        const float gv = up ? other : acc[mi][r];
        const float uv = up ? acc[mi][r + 8] : other;
        const int off = vgpr_offset(voff + (mi * 32 + 8 * (r >> 2) + (r & 3)) * 64);
        const float h = gv * __builtin_amdgcn_rcpf(1.0f + __expf(-gv)) * uv;
        const uint16_t hb = bf16_bits(h);
        __builtin_amdgcn_raw_buffer_store_b16(hb, rs_hi, off, 0, 0);
        if constexpr (SPLIT)
          __builtin_amdgcn_raw_buffer_store_b16(bf16_bits(h - __uint_as_float((uint32_t)hb << 16)),
                                                rs_lo, off, 0, 0);
      }
  } else {
    // y in f32; BF16 weights with BF16 activations: rounded to bf16.
    constexpr uint32_t esz = (SPLIT || Q8) ? 4 : 2;
    char* rows = reinterpret_cast<char*>(routed ? S.y : S.ys) + (size_t)(base + r0) * L.H * esz;
    const __amdgpu_buffer_rsrc_t rs = store_rsrc(rows, (uint32_t)mrows * L.H * esz);
    const uint32_t voff = ((uint32_t)(4 * fc) * L.H + wrow) * esz;
#pragma unroll
    for (int mi = 0; mi < MT; mi++)
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int off = vgpr_offset(
            (int)(voff + (uint32_t)(mi * 32 + 8 * (r >> 2) + (r & 3)) * L.H * esz));
        if constexpr (SPLIT || Q8)
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[mi][r]), rs, off, 0, 0);
        else
          __builtin_amdgcn_raw_buffer_store_b16(bf16_bits(acc[mi][r]), rs, off, 0, 0);
      }
  }
}

// Columns of a shared expert's item: the down GEMM's reduction is n_shared
// times a routed item's, so its items are half as wide and split K over two
// sets of waves (otherwise they end the launch by themselves: 61 tokens,
// BF16, down 48 us).
__host__ __device__ constexpr int shared_item_n(bool gateup, int S) {
  return !gateup && S % 128 == 0 ? kItemN / 2 : kItemN;
}

// Work items: the shared expert's (first: in the down GEMM they are the
// deeper ones), column tile by column tile, then the routed tiles', row tile
// by row tile. Each list is cut into 8 contiguous ranges, one per XCD
// (workgroup ids reach the XCDs round-robin), so the items that share
// weights (the shared expert's row tiles) or activations (an expert's column
// tiles) meet in one L2.
template <bool SPLIT, bool GATEUP, bool Q8>
__global__ __launch_bounds__(kThreads, 4) void stream_kernel(DeviceLayer L, Scratch S,
                                                             MfmaPlanes P, int T, int lists) {
  constexpr int kAP = SPLIT ? 2 : 1;
  __shared__ __attribute__((aligned(16))) char lds[(GATEUP ? 1 : 2) * 2 * 2 * kAP * kStreamBM * 64];
  const int shared_tiles = (lists & kListShared) ? (T + kStreamBM - 1) / kStreamBM : 0;
  const int routed_tiles = (lists & kListRouted) ? S.counters[1] : 0;
  const int n_routed = GATEUP ? 2 * L.I : L.H;
  const int n_shared = GATEUP ? 2 * L.S : L.H;
  const int nt_routed = (n_routed + kItemN - 1) / kItemN;
  const int shared_n = shared_item_n(GATEUP, L.S);
  const int nt_shared = (n_shared + shared_n - 1) / shared_n;
  auto cut = [](int n, int x) { return (int)((long long)n * x / kXcds); };
  const int xcd = blockIdx.x % kXcds;
  int j = blockIdx.x / kXcds;
  const int sh0 = cut(shared_tiles * nt_shared, xcd);
  const int n_sh = cut(shared_tiles * nt_shared, xcd + 1) - sh0;
  const int rt0 = cut(routed_tiles * nt_routed, xcd);
  const int n_rt = cut(routed_tiles * nt_routed, xcd + 1) - rt0;
  int g, r0, n0;
  if (j < n_sh) {
    g = L.E;
    r0 = (sh0 + j) % shared_tiles * kStreamBM;
    n0 = (sh0 + j) / shared_tiles * shared_n;
  } else {
    j -= n_sh;
    if (j >= n_rt) return;
    const int tile = (rt0 + j) / nt_routed;
    n0 = (rt0 + j) % nt_routed * kItemN;
    g = S.tiles[2 * tile];
    r0 = S.tiles[2 * tile + 1];
  }
  g = __builtin_amdgcn_readfirstlane(g);
  r0 = __builtin_amdgcn_readfirstlane(r0);
  const bool routed = g < L.E;
  const int base = routed ? S.offsets[g] : 0;
  const int rows = routed ? S.offsets[g + 1] - base : T;
  // Under DynamicActivations the small-batch engine's W8A8 path owns the
  // groups of one row.
  if (Q8 && routed && L.quant_mode == kQuantDynamic && rows == 1) return;
  const int mrows = min(kStreamBM, rows - r0);
  if constexpr (!GATEUP) {
    if (!routed && shared_n != kItemN) {
      if (mrows <= 32)
        stream_item<1, 2, SPLIT, GATEUP, Q8>(L, S, P, T, g, r0, n0, base, mrows, lds);
      else
        stream_item<2, 2, SPLIT, GATEUP, Q8>(L, S, P, T, g, r0, n0, base, mrows, lds);
      return;
    }
  }
  if (mrows <= 32)
    stream_item<1, 1, SPLIT, GATEUP, Q8>(L, S, P, T, g, r0, n0, base, mrows, lds);
  else
    stream_item<2, 1, SPLIT, GATEUP, Q8>(L, S, P, T, g, r0, n0, base, mrows, lds);
}

}  // namespace

template <bool GATEUP>
static void launch_stream(const DeviceLayer& L, const Scratch& S, const MfmaPlanes& P, int T,
                          int tiles_bound, bool bf16_only, int lists, hipStream_t s) {
  // An XCD takes an eighth of the shared items and of the routed ones, each
  // rounded up.
  const int n_routed = GATEUP ? 2 * L.I : L.H, n_shared = GATEUP ? 2 * L.S : L.H;
  const int shared_n = shared_item_n(GATEUP, L.S);
  const long long shared_tiles = lists & kListShared ? (T + kStreamBM - 1) / kStreamBM : 0;
  const long long shared = shared_tiles * ((n_shared + shared_n - 1) / shared_n);
  const long long routed = (lists & kListRouted ? tiles_bound - shared_tiles : 0) *
                           ((n_routed + kItemN - 1) / kItemN);
  const long long per_xcd = (shared + kXcds - 1) / kXcds + (routed + kXcds - 1) / kXcds;
  const dim3 grid((unsigned)(per_xcd * kXcds)), block(kThreads);
  const bool q8 = L.quant_mode != kQuantNone;
  if (q8 && bf16_only)
    stream_kernel<false, GATEUP, true><<<grid, block, 0, s>>>(L, S, P, T, lists);
  else if (q8)
    stream_kernel<true, GATEUP, true><<<grid, block, 0, s>>>(L, S, P, T, lists);
  else if (bf16_only)
    stream_kernel<false, GATEUP, false><<<grid, block, 0, s>>>(L, S, P, T, lists);
  else
    stream_kernel<true, GATEUP, false><<<grid, block, 0, s>>>(L, S, P, T, lists);
}

// Where this engine is the faster one. INT8 weights: everywhere (one layer,
// even routing, one box, against 64 x 512 items on two streams: 17 tokens 120
// -> 64 us, 273 134 -> 112, 512 145 -> 124, 1024 239 -> 195, 4096 675 -> 567).
// BF16 weights: up to the batch where 256 x 256 tiles fill (FP32 class, even /
// Zipf / hot: 64 tokens 149 -> 118 / 133 -> 115 / 131 -> 115 us, 512 169 ->
// 148 / 182 -> 152 / 186 -> 156, 768 179 -> 178 / 192 -> 178 / 193 -> 164, but
// 1024 189 -> 202 / 205 -> 211; BF16 activations, even: 256 133 -> 113, 512
// 135 -> 129, but 768 141 -> 152).
bool stream_preferred(const DeviceLayer& L, int T, bool bf16_only) {
  return L.quant_mode != kQuantNone || T <= (bf16_only ? 512 : 768);
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
