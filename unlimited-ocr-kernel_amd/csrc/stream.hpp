// Weight-streaming grouped GEMM for batches whose expert groups are small:
// every weight is used by a few dozen token rows at most, so the launch is
// bound by reading the weights from HBM and the matrix cores only have to
// keep up.
//
// Reference roles: the per-expert GEMMs of Decoder::experts / feed_forward
// (src/decoder/mod.rs:114-122, 197-218), as gemm.hip.
//
// A workgroup of 8 waves computes up to 64 token rows (in tiles of 16) x 256
// output features of one group with v_mfma_f32_16x16x32_bf16, activations the
// first operand; a wave owns 32 features (for gate/up 16 gate rows and the 16
// up rows beside them, so SiLU(g) u is register-local). The weights go from
// the k-blocked panels straight to the registers of the one wave that uses
// them, two 64-deep chunks ahead, and never through LDS; only the activation
// planes, which all waves read, are staged there (double buffered, one barrier
// per chunk). Two workgroups share a CU, four waves a SIMD, so one's waits,
// conversions and epilogue are covered by the others' loads and products. The
// routed and the shared expert's items run in one launch.
//
// What bounds it, one layer, even routing: 61 tokens BF16 gate/up, 302 MB in
// 55 us (5.5 TB/s, against 88 us of 128 x 512 items, with the shared expert's
// 122 us on a second stream); down, 151 MB in 35 us: one CU takes in 25-30
// B/ns, and the workgroups do not divide evenly over 256 CUs. 512 tokens INT8
// gate/up, 170 MB in 62-65 us (94): the matrix cores are busy 0.28 of the time
// and the VALU 0.41 (24 instructions of widening per 32 rows and 32-block, 8 of
// scaling per 16 tokens), so neither they nor HBM set the time; the waves wait.
// (An earlier form that took 74 us took 65 without its weight loads and 69
// without its activation loads.) What they wait for was not taken apart: a
// fragment is read from LDS right before the product that needs it, and each
// item starts with four dependent reads for its 20 (14) chunks. Measured and not
// kept: 32 x 32 MFMA tiles (up to 25% more padding: 512 tokens 122 against 116
// us a layer); 4 waves of 64 features (151 us); 7, 10 or 14 waves a workgroup,
// so that items divide the CUs evenly (one 14-wave workgroup a CU: gate/up 53
// against 58 us at 61 tokens, but 80 against 72 us at 512, its waves in step).
#pragma once

#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "mfma.hpp"
#include "moe_kernels.hpp"
#include "rowdot.hpp"

namespace uocr {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kStreamWaves = 8, kStreamThreads = 64 * kStreamWaves, kStreamN = 32 * kStreamWaves;

__device__ __forceinline__ u32x4 load16(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t soff) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, 0);
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

// One 32-deep stage of a wave's 32 weight rows, as loaded. BF16: fragment f
// (rows 16 f ..) with lane l holding row l % 16, k = 8 (l / 16) .. +7. INT8:
// lane l holds row l % 32, k = 16 (l / 32) .. +15, and the row's block scale;
// fragments() brings both to the same form.
template <bool Q8>
struct WeightStage {
  u32x4 w[Q8 ? 1 : 2];
  uint32_t scale;
};

// Rows r0 .. of group g (at most 16 RT), features n0 .. n0 + 256 / KS - 1.
// KS > 1: KS sets of kStreamWaves / KS waves take a part of K each; the first adds the
// others' sums.
template <int RT, int KS, bool SPLIT, bool GATEUP, bool Q8>
__device__ __forceinline__ void stream_item(const DeviceLayer& L, const Scratch& S,
                                            const MfmaPlanes& P, int T, int g, int r0, int n0,
                                            int base, int mrows, char* lds) {
  constexpr int kAP = SPLIT ? 2 : 1;
  constexpr int kSetWaves = kStreamWaves / KS;
  constexpr uint32_t kTile = 16 * 64;               // 16 rows of one plane and 32-block
  constexpr uint32_t kBuf = 2 * kAP * RT * kTile;   // a 64-deep chunk
  constexpr int kTiles = 2 * kAP * RT;              // its 1 KiB tiles, one wave's load each
  constexpr int kLoads = (kTiles + kSetWaves - 1) / kSetWaves;
  const bool routed = g < L.E;
  const int W = L.width(g);
  const int N = GATEUP ? 2 * W : L.H;
  const int K = GATEUP ? L.H : W;
  const int nc = K / 64 / KS;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int set = KS == 1 ? 0 : wave / kSetWaves, wn = KS == 1 ? wave : wave % kSetWaves;
  // A wave past the last column (N is a multiple of 64) multiplies zeros.
  const bool live = n0 + 32 * wn < N;
  char* ring = lds + set * 2 * kBuf;
  const int blk0 = set * nc * 2;  // the set's first 32-block of K

  // ---- activations: lane l brings 16-byte chunk l % 4 of row l / 4 of a
  // tile. Rows past the group read as zeros (offset outside the resource).
  // LDS: [block][plane][row][64 B], chunk c of row r at position
  // c ^ (-(r >> 2) & 3): a fragment read takes chunk l / 16 of row l % 16 in
  // lane l, and each group of 16 lanes that LDS serves at once (16 chunks of
  // one lane quarter, or lanes 0-3, 12-15, 20-27 and so on) covers all banks.
  const uint16_t* hi = GATEUP ? P.x_hi : routed ? P.h_hi : P.hs_hi;
  const uint16_t* lo = GATEUP ? P.x_lo : routed ? P.h_lo : P.hs_lo;
  const uint32_t a_rows = GATEUP || !routed ? (uint32_t)T : (uint32_t)T * L.K;
  // Tile (block * kAP + plane) * RT + rows / 16; waves past the last one load
  // another copy (the same bytes to the same place).
  auto tile = [&](int i) { return (wn + kSetWaves * i) % kTiles; };
  uint32_t a_off[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; i++) {
    const int row = 16 * (tile(i) % RT) + (lane >> 2);
    int src = -1;
    if (row < mrows) src = GATEUP && routed ? S.perm_rows[base + r0 + row] : base + r0 + row;
    a_off[i] = src >= 0 ? (uint32_t)src * 64u + 16u * (lane & 3) : kDmaOut;
  }
  const uint32_t a_lds = (uint32_t)(lane >> 2) * 64u + 16u * ((lane & 3) ^ (-(lane >> 4) & 3));
  u32x4 areg[kLoads];
  auto load_a = [&](int c) {
#pragma unroll
    for (int i = 0; i < kLoads; i++) {
      const int bp = tile(i) / RT;
      const int blk = blk0 + 2 * c + bp / kAP;
      // No record is in range past the set's last chunk.
      const __amdgpu_buffer_rsrc_t rs =
          load_rsrc(SPLIT && bp % kAP ? lo : hi, c < nc ? a_rows * (uint32_t)K * 2u : 0u);
      areg[i] = load16(rs, a_off[i], (uint32_t)blk * a_rows * 64u);
    }
  };
  auto store_a = [&](int buf) {
#pragma unroll
    for (int i = 0; i < kLoads; i++) {
      *reinterpret_cast<u32x4*>(ring + buf * kBuf + tile(i) * kTile + a_lds) = areg[i];
    }
  };

  // ---- weights, from the panels ([K/32][N][32]) and the block-major scales.
  // Gate/up: the wave's rows 0..15 are gate rows, 16..31 the up rows of the
  // same hidden columns (gate and up rows alternate in blocks of 32).
  const void* wmat;
  const float* wscale = nullptr;
  if constexpr (Q8) {
    wmat = GATEUP ? (const void*)(L.q13k + L.w13_offset(g)) : (const void*)(L.q2k + L.w2_offset(g));
    wscale = GATEUP ? L.s13k + L.s13_offset(g) : L.s2k + L.s2_offset(g);
  } else {
    wmat = GATEUP ? (const void*)(L.w13k + L.w13_offset(g)) : (const void*)(L.w2k + L.w2_offset(g));
  }
  constexpr uint32_t kRowB = Q8 ? 32 : 64;  // bytes of a row in one block
  constexpr int kStep = GATEUP ? 32 : 16;   // rows from fragment 0 to fragment 1
  const int unit = n0 / 32 + wn;            // 32 rows of the matrix
  const int wrow0 = GATEUP ? 64 * (unit >> 1) + 16 * (unit & 1) : 32 * unit;
  uint32_t w_off, s_off = 0;
  if constexpr (Q8) {
    const uint32_t row = wrow0 + (lane & 15) + (lane & 16 ? kStep : 0);
    w_off = row * kRowB + 16 * (lane >> 5);
    s_off = live ? row * 4 : kDmaOut;
  } else {
    w_off = (uint32_t)(wrow0 + (lane & 15)) * kRowB + 16 * (lane >> 4);
  }
  if (!live) w_off = kDmaOut;
  WeightStage<Q8> ws[2][2];  // [chunk parity][block of the chunk]
  auto load_w = [&](WeightStage<Q8>& st, int c, int b) {
    const uint32_t blk = (uint32_t)(blk0 + 2 * c + b);
    const __amdgpu_buffer_rsrc_t rs =
        load_rsrc(wmat, c < nc ? (uint32_t)N * K * (Q8 ? 1u : 2u) : 0u);
    st.w[0] = load16(rs, w_off, blk * N * kRowB);
    if constexpr (Q8) {
      const __amdgpu_buffer_rsrc_t rs_s =
          load_rsrc(wscale, c < nc ? (uint32_t)N * (K / kQBlock) * 4u : 0u);
      st.scale = __builtin_amdgcn_raw_buffer_load_b32(rs_s, s_off, blk * N * 4u, 0);
    } else {
      st.w[1] = load16(rs, w_off + kStep * kRowB, blk * N * kRowB);
    }
  };

  floatx4 acc[RT][2];
#pragma unroll
  for (int rt = 0; rt < RT; rt++)
#pragma unroll
    for (int f = 0; f < 2; f++) acc[rt][f] = floatx4{};

  // One 32-deep block: BF16 weights accumulate across blocks; an INT8
  // block's exact products go into a partial tile that its block scale folds
  // into the accumulator with one FMA per element.
  auto compute = [&](const WeightStage<Q8>& st, const char* a) {
    bf16x8 fb[2];
    float scale[2];
    if constexpr (Q8) {
      // (Opaque here, or the compiler keeps the widened bytes, not the
      // words, across iterations.) Lanes 16 g .. of the load hold rows 0..15
      // (g even) or 16..31 (g odd), k = 16 (g / 2) .. +15; swapping the odd
      // 16 lanes of the first eight k with the even 16 of the last eight
      // leaves rows 0..15 in the one and 16..31 in the other, with
      // k = 8 g ...
      u32x4 q = st.w[0];
      asm volatile("" : "+v"(q));
      const auto s02 = __builtin_amdgcn_permlane16_swap(q.x, q.z, false, false);
      const auto s13 = __builtin_amdgcn_permlane16_swap(q.y, q.w, false, false);
      const auto sc = __builtin_amdgcn_permlane16_swap(st.scale, st.scale, false, false);
#pragma unroll
      for (int f = 0; f < 2; f++) {
        fb[f] = widen_int8x8(s02[f], s13[f]);
        scale[f] = __uint_as_float(sc[f]);
      }
    } else {
      fb[0] = __builtin_bit_cast(bf16x8, st.w[0]);
      fb[1] = __builtin_bit_cast(bf16x8, st.w[1]);
    }
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
      bf16x8 fa[kAP];
#pragma unroll
      for (int p = 0; p < kAP; p++)
        fa[p] = as_bf16x8(*reinterpret_cast<const uint4*>(
            a + (p * RT + rt) * kTile + (lane & 15) * 64 + 16 * ((lane >> 4) ^ (-((lane >> 2) & 3) & 3))));
#pragma unroll
      for (int f = 0; f < 2; f++) {
        floatx4 sum = Q8 ? floatx4{} : acc[rt][f];
#pragma unroll
        for (int p = 0; p < kAP; p++)
          sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[p], fb[f], sum, 0, 0, 0);
        if constexpr (Q8) {
#pragma unroll
          for (int r = 0; r < 4; r++)
            acc[rt][f][r] = __builtin_fmaf(sum[r], scale[f], acc[rt][f][r]);
        } else {
          acc[rt][f] = sum;
        }
      }
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
      compute(ws[kPar][b], ring + kPar * kBuf + b * kAP * RT * kTile);
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

  if constexpr (KS > 1) {
    // The rings are free (every wave is past the last chunk's barrier). Sums
    // of sets 1 .. in set order.
    floatx4* sums = reinterpret_cast<floatx4*>(lds) + lane;
    if (set) {
#pragma unroll
      for (int i = 0; i < 2 * RT; i++)
        sums[(((set - 1) * kSetWaves + wn) * 2 * RT + i) * 64] = acc[i / 2][i % 2];
    }
    lds_barrier();
    if (set) return;
#pragma unroll
    for (int o = 0; o < KS - 1; o++)
#pragma unroll
      for (int i = 0; i < 2 * RT; i++)
        acc[i / 2][i % 2] += sums[((o * kSetWaves + wn) * 2 * RT + i) * 64];
  }
  if (!live) return;

  // Element (rt, f, r) of this lane: token row 16 rt + 4 (lane / 16) + r,
  // weight row lane % 16 of fragment f. Stores go through a resource over
  // exactly the item's rows (rows >= mrows fall past it and are dropped).
  const int row0 = 4 * (lane >> 4);
  if constexpr (GATEUP) {
    // Fragment 0 holds the gate values and 1 the up values of hidden column
    // 16 (unit % 2) + lane % 16 of a 32-column block; the item's rows of that
    // block of the h planes are one contiguous run of mrows x 64 bytes.
    uint16_t* h_hi = routed ? P.h_hi : P.hs_hi;
    uint16_t* h_lo = routed ? P.h_lo : P.hs_lo;
    const size_t hrows = routed ? (size_t)T * L.K : (size_t)T;
    const size_t run = ((size_t)(unit >> 1) * hrows + base + r0) * 32;
    const __amdgpu_buffer_rsrc_t rs_hi = store_rsrc(h_hi + run, (uint32_t)mrows * 64u);
    const __amdgpu_buffer_rsrc_t rs_lo = store_rsrc(h_lo + run, (uint32_t)mrows * 64u);
    const int voff = row0 * 64 + 2 * (16 * (unit & 1) + (lane & 15));
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int off = vgpr_offset(voff + (rt * 16 + r) * 64);
        const float gv = acc[rt][0][r];
        const float h = gv * __builtin_amdgcn_rcpf(1.0f + __expf(-gv)) * acc[rt][1][r];
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
    const uint32_t voff = ((uint32_t)row0 * L.H + wrow0 + (lane & 15)) * esz;
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
      for (int f = 0; f < 2; f++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int off =
              vgpr_offset((int)(voff + ((uint32_t)(rt * 16 + r) * L.H + 16 * f) * esz));
          if constexpr (SPLIT || Q8)
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[rt][f][r]), rs, off, 0, 0);
          else
            __builtin_amdgcn_raw_buffer_store_b16(bf16_bits(acc[rt][f][r]), rs, off, 0, 0);
        }
  }
}

template <int KS, bool SPLIT, bool GATEUP, bool Q8>
__device__ __forceinline__ void stream_rows(const DeviceLayer& L, const Scratch& S,
                                            const MfmaPlanes& P, int T, int g, int r0, int n0,
                                            int base, int mrows, char* lds) {
  if (mrows <= 16)
    stream_item<1, KS, SPLIT, GATEUP, Q8>(L, S, P, T, g, r0, n0, base, mrows, lds);
  else if (mrows <= 32)
    stream_item<2, KS, SPLIT, GATEUP, Q8>(L, S, P, T, g, r0, n0, base, mrows, lds);
  else if (mrows <= 48)
    stream_item<3, KS, SPLIT, GATEUP, Q8>(L, S, P, T, g, r0, n0, base, mrows, lds);
  else
    stream_item<4, KS, SPLIT, GATEUP, Q8>(L, S, P, T, g, r0, n0, base, mrows, lds);
}

// Work items: the shared expert's, column tile by column tile, and the routed
// tiles', row tile by row tile. Each list is cut into 8 contiguous ranges, one
// per XCD (workgroup ids reach the XCDs round-robin), so the items that share
// weights (the shared expert's row tiles) or activations (an expert's column
// tiles) meet in one L2. KR, KSH: the sets of waves that split K in a routed
// and in a shared item, which is then so much narrower and shorter.
// `block`: the workgroup's place among stream_blocks() of them.
template <int KR, int KSH, bool SPLIT, bool GATEUP, bool Q8>
__device__ __forceinline__ void stream_work(const DeviceLayer& L, const Scratch& S,
                                            const MfmaPlanes& P, int T, int lists, int block,
                                            char* lds) {
  constexpr int kRoutedN = kStreamN / KR, kSharedN = kStreamN / KSH;
  const int shared_tiles = (lists & kListShared) ? (T + kStreamBM - 1) / kStreamBM : 0;
  const int routed_tiles = (lists & kListRouted) ? S.counters[1] : 0;
  const int n_routed = GATEUP ? 2 * L.I : L.H;
  const int n_shared = GATEUP ? 2 * L.S : L.H;
  const int nt_routed = (n_routed + kRoutedN - 1) / kRoutedN;
  const int nt_shared = (n_shared + kSharedN - 1) / kSharedN;
  auto cut = [](int n, int x) { return (int)((long long)n * x / kXcds); };
  const int xcd = block % kXcds;
  int j = block / kXcds;
  const int sh0 = cut(shared_tiles * nt_shared, xcd);
  const int n_sh = cut(shared_tiles * nt_shared, xcd + 1) - sh0;
  const int rt0 = cut(routed_tiles * nt_routed, xcd);
  const int n_rt = cut(routed_tiles * nt_routed, xcd + 1) - rt0;
  if (j >= n_sh + n_rt) return;
  // The longer items first.
  constexpr bool kSharedLast = GATEUP;
  const bool shared = kSharedLast ? j >= n_rt : j < n_sh;
  if (shared) {
    if (kSharedLast) j -= n_rt;
    const int r0 = (sh0 + j) % shared_tiles * kStreamBM;
    const int n0 = (sh0 + j) / shared_tiles * kSharedN;
    stream_rows<KSH, SPLIT, GATEUP, Q8>(L, S, P, T, L.E, r0, n0, 0, min(kStreamBM, T - r0),
                                            lds);
    return;
  }
  if (!kSharedLast) j -= n_sh;
  const int tile = (rt0 + j) / nt_routed;
  const int n0 = (rt0 + j) % nt_routed * kRoutedN;
  const int g = __builtin_amdgcn_readfirstlane(S.tiles[2 * tile]);
  const int r0 = __builtin_amdgcn_readfirstlane(S.tiles[2 * tile + 1]);
  const int base = S.offsets[g];
  const int rows = S.offsets[g + 1] - base;
  // Under DynamicActivations the small-batch engine's W8A8 path owns the
  // groups of one row.
  if (Q8 && L.quant_mode == kQuantDynamic && rows == 1) return;
  stream_rows<KR, SPLIT, GATEUP, Q8>(L, S, P, T, g, r0, n0, base, min(kStreamBM, rows - r0),
                                         lds);
}

constexpr size_t stream_lds(int sets, bool split) {
  return (size_t)sets * 2 * 2 * (split ? 2 : 1) * kStreamBM * 64;
}

// Calls go(KR, KSH, SPLIT, Q8, workgroups, LDS bytes) with the kernel's
// template arguments as integral constants.
template <int KR, int KSH, bool GATEUP, typename Go>
void stream_shape(const DeviceLayer& L, int T, int tiles_bound, bool bf16_only, int lists, Go go) {
  if constexpr (KR > 1) {
    if ((GATEUP ? L.H : L.I) / 64 % KR)
      return stream_shape<1, KSH, GATEUP>(L, T, tiles_bound, bf16_only, lists, go);
  }
  // (Where I / 64 is even, so is S / 64: S is a multiple of I.)
  if constexpr (KSH > 1 && KR == 1) {
    if ((GATEUP ? L.H : L.S) / 64 % KSH)
      return stream_shape<KR, 1, GATEUP>(L, T, tiles_bound, bf16_only, lists, go);
  }
  // An XCD takes an eighth of the shared items and of the routed ones, each
  // rounded up.
  const int n_routed = GATEUP ? 2 * L.I : L.H, n_shared = GATEUP ? 2 * L.S : L.H;
  const int routed_n = kStreamN / KR, shared_n = kStreamN / KSH;
  const long long shared_tiles = (T + kStreamBM - 1) / kStreamBM;
  const long long shared =
      lists & kListShared ? shared_tiles * ((n_shared + shared_n - 1) / shared_n) : 0;
  const long long routed = lists & kListRouted
                               ? (tiles_bound - shared_tiles) * ((n_routed + routed_n - 1) / routed_n)
                               : 0;
  const long long per_xcd = (shared + kXcds - 1) / kXcds + (routed + kXcds - 1) / kXcds;
  if (per_xcd == 0) return;
  const unsigned blocks = (unsigned)(per_xcd * kXcds);
  const int sets = std::max(KR, lists & kListShared ? KSH : 1);
  const std::integral_constant<int, KR> kr;
  const std::integral_constant<int, KSH> ksh;
  const bool q8 = L.quant_mode != kQuantNone;
  if (q8 && bf16_only)
    go(kr, ksh, std::false_type{}, std::true_type{}, blocks, stream_lds(sets, false));
  else if (q8)
    go(kr, ksh, std::true_type{}, std::true_type{}, blocks, stream_lds(sets, true));
  else if (bf16_only)
    go(kr, ksh, std::false_type{}, std::false_type{}, blocks, stream_lds(sets, false));
  else
    go(kr, ksh, std::true_type{}, std::false_type{}, blocks, stream_lds(sets, true));
}

template <bool GATEUP, typename Go>
void stream_select(const DeviceLayer& L, int T, int tiles_bound, bool bf16_only, int lists, Go go) {
  // The shared items in two sets of waves: gate/up runs them last, where short
  // items fill the CUs that the routed ones leave (512 tokens, INT8: 69 -> 62
  // us; in one set and first, all but the last few ran in a first round of
  // two workgroups a CU), down first, where they are n_shared times as deep.
  // Down's routed items too at small batches: 320 workgroups of 256 features
  // leave most CUs one and some two (61 tokens, BF16: 39 -> 35 us; 273 tokens,
  // INT8, even routing: 30 -> 28 us, but Zipf routing 131 -> 135 us a layer,
  // 512 tokens 37 -> 45 us and 24 tokens with Zipf routing 78 -> 83 us a
  // layer: twice the activation reads).
  if constexpr (!GATEUP) {
    if (T > 32 && T <= 256)
      return stream_shape<2, 2, GATEUP>(L, T, tiles_bound, bf16_only, lists, go);
  }
  stream_shape<1, 2, GATEUP>(L, T, tiles_bound, bf16_only, lists, go);
}

}  // namespace uocr
