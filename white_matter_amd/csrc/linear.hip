// A feedback layer's products on a token group's rows, out = x W^T with bf16
// operands and fp32 sums, and what follows each product within its tile: the
// query's RMS norm and RoPE, or the gated activation of a pair of products
// (reference blocks/decoder_layer.py:51-72, layers/white_matter.py:105-118).
//
// These products are small (a group's 12 to 2,048 rows by widths of 128 to
// 3,072): a few us each, of which the library's call alone takes 19 us of host
// time, the three calls of a gated pair 44. Through the C++ operators a product
// takes 5 to 6 us of host time, and the norm, RoPE and activation kernels and
// their round trips go. GPU time in us, before (with the fused step's own kernel)
// and here, for widths 512 and 1536 (1024 and 3072):
//   rows   plain d -> d       plain 3d -> d      query              gated
//   1      3.7 3.0 (4.2 3.7)  4.9 4.4 (6.6 6.4)  5.9 4.4 (6.5 5.5)  9.3 3.9 (10.2 5.0)
//   128    6.6 3.2 (5.4 3.9)  5.0 4.5 (6.9 6.7)  9.2 4.6 (8.0 5.7)  15.4 4.1 (18.9 7.1)
//   1024   5.7 4.3 (7.8 6.5)  7.5 7.1 (14.8 14.4)  8.7 4.8 (11.2 7.8)  20.4 12.0 (32 25)
// They are bound by the latency of a workgroup's chain of stages: at most 64
// rows of operands a stage pass a CU's vector cache at 64 B a clock. Larger
// products, which are bound by the matrix cores, stay with the library
// (cyclic_pass.py).
#include "lds_tiles.h"
#include "wmx_kernels.h"

namespace wmx {

namespace {

constexpr int kStep = kRowElems;  // contraction elements of a stage
constexpr int kXcds = 8;

// The host pass needs the kernels' launch stubs only (it drops those of every
// instantiation after the first over the buffer-resource helpers).
#ifdef __HIP_DEVICE_COMPILE__
// Up to ROWS rows of one operand as the stages of a contraction over K. Rows
// past the last, elements past K and a stage past the last read as zeros:
// every stage issues the same loads, so that one wait count holds on every path
// (where the compiler sees paths with fewer loads behind a stage's, it waits
// for all loads before that stage is read).
template <int ROWS>
struct Operand {
  using DMA = TileDMA<kStep, 4, ROWS>;
  const bf16* base;
  int K, span;  // elements from the first row to the end of the last
  unsigned off[DMA::kInstr];

  __device__ __forceinline__ void init(const DMA& dma, const void* x, int64_t row, int64_t stride, int64_t rows, int K_) {
    base = (const bf16*)x + row * stride;
    K = K_;
    const int n = (int)min((int64_t)ROWS, rows - row);
    span = n > 0 ? (n - 1) * (int)stride + K : 0;
    dma.strided_offsets((int)stride * 2, off);
  }
  __device__ __forceinline__ void issue(const DMA& dma, int kt, bf16* tile) const {
    const int k0 = kt * kStep, left = K - k0;
    const rsrc_t rs = make_rsrc(base + (left > 0 ? k0 : 0), left > 0 ? max(span - k0, 0) * 2 : 0);
    unsigned part[DMA::kInstr];
#pragma unroll
    for (int r = 0; r < DMA::kInstr; ++r) part[r] = dma.chunk16(r) < 2 * left ? off[r] : kOutOfRange;
    dma.issue_strided(rs, tile, part);
  }
};

// Runs `stage(buffer, it)` for every stage of the contraction, buffers in turn.
template <int NS, class Stage>
__device__ __forceinline__ void for_stages(int count, Stage stage) {
  for (int it = 0;;) {
    stage(std::integral_constant<int, 0>{}, it);
    if (++it >= count) break;
    stage(std::integral_constant<int, 1>{}, it);
    if (++it >= count) break;
    if constexpr (NS > 2) {
      stage(std::integral_constant<int, 2>{}, it);
      if (++it >= count) break;
    }
    if constexpr (NS > 3) {
      stage(std::integral_constant<int, 3>{}, it);
      if (++it >= count) break;
    }
  }
}

// Roundings are the model's: each product to bf16 first (as silu_mul_kernel, query_norm_rope_kernel).
__device__ __forceinline__ float gated(float gate, float up) {
  const float g = round_bf16(gate);
  return round_bf16(g / (1.f + expf(-g))) * round_bf16(up);
}

// One head (D columns from n0) of ROWS rows: RMS norm, weight, bf16, RoPE.
// product(r, d0, q) gives elements d0 .. d0 + 7 of row r. D / 8 lanes (rounded up to a power of two)
// hold a row.
template <int D, int ROWS, class Product>
__device__ __forceinline__ void query_rows(const wmx_linear_args& a, int64_t m0, int n0, int mrows, Product product) {
#pragma clang fp contract(off)
  constexpr int L = D / 8, LPR = D == 96 ? 16 : L;
  const int l = threadIdx.x % LPR, lane = threadIdx.x & 63, from = l < L / 2 ? lane + L / 2 : lane - L / 2;
  const int d0 = l < L ? 8 * l : 0;
  float w[8];
  load8(a.norm, d0, a.norm_dtype == WMX_DTYPE_BF16, w);
  for (int r = threadIdx.x / LPR; r < ROWS; r += 256 / LPR) {
    const bool live = r < mrows && l < L;
    float q[8], c[8], s[8];
    product(r, d0, q);  // (rows past the last are zero)
#pragma unroll
    for (int e = 0; e < 8; ++e) q[e] = round_bf16(q[e]);
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) ss = fmaf(q[e], q[e], ss);
    ss = l < L ? ss : 0.f;
#pragma unroll
    for (int o = LPR / 2; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
    const float inv = rsqrtf(ss / (float)D + a.eps);
    const int64_t n = m0 + (live ? r : 0);
    const int64_t rope = n / a.tokens_per_row * a.rope_stride[0] + n % a.tokens_per_row * a.rope_stride[1] + d0;
    load8(a.cos, rope, false, c);
    load8(a.sin, rope, false, s);
    float y[8], out[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = round_bf16((q[e] * inv) * w[e]);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float p = __shfl(y[e], from);
      out[e] = y[e] * c[e] + (l < L / 2 ? -p : p) * s[e];
    }
    if (live)
      *reinterpret_cast<u32x4*>((bf16*)a.out + n * a.out_features + n0 + d0) =
          u32x4{pack_bf16x2(out[0], out[1]), pack_bf16x2(out[2], out[3]), pack_bf16x2(out[4], out[5]), pack_bf16x2(out[6], out[7])};
  }
}

// This workgroup's tile: consecutive tiles (rows first: they share weight rows)
// on one XCD.
__device__ __forceinline__ bool decode_tile(int64_t rows, int cols, int bm, int bn, int64_t& m0, int& n0) {
  const unsigned mt = (unsigned)((rows + bm - 1) / bm), total = mt * (unsigned)((cols + bn - 1) / bn);
  const unsigned u = blockIdx.x % kXcds * ((total + kXcds - 1) / kXcds) + blockIdx.x / kXcds;
  m0 = (int64_t)(u % mt) * bm;
  n0 = (int)(u / mt) * bn;
  return u < total;
}
#endif

// A workgroup computes 64 rows by 64 weight rows (WT = 2: of the gate's and of
// the up projection's weight). Four waves take 32 rows by 32 columns of every
// tile. NS stages of the contraction stream through LDS, NS - 1 of them in
// flight.
template <int WT, int NS>
__global__ __launch_bounds__(256, 1) void linear_kernel(const wmx_linear_args a) {
#ifdef __HIP_DEVICE_COMPILE__
  constexpr int BM = kTileRows, BN = 64, kStage = (1 + WT) * kTileElems;
  // separate arrays, so that the compiler sees that a stage that streams in
  // is not the one that is read
  __shared__ __attribute__((aligned(1024))) bf16 s0[kStage];
  __shared__ __attribute__((aligned(1024))) bf16 s1[kStage];
  __shared__ __attribute__((aligned(1024))) bf16 s2[kStage];
  __shared__ __attribute__((aligned(1024))) bf16 s3[NS > 3 ? kStage : 8];
  static_assert(NS == 3 || NS == 4, "stages");

  int64_t m0;
  int n0;
  if (!decode_tile(a.rows, a.out_features, BM, BN, m0, n0)) return;
  const int mrows = (int)min((int64_t)BM, a.rows - m0);
  const int lane = threadIdx.x & 63, wave = wave_id(), half = lane >> 5, col = lane & 31;
  const int wm = wave & 1, wn = wave >> 1;

  using Tile = Operand<BM>;
  typename Tile::DMA dma;
  dma.init(wave, lane);
  Tile x, w[WT];
  x.init(dma, a.x, m0, a.x_stride, a.rows, a.in_features);
#pragma unroll
  for (int j = 0; j < WT; ++j) w[j].init(dma, j ? a.weight2 : a.weight, n0, a.in_features, a.out_features, a.in_features);
  auto issue = [&](int kt, bf16* st) __attribute__((always_inline)) {
    x.issue(dma, kt, st);
#pragma unroll
    for (int j = 0; j < WT; ++j) w[j].issue(dma, kt, st + (1 + j) * kTileElems);
  };

  RowReads<kStep / 16> rd;
  rd.init(col, half);
  f32x16 acc[WT];
#pragma unroll
  for (int j = 0; j < WT; ++j) acc[j] = f32x16{};
  auto products = [&](const bf16* st) __attribute__((always_inline)) {
    constexpr int KS = kStep / 16, PF = 4;
    rd.refresh();
    const bf16* xt = st + wm * 32 * kRowElems;
    const bf16* wt = st + kTileElems + wn * 32 * kRowElems;
    bf16x8 xo[KS], wo[KS][WT];
    auto fetch = [&](int s) __attribute__((always_inline)) {
      xo[s] = rd.get(xt, s, 0);
#pragma unroll
      for (int j = 0; j < WT; ++j) wo[s][j] = rd.get(wt, s, 2 * j);
    };
#pragma unroll
    for (int s = 0; s < PF; ++s) fetch(s);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      __builtin_amdgcn_sched_barrier(0);
      if (s + PF < KS) fetch(s + PF);
#pragma unroll
      for (int j = 0; j < WT; ++j) acc[j] = mfma32(wo[s][j], xo[s], acc[j]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  issue(0, s0);
  issue(1, s1);
  if (NS > 3) issue(2, s2);
  for_stages<NS>((a.in_features + kStep - 1) / kStep, [&](auto bufc, int it) __attribute__((always_inline)) {
    constexpr int B = decltype(bufc)::value, BX = (B + NS - 1) % NS;
    // stage `it` has landed (the NS - 2 issued after it may still fly), and
    // every wave is done with the buffer that is filled next
    lds_sync<(NS - 2) * (1 + WT) * Tile::DMA::kInstr>();
    issue(it + NS - 1, BX == 0 ? s0 : BX == 1 ? s1 : BX == 2 ? s2 : s3);
    products(B == 0 ? s0 : B == 1 ? s1 : B == 2 ? s2 : s3);
  });
  dma_barrier();  // every wave is done with the stages: the tile's rows are laid out in the first

  // acc[j][r] is row 32 wm + col, column 32 wn + 8 (r / 4) + 4 half + r % 4
  constexpr int P = BN + 8;  // pitch
  bf16* const mine = s0 + (32 * wm + col) * P + 32 * wn + 4 * half;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    float y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      y[e] = acc[0][4 * g + e];
      if constexpr (WT == 2) y[e] = gated(y[e], acc[1][4 * g + e]);
    }
    *reinterpret_cast<u32x2*>(mine + 8 * g) = u32x2{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
  }
  lds_barrier();
  bf16* const orow = (bf16*)a.out + m0 * a.out_features + n0;
#pragma unroll
  for (int i = threadIdx.x; i < BM * 8; i += 256) {
    const int r = i >> 3, c = 8 * (i & 7);
    if (r < mrows && n0 + c < a.out_features)
      *reinterpret_cast<u32x4*>(orow + (int64_t)r * a.out_features + c) = *reinterpret_cast<const u32x4*>(s0 + r * P + c);
  }
#endif
}

// 32 rows by WT tiles of 32 weight rows (the gate's and the up projection's, or
// a head's), each of the four waves a quarter of every stage's contraction, the
// fp32 sums added through LDS at the end. A stage's time is its bytes through
// the CU's vector cache (64 B a clock), half of a 64-row stage's, and four times
// as many CUs take part.
template <int KIND, int WT, int NS>
__global__ __launch_bounds__(256, WT <= 2 ? 2 : 1) void linear_small_kernel(const wmx_linear_args a) {
#ifdef __HIP_DEVICE_COMPILE__
  constexpr bool kGated = KIND == WMX_LINEAR_GATED, kQuery = KIND == WMX_LINEAR_QUERY;
  constexpr int BM = 32, BN = kGated ? 32 : 32 * WT, kHalf = kTileElems / 2, kStage = (1 + WT) * kHalf;
  __shared__ __attribute__((aligned(1024))) bf16 s0[kStage];
  __shared__ __attribute__((aligned(1024))) bf16 s1[kStage];
  __shared__ __attribute__((aligned(1024))) bf16 s2[kStage];
  __shared__ __attribute__((aligned(1024))) bf16 s3[NS > 3 ? kStage : 8];
  static_assert(NS == 3 || NS == 4, "stages");
  int64_t m0;
  int n0;
  if (!decode_tile(a.rows, a.out_features, BM, BN, m0, n0)) return;
  const int mrows = (int)min((int64_t)BM, a.rows - m0);
  const int lane = threadIdx.x & 63, wave = wave_id(), half = lane >> 5, col = lane & 31;
  using Tile = Operand<32>;
  typename Tile::DMA dma;
  dma.init(wave, lane);
  Tile x, w[WT];
  x.init(dma, a.x, m0, a.x_stride, a.rows, a.in_features);
#pragma unroll
  for (int j = 0; j < WT; ++j) {
    if constexpr (kGated) w[j].init(dma, j ? a.weight2 : a.weight, n0, a.in_features, a.out_features, a.in_features);
    else w[j].init(dma, a.weight, n0 + 32 * j, a.in_features, a.out_features, a.in_features);
  }
  auto issue = [&](int kt, bf16* st) __attribute__((always_inline)) {
    x.issue(dma, kt, st);
#pragma unroll
    for (int j = 0; j < WT; ++j) w[j].issue(dma, kt, st + (1 + j) * kHalf);
  };
  constexpr int KS = kStep / 16 / 4;  // this wave's MFMA steps of a stage
  RowReads<KS> rd;
#pragma unroll
  for (int s = 0; s < KS; ++s) rd.off[s] = 2 * tile_elem(col, 2 * (KS * wave + s) + half);
  f32x16 acc[WT];
#pragma unroll
  for (int j = 0; j < WT; ++j) acc[j] = f32x16{};
  issue(0, s0);
  issue(1, s1);
  if (NS > 3) issue(2, s2);
  for_stages<NS>((a.in_features + kStep - 1) / kStep, [&](auto bufc, int it) __attribute__((always_inline)) {
    constexpr int B = decltype(bufc)::value, BX = (B + NS - 1) % NS;
    lds_sync<(NS - 2) * (1 + WT) * Tile::DMA::kInstr>();
    issue(it + NS - 1, BX == 0 ? s0 : BX == 1 ? s1 : BX == 2 ? s2 : s3);
    const bf16* st = B == 0 ? s0 : B == 1 ? s1 : B == 2 ? s2 : s3;
    rd.refresh();
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const bf16x8 xo = rd.get(st, s, 0);
#pragma unroll
      for (int j = 0; j < WT; ++j) acc[j] = mfma32(rd.get(st, s, 1 + j), xo, acc[j]);
    }
  });
  dma_barrier();  // every wave is done with the stages: they hold the waves' sums now

  // A wave's sums of one tile take 4 KB: row m, columns 4 c .. 4 c + 3 at chunk
  // c ^ (m / 2 % 8) (no bank conflicts). acc[j][r] is row col, column
  // 8 (r / 4) + 4 half + r % 4.
  auto sums = [&](int v, int j) { return (float*)(WT * v + j < 2 * (1 + WT) ? s0 : s1) + 1024 * ((WT * v + j) % (2 * (1 + WT))); };
#pragma unroll
  for (int j = 0; j < WT; ++j) {
    float* const f = sums(wave, j) + 32 * col;
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(f + 4 * ((2 * g + half) ^ (col >> 1 & 7))) =
          f32x4{acc[j][4 * g], acc[j][4 * g + 1], acc[j][4 * g + 2], acc[j][4 * g + 3]};
  }
  lds_barrier();
  // the product's row r, columns 4 c .. 4 c + 3 of tile j
  auto product = [&](int j, int r, int c) {
    const int at = 32 * r + 4 * (c ^ (r >> 1 & 7));
    f32x4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = *reinterpret_cast<const f32x4*>(sums(k, j) + at);
    return (v[0] + v[1]) + (v[2] + v[3]);
  };
  bf16* const orow = (bf16*)a.out + m0 * a.out_features + n0;
  if constexpr (!kQuery) {
    const int r = threadIdx.x >> 3, c = threadIdx.x & 7;
    if (r >= mrows || n0 + 4 * c >= a.out_features) return;
    f32x4 y = product(0, r, c);
    if constexpr (kGated) {
      const f32x4 up = product(1, r, c);
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = gated(y[e], up[e]);
    }
    *reinterpret_cast<u32x2*>(orow + (int64_t)r * a.out_features + 4 * c) = u32x2{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
  } else {
    query_rows<BN, BM>(a, m0, n0, mrows, [&](int r, int d0, float (&q)[8]) {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const f32x4 v = product(d0 >> 5, r, (d0 >> 2 & 7) + e);
        q[4 * e] = v[0], q[4 * e + 1] = v[1], q[4 * e + 2] = v[2], q[4 * e + 3] = v[3];
      }
    });
  }
#endif
}

// The pool's channel projections, out[c] = x[c] W[c] with W (in, out) rows, both
// sides of every channel in one launch: 64 rows by 128 columns. A stage's weight
// rows are the contraction, read transposed from LDS (ds_read_b64_tr_b16); the
// rows' operand is read in the same order of k. The two batched library products
// take 36 us of host time, this launch 6. GPU time, before and here, in us, of
// both sides: four channels of 512 -> 256, 16 rows 17.4 and 5.9, 1,024 rows 14.6
// and 7.0; eight of 1024 -> 512, 16 rows 10.0 and 8.9, 512 rows 23.0 and 21.4.
__global__ __launch_bounds__(256, 1) void pool_project_kernel(const wmx_pool_project_args a) {
#ifdef __HIP_DEVICE_COMPILE__
  constexpr int BM = kTileRows, BN = kRowElems, NS = 3, kStage = 3 * kTileElems;
  __shared__ __attribute__((aligned(1024))) bf16 s0[kStage];
  __shared__ __attribute__((aligned(1024))) bf16 s1[kStage];
  __shared__ __attribute__((aligned(1024))) bf16 s2[kStage];
  int64_t m0;
  int n0;
  if (!decode_tile(a.rows, a.out_features, BM, BN, m0, n0)) return;
  const int side = blockIdx.y & 1;
  const int64_t ch = blockIdx.y >> 1;
  const int K = a.in_features, N = a.out_features;
  const bf16* const weight = (const bf16*)(side ? a.weight_v : a.weight_k) + ch * K * N + n0;
  bf16* const orow = (bf16*)(side ? a.out_v : a.out_k) + (ch * a.rows + m0) * N + n0;
  const int mrows = (int)min((int64_t)BM, a.rows - m0), cols = min(BN, N - n0);
  const int lane = threadIdx.x & 63, wave = wave_id(), half = lane >> 5, col = lane & 31;
  const int wm = wave & 1, wn = wave >> 1;

  using Tile = Operand<BM>;
  typename Tile::DMA dma;
  dma.init(wave, lane);
  Tile x;
  x.init(dma, (const bf16*)(side ? a.x_v : a.x_k) + ch * a.rows * K, m0, K, a.rows, K);
  unsigned woff[Tile::DMA::kInstr];
  dma.strided_offsets(N * 2, woff);
#pragma unroll
  for (int r = 0; r < Tile::DMA::kInstr; ++r) woff[r] = dma.chunk16(r) < 2 * cols ? woff[r] : kOutOfRange;
  auto issue = [&](int kt, bf16* st) __attribute__((always_inline)) {
    x.issue(dma, kt, st);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int k0 = kt * kStep + 64 * j, left = min(64, K - k0);
      dma.issue_strided(make_rsrc(weight + (left > 0 ? (int64_t)k0 * N : 0), left > 0 ? ((left - 1) * N + cols) * 2 : 0),
                        st + (1 + j) * kTileElems, woff);
    }
  };
  TrReads<2> wr;
  wr.init(lane, 64 * wn);
  const int swz = tile_swz(col);
  f32x16 acc[2] = {f32x16{}, f32x16{}};
  issue(0, s0);
  issue(1, s1);
  for_stages<NS>((K + kStep - 1) / kStep, [&](auto bufc, int it) __attribute__((always_inline)) {
    constexpr int B = decltype(bufc)::value, BX = (B + NS - 1) % NS;
    lds_sync<(NS - 2) * 3 * Tile::DMA::kInstr>();
    issue(it + NS - 1, BX == 0 ? s0 : BX == 1 ? s1 : s2);
    const bf16* const st = B == 0 ? s0 : B == 1 ? s1 : s2;
    const bf16* const xr = st + (32 * wm + col) * kRowElems + 4 * half;
    wr.refresh();
    constexpr int KS = kStep / 16, PF = 3;
    bf16x8 xo[KS], wo[KS][2];
    auto fetch = [&](int s) __attribute__((always_inline)) {
      // k of element e: 16 s + 8 (e / 4) + 4 half + e % 4, as the transposed reads'
      const u32x2 lo = *reinterpret_cast<const u32x2*>(xr + 8 * ((2 * s) ^ swz));
      const u32x2 hi = *reinterpret_cast<const u32x2*>(xr + 8 * ((2 * s + 1) ^ swz));
      xo[s] = as_bf16x8(u32x4{lo[0], lo[1], hi[0], hi[1]});
#pragma unroll
      for (int d = 0; d < 2; ++d) wo[s][d] = wr.get(st + (1 + s / 4) * kTileElems, d, s % 4);
    };
#pragma unroll
    for (int s = 0; s < PF; ++s) fetch(s);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      __builtin_amdgcn_sched_barrier(0);
      if (s + PF < KS) fetch(s + PF);
#pragma unroll
      for (int d = 0; d < 2; ++d) acc[d] = mfma32(wo[s][d], xo[s], acc[d]);
    }
    __builtin_amdgcn_sched_barrier(0);
  });
  dma_barrier();  // every wave is done with the stages: the tile's rows are laid out in the first

  // acc[d][r] is row 32 wm + col, column 64 wn + 32 d + 8 (r / 4) + 4 half + r % 4
  constexpr int P = BN + 8;  // pitch
  bf16* const mine = s0 + (32 * wm + col) * P + 64 * wn + 4 * half;
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<u32x2*>(mine + 32 * d + 8 * g) =
          u32x2{pack_bf16x2(acc[d][4 * g], acc[d][4 * g + 1]), pack_bf16x2(acc[d][4 * g + 2], acc[d][4 * g + 3])};
  lds_barrier();
#pragma unroll
  for (int i = threadIdx.x; i < BM * 16; i += 256) {
    const int r = i >> 4, c = 8 * (i & 15);
    if (r < mrows && c < cols) *reinterpret_cast<u32x4*>(orow + (int64_t)r * N + c) = *reinterpret_cast<const u32x4*>(s0 + r * P + c);
  }
#endif
}

int64_t grid_of(int64_t rows, int64_t cols) { return (rows * cols + kXcds - 1) / kXcds * kXcds; }

template <int WT, int NS>
int run(const wmx_linear_args& a, hipStream_t stream) {
  const int64_t grid = grid_of((a.rows + 63) / 64, (a.out_features + 63) / 64);
  if (grid > INT32_MAX) return WMX_E_UNSUPPORTED;
  hipLaunchKernelGGL((linear_kernel<WT, NS>), dim3((unsigned)grid), dim3(256), 0, stream, a);
  return WMX_OK;
}

template <int KIND, int WT, int NS>
int run_small(const wmx_linear_args& a, hipStream_t stream) {
  constexpr int BN = KIND == WMX_LINEAR_GATED ? 32 : 32 * WT;
  const int64_t grid = grid_of((a.rows + 31) / 32, (a.out_features + BN - 1) / BN);
  if (grid > INT32_MAX) return WMX_E_UNSUPPORTED;
  hipLaunchKernelGGL((linear_small_kernel<KIND, WT, NS>), dim3((unsigned)grid), dim3(256), 0, stream, a);
  return WMX_OK;
}

}  // namespace

// Up to this many 64 x 64 tiles the 32-row kernel is the faster one (us, 32-row
// and 64-row; features in -> out): plain 128 x 3072 -> 1024 (32 tiles) 6.7 and
// 12.3, 1024 x 1536 -> 512 (128 tiles) 7.1 and 7.9, 1024 x 1024 -> 1024 (256
// tiles) 9.1 and 6.4; gated 256 x 512 -> 1536 (96 tiles) 5.5 and 6.4, 512 rows
// (192 tiles) 7.9 and 6.7.
constexpr int64_t kFewTiles = 128;

int launch_linear(const wmx_linear_args& a, hipStream_t stream) {
  if (a.kind == WMX_LINEAR_QUERY) {
    // (32 rows throughout: 64-row tiles took 5.9 and 34.4 us where these take
    // 4.7 and 32.0, at 512 x 512 and 4096 x 1024)
    switch (a.head_dim) {
      case 64: return run_small<WMX_LINEAR_QUERY, 2, 3>(a, stream);
      case 96: return run_small<WMX_LINEAR_QUERY, 3, 3>(a, stream);
      case 128: return run_small<WMX_LINEAR_QUERY, 4, 3>(a, stream);
      default: return WMX_E_UNSUPPORTED;
    }
  }
  const bool few = (a.rows + 63) / 64 * ((a.out_features + 63) / 64) <= kFewTiles;
  if (a.kind == WMX_LINEAR_GATED) return few ? run_small<WMX_LINEAR_GATED, 2, 3>(a, stream) : run<2, 3>(a, stream);
  return few ? run_small<WMX_LINEAR_PLAIN, 1, 4>(a, stream) : run<1, 4>(a, stream);
}

int launch_pool_project(const wmx_pool_project_args& a, hipStream_t stream) {
  const int64_t grid = grid_of((a.rows + 63) / 64, (a.out_features + kRowElems - 1) / kRowElems);
  if (grid > INT32_MAX) return WMX_E_UNSUPPORTED;
  hipLaunchKernelGGL(pool_project_kernel, dim3((unsigned)grid, 2 * a.channels), dim3(256), 0, stream, a);
  return WMX_OK;
}

}  // namespace wmx
