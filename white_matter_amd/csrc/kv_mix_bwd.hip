// Backward of the KV-pool producer (wmx_kv_mix_bwd_args): the gradients of
// the sources, pre-mix weights, router weights and biases, and gains, from the
// gradients of the mixtures. With, per token n and side,
//   p = bf16(x * inv * pre), z = p[read sources] . W^T + b, m = bf16(sum z p),
//   h = bf16(m * minv * gain)
// the steps are
//   mix     - per token and side: m again from p and the logits, the norm's
//             backward dm (bf16, as autograd's through the bf16 mixture), the
//             gain's gradient, and dz = dm . p^T on the MFMA units (bf16);
//   context - dctx = dz . W, an MFMA GEMM of few inputs (the logits);
//   sources - per token and source: dp = sum over channels of z dm, plus dctx
//             on the sources that the router reads; the pre-mix gradient, and
//             the source norm's backward;
//   weight  - dW = dz^T . p over the tokens, p read in place;
//   reduce  - the sums over tokens of the small gradients, in a fixed order.
// All of them stream: the sources are read once, p once by mix and its read
// half once by weight, dm once per group of sources. As torch operations on the
// recomputed steps the backward took 134 launches, most over every source in
// fp32. 1,024 tokens, 25 sources of 1,024, 8 channels, both sides: 2.8 ms as
// torch operations, 0.31 ms here (see launch_kv_mix_bwd).
#include "lds_tiles.h"
#include "wmx_kernels.h"

namespace wmx {

namespace {

constexpr int kMixRows = 4;      // tokens per mix workgroup (each leaves one partial gain gradient)
constexpr int kSourceRows = 16;  // most tokens per sources workgroup (each leaves one partial pre-mix gradient)
constexpr int kGroup = 2;        // sources per sources workgroup
constexpr int kContextRows = 128;
constexpr int kMaxLogits = WMX_KV_ROUTER_MAX_LOGITS;

__host__ __device__ inline int64_t pad(int64_t x, int64_t to) { return (x + to - 1) / to * to; }

struct BwdLayout {
  int64_t rows, logits, kp, inputs;
  int64_t mix_blocks, groups, source_rows, source_blocks;
  int64_t dm, dz, dctx, gain_parts, pre_parts, bytes;  // byte offsets
  __host__ __device__ explicit BwdLayout(const wmx_kv_mix_bwd_args& a) {
    rows = (int64_t)a.batch * a.tokens;
    logits = (int64_t)a.channels * a.num_sources;
    kp = pad(logits, 16);  // dz row: whole MFMA k-steps, zeros past the logits
    inputs = (int64_t)a.read_sources * a.hidden;
    mix_blocks = pad(rows, kMixRows) / kMixRows;
    // sources workgroups: one (token block, source group) each; blocks of 4 to
    // 16 tokens, as long as about 2,048 workgroups remain (few tokens leave more
    // partial sums, many leave the last round of workgroups half empty)
    groups = (a.num_sources + kGroup - 1) / kGroup;
    const int64_t fill = (rows * groups + 2047) / 2048;
    source_rows = fill < 4 ? 4 : fill > kSourceRows ? kSourceRows : fill;
    source_blocks = (rows + source_rows - 1) / source_rows;
    dm = 0;                                                                   // bf16 [side][row][channel][hidden]
    dz = pad(dm + 2 * rows * a.channels * a.hidden * 2, 256);                 // bf16 [side][row][kp]
    dctx = pad(dz + 2 * rows * kp * 2, 256);                                  // bf16 [side][row][inputs]
    gain_parts = pad(dctx + 2 * rows * inputs * 2, 256);                      // fp32 [mix block][side][channel][hidden]
    pre_parts = pad(gain_parts + mix_blocks * 2 * a.channels * a.hidden * 4, 256);  // fp32 [source block][side][source][hidden]
    bytes = pad(pre_parts + source_blocks * 2 * a.num_sources * a.hidden * 4, 256);
  }
};

__device__ __forceinline__ void unpack4(const u32x2& w, float (&v)[4]) {
  v[0] = bf16_lo(w[0]);
  v[1] = bf16_hi(w[0]);
  v[2] = bf16_lo(w[1]);
  v[3] = bf16_hi(w[1]);
}
__device__ __forceinline__ u32x2 pack4(const float (&v)[4]) { return u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])}; }
__device__ __forceinline__ u32x2 load8b(const bf16* p) { return *reinterpret_cast<const u32x2*>(p); }

// Four consecutive elements as fp32 from an fp32 or bf16 array.
__device__ __forceinline__ void load4(const void* base, int64_t off, bool bf16_src, float (&v)[4]) {
  if (bf16_src) {
    unpack4(load8b((const bf16*)base + off), v);
  } else {
    const f32x4 x = *reinterpret_cast<const f32x4*>((const float*)base + off);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = x[e];
  }
}

// The sums over the wave of N values per lane (N a power of two up to 64):
// each step hands half of the values to the partner lane and keeps the sum of
// the other half, N - 1 exchanges instead of 6 N; then lanes that hold the same
// value add up. Returns value (lane / (64 / N)) to its 64 / N lanes.
template <int N>
__device__ __forceinline__ float wave_sums(float (&v)[N], int lane) {
  int o = 32;
#pragma unroll
  for (int n = N / 2; n >= 1; n >>= 1, o >>= 1) {
    const bool upper = lane & o;
#pragma unroll
    for (int i = 0; i < n; ++i) {
      const float send = upper ? v[i] : v[i + n];
      v[i] = (upper ? v[i + n] : v[i]) + __shfl_xor(send, o);
    }
  }
  float x = v[0];
#pragma unroll
  for (; o > 0; o >>= 1) x += __shfl_xor(x, o);
  return x;
}

// EPT consecutive elements of a bf16 row, as words and as fp32.
constexpr int EPT = 4;
__device__ __forceinline__ void unpack(const uint32_t (&w)[EPT / 2], float (&v)[EPT]) {
#pragma unroll
  for (int i = 0; i < EPT / 2; ++i) {
    v[2 * i] = bf16_lo(w[i]);
    v[2 * i + 1] = bf16_hi(w[i]);
  }
}
__device__ __forceinline__ void load_words(const bf16* p, uint32_t (&w)[EPT / 2]) {
  const u32x2 x = load8b(p);
  w[0] = x[0];
  w[1] = x[1];
}

// mix: workgroup (kMixRows tokens, side) of NT threads; thread t holds elements
// EPT t + [0, EPT) of a row (hidden <= NT EPT) for up to CM channels. What bounds
// it is latency: a token is a chain of loads, two reductions and a product,
// hence eight source rows in flight at a time (four: 132 us against 92) and
// barriers that wait for LDS only, not for the stores. Eight waves of half the
// elements measured 118 us, three workgroups per CU in fewer registers 143 (spills). dm of a token is staged in LDS as the A operand (16 channel
// rows) of dz = dm . p^T, 16x16x32 MFMA blocks of 16 sources whose k-steps are
// dealt over the waves; B operands come from the token's p rows, which the
// first half has just read (64 consecutive bytes per row and k-step).
template <int NT, int CM>
__global__ __launch_bounds__(NT, NT == 256 && CM == 8 ? 2 : NT / 256) void mix_bwd_kernel(const wmx_kv_mix_bwd_args a) {
  constexpr int NW = NT / 64;
  constexpr int LDK = NT * EPT + 8;
  constexpr int SB = 4;  // source blocks summed over the waves together
  constexpr int kBatch = 8;
  __shared__ __attribute__((aligned(16))) bf16 dm_lds[16 * LDK];
  __shared__ __attribute__((aligned(16))) float z_lds[(kMaxLogits + 16) * CM];  // [source][channel]
  __shared__ __attribute__((aligned(16))) float red[2 * CM][NW];
  __shared__ float part[NW][SB][256];
  const BwdLayout L(a);
  const int side = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int H = a.hidden, S = a.num_sources, C = a.channels;
  char* ws = (char*)a.workspace;
  bf16* dm_out = (bf16*)(ws + L.dm) + side * L.rows * C * H;
  bf16* dz_out = (bf16*)(ws + L.dz) + side * L.rows * L.kp;
  const int64_t r0 = (int64_t)blockIdx.x * kMixRows, r1 = min(r0 + kMixRows, L.rows);
  for (int i = tid; i < 16 * LDK / 8; i += NT) reinterpret_cast<u32x4*>(dm_lds)[i] = u32x4{0u, 0u, 0u, 0u};
  // channels past the last repeat it and elements past the row read its end:
  // loads need no predicate; `in` zeroes what the sums take
  const bool in = EPT * tid < H;
  const unsigned d = (unsigned)(in ? EPT * tid : H - EPT);  // unsigned: uniform base + 32-bit lane offset
  float gain[CM][EPT], dgain[CM][EPT];
#pragma unroll
  for (int c = 0; c < CM; ++c) {
    const int64_t at = (int64_t)min(c, C - 1) * H;
    if (a.weight_dtype == WMX_DTYPE_BF16) {
      uint32_t w[EPT / 2];
      load_words(((const bf16*)a.gain[side] + at) + d, w);
      unpack(w, gain[c]);
    } else {
#pragma unroll
      for (int e = 0; e < EPT; ++e) gain[c][e] = (((const float*)a.gain[side]) + at)[d + e];
    }
#pragma unroll
    for (int e = 0; e < EPT; ++e) dgain[c][e] = 0.f;
  }
  const float rh = 1.f / (float)H;
  // kBatch source rows in flight while the batch before is summed
  uint32_t pw[kBatch][EPT / 2];
  auto load_rows = [&](const bf16* p, int s0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kBatch; ++u) load_words((p + (int64_t)min(s0 + u, S - 1) * H) + d, pw[u]);
  };
#pragma unroll 1
  for (int64_t r = r0; r < r1; ++r) {
    const bf16* p = (const bf16*)a.premixed[side] + r * S * H;
    const bf16* z = (const bf16*)a.alpha[side] + r * a.alpha_stride;
    // (sources past the last have zero logits)
    for (int i = tid; i < (S + kBatch) * CM; i += NT) {
      const int s = i / CM, c = i % CM;
      z_lds[i] = c < C && s < S ? (float)z[c * S + s] : 0.f;
    }
    uint32_t g[CM][EPT / 2];
    const bf16* grow = (const bf16*)a.grad[side] + r * H;
    const int64_t gstep = L.rows * H;
#pragma unroll
    for (int c = 0; c < CM; ++c) {
      load_words((grow + min(c, C - 1) * gstep) + d, g[c]);
#pragma unroll
      for (int i = 0; i < EPT / 2; ++i) g[c][i] = in ? g[c][i] : 0u;
    }
    load_rows(p, 0);
    lds_barrier();  // the logits; the previous token's operands and sums are read
    float m[CM][EPT];
#pragma unroll
    for (int c = 0; c < CM; ++c)
#pragma unroll
      for (int e = 0; e < EPT; ++e) m[c][e] = 0.f;
#pragma unroll 1
    for (int s0 = 0; s0 < S; s0 += kBatch) {
      uint32_t now[kBatch][EPT / 2];
#pragma unroll
      for (int u = 0; u < kBatch; ++u)
#pragma unroll
        for (int i = 0; i < EPT / 2; ++i) now[u][i] = pw[u][i];
      if (s0 + kBatch < S) load_rows(p, s0 + kBatch);
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        float pv[EPT];
        unpack(now[u], pv);
#pragma unroll
        for (int c0 = 0; c0 < CM; c0 += 4) {
          const f32x4 al = *reinterpret_cast<const f32x4*>(z_lds + (s0 + u) * CM + c0);
#pragma unroll
          for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int e = 0; e < EPT; ++e) m[c0 + c][e] = fmaf(al[c], pv[e], m[c0 + c][e]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    float sums[2 * CM];
#pragma unroll
    for (int c = 0; c < CM; ++c) {
      float ss = 0.f, um = 0.f, gv[EPT];
      __builtin_amdgcn_sched_barrier(0);
      unpack(g[c], gv);
#pragma unroll
      for (int e = 0; e < EPT; ++e) {
        m[c][e] = in ? round_bf16(m[c][e]) : 0.f;
        ss = fmaf(m[c][e], m[c][e], ss);
        um = fmaf(gv[e] * gain[c][e], m[c][e], um);
      }
      sums[2 * c] = ss;
      sums[2 * c + 1] = um;
    }
    const float sum = wave_sums<2 * CM>(sums, lane);
    if (lane % (32 / CM) == 0) red[lane / (32 / CM)][wave] = sum;
    lds_barrier();
#pragma unroll
    for (int c = 0; c < CM; ++c) {
      __builtin_amdgcn_sched_barrier(0);  // one channel's sums and rows at a time
      float ss = 0.f, um = 0.f, gv[EPT], dm[EPT];
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        ss += red[2 * c][w];
        um += red[2 * c + 1][w];
      }
      const float minv = 1.f / sqrtf(ss * rh + a.mix_eps);
      const float k = um * rh * minv * minv * minv;
      unpack(g[c], gv);
#pragma unroll
      for (int e = 0; e < EPT; ++e) {
        dgain[c][e] = fmaf(gv[e], m[c][e] * minv, dgain[c][e]);
        dm[e] = gv[e] * gain[c][e] * minv - m[c][e] * k;
      }
      if (c < C && in) {
#pragma unroll
        for (int e = 0; e < EPT; e += 2) {
          const uint32_t w = pack_bf16x2(dm[e], dm[e + 1]);
          *reinterpret_cast<uint32_t*>(dm_lds + c * LDK + d + e) = w;
          *reinterpret_cast<uint32_t*>((dm_out + (r * C + c) * H) + (d + e)) = w;
        }
      }
    }
    lds_barrier();  // the channel rows of dm
    const int row = lane & 15, k8 = 8 * (lane >> 4);
    for (int b0 = 0; b0 * 16 < S; b0 += SB) {
      // the group's source blocks share each A operand
      f32x4 acc[SB];
      const bf16* ps[SB];
#pragma unroll
      for (int sb = 0; sb < SB; ++sb) {
        acc[sb] = f32x4{0.f, 0.f, 0.f, 0.f};
        ps[sb] = p + (int64_t)min((b0 + sb) * 16 + row, S - 1) * H + k8;
      }
#pragma unroll 2
      for (int k0 = 32 * wave; k0 < H; k0 += 32 * NW) {
        const bf16x8 av = as_bf16x8(*reinterpret_cast<const u32x4*>(dm_lds + row * LDK + k0 + k8));
#pragma unroll
        for (int sb = 0; sb < SB; ++sb) {
          if (sb > 0 && (b0 + sb) * 16 >= S) continue;  // uniform
          const u32x4 bw = k0 + k8 < H ? load16(ps[sb] + k0) : u32x4{0u, 0u, 0u, 0u};
          acc[sb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, as_bf16x8(bw), acc[sb], 0, 0, 0);
        }
      }
#pragma unroll
      for (int sb = 0; sb < SB; ++sb)
#pragma unroll
        for (int i = 0; i < 4; ++i) part[wave][sb][(4 * (lane >> 4) + i) * 16 + row] = acc[sb][i];
      lds_barrier();
#pragma unroll
      for (int sb = tid >> 8; sb < SB; sb += NT / 256) {
        const int at = tid & 255, c = at >> 4, s = (b0 + sb) * 16 + (at & 15);
        if (c < C && s < S) {
          float x = 0.f;
#pragma unroll
          for (int w = 0; w < NW; ++w) x += part[w][sb][at];
          dz_out[r * L.kp + c * S + s] = (bf16)x;
        }
      }
      if ((b0 + SB) * 16 < S) lds_barrier();
    }
    if (tid < L.kp - L.logits) dz_out[r * L.kp + L.logits + tid] = (bf16)0.f;
  }
  float* out = (float*)(ws + L.gain_parts) + ((int64_t)blockIdx.x * 2 + side) * C * H;
#pragma unroll
  for (int c = 0; c < CM; ++c)
#pragma unroll
    for (int e = 0; e < EPT; ++e)
      if (c < C && in) (out + (int64_t)c * H)[d + e] = dgain[c][e];
}

// A 64-row x 128-column tile of a row-major bf16 matrix in the layout of
// lds_tiles.h: lane chunks of 8 columns from column n0 on, rows from row0 on;
// rows and columns outside the matrix read as zeros. `chunk_at` maps a chunk's
// first column to its element offset in a row (a chunk never straddles two
// sources: their width is a multiple of 8).
template <class ChunkAt>
__device__ __forceinline__ void issue_matrix_tile(const TileDMA<128, 4>& dma, const bf16* base, int64_t row_elems,
                                                  int64_t row0, int64_t rows, int n0, int columns, ChunkAt chunk_at,
                                                  bf16* tile) {
  const int nvalid = (int)min((int64_t)kTileRows, max((int64_t)0, rows - row0));
  // the buffer ends with the last valid row: later rows are out of range
  const rsrc_t rs = make_rsrc(base + row0 * row_elems, (int)(nvalid * row_elems * 2));
#pragma unroll
  for (int i = 0; i < TileDMA<128, 4>::kInstr; ++i) {
    const int col = n0 + dma.chunk16(i) / 2;
    const unsigned off = col < columns ? (unsigned)(dma.row(i) * (int)row_elems + chunk_at(col)) * 2u : kOutOfRange;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, dma.dst(tile, i), 16, off, 0, 0, 0);
  }
}

// context: dctx = dz . W for 128 columns and kContextRows tokens per step.
// The workgroup keeps its columns of W (up to four 64-row tiles) in LDS and
// walks the token blocks; waves own 32 tokens, whose dz rows are read straight
// from memory in the k order of the transposed W operand.
__global__ __launch_bounds__(256) void context_bwd_kernel(const wmx_kv_mix_bwd_args a) {
  __shared__ __attribute__((aligned(1024))) bf16 w_lds[kMaxLogits / kTileRows][kTileElems];
  const BwdLayout L(a);
  const int side = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int col = lane & 31, half = lane >> 5;
  const int n0 = blockIdx.x * 128;
  char* ws = (char*)a.workspace;
  const bf16* dz = (const bf16*)(ws + L.dz) + side * L.rows * L.kp;
  bf16* out = (bf16*)(ws + L.dctx) + side * L.rows * L.inputs;
  TileDMA<128, 4> dma;
  dma.init(wave, lane);
  const int tiles = (int)((L.logits + kTileRows - 1) / kTileRows);
  for (int t = 0; t < tiles; ++t)
    issue_matrix_tile(dma, (const bf16*)a.weight[side], L.inputs, t * kTileRows, L.logits, n0, (int)L.inputs,
                      [](int c) { return c; }, w_lds[t]);
  dma_barrier();
  TrReads<4> rd;
  rd.init(lane);
  const int steps = (int)(L.kp / 16);
  for (int64_t m0 = (int64_t)blockIdx.z * kContextRows; m0 < L.rows; m0 += (int64_t)gridDim.z * kContextRows) {
    const int64_t r = m0 + wave * 32 + col;
    const bf16* zr = dz + (r < L.rows ? r : L.rows - 1) * L.kp;
    f32x16 acc[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) acc[d] = f32x16{};
    for (int s = 0; s < steps; ++s) {
      const u32x2 lo = load8b(zr + 16 * s + 4 * half), hi = load8b(zr + 16 * s + 8 + 4 * half);
      const bf16x8 b = as_bf16x8(u32x4{lo[0], lo[1], hi[0], hi[1]});
#pragma unroll
      for (int d = 0; d < 4; ++d) acc[d] = mfma32(rd.get(w_lds[s >> 2], d, s & 3), b, acc[d]);
    }
    if (r < L.rows) {
      // both lanes of a pair hold the same token: whole blocks, then the tail by columns
      bf16* to = out + r * L.inputs + n0;
#pragma unroll
      for (int d = 0; d < 4; ++d) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int e = 8 * t;
          const u32x4 w = {pack_bf16x2(acc[d][e], acc[d][e + 1]), pack_bf16x2(acc[d][e + 2], acc[d][e + 3]),
                           pack_bf16x2(acc[d][e + 4], acc[d][e + 5]), pack_bf16x2(acc[d][e + 6], acc[d][e + 7])};
          const auto x = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
          const auto y = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
          const int n = d * 32 + 16 * t + 8 * half;
          if (n0 + n < L.inputs) *reinterpret_cast<u32x4*>(to + n) = u32x4{x[0], y[0], x[1], y[1]};
        }
      }
    }
  }
}

// sources: workgroup (a block of tokens, G sources), both sides; thread t
// holds elements 1024 v + 4 t + [0, 4). A token's channel rows dm are read once
// for G sources, from the L2 of the XCD that runs the block's groups one after
// another. Bound by latency too: with five sources per workgroup (fewer reads of
// dm, 253 registers) it took 146-159 us, with four 139, with two 83-88, with one
// 111-120; the barrier of a token waits for LDS only, so its stores fly on.
template <int VPT, int CM, bool SRC_BF16>
__global__ __launch_bounds__(256, VPT * CM <= 8 ? 2 : 1) void sources_bwd_kernel(const wmx_kv_mix_bwd_args a) {
  constexpr int G = kGroup, NS = 2 * G;
  static_assert(G == 2, "a channel's logits of the group are one vector read");
  __shared__ __attribute__((aligned(16))) float z_lds[kSourceRows][2][CM * G];
  __shared__ float red[2][4][NS];
  const BwdLayout L(a);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int H = a.hidden, S = a.num_sources, C = a.channels;
  // workgroups go to the XCDs round-robin: the source groups of a token block
  // follow each other on one XCD, whose L2 then holds the block's channel rows
  const int64_t slot = blockIdx.x >> 3;
  const int64_t block = slot / L.groups * 8 + (blockIdx.x & 7);
  if (block >= L.source_blocks) return;
  const int s0 = (int)(slot % L.groups) * G;
  const char* ws = (const char*)a.workspace;
  const bf16* dm = (const bf16*)(ws + L.dm);
  const bf16* dctx = (const bf16*)(ws + L.dctx);
  const int64_t r0 = block * L.source_rows;
  const int nrows = (int)min(L.source_rows, L.rows - r0);
  for (int i = tid; i < nrows * 2 * CM * G; i += 256) {
    const int g = i % G, c = i / G % CM, side = i / (G * CM) % 2, rr = i / (G * CM * 2);
    const bool in = s0 + g < S && c < C;
    z_lds[rr][side][c * G + g] = in ? (float)((const bf16*)a.alpha[side])[(r0 + rr) * a.alpha_stride + c * S + s0 + g] : 0.f;
  }
  // sources and channels past the last repeat it (with zero logits), elements
  // past the row read its end (with zero sources and weights)
  unsigned d[VPT];  // unsigned: uniform base + 32-bit lane offset
  int src_at[G];
  bool in[VPT];
#pragma unroll
  for (int v = 0; v < VPT; ++v) {
    in[v] = 1024 * v + 4 * tid < H;
    d[v] = (unsigned)(in[v] ? 1024 * v + 4 * tid : H - 4);
  }
  float pre[2][G][VPT][4], dpre[2][G][VPT][4];
  int read_at[G];  // place of the source among those that the router reads, or -1
#pragma unroll
  for (int g = 0; g < G; ++g) {
    src_at[g] = min(s0 + g, S - 1);
    const int rel = src_at[g] - a.read_start;
    const bool read = rel >= 0 && rel % a.read_stride == 0 && rel / a.read_stride < a.read_sources;
    read_at[g] = read ? rel / a.read_stride : -1;
#pragma unroll
    for (int side = 0; side < 2; ++side)
#pragma unroll
      for (int v = 0; v < VPT; ++v) {
        load4(a.pre_mix[side], (int64_t)src_at[g] * H + d[v], a.weight_dtype == WMX_DTYPE_BF16, pre[side][g][v]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          pre[side][g][v][e] = in[v] ? pre[side][g][v][e] : 0.f;
          dpre[side][g][v][e] = 0.f;
        }
      }
  }
  lds_barrier();
  const float rh = 1.f / (float)H;
  // a token's loads, all in flight together
  uint32_t xw[G][VPT][SRC_BF16 ? 2 : 4];
  u32x2 wr[2][CM][VPT], cx[2][G][VPT];
  auto load_token = [&](int rr) __attribute__((always_inline)) {
    const int64_t r = r0 + rr;
    const int64_t b = r / a.tokens, t = r - b * a.tokens;
    const int64_t src = b * a.source_stride[0] + t * a.source_stride[1];
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      const bf16* row = dm + (side * L.rows + r) * C * H;
#pragma unroll
      for (int c = 0; c < CM; ++c)
#pragma unroll
        for (int v = 0; v < VPT; ++v) wr[side][c][v] = load8b((row + min(c, C - 1) * H) + d[v]);
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int v = 0; v < VPT; ++v) {
          cx[side][g][v] = u32x2{0u, 0u};
          if (read_at[g] >= 0)
            cx[side][g][v] = load8b((dctx + (side * L.rows + r) * L.inputs + (int64_t)read_at[g] * H) + d[v]);
        }
    }
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int v = 0; v < VPT; ++v) {
        const int64_t at = src + src_at[g] * a.source_stride[2];
        if constexpr (SRC_BF16) {
          const u32x2 w = load8b(((const bf16*)a.sources + at) + d[v]);
          xw[g][v][0] = w[0];
          xw[g][v][1] = w[1];
        } else {
          const u32x4 w = *reinterpret_cast<const u32x4*>(((const float*)a.sources + at) + d[v]);
#pragma unroll
          for (int e = 0; e < 4; ++e) xw[g][v][e] = w[e];
        }
      }
  };
#pragma unroll 1
  for (int rr = 0; rr < nrows; ++rr) {
    const int64_t r = r0 + rr;
    load_token(rr);
    float x[G][VPT][4], dp[2][G][VPT][4];
#pragma unroll
    for (int side = 0; side < 2; ++side) {
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int v = 0; v < VPT; ++v) unpack4(cx[side][g][v], dp[side][g][v]);
#pragma unroll
      for (int c = 0; c < CM; ++c) {
        float z[G];
        const float2 w2 = *reinterpret_cast<const float2*>(&z_lds[rr][side][c * G]);
        z[0] = w2.x;
        z[1] = w2.y;
#pragma unroll
        for (int v = 0; v < VPT; ++v) {
          float w[4];
          unpack4(wr[side][c][v], w);
#pragma unroll
          for (int g = 0; g < G; ++g)
#pragma unroll
            for (int e = 0; e < 4; ++e) dp[side][g][v][e] = fmaf(z[g], w[e], dp[side][g][v][e]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int v = 0; v < VPT; ++v) {
        if constexpr (SRC_BF16) unpack4(u32x2{xw[g][v][0], xw[g][v][1]}, x[g][v]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (!SRC_BF16) x[g][v][e] = __uint_as_float(xw[g][v][e]);
          x[g][v][e] = in[v] ? x[g][v][e] : 0.f;
        }
      }
    // the norm's backward: dx = inv dy - x inv^3 mean(dy x), dy = sum of pre dp
    float sums[NS];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float ss = 0.f, yx = 0.f;
#pragma unroll
      for (int v = 0; v < VPT; ++v)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float dy = pre[0][g][v][e] * dp[0][g][v][e] + pre[1][g][v][e] * dp[1][g][v][e];
          ss = fmaf(x[g][v][e], x[g][v][e], ss);
          yx = fmaf(dy, x[g][v][e], yx);
        }
      sums[2 * g] = ss;
      sums[2 * g + 1] = yx;
    }
    const float sum = wave_sums<NS>(sums, lane);
    if (lane % (64 / NS) == 0) red[rr & 1][wave][lane / (64 / NS)] = sum;
    lds_barrier();  // (the other buffer is read again two tokens on, past the next barrier)
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const float(&s)[4][NS] = red[rr & 1];
      const float ss = s[0][2 * g] + s[1][2 * g] + s[2][2 * g] + s[3][2 * g];
      const float yx = s[0][2 * g + 1] + s[1][2 * g + 1] + s[2][2 * g + 1] + s[3][2 * g + 1];
      const float inv = 1.f / sqrtf(ss * rh + a.eps);
      const float k = yx * rh * inv * inv * inv;
#pragma unroll
      for (int v = 0; v < VPT; ++v) {
        float dx[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float y = x[g][v][e] * inv;
          dpre[0][g][v][e] = fmaf(dp[0][g][v][e], y, dpre[0][g][v][e]);
          dpre[1][g][v][e] = fmaf(dp[1][g][v][e], y, dpre[1][g][v][e]);
          const float dy = pre[0][g][v][e] * dp[0][g][v][e] + pre[1][g][v][e] * dp[1][g][v][e];
          dx[e] = dy * inv - x[g][v][e] * k;
        }
        if (s0 + g < S && in[v]) {
          const int64_t to = (r * S + s0 + g) * H;
          if constexpr (SRC_BF16) *reinterpret_cast<u32x2*>(((bf16*)a.grad_sources + to) + d[v]) = pack4(dx);
          else *reinterpret_cast<f32x4*>(((float*)a.grad_sources + to) + d[v]) = f32x4{dx[0], dx[1], dx[2], dx[3]};
        }
      }
    }
  }
  float* out = (float*)((char*)a.workspace + L.pre_parts) + block * 2 * S * H;
#pragma unroll
  for (int side = 0; side < 2; ++side)
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int v = 0; v < VPT; ++v)
        if (s0 + g < S && in[v])
          *reinterpret_cast<f32x4*>(out + ((int64_t)side * S + s0 + g) * H + d[v]) =
              f32x4{dpre[side][g][v][0], dpre[side][g][v][1], dpre[side][g][v][2], dpre[side][g][v][3]};
}

// weight: dW = dz^T . p for 128 columns of the router's view, all logits, one
// workgroup over every token: tiles of 64 tokens of p (its columns in place) and of dz, both
// read transposed; wave w owns columns 32 w .. 32 w + 31. Two buffers, the next
// tiles stream in during the products.
template <int NB>
__global__ __launch_bounds__(256) void weight_bwd_kernel(const wmx_kv_mix_bwd_args a) {
  constexpr int ZT = (NB + 3) / 4;  // 128-column tiles of dz
  // one array per buffer: the compiler then sees that a prefetch into one
  // buffer never aliases reads of the other
  __shared__ __attribute__((aligned(1024))) bf16 p_lds0[kTileElems];
  __shared__ __attribute__((aligned(1024))) bf16 p_lds1[kTileElems];
  __shared__ __attribute__((aligned(1024))) bf16 z_lds0[ZT * kTileElems];
  __shared__ __attribute__((aligned(1024))) bf16 z_lds1[ZT * kTileElems];
  const BwdLayout L(a);
  const int side = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int col = lane & 31, half = lane >> 5;
  const int n0 = blockIdx.x * 128;
  const bf16* dz = (const bf16*)((const char*)a.workspace + L.dz) + side * L.rows * L.kp;
  const bf16* p = (const bf16*)a.premixed[side];
  const int64_t row_elems = (int64_t)a.num_sources * a.hidden;
  const int H = a.hidden, start = a.read_start, stride = a.read_stride;
  auto place = [&](int c) {
    const int source = c / H;
    return (start + stride * source) * H + (c - source * H);
  };
  TileDMA<128, 4> dma;
  dma.init(wave, lane);
  auto issue = [&](int64_t r, bf16* pt, bf16* zt) {
    issue_matrix_tile(dma, p, row_elems, r, L.rows, n0, (int)L.inputs, place, pt);
#pragma unroll
    for (int t = 0; t < ZT; ++t)
      issue_matrix_tile(dma, dz, L.kp, r, L.rows, t * 128, (int)L.kp, [](int c) { return c; }, zt + t * kTileElems);
  };
  TrReads<1> prd;
  prd.init(lane, 32 * wave);
  TrReads<4> zrd;
  zrd.init(lane);
  f32x16 acc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) acc[nb] = f32x16{};
  auto step = [&](int64_t r, const bf16* pt, const bf16* zt, bf16* pnext, bf16* znext) __attribute__((always_inline)) {
    dma_barrier();
    if (r + kTileRows < L.rows) issue(r + kTileRows, pnext, znext);
#pragma unroll
    for (int s = 0; s < kTileRows / 16; ++s) {
      const bf16x8 b = prd.get(pt, 0, s);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) acc[nb] = mfma32(zrd.get(zt + (nb >> 2) * kTileElems, nb & 3, s), b, acc[nb]);
    }
  };
  issue(0, p_lds0, z_lds0);
  for (int64_t r = 0; r < L.rows; r += 2 * kTileRows) {
    step(r, p_lds0, z_lds0, p_lds1, z_lds1);
    if (r + kTileRows < L.rows) step(r + kTileRows, p_lds1, z_lds1, p_lds0, z_lds0);
  }
  const int n = n0 + 32 * wave + col;
  if (n >= L.inputs) return;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int l = nb * 32 + 8 * (i >> 2) + 4 * half + (i & 3);
      if (l >= L.logits) continue;
      if (a.grad_weight_dtype == WMX_DTYPE_BF16) ((bf16*)a.grad_weight[side])[l * L.inputs + n] = (bf16)acc[nb][i];
      else ((float*)a.grad_weight[side])[l * L.inputs + n] = acc[nb][i];
    }
}

// reduce: 64 columns of one sum per workgroup, 16 phases of its terms: the
// pre-mix gradients' and the gains' partials, and the biases' dz rows.
__global__ __launch_bounds__(1024) void reduce_bwd_kernel(const wmx_kv_mix_bwd_args a, int pre_blocks, int gain_blocks) {
  __shared__ float sums[16][64];
  const BwdLayout L(a);
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  const char* ws = (const char*)a.workspace;
  int64_t width;
  float acc = 0.f;
  int64_t e, at;
  void* out;
  int dtype = a.weight_dtype;
  if ((int)blockIdx.x < pre_blocks + gain_blocks) {
    const bool is_pre = (int)blockIdx.x < pre_blocks;
    const int64_t one = (int64_t)(is_pre ? a.num_sources : a.channels) * a.hidden;
    const int64_t count = is_pre ? L.source_blocks : L.mix_blocks;
    const float* parts = (const float*)(ws + (is_pre ? L.pre_parts : L.gain_parts));
    width = 2 * one;
    e = (int64_t)(is_pre ? blockIdx.x : blockIdx.x - pre_blocks) * 64 + tx;
    if (e < width)
#pragma unroll 4
      for (int64_t k = ty; k < count; k += 16) acc += parts[k * width + e];
    out = (is_pre ? a.grad_pre_mix : a.grad_gain)[e >= one];
    at = e >= one ? e - one : e;
  } else {
    width = 2 * L.logits;
    e = (int64_t)(blockIdx.x - pre_blocks - gain_blocks) * 64 + tx;
    const int side = e >= L.logits;
    const int64_t l = side ? e - L.logits : e;
    const bf16* dz = (const bf16*)(ws + L.dz) + side * L.rows * L.kp + l;
    if (e < width)
#pragma unroll 8
      for (int64_t r = ty; r < L.rows; r += 16) acc += (float)dz[r * L.kp];
    out = a.grad_bias[side];
    at = l;
    dtype = a.grad_weight_dtype;
  }
  sums[ty][tx] = acc;
  __syncthreads();
  if (ty == 0 && e < width) {
    float total = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) total += sums[k][tx];
    if (dtype == WMX_DTYPE_BF16) ((bf16*)out)[at] = (bf16)total;
    else ((float*)out)[at] = total;
  }
}

template <int NT, int CM>
void launch_mix(const wmx_kv_mix_bwd_args& a, const BwdLayout& L, hipStream_t stream) {
  hipLaunchKernelGGL((mix_bwd_kernel<NT, CM>), dim3((unsigned)L.mix_blocks, 2), dim3(NT), 0, stream, a);
}

template <int VPT, int CM>
void launch_sources(const wmx_kv_mix_bwd_args& a, const BwdLayout& L, hipStream_t stream) {
  const dim3 grid((unsigned)((L.source_blocks + 7) / 8 * 8 * L.groups));
  if (a.source_dtype == WMX_DTYPE_BF16) hipLaunchKernelGGL((sources_bwd_kernel<VPT, CM, true>), grid, dim3(256), 0, stream, a);
  else hipLaunchKernelGGL((sources_bwd_kernel<VPT, CM, false>), grid, dim3(256), 0, stream, a);
}

template <int NB>
void launch_weight(const wmx_kv_mix_bwd_args& a, const BwdLayout& L, hipStream_t stream) {
  hipLaunchKernelGGL((weight_bwd_kernel<NB>), dim3((unsigned)((L.inputs + 127) / 128), 2), dim3(256), 0, stream, a);
}

}  // namespace

int64_t kv_mix_bwd_workspace_size(const wmx_kv_mix_bwd_args& a) { return BwdLayout(a).bytes; }

// Measured at 1,024 tokens, 25 sources of 1,024, 8 channels: mix 92 us, context
// 37, sources 83-88, weight 38, reduce 17-19 us, after 38 us for the premixed rows
// again; forward and backward with the key transform 3.0 ms -> 0.57-0.66 ms.
int launch_kv_mix_bwd(const wmx_kv_mix_bwd_args& a, hipStream_t stream) {
  const BwdLayout L(a);
  if (L.mix_blocks > INT32_MAX) return WMX_E_UNSUPPORTED;
  const bool wide = a.hidden > 1024;
  if (a.channels <= 8) wide ? launch_mix<512, 8>(a, L, stream) : launch_mix<256, 8>(a, L, stream);
  else wide ? launch_mix<512, 16>(a, L, stream) : launch_mix<256, 16>(a, L, stream);
  const unsigned columns = (unsigned)((L.inputs + 127) / 128);
  // enough workgroups for every CU (W's columns are read again by each)
  const unsigned blocks = (unsigned)((L.rows + kContextRows - 1) / kContextRows);
  const unsigned want = (1024 + 2 * columns - 1) / (2 * columns);
  hipLaunchKernelGGL(context_bwd_kernel, dim3(columns, 2, want < blocks ? want : blocks), dim3(256), 0, stream, a);
  if (a.channels <= 8) wide ? launch_sources<2, 8>(a, L, stream) : launch_sources<1, 8>(a, L, stream);
  else wide ? launch_sources<2, 16>(a, L, stream) : launch_sources<1, 16>(a, L, stream);
  switch ((L.logits + 31) / 32) {
    case 1: launch_weight<1>(a, L, stream); break;
    case 2: launch_weight<2>(a, L, stream); break;
    case 3: launch_weight<3>(a, L, stream); break;
    case 4: launch_weight<4>(a, L, stream); break;
    case 5: launch_weight<5>(a, L, stream); break;
    case 6: launch_weight<6>(a, L, stream); break;
    case 7: launch_weight<7>(a, L, stream); break;
    default: launch_weight<8>(a, L, stream); break;
  }
  const int pre_blocks = (int)((2 * (int64_t)a.num_sources * a.hidden + 63) / 64);
  const int gain_blocks = (int)((2 * (int64_t)a.channels * a.hidden + 63) / 64);
  const int bias_blocks = (int)((2 * L.logits + 63) / 64);
  hipLaunchKernelGGL(reduce_bwd_kernel, dim3((unsigned)(pre_blocks + gain_blocks + bias_blocks)), dim3(1024), 0, stream, a,
                     pre_blocks, gain_blocks);
  return WMX_OK;
}

}  // namespace wmx
