// Plans of packed attention calls on the device: the kernel form of cyclic
// document metadata, and the covering schedule, work lists and dS layout of a
// packed schedule (wmx_plan_args). The same plans as the host's
// _build_packed_schedule / _covering_schedule, _work_units, _fused_units and
// _segment_fields, entry for entry.
//
// A step of training or a prefill has new documents, so its plans are built
// once per step and residue. As torch operations with host lists a plan took
// 2.7 ms (packed, 249 launches and 64 copies) to 3.4 ms (a cyclic residue, 334
// and 66), with Python loops over the segments, beside 0.1 ms of attention that
// it serves; here (0.12 and 0.13 ms) it is a count
// pass, one read of the counts by the host, which sizes the outputs, and
// three kernels:
//   count - one workgroup per batch row: scans over its queries and keys find
//           the segments, the runs that no segment holds and the number of
//           work units (packed schedules: one workgroup per segment marks its
//           rows first);
//   fill  - the covering schedule's indices and bounds, at offsets from the
//           counts of the rows before;
//   units - one workgroup: a scan over the segments gives dS offsets, each
//           segment's fields and one 64-bit sort key per work unit;
//   rank  - each unit's place is the number of larger keys of its list
//           (counted against all of them from LDS), where its entry goes.
// All of it is integer work on a few KB per row, bound by the latency of the
// scans and of the launches (measured at launch_plan_fill).
#include "wmx_kernels.h"

namespace wmx {

namespace {

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / 64;
constexpr int kTile = 128;  // query rows (and dS padding) of a work unit
constexpr int kStep = 64;   // rows of the tiles that the kernels' loops step over

__host__ __device__ constexpr int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Inclusive sum over the workgroup's 1024 threads in thread order; `total`
// receives the sum over all of them. Every thread must call it.
__device__ int64_t block_scan(int64_t x, int64_t& total, int64_t* sh) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int64_t y = __shfl_up(x, o);
    if (lane >= o) x += y;
  }
  if (lane == 63) sh[w] = x;
  __syncthreads();
  int64_t before = 0, all = 0;
#pragma unroll
  for (int i = 0; i < kWaves; ++i) {
    if (i < w) before += sh[i];
    all += sh[i];
  }
  __syncthreads();  // sh is free again
  total = all;
  return before + x;
}

// Up to three counts below 2^21 (the host's limit on rows, keys and units)
// summed in one scan.
constexpr int kCountBits = 21;
__device__ __forceinline__ int64_t pack3(int a, int b, int c = 0) {
  return (int64_t)a | (int64_t)b << kCountBits | (int64_t)c << 2 * kCountBits;
}
__device__ __forceinline__ int count_of(int64_t packed, int which) {
  return (int)(packed >> which * kCountBits) & ((1 << kCountBits) - 1);
}

constexpr int kItems = 4;  // consecutive entries per thread of a scan: rows of up to 4,096 take one
constexpr int kChunk = kItems * kThreads;

// int32 scratch of one batch row. Cyclic rows use all of it; packed schedules
// the seen counters (in place of `cover` and of the query flags), the
// positions and the runs.
struct RowLayout {
  int64_t cover, run, qseen, qpos, kpos, segs, qruns, kruns, row_ints;
  __host__ __device__ explicit RowLayout(const wmx_plan_args& a) {
    const int64_t q = a.q_len, k = a.k_len;
    cover = 0;                 // k + 1: coverage differences (packed: seen keys)
    run = cover + k + 1;       // k: number of the run of equal key ids
    qseen = run + k;           // q (packed: seen queries)
    qpos = qseen + q;          // q: place among the row's valid queries, or ~place among the idle ones
    kpos = qpos + q;           // k: place among the row's idle keys, or -1
    segs = kpos + k;           // 4 q: first query, last query, first key, real keys
    qruns = segs + 4 * q;      // 2 q: first and last query
    kruns = qruns + 2 * q;     // 2 k: first and last key
    row_ints = (kruns + 2 * k + 3) & ~(int64_t)3;
  }
};

// One row's counts (wmx_plan_args counts), kept in LDS while it is counted.
struct Tally {
  unsigned long long v[WMX_PLAN_COUNTS];
};

__device__ __forceinline__ void tally_add(Tally& t, int what, int64_t x) {
  if (x) atomicAdd(&t.v[what], (unsigned long long)x);
}
__device__ __forceinline__ void tally_max(Tally& t, int what, int64_t x) {
  atomicMax(&t.v[what], (unsigned long long)x);
}
__device__ __forceinline__ void tally_flag(Tally& t, int bit) { atomicOr(&t.v[WMX_PLAN_FLAGS], (unsigned long long)bit); }

// What a segment of nq queries and nk keys adds to the plan.
__device__ void tally_segment(Tally& t, const wmx_plan_args& a, int64_t nq, int64_t nk) {
  const int64_t qt = ceil_div(nq, kTile), kt = ceil_div(nk, a.key_tile);
  const bool fused = nq >= 1 && nq <= a.fused_rows && nk > 0;
  tally_max(t, WMX_PLAN_MAX_QUERIES, nq);
  tally_max(t, WMX_PLAN_MAX_KEYS, nk);
  tally_add(t, WMX_PLAN_Q_UNITS, qt);
  tally_add(t, WMX_PLAN_K_UNITS, kt);
  tally_add(t, fused ? WMX_PLAN_F_UNITS : WMX_PLAN_BQ_UNITS, fused ? 1 : qt);
  if (!fused) tally_add(t, WMX_PLAN_BK_UNITS, kt);
  tally_add(t, WMX_PLAN_DS_ELEMENTS, nk * qt * kTile);
}

// The row's runs of entries that `covered` does not hold: their places in
// order (pos, through `place`) and their first and last entries.
template <class Covered, class Place>
__device__ void idle_runs(int n, Covered covered, Place place, int32_t* runs, int& idle_total, int& run_total, int64_t* sh) {
  int carry = 0, carry_run = 0;
  for (int j0 = 0; j0 < n; j0 += kChunk) {
    const int j = j0 + kItems * (int)threadIdx.x;
    bool idle[kItems + 2];  // entries j - 1 .. j + kItems; outside the row: covered
#pragma unroll
    for (int e = 0; e < kItems + 2; ++e) idle[e] = j + e - 1 >= 0 && j + e - 1 < n && !covered(j + e - 1);
    int mine = 0, firsts = 0;
#pragma unroll
    for (int e = 1; e <= kItems; ++e) {
      mine += idle[e];
      firsts += idle[e] && !idle[e - 1];
    }
    int64_t total;
    const int64_t incl = block_scan(pack3(mine, firsts), total, sh);
    int at = carry + count_of(incl, 0) - mine, run = carry_run + count_of(incl, 1) - firsts;
#pragma unroll
    for (int e = 1; e <= kItems; ++e) {
      const int i = j + e - 1;
      if (i < n) place(i, idle[e], at);
      if (idle[e]) {
        if (!idle[e - 1]) runs[2 * run++] = i;
        if (!idle[e + 1]) runs[2 * run - 1] = i;
        ++at;
      }
    }
    carry += count_of(total, 0);
    carry_run += count_of(total, 1);
  }
  idle_total = carry;
  run_total = carry_run;
}

// The runs of idle rows as segments, once they are written.
__device__ void tally_runs(Tally& t, const wmx_plan_args& a, const int32_t* ws, const RowLayout& L, int q_runs, int k_runs) {
  for (int r = threadIdx.x; r < q_runs; r += kThreads)
    tally_segment(t, a, ws[L.qruns + 2 * (int64_t)r + 1] - ws[L.qruns + 2 * (int64_t)r] + 1, 0);
  for (int r = threadIdx.x; r < k_runs; r += kThreads)
    tally_segment(t, a, 0, ws[L.kruns + 2 * (int64_t)r + 1] - ws[L.kruns + 2 * (int64_t)r] + 1);
}

__device__ void store_counts(const wmx_plan_args& a, int row, const Tally& t) {
  for (int c = threadIdx.x; c < WMX_PLAN_COUNTS; c += kThreads)
    a.counts[(int64_t)row * WMX_PLAN_COUNTS + c] = (int64_t)t.v[c];
}

// ---------------------------------------------------------------- cyclic ----
// One batch row of cyclic document metadata. Segments are the runs of valid
// queries (those that see a key) of one document; see the packed schedule's
// conditions in cyclic_attention.py (_build_packed_schedule). A row that
// breaks one sets WMX_PLAN_REFUSED (the document-mode kernels take the call);
// a form that the host's builder decides sets WMX_PLAN_GENERAL.
__global__ __launch_bounds__(kThreads) void cyclic_count_kernel(const wmx_plan_args a) {
  __shared__ int64_t sh[kWaves];
  __shared__ Tally tally;
  const int b = blockIdx.x, tid = threadIdx.x;
  const RowLayout L(a);
  int32_t* ws = (int32_t*)a.workspace + (int64_t)b * L.row_ints;
  const int Q = a.q_len, K = a.k_len;
  const int32_t* qseg = a.q_seg + (int64_t)b * Q;
  const int32_t* kseg = a.k_seg + (int64_t)b * K;
  const int32_t* qstart = a.q_start + (int64_t)b * Q;
  const int32_t* kqend = a.k_qend + (int64_t)b * K;
  for (int c = tid; c < WMX_PLAN_COUNTS; c += kThreads) tally.v[c] = 0;

  // keys: the dummy prefix, the runs of equal ids
  int carry_run = 0, nd = 0, bad = 0;
  for (int j0 = 0; j0 < K; j0 += kChunk) {
    const int j = j0 + kItems * tid;
    int opens = 0, dummies = 0;
    bool open[kItems];
    int before = j > 0 && j <= K ? kseg[j - 1] : 0, end_before = j > 0 && j <= K ? kqend[j - 1] : 0;
#pragma unroll
    for (int e = 0; e < kItems; ++e) {
      const int i = j + e;
      open[e] = false;
      if (i < K) {
        const int id = kseg[i], end = kqend[i];
        open[e] = i == 0 || before != id;
        opens += open[e];
        dummies += id < 0;
        bad |= i > 0 && id < 0 && before >= 0;  // the dummies are one leading prefix
        bad |= id < 0 && end < Q;               // every query may see them
        bad |= !open[e] && end != end_before;   // one query end per run
        before = id;
        end_before = end;
        ws[L.cover + i] = 0;
      }
    }
    int64_t total;
    int run = carry_run + count_of(block_scan(pack3(opens, dummies), total, sh), 0) - opens;
#pragma unroll
    for (int e = 0; e < kItems; ++e) {
      run += open[e];
      if (j + e < K) ws[L.run + j + e] = run;
    }
    carry_run += count_of(total, 0);
    nd += count_of(total, 1);
  }
  if (tid == 0) ws[L.cover + K] = 0;
  __threadfence();  // the zeroed coverage is written before the atomics below
  __syncthreads();  // run numbers are read at arbitrary slots below

  // queries: validity and segments
  auto slot_of = [&](int i) { return (int64_t)a.query_offset + (int64_t)a.query_stride * i; };
  int carry_pos = 0, carry_seg = 0, carry_idle_run = 0, general = 0;
  for (int i0 = 0; i0 < Q; i0 += kChunk) {
    const int i = i0 + kItems * tid;
    // entries i - 1 .. i + kItems; those outside the row are neither valid nor idle
    bool valid[kItems + 2], inside[kItems + 2];
    int start[kItems + 2], doc[kItems + 2];
#pragma unroll
    for (int e = 0; e < kItems + 2; ++e) {
      const int x = i + e - 1;
      inside[e] = x >= 0 && x < Q;
      start[e] = inside[e] ? qstart[x] : 0;
      doc[e] = inside[e] ? qseg[x] : 0;
      const int64_t slot = slot_of(x);
      valid[e] = inside[e] && slot >= 0 && (nd > 0 || slot >= (int64_t)start[e]);
    }
    auto joined = [&](int e) {  // entries e and e + 1 are queries of one segment
      return valid[e] && valid[e + 1] && start[e] == start[e + 1] && doc[e] == doc[e + 1];
    };
    int mine = 0, firsts = 0, idle_firsts = 0;
#pragma unroll
    for (int e = 1; e <= kItems; ++e) {
      mine += valid[e];
      firsts += valid[e] && !joined(e - 1);
      idle_firsts += inside[e] && !valid[e] && (!inside[e - 1] || valid[e - 1]);
    }
    int64_t total;
    const int64_t incl = block_scan(pack3(mine, firsts, idle_firsts), total, sh);
    int pos = carry_pos + count_of(incl, 0) - mine, seg = carry_seg + count_of(incl, 1) - firsts;
    int idle_run = carry_idle_run + count_of(incl, 2) - idle_firsts;
#pragma unroll
    for (int e = 1; e <= kItems; ++e) {
      const int x = i + e - 1;
      if (!inside[e]) continue;
      const int64_t slot = slot_of(x);
      bad |= doc[e] < 0;
      if (slot >= (int64_t)start[e]) {
        const int at = (int)(slot < 0 ? 0 : slot < K ? slot : K - 1);
        const int from = start[e] < 0 ? 0 : start[e] < at ? start[e] : at;
        // [start, slot] lies in one run, of this document, that the query may see
        bad |= kseg[at] != doc[e] || ws[L.run + from] != ws[L.run + at] || start[e] < nd || kqend[at] <= x;
      }
      bad |= valid[e] && nd > 0 && slot < (int64_t)start[e] - 1;
      general |= slot >= K;
      ws[L.qpos + x] = valid[e] ? pos : ~(x - pos);
      if (valid[e]) {
        if (!joined(e - 1)) ws[L.segs + 4 * (int64_t)seg++] = x;
        if (!joined(e)) {
          const int64_t reach = slot - start[e] + 1;
          const int real = reach > 0 ? (int)reach : 0;
          int32_t* s = ws + L.segs + 4 * (int64_t)(seg - 1);
          s[1] = x;
          s[2] = start[e];
          s[3] = real;
          if (real > 0) {
            if (start[e] >= 0 && slot < K) {
              atomicAdd(&ws[L.cover + start[e]], 1);
              atomicAdd(&ws[L.cover + slot + 1], -1);
            } else {
              general = 1;
            }
          }
        }
        ++pos;
      } else {
        if (!inside[e - 1] || valid[e - 1]) ws[L.qruns + 2 * (int64_t)idle_run++] = x;
        if (!inside[e + 1] || valid[e + 1]) ws[L.qruns + 2 * (int64_t)idle_run - 1] = x;
      }
    }
    carry_pos += count_of(total, 0);
    carry_seg += count_of(total, 1);
    carry_idle_run += count_of(total, 2);
  }
  __threadfence();
  __syncthreads();  // coverage differences, segments and query runs are complete
  for (int s = tid; s < carry_seg; s += kThreads) {
    const int32_t* e = ws + L.segs + 4 * (int64_t)s;
    tally_segment(tally, a, e[1] - e[0] + 1, (int64_t)e[3] + nd);
    tally_add(tally, WMX_PLAN_KEYS, (int64_t)e[3] + nd);
  }

  // keys that no segment holds
  int carry_cover = 0, idle_k, k_runs;
  for (int j0 = 0; j0 < K; j0 += kChunk) {
    const int j = j0 + kItems * tid;
    int d[kItems], sum = 0;
#pragma unroll
    for (int e = 0; e < kItems; ++e) {
      d[e] = j + e < K ? ws[L.cover + j + e] : 0;
      sum += d[e];
    }
    int64_t total;
    int c = carry_cover + (int)block_scan(sum, total, sh) - sum;
#pragma unroll
    for (int e = 0; e < kItems; ++e) {
      c += d[e];
      if (j + e < K) {
        ws[L.run + j + e] = c > 0 || kseg[j + e] < 0 ? 1 : 0;  // the run numbers are done with
        general |= c > 1;  // two segments hold this key row
      }
    }
    carry_cover += (int)total;
  }
  __syncthreads();
  idle_runs(
      K, [&](int j) { return ws[L.run + j] != 0; },
      [&](int j, bool idle, int at) { ws[L.kpos + j] = idle ? at : -1; }, ws + L.kruns, idle_k, k_runs, sh);
  __syncthreads();
  tally_runs(tally, a, ws, L, carry_idle_run, k_runs);
  if (bad) tally_flag(tally, WMX_PLAN_REFUSED);
  if (general || nd > 1) tally_flag(tally, WMX_PLAN_GENERAL);
  if (tid == 0) {
    tally.v[WMX_PLAN_QUERIES] = carry_pos;
    tally.v[WMX_PLAN_SEGMENTS] = carry_seg;
    tally.v[WMX_PLAN_IDLE_QUERIES] = Q - carry_pos;
    tally.v[WMX_PLAN_QUERY_RUNS] = carry_idle_run;
    tally.v[WMX_PLAN_IDLE_KEYS] = idle_k;
    tally.v[WMX_PLAN_KEY_RUNS] = k_runs;
    tally.v[WMX_PLAN_DUMMIES] = nd;
  }
  __syncthreads();
  store_counts(a, b, tally);
}

// Totals over all rows, and over the rows before this one, of the counts that
// place a row's outputs: one wave per count.
struct RowOffsets {
  int64_t before[WMX_PLAN_KEY_RUNS + 1], total[WMX_PLAN_KEY_RUNS + 1];
  __device__ void init(const wmx_plan_args& a, int b) {
    const int what = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (what <= WMX_PLAN_KEY_RUNS) {
      int64_t mine = 0, all = 0;
      for (int r = lane; r < a.batch; r += 64) {
        const int64_t c = a.counts[(int64_t)r * WMX_PLAN_COUNTS + what];
        all += c;
        if (r < b) mine += c;
      }
      for (int o = 32; o > 0; o >>= 1) {
        mine += __shfl_xor(mine, o);
        all += __shfl_xor(all, o);
      }
      if (lane == 0) {
        before[what] = mine;
        total[what] = all;
      }
    }
    __syncthreads();
  }
};

// The idle rows of batch row b as segments after the first `segments` ones,
// whose queries and keys come first: the queries' runs, then the keys'.
__device__ void fill_idle(const wmx_plan_args& a, int b, const int32_t* ws, const RowLayout& L, const RowOffsets& at,
                          int64_t segments, int64_t queries, int64_t keys) {
  const int64_t iq = queries + at.before[WMX_PLAN_IDLE_QUERIES], ik = keys + at.before[WMX_PLAN_IDLE_KEYS];
  const int64_t rq = segments + at.before[WMX_PLAN_QUERY_RUNS];
  const int64_t rk = segments + at.total[WMX_PLAN_QUERY_RUNS] + at.before[WMX_PLAN_KEY_RUNS];
  const int64_t all_queries = queries + at.total[WMX_PLAN_IDLE_QUERIES];
  const int64_t* mine = a.counts + (int64_t)b * WMX_PLAN_COUNTS;
  for (int i = threadIdx.x; i < a.q_len; i += kThreads) {
    const int p = ws[L.qpos + i];
    if (p < 0) a.out_query_indices[iq + ~p] = (int64_t)b * a.q_len + i;
  }
  for (int j = threadIdx.x; j < a.k_len; j += kThreads) {
    const int p = ws[L.kpos + j];
    if (p >= 0) a.out_key_indices[ik + p] = (int64_t)b * a.k_len + j;
  }
  for (int64_t r = threadIdx.x; r < mine[WMX_PLAN_QUERY_RUNS]; r += kThreads) {
    a.out_cu_queries[rq + r] = (int32_t)(iq + ~ws[L.qpos + ws[L.qruns + 2 * r]]);
    a.out_cu_keys[rq + r] = (int32_t)keys;
  }
  for (int64_t r = threadIdx.x; r < mine[WMX_PLAN_KEY_RUNS]; r += kThreads) {
    a.out_cu_queries[rk + r] = (int32_t)all_queries;
    a.out_cu_keys[rk + r] = (int32_t)(ik + ws[L.kpos + ws[L.kruns + 2 * r]]);
  }
  if (b == a.batch - 1 && threadIdx.x == 0) {
    const int64_t end = segments + at.total[WMX_PLAN_QUERY_RUNS] + at.total[WMX_PLAN_KEY_RUNS];
    a.out_cu_queries[end] = (int32_t)all_queries;
    a.out_cu_keys[end] = (int32_t)(keys + at.total[WMX_PLAN_IDLE_KEYS]);
  }
}

__global__ __launch_bounds__(kThreads) void cyclic_fill_kernel(const wmx_plan_args a) {
  __shared__ int64_t sh[kWaves];
  __shared__ RowOffsets at;
  const int b = blockIdx.x, tid = threadIdx.x;
  const RowLayout L(a);
  const int32_t* ws = (const int32_t*)a.workspace + (int64_t)b * L.row_ints;
  at.init(a, b);
  const int64_t q0 = at.before[WMX_PLAN_QUERIES], s0 = at.before[WMX_PLAN_SEGMENTS], k0 = at.before[WMX_PLAN_KEYS];
  const int64_t* mine = a.counts + (int64_t)b * WMX_PLAN_COUNTS;
  const int nseg = (int)mine[WMX_PLAN_SEGMENTS], nd = (int)mine[WMX_PLAN_DUMMIES];
  for (int i = tid; i < a.q_len; i += kThreads) {
    const int p = ws[L.qpos + i];
    if (p >= 0) a.out_query_indices[q0 + p] = (int64_t)b * a.q_len + i;
  }
  fill_idle(a, b, ws, L, at, at.total[WMX_PLAN_SEGMENTS], at.total[WMX_PLAN_QUERIES], at.total[WMX_PLAN_KEYS]);
  int64_t carry = 0;
  for (int t0 = 0; t0 < nseg; t0 += kThreads) {
    const int s = t0 + tid;
    const bool in = s < nseg;
    const int32_t* e = ws + L.segs + 4 * (int64_t)(in ? s : 0);
    int64_t total;
    const int64_t nk = in ? (int64_t)e[3] + nd : 0;
    const int64_t end = carry + block_scan(nk, total, sh);
    if (in) {
      a.out_cu_queries[s0 + s] = (int32_t)(q0 + ws[L.qpos + e[0]]);
      a.out_cu_keys[s0 + s] = (int32_t)(k0 + end - nk);
    }
    carry += total;
  }
  __threadfence_block();
  __syncthreads();  // this row's key starts are read below
  const int wave = tid >> 6, lane = tid & 63;
  for (int s = wave; s < nseg; s += kWaves) {
    const int32_t* e = ws + L.segs + 4 * (int64_t)s;
    const int first = e[2], nk = e[3] + nd;
    const int64_t to = a.out_cu_keys[s0 + s];
    for (int j = lane; j < nk; j += 64)
      a.out_key_indices[to + j] = (int64_t)b * a.k_len + (j < nd ? j : first + j - nd);
  }
}

// ------------------------------------------------------- packed schedules ----
// One segment of the given schedule: its bounds, its layout (queries one
// after another in one row; keys likewise from the second on) and its marks
// in the rows' seen counters. What the host's planner has to decide or refuse
// sets WMX_PLAN_GENERAL. The counts go to row `batch`; only bounds that were
// checked here are followed.
__global__ __launch_bounds__(256) void packed_mark_kernel(const wmx_plan_args a) {
  __shared__ int general_lds;
  const int s = blockIdx.x, tid = threadIdx.x;
  const RowLayout L(a);
  int32_t* ws = (int32_t*)a.workspace;
  unsigned long long* counts = (unsigned long long*)a.counts + (int64_t)a.batch * WMX_PLAN_COUNTS;
  const int64_t qs = a.cu_queries[s], qe = a.cu_queries[s + 1], ks = a.cu_keys[s], ke = a.cu_keys[s + 1];
  const bool bounded = 0 <= qs && qs <= qe && qe <= a.num_queries && 0 <= ks && ks <= ke && ke <= a.num_keys &&
                       (s + 1 < a.num_segments || (qe == a.num_queries && ke == a.num_keys)) &&
                       (s > 0 || (qs == 0 && ks == 0));
  if (tid == 0) general_lds = bounded ? 0 : 1;
  __syncthreads();
  if (bounded) {
    const int64_t nq = qe - qs, nk = ke - ks;
    const int64_t q_slots = (int64_t)a.batch * a.q_len, k_slots = (int64_t)a.batch * a.k_len;
    int general = 0;
    int64_t slot0 = 0;
    if (nq > 0) {
      const int64_t first = a.query_indices[qs];
      const bool ok = first >= 0 && first + nq <= q_slots && first / a.q_len == (first + nq - 1) / a.q_len;
      general |= !ok;
      if (ok) {
        int32_t* seen = ws + first / a.q_len * L.row_ints + L.qseen + first % a.q_len;
        for (int64_t e = tid; e < nq; e += 256) {
          general |= a.query_indices[qs + e] != first + e;
          general |= atomicAdd(&seen[e], 1) != 0;  // a query row of two segments
        }
      }
    }
    if (nk > 0) {
      const int64_t key0 = a.key_indices[ks], second = nk > 1 ? a.key_indices[ks + 1] : key0 + 1;
      bool ok = key0 >= 0 && key0 < k_slots;
      ok = ok && (nk == 1 || (second >= 0 && second + nk - 1 <= k_slots &&
                              second / a.k_len == key0 / a.k_len && (second + nk - 2) / a.k_len == key0 / a.k_len));
      general |= !ok;
      if (ok) {
        int32_t* row = ws + key0 / a.k_len * L.row_ints + L.cover;
        slot0 = key0 % a.k_len;
        general |= nk > 1 && slot0 == 0 && second % a.k_len == 0;  // slot 0 twice in this segment
        if (tid == 0 && atomicAdd(&row[slot0], 1) != 0) {
          // a shared slot 0 (a leading dummy) is a layout of its own
          if (slot0 == 0) atomicAdd(&counts[WMX_PLAN_DUMMIES], 1ull);
          else general = 1;
        }
        int32_t* rest = row + (nk > 1 ? second % a.k_len : 0);
        for (int64_t e = tid; e + 1 < nk; e += 256) {
          general |= a.key_indices[ks + 1 + e] != second + e;
          general |= atomicAdd(&rest[e], 1) != 0;
        }
      }
    }
    if (general) atomicOr(&general_lds, 1);
    if (tid == 0) {
      const int64_t qt = ceil_div(nq, kTile);
      atomicMax(&counts[WMX_PLAN_MAX_QUERIES], (unsigned long long)nq);
      atomicMax(&counts[WMX_PLAN_MAX_KEYS], (unsigned long long)nk);
      atomicAdd(&counts[WMX_PLAN_Q_UNITS], (unsigned long long)qt);
      atomicAdd(&counts[WMX_PLAN_K_UNITS], (unsigned long long)ceil_div(nk, a.key_tile));
      atomicAdd(&counts[WMX_PLAN_DS_ELEMENTS], (unsigned long long)(nk * qt * kTile));
    }
  }
  __syncthreads();
  if (tid == 0 && general_lds) atomicOr(&counts[WMX_PLAN_FLAGS], (unsigned long long)WMX_PLAN_GENERAL);
}

__global__ __launch_bounds__(kThreads) void packed_count_kernel(const wmx_plan_args a) {
  __shared__ int64_t sh[kWaves];
  __shared__ Tally tally;
  const int b = blockIdx.x, tid = threadIdx.x;
  const RowLayout L(a);
  int32_t* ws = (int32_t*)a.workspace + (int64_t)b * L.row_ints;
  for (int c = tid; c < WMX_PLAN_COUNTS; c += kThreads) tally.v[c] = 0;
  int idle_q, q_runs, idle_k, k_runs;
  idle_runs(
      a.q_len, [&](int i) { return ws[L.qseen + i] != 0; },
      [&](int i, bool idle, int at) { ws[L.qpos + i] = idle ? ~at : 0; }, ws + L.qruns, idle_q, q_runs, sh);
  idle_runs(
      a.k_len, [&](int j) { return ws[L.cover + j] != 0; },
      [&](int j, bool idle, int at) { ws[L.kpos + j] = idle ? at : -1; }, ws + L.kruns, idle_k, k_runs, sh);
  __syncthreads();
  tally_runs(tally, a, ws, L, q_runs, k_runs);
  if (tid == 0) {
    tally.v[WMX_PLAN_IDLE_QUERIES] = idle_q;
    tally.v[WMX_PLAN_QUERY_RUNS] = q_runs;
    tally.v[WMX_PLAN_IDLE_KEYS] = idle_k;
    tally.v[WMX_PLAN_KEY_RUNS] = k_runs;
  }
  __syncthreads();
  store_counts(a, b, tally);
}

// The covering schedule: the given one (copied by the workgroups past the
// batch's), then the idle rows.
__global__ __launch_bounds__(kThreads) void packed_fill_kernel(const wmx_plan_args a) {
  __shared__ RowOffsets at;
  if ((int)blockIdx.x < a.batch) {
    const RowLayout L(a);
    const int b = blockIdx.x;
    at.init(a, b);
    fill_idle(a, b, (const int32_t*)a.workspace + (int64_t)b * L.row_ints, L, at, a.num_segments, a.num_queries, a.num_keys);
    return;
  }
  const int64_t mine = (int64_t)(blockIdx.x - a.batch) * kThreads + threadIdx.x;
  const int64_t step = (int64_t)(gridDim.x - a.batch) * kThreads;
  for (int64_t e = mine; e < a.num_queries; e += step) a.out_query_indices[e] = a.query_indices[e];
  for (int64_t e = mine; e < a.num_keys; e += step) a.out_key_indices[e] = a.key_indices[e];
  for (int64_t e = mine; e < a.num_segments; e += step) {
    a.out_cu_queries[e] = a.cu_queries[e];
    a.out_cu_keys[e] = a.cu_keys[e];
  }
}

// ------------------------------------------------------------- work lists ----
// A unit's sort key: steps its loop visits (20 bits), its rows (8), then
// earlier segments (20) and tiles (15) first, and the mark of a segment that
// the fused backward takes. The host checks that the schedule fits.
__device__ __forceinline__ uint64_t unit_key(int64_t steps, int64_t rows, int64_t seg, int64_t tile, bool fused) {
  return (uint64_t)steps << 44 | (uint64_t)rows << 36 | (uint64_t)((1 << 20) - 1 - seg) << 16 |
         (uint64_t)((1 << 15) - 1 - tile) << 1 | (fused ? 1u : 0u);
}

struct UnitsLayout {
  int64_t fields, q_keys, k_keys, f_keys, bytes;
  __host__ __device__ explicit UnitsLayout(const wmx_plan_args& a) {
    fields = 0;
    q_keys = fields + (int64_t)a.total_segments * WMX_UNIT_FIELDS * (int64_t)sizeof(int32_t);
    k_keys = q_keys + (int64_t)a.num_q_units * 8;
    f_keys = k_keys + (int64_t)a.num_k_units * 8;
    bytes = f_keys + (int64_t)a.num_f_units * 8;
  }
};

__global__ __launch_bounds__(kThreads) void units_kernel(const wmx_plan_args a) {
  __shared__ int64_t sh[kWaves];
  const UnitsLayout U(a);
  char* base = (char*)a.unit_workspace;
  int32_t* fields = (int32_t*)(base + U.fields);
  uint64_t* q_keys = (uint64_t*)(base + U.q_keys);
  uint64_t* k_keys = (uint64_t*)(base + U.k_keys);
  uint64_t* f_keys = (uint64_t*)(base + U.f_keys);
  int64_t c_ds = 0;
  int c_q = 0, c_k = 0, c_f = 0;
  const int stride = a.query_stride, key_tile = a.key_tile;
  for (int s0 = 0; s0 < a.total_segments; s0 += kThreads) {
    const int s = s0 + (int)threadIdx.x;
    const bool in = s < a.total_segments;
    int qs = 0, ks = 0, nq = 0, nk = 0;
    if (in) {
      qs = a.out_cu_queries[s];
      nq = a.out_cu_queries[s + 1] - qs;
      ks = a.out_cu_keys[s];
      nk = a.out_cu_keys[s + 1] - ks;
    }
    const int qt = (nq + kTile - 1) / kTile, kt = (nk + key_tile - 1) / key_tile;
    const bool fused = nq >= 1 && nq <= a.fused_rows && nk > 0;
    int64_t t_ds, t_units;
    const int64_t blk = (int64_t)nk * qt * kTile;
    const int64_t ds = c_ds + block_scan(blk, t_ds, sh) - blk;
    const int64_t units = block_scan(pack3(qt, kt, fused ? 1 : 0), t_units, sh);
    const int qu = c_q + count_of(units, 0) - qt, ku = c_k + count_of(units, 1) - kt;
    const int fu = c_f + count_of(units, 2) - (fused ? 1 : 0);
    if (in) {
      a.ds_offsets[s] = ds;
      int32_t e[WMX_UNIT_FIELDS] = {};
      e[WMX_UNIT_SEGMENT] = s;
      e[WMX_UNIT_QUERY_START] = qs;
      e[WMX_UNIT_QUERIES] = nq;
      e[WMX_UNIT_KEY_START] = ks;
      e[WMX_UNIT_KEYS] = nk;
      // rows and slots fit 32 bits (the host's limit)
      if (nq > 0) {
        const uint32_t at = (uint32_t)a.out_query_indices[qs], row = at / (uint32_t)a.q_len;
        e[WMX_UNIT_QUERY_ROW] = (int32_t)row;
        e[WMX_UNIT_QUERY_SLOT0] = (int32_t)(at - row * a.q_len);
        e[WMX_UNIT_QUERY_SLOT1] =
            nq > 1 ? (int32_t)((uint32_t)a.out_query_indices[qs + 1] - row * a.q_len) : e[WMX_UNIT_QUERY_SLOT0] + 1;
      }
      if (nk > 0) {
        const uint32_t at = (uint32_t)a.out_key_indices[ks], row = at / (uint32_t)a.k_len;
        e[WMX_UNIT_KEY_ROW] = (int32_t)row;
        e[WMX_UNIT_KEY_SLOT0] = (int32_t)(at - row * a.k_len);
        e[WMX_UNIT_KEY_SLOT1] =
            nk > 1 ? (int32_t)((uint32_t)a.out_key_indices[ks + 1] - row * a.k_len) : e[WMX_UNIT_KEY_SLOT0] + 1;
      }
      e[WMX_UNIT_DS_LO] = (int32_t)(uint32_t)ds;
      e[WMX_UNIT_DS_HI] = (int32_t)(ds >> 32);
      int4* to = (int4*)(fields + (int64_t)s * WMX_UNIT_FIELDS);
#pragma unroll
      for (int v = 0; v < WMX_UNIT_FIELDS / 4; ++v) to[v] = make_int4(e[4 * v], e[4 * v + 1], e[4 * v + 2], e[4 * v + 3]);
      // query i of the segment sees keys 0 .. off + stride * i
      const int64_t off = (int64_t)nk - 1 - (int64_t)stride * (nq - 1);
      for (int t = 0; t < qt; ++t) {
        const int end = min(nq, (t + 1) * kTile);
        int64_t reach = off + (int64_t)stride * (end - 1) + 1;
        reach = reach < 0 ? 0 : reach < nk ? reach : nk;
        q_keys[qu + t] = unit_key(((int)reach + kStep - 1) / kStep, end - t * kTile, s, t, fused);
      }
      for (int t = 0; t < kt; ++t) {
        const int end = min(nk, (t + 1) * key_tile);
        const int64_t need = (int64_t)t * key_tile - off;
        // a 32-bit division where the operands fit
        const int64_t first = need <= 0           ? 0
                              : need <= INT32_MAX ? (int64_t)(((uint32_t)need + (uint32_t)stride - 1) / (uint32_t)stride)
                                                  : ceil_div(need, stride);
        const int steps = first < nq ? (nq - (int)first / kStep * kStep + kStep - 1) / kStep : 0;
        k_keys[ku + t] = unit_key(steps, end - t * key_tile, s, t, fused);
      }
      if (fused) f_keys[fu] = unit_key((nk + kStep - 1) / kStep, nq, s, 0, true);
    }
    c_ds += t_ds;
    c_q += count_of(t_units, 0);
    c_k += count_of(t_units, 1);
    c_f += count_of(t_units, 2);
  }
  if (threadIdx.x == 0) a.ds_offsets[a.total_segments] = c_ds;
}

// One workgroup places 256 units of one list (grid.y: query tiles, key tiles,
// fused segments) in it and, for the first two, in the list of the backward
// without the fused segments.
__global__ __launch_bounds__(256) void rank_kernel(const wmx_plan_args a) {
  __shared__ uint64_t keys_lds[256];
  const UnitsLayout U(a);
  const char* base = (const char*)a.unit_workspace;
  const int which = blockIdx.y, tid = threadIdx.x;
  const int n = which == 0 ? a.num_q_units : which == 1 ? a.num_k_units : a.num_f_units;
  if ((int64_t)blockIdx.x * 256 >= n) return;
  const uint64_t* keys = (const uint64_t*)(base + (which == 0 ? U.q_keys : which == 1 ? U.k_keys : U.f_keys));
  int32_t* list = which == 0 ? a.q_units : which == 1 ? a.k_units : a.f_units;
  int32_t* rest = which == 0 ? a.bq_units : which == 1 ? a.bk_units : nullptr;
  const int u = blockIdx.x * 256 + tid;
  const uint64_t mine = u < n ? keys[u] : 0;
  int rank = 0, rest_rank = 0;
  for (int v0 = 0; v0 < n; v0 += 256) {
    const int m = min(256, n - v0);
    if (tid < m) keys_lds[tid] = keys[v0 + tid];
    __syncthreads();
    for (int v = 0; v < m; ++v) {
      const uint64_t k = keys_lds[v];
      rank += k > mine ? 1 : 0;
      rest_rank += k > mine && !(k & 1) ? 1 : 0;
    }
    __syncthreads();
  }
  if (u >= n) return;
  const int seg = (1 << 20) - 1 - (int)(mine >> 16 & ((1 << 20) - 1));
  const int tile = (1 << 15) - 1 - (int)(mine >> 1 & ((1 << 15) - 1));
  const int4* from = (const int4*)((const int32_t*)(base + U.fields) + (int64_t)seg * WMX_UNIT_FIELDS);
  int4 e[WMX_UNIT_FIELDS / 4];
#pragma unroll
  for (int v = 0; v < WMX_UNIT_FIELDS / 4; ++v) e[v] = from[v];
  e[0].y = tile;  // WMX_UNIT_TILE
  int4* to = (int4*)(list + (int64_t)rank * WMX_UNIT_FIELDS);
#pragma unroll
  for (int v = 0; v < WMX_UNIT_FIELDS / 4; ++v) to[v] = e[v];
  if (rest && !(mine & 1)) {
    to = (int4*)(rest + (int64_t)rest_rank * WMX_UNIT_FIELDS);
#pragma unroll
    for (int v = 0; v < WMX_UNIT_FIELDS / 4; ++v) to[v] = e[v];
  }
}

}  // namespace

int64_t plan_workspace_size(const wmx_plan_args& a) {
  return (int64_t)a.batch * RowLayout(a).row_ints * (int64_t)sizeof(int32_t);
}

int64_t plan_unit_workspace_size(const wmx_plan_args& a) { return UnitsLayout(a).bytes; }

int launch_plan_count(const wmx_plan_args& a, hipStream_t stream) {
  if (a.q_seg) {
    hipLaunchKernelGGL(cyclic_count_kernel, dim3(a.batch), dim3(kThreads), 0, stream, a);
    return WMX_OK;
  }
  hipLaunchKernelGGL(packed_mark_kernel, dim3(a.num_segments), dim3(256), 0, stream, a);
  hipLaunchKernelGGL(packed_count_kernel, dim3(a.batch), dim3(kThreads), 0, stream, a);
  return WMX_OK;
}

// Measured (4 rows of 1,027 tokens, stride 8, dummy, about 20 documents): count
// 27, fill 6, units 11 and rank 5 us per residue. Metadata and plans of all
// eight residues with four layers of attention behind them: 24.3-27 ms with the
// host builders, 1.7 ms here. The Jacobi plan of 4 x 1,531 tokens: mark and
// count 15, fill 7, units 13, rank 5 us; its step over four layers 3.46 ->
// 0.95 ms.
int launch_plan_fill(const wmx_plan_args& a, hipStream_t stream) {
  wmx_plan_args u = a;
  if (a.q_seg) {
    hipLaunchKernelGGL(cyclic_fill_kernel, dim3(a.batch), dim3(kThreads), 0, stream, a);
  } else if (a.out_query_indices) {
    const int64_t elements = a.num_queries > a.num_keys ? a.num_queries : a.num_keys;
    const int64_t blocks = ceil_div(elements, 4 * kThreads);
    hipLaunchKernelGGL(packed_fill_kernel, dim3((unsigned)(a.batch + (blocks < 256 ? blocks : 256))), dim3(kThreads), 0,
                       stream, a);
  } else {
    // nothing to add: the given schedule runs as it is
    u.out_query_indices = const_cast<int64_t*>(a.query_indices);
    u.out_key_indices = const_cast<int64_t*>(a.key_indices);
    u.out_cu_queries = const_cast<int32_t*>(a.cu_queries);
    u.out_cu_keys = const_cast<int32_t*>(a.cu_keys);
  }
  hipLaunchKernelGGL(units_kernel, dim3(1), dim3(kThreads), 0, stream, u);
  const int64_t longest = a.num_q_units > a.num_k_units ? a.num_q_units : a.num_k_units;
  const int64_t blocks = ceil_div(longest > a.num_f_units ? longest : a.num_f_units, 256);
  if (blocks > 0) hipLaunchKernelGGL(rank_kernel, dim3((unsigned)blocks, 3), dim3(256), 0, stream, u);
  return WMX_OK;
}

}  // namespace wmx
