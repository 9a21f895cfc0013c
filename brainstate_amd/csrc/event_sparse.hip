// N2a / N2b: event-driven sparse mat-vec for fixed-num and CSR connectivity.
//
// Scatter (pre-major): waves stride over (active row, 64-synapse chunk) work items; each
// lane loads one target index and weight (a row's synapses are contiguous, so a wave
// reads 256 B of indices and 256 B of weights per chunk) and issues one hardware fp32
// atomic add.  The number of active rows is read on the device, so the launch needs
// no host synchronisation.
//
// Gather (post-major, SELL-64x4): one wave per slice of 64 posts, lane = post.  Each step
// loads the lane's next 4 columns of pre indices as one 16-byte word (1 KB per wave), tests
// the spike of each and adds the weight in column order, so every post accumulates its
// incoming synapses in ascending (pre, k) order -- bit-identical to a sequential pre-major
// scatter, with no atomics.
#include <cmath>
#include <type_traits>

#include "common.h"

namespace {

constexpr int kBlock = 256;

__global__ __launch_bounds__(kBlock) void k_fill_f32(float* __restrict__ p, int64_t n, float v) {
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kBlock)
    p[i] = v;
}

template <bool kCsr, bool kHet>
__global__ __launch_bounds__(kBlock) void k_scatter(const int32_t* __restrict__ active,
                                                    const int32_t* __restrict__ n_active_p,
                                                    int32_t n_pre,
                                                    const int32_t* __restrict__ indptr,
                                                    const int32_t* __restrict__ indices,
                                                    int32_t k, const float* __restrict__ w,
                                                    float w_homo, int32_t n_post,
                                                    float* __restrict__ out) {
  int32_t na = *n_active_p;
  na = na < 0 ? 0 : (na > n_pre ? n_pre : na);
  const int lane = bs_lane();
  const int64_t wave = ((int64_t)blockIdx.x * kBlock + threadIdx.x) / BS_WAVE;
  const int64_t nwaves = (int64_t)gridDim.x * (kBlock / BS_WAVE);
  if (!kCsr) {
    const int32_t cpr = (k + BS_WAVE - 1) / BS_WAVE;  // 64-synapse chunks per row
    const int64_t items = (int64_t)na * cpr;
    for (int64_t it = wave; it < items; it += nwaves) {
      const int32_t a = (int32_t)(it / cpr);
      const int32_t c = (int32_t)(it - (int64_t)a * cpr);
      const int32_t row = active[a];
      const int32_t t = c * BS_WAVE + lane;
      if ((uint32_t)row < (uint32_t)n_pre && t < k) {
        const int64_t s = (int64_t)row * k + t;
        const int32_t j = indices[s];
        const float v = kHet ? w[s] : w_homo;
        if ((uint32_t)j < (uint32_t)n_post) bs_atomic_add_f32(out + j, v);
      }
    }
  } else {
    const int32_t nnz = indptr[n_pre];
    for (int64_t a = wave; a < na; a += nwaves) {
      const int32_t row = active[a];
      if ((uint32_t)row >= (uint32_t)n_pre) continue;
      int32_t beg = indptr[row], end = indptr[row + 1];
      beg = beg < 0 ? 0 : beg;
      end = end > nnz ? nnz : end;
      for (int32_t s = beg + lane; s < end; s += BS_WAVE) {
        const int32_t j = indices[s];
        const float v = kHet ? w[s] : w_homo;
        if ((uint32_t)j < (uint32_t)n_post) bs_atomic_add_f32(out + j, v);
      }
    }
  }
}

// Spikes -> bitmap, one ballot per 64 spikes: bits[w] bit l <=> spk[32*w + l] != 0.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_pack(const T* __restrict__ spk, int32_t n,
                                                 uint32_t* __restrict__ bits) {
  const int lane = bs_lane();
  const int64_t nwords = ((int64_t)n + 31) / 32;
  for (int64_t base = ((int64_t)blockIdx.x * kBlock + threadIdx.x) - lane;
       base < (int64_t)n; base += (int64_t)gridDim.x * kBlock) {
    const int64_t i = base + lane;
    const bool a = i < n && spk[i] != T(0);
    const uint64_t m = bs_ballot(a);
    const int64_t w = base / 32;
    if (lane == 0 && w < nwords) bits[w] = (uint32_t)m;
    if (lane == 1 && w + 1 < nwords) bits[w + 1] = (uint32_t)(m >> 32);
  }
}

// Gather over SELL-64x4: wave = slice of 64 posts, lane = post; kU 16-byte groups of 4 pre
// indices in flight per lane; the spike test reads a bitmap held in LDS (kLds) or global
// memory.
template <bool kHet, bool kLds>
__global__ __launch_bounds__(kBlock) void k_gather(const uint32_t* __restrict__ bits,
                                                   int32_t n_pre,
                                                   const int64_t* __restrict__ slice_ptr,
                                                   const int32_t* __restrict__ sell_pre,
                                                   const float* __restrict__ sell_w,
                                                   float w_homo, int32_t n_post,
                                                   float* __restrict__ out) {
  constexpr int kGU = 8;  // 16-byte index groups per stage (16: slower, 2x the registers)
  extern __shared__ uint32_t s_bits[];
  const int32_t nwords = (n_pre + 31) / 32;
  if (kLds) {
    for (int32_t w = threadIdx.x; w < nwords; w += kBlock) s_bits[w] = bits[w];
    __syncthreads();
  }
  const uint32_t* bm = kLds ? s_bits : bits;
  const int lane = bs_lane();
  const int64_t slice = ((int64_t)blockIdx.x * kBlock + threadIdx.x) / BS_WAVE;
  const int64_t n_slices = ((int64_t)n_post + BS_WAVE - 1) / BS_WAVE;
  if (slice >= n_slices) return;
  const int64_t beg = slice_ptr[slice];
  const int64_t ngrp = (slice_ptr[slice + 1] - beg) / (4 * BS_WAVE);  // groups of 4 columns
  const int4* pre4 = (const int4*)(sell_pre + beg) + lane;
  float acc = 0.0f;
  const auto on = [&](int32_t i) {
    return (uint32_t)i < (uint32_t)n_pre && ((bm[i >> 5] >> (i & 31)) & 1u);
  };
  const float4* w4 = kHet ? (const float4*)(sell_w + beg) + lane : nullptr;
  int64_t g = 0;
  // two stages of kGU 16-byte index groups: the next stage's indices are loaded before this
  // stage's spike lookups, weight loads and adds, which stay in column order (100k x 100k,
  // K = 1000: 121 / 146 / 165 -> 112 / 125 / 158 us at p = 0.001 / 0.01 / 0.1; a third stage
  // for the weights, loaded one block ahead of their adds, measured slower)
  auto ld = [&](int64_t g0, int4 (&q)[kGU]) {
#pragma unroll
    for (int u = 0; u < kGU; ++u) q[u] = pre4[(g0 + u) * BS_WAVE];
  };
  auto use = [&](int64_t g0, const int4 (&q)[kGU]) {
    uint32_t act[kGU];  // bit e: column 4(g0+u)+e is an active synapse
    float4 wq[kGU];
#pragma unroll
    for (int u = 0; u < kGU; ++u) {
      act[u] = (uint32_t)on(q[u].x) | ((uint32_t)on(q[u].y) << 1) | ((uint32_t)on(q[u].z) << 2) |
               ((uint32_t)on(q[u].w) << 3);
      wq[u] = make_float4(w_homo, w_homo, w_homo, w_homo);
      if (kHet && act[u]) wq[u] = w4[(g0 + u) * BS_WAVE];  // this lane's 4 weights, one load
    }
#pragma unroll
    for (int u = 0; u < kGU; ++u) {
      if (act[u] & 1u) acc += wq[u].x;
      if (act[u] & 2u) acc += wq[u].y;
      if (act[u] & 4u) acc += wq[u].z;
      if (act[u] & 8u) acc += wq[u].w;
    }
  };
  if (kGU <= ngrp) {
    int4 qa[kGU], qb[kGU];
    ld(0, qa);
    for (; g + 2 * kGU <= ngrp; g += 2 * kGU) {
      __builtin_amdgcn_sched_barrier(0);
      ld(g + kGU, qb);
      __builtin_amdgcn_sched_barrier(0);
      use(g, qa);
      if (g + 3 * kGU <= ngrp) {
        __builtin_amdgcn_sched_barrier(0);
        ld(g + 2 * kGU, qa);
        __builtin_amdgcn_sched_barrier(0);
      }
      use(g + kGU, qb);
    }
    if (g + kGU <= ngrp) {  // qa holds stage g (loaded above, or before the loop)
      use(g, qa);
      g += kGU;
    }
  }
  for (; g < ngrp; ++g) {
    const int4 q = pre4[g * BS_WAVE];
    const int32_t iv[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (on(iv[e])) acc += kHet ? sell_w[beg + (g * BS_WAVE + lane) * 4 + e] : w_homo;
  }
  const int64_t j = slice * BS_WAVE + lane;
  if (j < n_post) out[j] = acc;
}

// Fused event mat-vec straight from the spike vector: workgroup w owns pre rows
// [w*rows, (w+1)*rows); it compacts its active rows into LDS (wave ballots), then adds the
// synapses of those rows.  If the whole output fits in LDS (n_post <= kLdsPosts) and the
// workgroup has at least kLdsRatio events per output, the events of per-synapse weights are
// first aggregated with LDS atomics and each touched output receives one global atomic;
// otherwise every event is one global atomic.  The choice is made per workgroup from its own
// event count.
constexpr int kLdsPosts = 16384;
constexpr int kLdsRatio = 4;
constexpr int kRowsCap = 1024;

// kVal: each event is weighted by its spike value (sum_i x[i] * w[i,k]); otherwise by 1.
// Batched: blockIdx.y selects the batch row (spike row b at spk + b * n_pre, output row at
// out + b * n_post); the connectivity is shared by every row.
template <typename T, bool kCsr, bool kHet, bool kVal = false>
__global__ __launch_bounds__(kBlock) void k_matvec(const T* __restrict__ spk, int32_t n_pre,
                                                   int32_t rows, const int32_t* __restrict__ indptr,
                                                   const int32_t* __restrict__ indices, int32_t k,
                                                   const float* __restrict__ w, float w_homo,
                                                   int32_t n_post, float* __restrict__ out) {
  spk += (int64_t)blockIdx.y * n_pre;
  out += (int64_t)blockIdx.y * n_post;
  __shared__ int32_t s_rows[kRowsCap];
  __shared__ int32_t s_wave[kBlock / BS_WAVE];
  __shared__ int32_t s_nev;
  extern __shared__ float s_acc[];
  const int lane = bs_lane();
  const int wid = threadIdx.x / BS_WAVE;
  const int64_t r0 = (int64_t)blockIdx.x * rows;
  int32_t count = 0;
  for (int32_t off = 0; off < rows; off += kBlock) {
    const int64_t r = r0 + off + threadIdx.x;
    const bool a = off + (int32_t)threadIdx.x < rows && r < n_pre && spk[r] != T(0);
    const uint64_t m = bs_ballot(a);
    if (lane == 0) s_wave[wid] = __popcll(m);
    __syncthreads();
    int32_t pos = count, tot = 0;
#pragma unroll
    for (int v = 0; v < kBlock / BS_WAVE; ++v) {
      pos += v < wid ? s_wave[v] : 0;
      tot += s_wave[v];
    }
    if (a) s_rows[pos + bs_rank_below(m)] = (int32_t)r;
    count += tot;
    __syncthreads();
  }
  if (count == 0) return;
  // events of this workgroup
  if (threadIdx.x == 0) {
    int64_t ev = 0;
    if (!kCsr) {
      ev = (int64_t)count * k;
    } else {
      for (int32_t i = 0; i < count; ++i) ev += indptr[s_rows[i] + 1] - indptr[s_rows[i]];
    }
    s_nev = ev > 0x7FFFFFFF ? 0x7FFFFFFF : (int32_t)ev;
  }
  __syncthreads();
  // Homogeneous weights always go direct: sums of one repeated value are order-free and exact
  // only as a single chain of +w, which LDS partial sums would break.
  const bool use_lds =
      (kHet || kVal) && n_post <= kLdsPosts && (int64_t)s_nev >= (int64_t)kLdsRatio * n_post;
  if (use_lds) {
    for (int32_t j = threadIdx.x; j < n_post; j += kBlock) s_acc[j] = 0.0f;
    __syncthreads();
  }
  const int32_t nnz = kCsr ? indptr[n_pre] : 0;
  for (int32_t a = wid; a < count; a += kBlock / BS_WAVE) {  // one wave per active row
    const int32_t row = s_rows[a];
    const float xv = kVal ? (float)spk[row] : 1.0f;
    int64_t beg, end;
    if (kCsr) {
      beg = indptr[row];
      end = indptr[row + 1];
      beg = beg < 0 ? 0 : beg;
      end = end > nnz ? nnz : end;
    } else {
      beg = (int64_t)row * k;
      end = beg + k;
    }
    for (int64_t s = beg + lane; s < end; s += BS_WAVE) {
      const int32_t j = indices[s];
      const float v = kVal ? (kHet ? w[s] : w_homo) * xv : (kHet ? w[s] : w_homo);
      if ((uint32_t)j < (uint32_t)n_post) {
        if (use_lds) atomicAdd(&s_acc[j], v);
        else bs_atomic_add_f32(out + j, v);
      }
    }
  }
  if (use_lds) {
    __syncthreads();
    for (int32_t j = threadIdx.x; j < n_post; j += kBlock) {
      const float v = s_acc[j];
      if (v != 0.0f) bs_atomic_add_f32(out + j, v);
    }
  }
}

// The mat-vec (fixed fan-out) with the sums in LDS instead of global fp32 atomics, which run at
// ~2e10/s over the whole chip.  Workgroup (range q, row group r) of batch row blockIdx.y lists
// its active rows, reads all their synapses and adds those that hit its `len` posts; with one
// row group it writes the outputs, else a partial row that k_mv_finish adds (header, then
// [R][n_post] per batch row).  As in the bucketed operator, the row groups in use follow the
// spikes: every workgroup estimates the active synapses from the same spikes (the leading ones
// of every batch row), groups past R_eff return, and R_eff = 1 writes the outputs.  When the
// estimate says that atomics are the faster way for so few events (MvCost), the workgroups
// clear the outputs instead, R_eff is 0 and k_mv_finish adds the events.
// A shared event weight is counted and added in one chain afterwards (the sequential sum, as
// k_matvec and the bucketed operator give it); other sums are fp32 in no fixed order.
// The workgroups of a row group read the same synapses: they are placed on one XCD.
// Bound by the LDS fp32 adds (84 instead of 112 us with integer ones) and the re-reads of the
// synapses by every range.
constexpr int kMvB = 1024;
constexpr int kMvPosts = 16000;        // posts per range at most (two workgroups per CU)
constexpr int kMvSpan = 4096;          // rows listed at a time
constexpr int kMvSample = 4096;        // spikes the estimate reads: one load per thread
constexpr int kMvSyn = 8192;           // active synapses per row group the estimate aims for,
                                       // plus n_post / 4 (a group's partials cost that much)
constexpr int kMvHdr = 64;             // header words ahead of a batch row's partials

// Costs in us of the two ways, from the events ev of a batch row (filled in by mv_plan).
struct MvCost {
  int32_t R, rs;       // row groups at most, and with one span of rows each
  float per;           // events of a batch row per spike of the sample
  float group;         // 1 / events a row group aims for
  float direct0, direct1, lds0, span, last, read, part;
  // row groups for ev events: no group lists more than one span of rows if R allows
  __host__ __device__ int32_t groups(float ev) const {
    const int32_t re = (int32_t)fminf(ceilf(ev * group), (float)R);
    const int32_t g = re > rs ? re : rs;
    return g > R ? R : g;
  }
  // atomics: a rate; LDS: spans of rows listed one after another, then the synapses of a
  // group's events, then its partial sums
  __host__ __device__ float direct_us(float ev) const { return direct0 + ev * direct1; }
  __host__ __device__ float lds_us(float ev, int32_t g) const {
    return lds0 + (g >= rs ? span : last) + read * (ev / (float)g) +
           (g > 1 ? (float)g * part : 0.0f);
  }
};

// Batch rows the estimate reads with `sample` threads, kE spikes each, on one of them.
__host__ __device__ __forceinline__ int32_t mv_sample_rows(int32_t sample, int32_t kE) {
  const int32_t n = kMvSample / kE / sample;
  return n < 1 ? 1 : n;
}

struct __attribute__((packed, aligned(1))) Any16 {
  uint4 v;
};

// Nonzero ones among 16 bytes of spikes.
template <typename T>
__device__ __forceinline__ int32_t nonzeros(uint4 v) {
  const uint32_t x[4] = {v.x, v.y, v.z, v.w};
  int32_t c = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (sizeof(T) == 4) c += (x[e] & 0x7fffffffu) != 0u;
    else c += __popc((((x[e] & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x[e]) & 0x80808080u);
  }
  return c;
}

template <typename T, bool kHet, bool kVal>
__global__ __launch_bounds__(kMvB) void k_mv_lds(
    const T* __restrict__ spk, int32_t n_pre, const int32_t* __restrict__ indices, int32_t k,
    const float* __restrict__ w, float w_homo, int32_t n_post, int32_t nr, int32_t len,
    int32_t R, int32_t sample, MvCost cost, int32_t accumulate, float* __restrict__ out,
    uint32_t* __restrict__ ws) {
  constexpr bool kCount = !kHet && !kVal;
  constexpr int kWv = kMvB / BS_WAVE, kU = kMvSpan / kMvB;
  __shared__ __align__(16) uint32_t s_acc[kMvPosts];
  __shared__ int32_t s_list[kMvSpan];
  __shared__ int32_t s_wave[kU][kWv];
  const int lane = bs_lane();
  const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / BS_WAVE));
  const T* all = spk;
  spk += (int64_t)blockIdx.y * n_pre;
  out += (int64_t)blockIdx.y * n_post;
  ws += (int64_t)blockIdx.y * (kMvHdr + (R > 1 ? (int64_t)R * n_post : 0));
  // workgroup x -> (r, q): the ranges of a row group share x mod 8, the XCD
  const int32_t x = blockIdx.x;
  const int32_t r = R == 1 ? 0 : x / (8 * nr) * 8 + x % 8, q = R == 1 ? x : x / 8 % nr;
  if (r >= R) return;
  const int32_t p0 = q * len;
  const int32_t rest = n_post - p0 > 0 ? n_post - p0 : 0;     // 0: a last range left empty
  const int32_t pn = rest < len ? rest : len;
  int32_t Reff = 1;
  if (sample > 0) {                    // threads per batch row, 16 bytes of its spikes each
    constexpr int32_t kE = 16 / sizeof(T);
    const int32_t b = (int32_t)threadIdx.x / sample, i = (int32_t)threadIdx.x % sample * kE;
    int32_t c = 0;
    if (b < (int32_t)gridDim.y && b < mv_sample_rows(sample, kE)) {
      const T* p = all + (int64_t)b * n_pre;
      if (i + kE <= n_pre) c = nonzeros<T>(((const Any16*)(p + i))->v);
      else for (int32_t e = i; e < n_pre; ++e) c += p[e] != T(0) ? 1 : 0;
    }
#pragma unroll
    for (int o = BS_WAVE / 2; o > 0; o >>= 1) c += __shfl_xor(c, o);
    if (lane == 0) s_wave[0][wid] = c;
    __syncthreads();
    c = 0;
#pragma unroll
    for (int v = 0; v < kWv; ++v) c += s_wave[0][v];
    __syncthreads();
    const float ev = (float)c * cost.per;               // the same in every workgroup, so all
                                                        // batch rows take the same way
    Reff = cost.groups(ev);
    if (cost.direct_us(ev) < cost.lds_us(ev, Reff)) Reff = 0;
    if (x == 0 && threadIdx.x == 0) ws[0] = (uint32_t)Reff;
    if (Reff == 0) {                   // this workgroup's share of its range cleared
      if (accumulate) return;
      const int32_t j0 = (int32_t)((int64_t)pn * r / R), j1 = (int32_t)((int64_t)pn * (r + 1) / R);
      for (int32_t j = j0 + threadIdx.x; j < j1; j += kMvB) out[p0 + j] = 0.0f;
      return;
    }
    if (r >= Reff) return;             // whole workgroup
  }
  for (int j = threadIdx.x; j < pn; j += kMvB) s_acc[j] = 0u;
  const int64_t r0 = (int64_t)n_pre * r / Reff, r1 = (int64_t)n_pre * (r + 1) / Reff;
  T next[kU];                          // the next span's spikes, in flight over this one's rows
  auto ahead = [&](int64_t c0) {
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int64_t i = c0 + u * kMvB + threadIdx.x;
      next[u] = spk[i < r1 ? i : r0];  // repeated past the end
    }
  };
  if (r0 < r1) ahead(r0);
  for (int64_t c0 = r0; c0 < r1; c0 += kMvSpan) {
    uint64_t m[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      m[u] = bs_ballot(c0 + u * kMvB + threadIdx.x < r1 && next[u] != T(0));
      if (lane == 0) s_wave[u][wid] = __popcll(m[u]);
    }
    if (c0 + kMvSpan < r1) ahead(c0 + kMvSpan);
    __syncthreads();                   // also: s_acc is zero, the last span's rows are done
    int32_t count = 0;
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      int32_t pos = count;
#pragma unroll
      for (int v = 0; v < kWv; ++v) {
        const int32_t n = s_wave[u][v];
        pos += v < wid ? n : 0;
        count += n;
      }
      if ((m[u] >> lane) & 1ull)
        s_list[pos + bs_rank_below(m[u])] = (int32_t)(c0 + u * kMvB + threadIdx.x);
    }
    __syncthreads();
    // eight 64-synapse chunks in flight per wave: two of each of four rows, or, when that would
    // leave waves without rows, eight of one
    auto rows = [&](auto nrow) {
      constexpr int kRows = decltype(nrow)::value, kPass = 8 / kRows;
      for (int32_t a0 = wid * kRows; a0 < count; a0 += kWv * kRows) {
        int32_t row[kRows];
        float xv[kRows];
#pragma unroll
        for (int e = 0; e < kRows; ++e) {
          row[e] = __builtin_amdgcn_readfirstlane(s_list[a0 + e < count ? a0 + e : a0]);
          xv[e] = kVal ? (float)spk[row[e]] : 1.0f;
        }
        for (int32_t t0 = 0; t0 < k; t0 += kPass * BS_WAVE) {
          int32_t jj[kRows][kPass];
          float vv[kRows][kPass];
#pragma unroll
          for (int e = 0; e < kRows; ++e)
#pragma unroll
            for (int u = 0; u < kPass; ++u) {
              const int32_t t = t0 + u * BS_WAVE + lane;
              const bool ok = t < k && a0 + e < count;
              const int64_t o = (int64_t)row[e] * k + t;
              jj[e][u] = ok ? indices[o] : -1;
              vv[e][u] = kHet && ok ? w[o] : w_homo;
            }
#pragma unroll
          for (int e = 0; e < kRows; ++e)
#pragma unroll
            for (int u = 0; u < kPass; ++u) {
              const uint32_t j = (uint32_t)jj[e][u] - (uint32_t)p0;
              if (jj[e][u] >= 0 && j < (uint32_t)pn) {
                if (kCount) atomicAdd(&s_acc[j], 1u);
                else unsafeAtomicAdd((float*)&s_acc[j], kVal ? vv[e][u] * xv[e] : vv[e][u]);
              }
            }
        }
      }
    };
    if (count <= 3 * kWv) rows(std::integral_constant<int, 1>());
    else rows(std::integral_constant<int, 4>());
    __syncthreads();                   // the list is rewritten next
  }
  __syncthreads();                     // a group without rows: s_acc is zero
  if (Reff > 1) {
    uint32_t* dst = ws + kMvHdr + (int64_t)r * n_post + p0;
    for (int j = threadIdx.x; j < pn; j += kMvB) dst[j] = s_acc[j];
    return;
  }
  for (int j = threadIdx.x; j < pn; j += kMvB) {
    float acc = accumulate ? out[p0 + j] : 0.0f;
    if (kCount) {
      const uint32_t c = s_acc[j];
      for (uint32_t u = 0; u < c; ++u) acc += w_homo;
    } else {
      acc += __uint_as_float(s_acc[j]);
    }
    out[p0 + j] = acc;
  }
}

// R_eff > 1: out[j] = (accumulate ? out[j] : 0) + the R_eff partials of j.  A workgroup takes 64
// posts; thread (c, j) adds every fourth partial from c on, 16 in flight, and the four sums meet
// in order.  R_eff = 0: a workgroup lists the active ones of its `rows` pre rows and adds their
// synapses to the outputs with global atomics, a wave 4 x 64 of one row at a time (k_matvec
// gives a wave the whole row: 12.1 us for 12 rows of 1,000 synapses, 10.0 here for both launches).
template <typename T, bool kHet, bool kVal>
__global__ __launch_bounds__(kBlock) void k_mv_finish(
    const T* __restrict__ spk, int32_t n_pre, int32_t rows, const int32_t* __restrict__ indices,
    int32_t k, const float* __restrict__ w, int32_t n_post, int32_t R, float w_homo,
    int32_t accumulate, const uint32_t* __restrict__ ws, float* __restrict__ out) {
  constexpr bool kCount = !kHet && !kVal;
  constexpr int kC = kBlock / BS_WAVE, kF = 16, kQ = 4;
  __shared__ uint32_t s_p[kC][BS_WAVE];
  __shared__ int32_t s_rows[kRowsCap];
  const int c = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / BS_WAVE)), lane = bs_lane();
  ws += (int64_t)blockIdx.y * (kMvHdr + (R > 1 ? (int64_t)R * n_post : 0));
  out += (int64_t)blockIdx.y * n_post;
  const int32_t Reff = (int32_t)__builtin_amdgcn_readfirstlane(ws[0]);
  if (Reff == 0) {
    spk += (int64_t)blockIdx.y * n_pre;
    const int64_t r0 = (int64_t)blockIdx.x * rows;
    int32_t count = 0;
    for (int32_t off = 0; off < rows; off += kBlock) {
      const int64_t r = r0 + off + threadIdx.x;
      const bool a = off + (int32_t)threadIdx.x < rows && r < n_pre && spk[r] != T(0);
      const uint64_t m = bs_ballot(a);
      if (lane == 0) s_p[c][0] = (uint32_t)__popcll(m);
      __syncthreads();
      int32_t pos = count;
#pragma unroll
      for (int v = 0; v < kC; ++v) {
        const int32_t n = (int32_t)s_p[v][0];
        pos += v < c ? n : 0;
        count += n;
      }
      if (a) s_rows[pos + bs_rank_below(m)] = (int32_t)r;
      __syncthreads();
    }
    const int32_t per = (k - 1) / (kQ * BS_WAVE) + 1;        // items of a row
    for (int32_t a = 0, q = c;; q += kC) {                   // item q of active row a
      while (q >= per && a < count) {
        q -= per;
        ++a;
      }
      if (a >= count) break;
      const int32_t row = __builtin_amdgcn_readfirstlane(s_rows[a]);
      const float xv = kVal ? (float)spk[row] : 1.0f;
      const int32_t t0 = q * (kQ * BS_WAVE) + lane;
      int32_t jj[kQ];
      float vv[kQ];
#pragma unroll
      for (int u = 0; u < kQ; ++u) {
        const int32_t t = t0 + u * BS_WAVE;
        const int64_t o = (int64_t)row * k + t;
        jj[u] = t < k ? indices[o] : -1;
        vv[u] = kHet && t < k ? w[o] : w_homo;
      }
#pragma unroll
      for (int u = 0; u < kQ; ++u)
        if ((uint32_t)jj[u] < (uint32_t)n_post)
          bs_atomic_add_f32(out + jj[u], kVal ? vv[u] * xv : vv[u]);
    }
    return;
  }
  const int64_t j = (int64_t)blockIdx.x * BS_WAVE + lane;
  if (Reff == 1 || (int64_t)blockIdx.x * BS_WAVE >= n_post) return;
  const uint32_t* p = ws + kMvHdr + (j < n_post ? j : 0);
  float sum = 0.0f;
  uint32_t cnt = 0;
  for (int32_t g = c; g < Reff; g += kC * kF) {
    uint32_t v[kF];
#pragma unroll
    for (int u = 0; u < kF; ++u)
      v[u] = g + u * kC < Reff ? p[(int64_t)(g + u * kC) * n_post] : 0u;
#pragma unroll
    for (int u = 0; u < kF; ++u) {
      if (kCount) cnt += v[u];
      else sum += __uint_as_float(v[u]);
    }
  }
  s_p[c][lane] = kCount ? cnt : __float_as_uint(sum);
  __syncthreads();
  if (c != 0 || j >= n_post) return;
  float acc = accumulate ? out[j] : 0.0f;
  if (kCount) {
    cnt = s_p[0][lane] + s_p[1][lane] + s_p[2][lane] + s_p[3][lane];
    for (uint32_t u = 0; u < cnt; ++u) acc += w_homo;
  } else {
    sum = __uint_as_float(s_p[0][lane]);
    for (int u = 1; u < kC; ++u) sum += __uint_as_float(s_p[u][lane]);
    acc += sum;
  }
  out[j] = acc;
}

// gw[0] += the sum over the workgroup's waves of their (wave-uniform) v: one atomic per
// workgroup.  The terms of this one sum mostly cancel, so it is carried in 64 bits over the rows
// of a workgroup (a row's own sum of g is formed as the kernel forms grad_x, and the workgroups'
// sums meet in fp32).  Called by every wave that has not ended.  (One fp32 atomic per active
// row made the shared weight's gradient of 100k rows of 128 synapses take 1.27 ms, and that of
// two batch rows of 100k x 100 take 266 us; 91 this way.)
template <int kWaves>
__device__ __forceinline__ void block_atomic_sum(double v, float* gw) {
  __shared__ double s_v[kWaves];
  const int wid = threadIdx.x / BS_WAVE;
  if (bs_lane() == 0) s_v[wid] = v;
  __syncthreads();
  if (threadIdx.x != 0) return;
  double t = s_v[0];
  for (int u = 1; u < kWaves; ++u) t += s_v[u];
  if (t != 0.0) bs_atomic_add_f32(gw, (float)t);
}

constexpr int kVjpU = 8;  // 64-synapse chunks per wave and round in k_matvec_vjp

// Reverse mode of the event mat-vec y[j] = sum_{i,k: idx[i,k]=j} x[i] * w[i,k] (x = spike
// value; 1 for byte spikes): one wave per pre row i gathers g[idx[i,k]] over the row and
//   grad_x[i]   = sum_k w[i,k] * g[idx[i,k]]            (lane partials, then a wave sum)
//   grad_w[i,k] = x[i] * g[idx[i,k]]                    (per-synapse weights)
//   grad_w[0]  += x[i] * sum_k g[idx[i,k]]              (homogeneous weight)
// Synapses with out-of-range targets contribute nothing, as in the forward pass.
template <typename T, bool kCsr, bool kHet>
__global__ __launch_bounds__(kBlock) void k_matvec_vjp(const T* __restrict__ spk, int32_t n_pre,
                                                       const int32_t* __restrict__ indptr,
                                                       const int32_t* __restrict__ indices,
                                                       int32_t k, const float* __restrict__ w,
                                                       float w_homo, int32_t n_post,
                                                       const float* __restrict__ g,
                                                       float* __restrict__ gx,
                                                       float* __restrict__ gw) {
  const int lane = bs_lane();
  const int64_t nw = (int64_t)gridDim.x * (kBlock / BS_WAVE);
  const int32_t nnz = kCsr ? indptr[n_pre] : 0;
  double sw = 0.0;
  for (int64_t row = ((int64_t)blockIdx.x * kBlock + threadIdx.x) / BS_WAVE; row < n_pre;
       row += nw) {
    int64_t beg, end;
    if (kCsr) {
      beg = indptr[row];
      end = indptr[row + 1];
      beg = beg < 0 ? 0 : beg;
      end = end > nnz ? nnz : end;
    } else {
      beg = row * k;
      end = beg + k;
    }
    const float xv = (float)spk[row];
    float sx = 0.0f, sg = 0.0f;
    // kVjpU chunks of 64 synapses per round, every index, weight and gathered g of the round
    // loaded before any is added (one dependent pair of round trips per round instead of one
    // per chunk); each lane still adds its synapses in ascending order (100k x 100k, K = 1000:
    // 774 -> 712 us; what remains is ~1e8 random 4-byte gathers of g from L2 per call)
    for (int64_t s0 = beg + lane; s0 < end; s0 += BS_WAVE * kVjpU) {
      int32_t jj[kVjpU];
      float wv[kVjpU], gj[kVjpU];
#pragma unroll
      for (int u = 0; u < kVjpU; ++u) {
        const int64_t s = s0 + (int64_t)u * BS_WAVE;
        jj[u] = s < end ? indices[s] : -1;
        wv[u] = kHet && gx && s < end ? w[s] : w_homo;
      }
#pragma unroll
      for (int u = 0; u < kVjpU; ++u) gj[u] = (uint32_t)jj[u] < (uint32_t)n_post ? g[jj[u]] : 0.0f;
#pragma unroll
      for (int u = 0; u < kVjpU; ++u) {
        const int64_t s = s0 + (int64_t)u * BS_WAVE;
        if (s < end) {
          if (gx) sx += wv[u] * gj[u];
          if (kHet && gw) gw[s] = xv * gj[u];
          sg += gj[u];
        }
      }
    }
#pragma unroll
    for (int o = BS_WAVE / 2; o > 0; o >>= 1) {
      sx += __shfl_xor(sx, o);
      sg += __shfl_xor(sg, o);
    }
    if (lane == 0 && gx) gx[row] = sx;
    if (!kHet && xv != 0.0f) sw += (double)xv * (double)sg;
  }
  if (!kHet && gw) block_atomic_sum<kBlock / BS_WAVE>(sw, gw);
}

// Sum over the wave in k_matvec_vjp's order (lane l with l ^ 32, then 16, 8, 4, 2, 1): after the
// exchange at distance 8 the values repeat every 8 lanes, so a rotation by 4 inside 16 lanes
// meets the same value as the exchange at distance 4.
__device__ __forceinline__ float wave_sum_xor(float v) {
  v += __shfl_xor(v, 32);
  v += __shfl_xor(v, 16);
#define BS_DPP(x, ctrl) \
  __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), ctrl, 0xF, 0xF, true))
  v += BS_DPP(v, 0x128);  // row_ror:8
  v += BS_DPP(v, 0x124);  // row_ror:4
  v += BS_DPP(v, 0x4E);   // quad_perm [2, 3, 0, 1]
  v += BS_DPP(v, 0xB1);   // quad_perm [1, 0, 3, 2]
#undef BS_DPP
  return v;
}

// The same gradients (fixed fan-out) with g read from LDS.  A gather of g from L2 moves a whole
// 128-byte line for 4 bytes, which holds k_matvec_vjp at ~2e11 gathers/s, fewer when the
// synapses come from HBM.  Here one workgroup per compute unit streams the synapses of its
// rows while ranges of kLvR posts of g pass through two LDS buffers: 4 waves load the next
// range into one buffer while 12 waves pick the values of their targets out of the other, with
// one barrier per range.  Each of the 12 waves holds kLvS chunks of 64 synapses at a time --
// kLvS / CP rows of CP chunks, or 16 chunks of a longer row -- with the next pass's indices
// and this pass's weights in flight.  An index outside the range reads the zero slot behind
// it; at most one range holds a target, so OR-ing the bits of all ranges is exact.  Up to two
// ranges stay in LDS for the whole launch.
// Loads and stores of a pass are unconditional (lanes past the row's end repeat its last
// synapse, rows past the wave's last repeat that row, with the same values), so that the wait
// for the next indices counts only what was issued after them.
// Every row is summed as k_matvec_vjp sums it, bit for bit.
constexpr int kLvB = 1024;
constexpr int kLvR = 20416;                       // posts per range (two ranges fill LDS)
template <typename T, int CP, bool kHet, bool kGw, bool kMulti>
__global__ __launch_bounds__(kLvB) void k_matvec_vjp_lds(
    const T* __restrict__ spk, int32_t n_pre, const int32_t* __restrict__ indices, int32_t k,
    const float* __restrict__ w, float w_homo, int32_t n_post, const float* __restrict__ g,
    float* __restrict__ gx, float* __restrict__ gw) {
  constexpr int kLvS = kMulti ? 32 : 16;              // chunks per wave and pass
  constexpr int kLvW = kMulti ? 12 : 16;              // waves that own rows
  constexpr int kLvF = kMulti ? 256 : kLvB;           // threads that fill LDS (the last ones)
  constexpr int kR = kLvS / CP;                       // rows per pass
  __shared__ __align__(16) uint32_t s_g[2][kLvR + 16];  // [kLvR]: the zero slot
  const int lane = bs_lane();
  const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / BS_WAVE));
  const int64_t nw = (int64_t)gridDim.x * kLvW;
  const int32_t nblk = (k + CP * BS_WAVE - 1) / (CP * BS_WAVE);  // > 1 only for CP = 16
  // the same number of passes in every wave: the ranges change at barriers
  const int32_t passes = (int32_t)(((n_pre + nw - 1) / nw + kR - 1) / kR) * nblk;
  const int32_t nr = (n_post + kLvR - 1) / kLvR;      // at most 2 unless kMulti
  // range q by kLvF threads: into registers (16-byte loads, all in flight), then to s_g[buf]
  constexpr int kU = (kLvR / 4 + kLvF - 1) / kLvF;
  static_assert(4 * kU * kLvF >= kLvR + 4, "the zero slot is written with its range");
  const bool al = ((uintptr_t)g & 15) == 0;
  auto length = [&](int32_t q) { return n_post - q * kLvR < kLvR ? n_post - q * kLvR : kLvR; };
  auto load = [&](int32_t q, int tid, uint4 (&v)[kU], uint32_t (&tail)[3]) {
    const int32_t len = length(q), len4 = len & ~3;
    const uint32_t* p = (const uint32_t*)g + (int64_t)q * kLvR;
    if (!al || len4 == 0) return;                     // store() reads g itself
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int i = 4 * (tid + u * kLvF);
      v[u] = *(const uint4*)(p + (i < len4 ? i : len4 - 4));
    }
#pragma unroll
    for (int e = 0; e < 3; ++e) tail[e] = p[len4 + e < len ? len4 + e : len - 1];
  };
  auto store = [&](int32_t q, int buf, int tid, const uint4 (&v)[kU], const uint32_t (&tail)[3]) {
    const int32_t len = length(q), len4 = len & ~3;
    if (!al || len4 == 0) {
      const uint32_t* p = (const uint32_t*)g + (int64_t)q * kLvR;
      for (int i = tid; i < kLvR + 16; i += kLvF) s_g[buf][i] = i < len ? p[i] : 0u;
      return;
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int i = 4 * (tid + u * kLvF);
      const bool full = i < len4, cut = i == len4;
      uint4 x;
      x.x = full ? v[u].x : (cut && len4 < len ? tail[0] : 0u);
      x.y = full ? v[u].y : (cut && len4 + 1 < len ? tail[1] : 0u);
      x.z = full ? v[u].z : (cut && len4 + 2 < len ? tail[2] : 0u);
      x.w = full ? v[u].w : 0u;
      if (i < kLvR + 16) *(uint4*)(s_g[buf] + i) = x;
    }
  };
  // compute units of one XCD start at different ranges, so that they do not all read the same
  // lines of g at once
  const int32_t q0 = kMulti ? (int32_t)((blockIdx.x / 8) % nr) : 0;
  if (kLvF == kLvB || wid >= kLvW) {  // the filling waves
    const int tid = (int)threadIdx.x - (kLvB - kLvF);
    uint4 v[kU];
    uint32_t tail[3];
    int32_t q = q0;
    load(q, tid, v, tail);
    store(q, 0, tid, v, tail);
    if constexpr (!kMulti) {
      if (nr == 2) {
        load(1, tid, v, tail);
        store(1, 1, tid, v, tail);
      }
    } else {
      // step t reads range q0 + t (mod nr) from s_g[t & 1]; the next one is stored meanwhile,
      // and the one after it is on its way across the barrier
      const int64_t steps = (int64_t)passes * nr;
      auto ahead = [&](int64_t t) {
        q = q + 1 == nr ? 0 : q + 1;
        if (t < steps) load(q, tid, v, tail);
      };
      ahead(1);
      __syncthreads();
      for (int64_t t = 0; t < steps; ++t) {
        if (t + 1 < steps) store(q, (int)((t + 1) & 1), tid, v, tail);
        ahead(t + 2);
        __syncthreads();
      }
      if (!kHet && gw) block_atomic_sum<kLvB / BS_WAVE>(0.0, gw);
      return;
    }
  }
  __syncthreads();
  const int64_t wv = (int64_t)blockIdx.x * kLvW + wid;
  const int64_t r0 = n_pre * wv / nw;                 // this wave's rows [r0, r0 + rows)
  const int32_t rows = (int32_t)(n_pre * (wv + 1) / nw - r0);
  const int32_t lastr = rows > 0 ? rows - 1 : 0;      // repeated past the end (r0 < n_pre)
  auto rowat = [&](int32_t r) -> int64_t { return (r0 + (r < lastr ? r : lastr)) * k; };
  // byte offset in its row of this lane's synapse in chunk c of a block that starts at kb
  auto syn = [&](int32_t kb, int c, int ln) -> uint32_t {
    const int32_t t = kb + c * BS_WAVE + ln;
    return (uint32_t)(t < k ? t : k - 1) * 4u;
  };
  // the lane number, hidden from the compiler: it would keep the offsets of one walk over the
  // chunks for the next and spill
  auto hidden = [&]() {
    int ln = lane;
    asm volatile("" : "+v"(ln));
    return ln;
  };
  auto rd = [](const void* p, uint32_t off) { return *(const uint32_t*)((const char*)p + off); };
  uint32_t jj[kLvS];
  auto load_idx = [&](int32_t r, int32_t b) {
    const int ln = hidden();
#pragma unroll
    for (int s = 0; s < kLvS; ++s) jj[s] = rd(indices + rowat(r + s / CP), syn(b, s % CP, ln));
  };
  load_idx(0, 0);
  float cx[kR], cg[kR];                               // lane sums carried over a row's blocks
  double sw = 0.0;
  int32_t row = 0, kb = 0;                            // this pass: rows row .. row + kR - 1
  int step = 0;
  for (int32_t pass = 0; pass < passes; ++pass) {
    uint32_t gj[kLvS];
    float wt[kLvS];
    // lane r: the spike value of row r of the pass
    const float xl = (float)spk[r0 + (row + lane < lastr ? row + lane : lastr)];
#pragma unroll
    for (int s = 0; s < kLvS; ++s) {
      jj[s] = (jj[s] < (1u << 29) ? jj[s] : 1u << 29) * 4u;   // byte offset in g
      gj[s] = 0u;
    }
    for (int32_t qq = 0, q = q0; qq < nr; ++qq, q = q + 1 == nr ? 0 : q + 1) {
      const uint32_t lo = (uint32_t)q * kLvR * 4u;
      const char* sgp = (const char*)s_g[kMulti ? step & 1 : q];
      if (qq + 1 == nr) {                             // weights: in flight during the last range
        const int ln = hidden();
#pragma unroll
        for (int s = 0; s < kLvS; ++s)
          wt[s] = kHet ? __uint_as_float(rd(w + rowat(row + s / CP), syn(kb, s % CP, ln)))
                       : w_homo;
      }
#pragma unroll
      for (int s = 0; s < kLvS; ++s) {
        const uint32_t u = jj[s] - lo;
        gj[s] |= *(const uint32_t*)(sgp + (u < kLvR * 4u ? u : kLvR * 4u));
      }
      ++step;
      if (kMulti) __syncthreads();
    }
    // the next pass's indices (past the end: the last row's again), in flight from here
    const bool wrap = CP < 16 || kb + CP * BS_WAVE >= k;
    const int32_t nrow = wrap ? row + kR : row, nkb = wrap ? 0 : kb + CP * BS_WAVE;
    load_idx(nrow, nkb);
    const int ln = hidden();
#pragma unroll
    for (int r = 0; r < kR; ++r) {
      const float xv = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(xl), r));
      float sx = kb ? cx[r] : 0.0f, sg = kb ? cg[r] : 0.0f;
#pragma unroll
      for (int c = 0; c < CP; ++c) {
        const float gv = __uint_as_float(gj[r * CP + c]);
        const bool in = kb + c * BS_WAVE + ln < k;
        if (kGw) *(float*)((char*)(gw + rowat(row + r)) + syn(kb, c, ln)) = xv * gv;
        sx += in ? wt[r * CP + c] * gv : 0.0f;
        if (!kHet) sg += in ? gv : 0.0f;
      }
      if (CP == 16) {
        cx[r] = sx;
        cg[r] = sg;
      }
      if (wrap) {
        const bool own = row + r < rows;
        const float vx = wave_sum_xor(sx);
        if (gx && own && lane == 0) gx[r0 + row + r] = vx;
        if (!kHet && own && xv != 0.0f) sw += (double)xv * (double)wave_sum_xor(sg);
      }
    }
    row = nrow;
    kb = nkb;
  }
  if (!kHet && gw) block_atomic_sum<kLvB / BS_WAVE>(sw, gw);
}

// The same gradients for B batch rows in one launch (spk [B, n_pre], g [B, n_post]): one wave
// per pre row i, the row's synapses read once per batch row (from cache after the first):
//   grad_x[b, i] as k_matvec_vjp forms it for row b (lane partials, then a wave sum);
//   grad_w[i, k] = sum_b x[b, i] * g[b, idx[i, k]], the products added in b order, as adding
//   the per-row gradients one after another does (fp32, no contraction);
//   homogeneous: grad_w[0] += x[b, i] * sum_k g[b, idx[i, k]], summed over (row, b) in 64 bits.
template <typename T, bool kCsr, bool kHet>
__global__ __launch_bounds__(kBlock) void k_matvec_vjp_batch(
    const T* __restrict__ spk, int32_t batch, int32_t n_pre, const int32_t* __restrict__ indptr,
    const int32_t* __restrict__ indices, int32_t k, const float* __restrict__ w, float w_homo,
    int32_t n_post, const float* __restrict__ g, float* __restrict__ gx,
    float* __restrict__ gw) {
  const int lane = bs_lane();
  const int64_t nw = (int64_t)gridDim.x * (kBlock / BS_WAVE);
  const int32_t nnz = kCsr ? indptr[n_pre] : 0;
  double sw = 0.0;
  for (int64_t row = ((int64_t)blockIdx.x * kBlock + threadIdx.x) / BS_WAVE; row < n_pre;
       row += nw) {
    int64_t beg, end;
    if (kCsr) {
      beg = indptr[row];
      end = indptr[row + 1];
      beg = beg < 0 ? 0 : beg;
      end = end > nnz ? nnz : end;
    } else {
      beg = row * k;
      end = beg + k;
    }
    for (int32_t b = 0; b < batch; ++b) {
      const float xv = (float)spk[(int64_t)b * n_pre + row];
      const float* gb = g + (int64_t)b * n_post;
      float sx = 0.0f, sg = 0.0f;
      for (int64_t s = beg + lane; s < end; s += BS_WAVE) {
        const int32_t j = indices[s];
        const float gj = (uint32_t)j < (uint32_t)n_post ? gb[j] : 0.0f;
        if (gx) sx += (kHet ? w[s] : w_homo) * gj;
        sg += gj;
      }
#pragma unroll
      for (int o = BS_WAVE / 2; o > 0; o >>= 1) {
        sx += __shfl_xor(sx, o);
        sg += __shfl_xor(sg, o);
      }
      if (lane == 0 && gx) gx[(int64_t)b * n_pre + row] = sx;
      if (!kHet && xv != 0.0f) sw += (double)xv * (double)sg;
    }
    if (kHet && gw) {
      for (int64_t s = beg + lane; s < end; s += BS_WAVE) {
        const int32_t j = indices[s];
        float acc = 0.0f;
        for (int32_t b = 0; b < batch; ++b) {
          const float gj = (uint32_t)j < (uint32_t)n_post ? g[(int64_t)b * n_post + j] : 0.0f;
          const float prod = (float)spk[(int64_t)b * n_pre + row] * gj;
          acc = acc + prod;
        }
        gw[s] = acc;
      }
    }
  }
  if (!kHet && gw) block_atomic_sum<kBlock / BS_WAVE>(sw, gw);
}

// ---- the same with g transposed: gT[j][b], Bp columns (a multiple of LB), row n_post zero ----
// A 4-byte gather of g moves a line for each (synapse, batch row); transposed, the batch values
// of a synapse's target lie side by side.
constexpr int kTr = 64;        // tile of the transposition
constexpr int kTrWgs = 2048;   // its workgroups at most, a flag each: k_matvec_vjp_bt reads them all
// Tiles in one dimension, tj across the posts: a grid in y ends at 65,536 x 64 batch rows.
__global__ __launch_bounds__(kBlock) void k_transpose_g(const float* __restrict__ g, int32_t batch,
                                                        int32_t n_post, int32_t Bp, int32_t tj,
                                                        int32_t tiles, float* __restrict__ gT,
                                                        uint32_t* __restrict__ odd) {
  constexpr int kS = kBlock / 64;
  __shared__ float s_t[kTr][kTr + 1];
  __shared__ uint32_t s_odd;
  const int c = threadIdx.x & 63, r0 = threadIdx.x >> 6;
  if (threadIdx.x == 0) s_odd = 0u;
  __syncthreads();
  bool bad = false;
  for (int32_t t = blockIdx.x; t < tiles; t += gridDim.x) {
    const int64_t j0 = (int64_t)(t % tj) * kTr, b0 = (int64_t)(t / tj) * kTr;
#pragma unroll
    for (int u = 0; u < kTr / kS; ++u) {
      const int r = r0 + u * kS;
      const int64_t b = b0 + r, j = j0 + c;
      const float v = b < batch && j < n_post ? g[b * n_post + j] : 0.0f;
      bad |= (__float_as_uint(v) & 0x7f800000u) == 0x7f800000u;
      s_t[r][c] = v;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kTr / kS; ++u) {
      const int r = r0 + u * kS;
      const int64_t j = j0 + r, b = b0 + c;
      if (j <= n_post && b < Bp) gT[j * Bp + b] = s_t[c][r];
    }
    __syncthreads();                     // the tile is rewritten next
  }
  if (bad) s_odd = 1u;
  __syncthreads();
  if (threadIdx.x == 0) odd[blockIdx.x] = s_odd;   // an inf or NaN among its values
}

// One wave per pre row i.
//   grad_x[b, i]: lane (q, b) = (lane / LB, lane % LB) sums the row's synapses l = a G + q of
//   every 64 (G = 64 / LB) into its own accumulator a -- the lane sums of k_matvec_vjp, held
//   by a instead of by lane -- and adds them in k_matvec_vjp's order: bit for bit its value.
//   grad_w[i, k]: lane = synapse, the products x[b, i] g[b, idx] added in b order over the
//   batch rows whose x is not zero (the others add +-0; unless some g is inf or NaN, `odd`:
//   then over all).
// 64 rows of 3200 -> 4000, K = 80: 101 us with per-row 4-byte gathers of g for both, 16 (and 7
// for the transposition) here; bound by latency at that size, by L2 at 128 x 10k.
template <typename T, bool kCsr, bool kHet, int LB>
__global__ __launch_bounds__(kBlock) void k_matvec_vjp_bt(
    const T* __restrict__ spk, int32_t batch, int32_t n_pre, const int32_t* __restrict__ indptr,
    const int32_t* __restrict__ indices, int32_t k, const float* __restrict__ w, float w_homo,
    int32_t n_post, const float* __restrict__ gT, int32_t Bp, const uint32_t* __restrict__ odd,
    int32_t n_odd, float* __restrict__ gx, float* __restrict__ gw) {
  constexpr int G = BS_WAVE / LB, A = LB, kU = 16;
  const int lane = bs_lane();
  const int q = lane / LB, bl = lane % LB;
  const int64_t nw = (int64_t)gridDim.x * (kBlock / BS_WAVE);
  const int32_t nnz = kCsr ? indptr[n_pre] : 0;
  bool all = false;
  if (kHet && gw)
    for (int32_t t = lane; t < n_odd; t += BS_WAVE) all |= odd[t] != 0u;
  all = bs_ballot(all) != 0ull;
  double sw = 0.0;
  for (int64_t row = __builtin_amdgcn_readfirstlane(
           (int)(((int64_t)blockIdx.x * kBlock + threadIdx.x) / BS_WAVE));
       row < n_pre; row += nw) {
    int64_t beg, end;
    if (kCsr) {
      beg = indptr[row];
      end = indptr[row + 1];
      beg = beg < 0 ? 0 : beg;
      end = end > nnz ? nnz : end;
    } else {
      beg = row * k;
      end = beg + k;
    }
    if (gx || !kHet) {
      for (int32_t b0 = 0; b0 < batch; b0 += LB) {
        const int32_t b = b0 + bl;
        const float* gb = gT + b;                      // b < Bp
        float acc[A];
        double tot = 0.0;
#pragma unroll
        for (int a = 0; a < A; ++a) acc[a] = 0.0f;
        for (int64_t s0 = beg; s0 < end; s0 += BS_WAVE) {
          const int cnt = (int)(end - s0 < BS_WAVE ? end - s0 : BS_WAVE);
          const bool in = lane < cnt;
          const int32_t js = in ? indices[s0 + lane] : n_post;
          const int32_t jl = (uint32_t)js < (uint32_t)n_post ? js : n_post;   // the zero row
          const float wl = !in ? 0.0f : (kHet ? w[s0 + lane] : w_homo);
#pragma unroll
          for (int a0 = 0; a0 < A; a0 += kU) {
            if (a0 * G >= cnt) break;                  // uniform
            float v[kU];
#pragma unroll
            for (int u = 0; u < kU; ++u) {
              const int l = (a0 + u) * G;
              const int32_t j = G == 1 ? __builtin_amdgcn_readlane(jl, l) : __shfl(jl, l + q);
              v[u] = gb[(uint32_t)j * (uint32_t)Bp];
            }
#pragma unroll
            for (int u = 0; u < kU; ++u) {
              const int l = (a0 + u) * G;
              const float ws = G == 1 ? __uint_as_float(__builtin_amdgcn_readlane(
                                            __float_as_uint(wl), l))
                                      : __shfl(wl, l + q);
              acc[a0 + u] += ws * v[u];
              if (!kHet) tot += (double)v[u];
            }
          }
        }
#pragma unroll
        for (int o = A / 2; o > 0; o >>= 1)
#pragma unroll
          for (int a = 0; a < o; ++a) acc[a] += acc[a + o];
        float sx = acc[0];
#pragma unroll
        for (int o = BS_WAVE / 2; o >= LB; o >>= 1) sx += __shfl_xor(sx, o);
        if (b < batch) {
          if (gx && q == 0) gx[(int64_t)b * n_pre + row] = sx;
          if (!kHet && gw) {
            const float xv = (float)spk[(int64_t)b * n_pre + row];
            if (xv != 0.0f) sw += (double)xv * tot;    // this lane's share of the row's g
          }
        }
      }
    }
    if (kHet && gw) {
      for (int64_t s = beg + lane; s - lane < end; s += BS_WAVE) {
        const int32_t js = s < end ? indices[s] : n_post;
        const float* gj = gT + (uint32_t)((uint32_t)js < (uint32_t)n_post ? js : n_post) *
                                   (uint32_t)Bp;
        float acc = 0.0f;
        for (int32_t b0 = 0; b0 < batch; b0 += BS_WAVE) {
          const int32_t bx = b0 + lane;
          const float xl = bx < batch ? (float)spk[(int64_t)bx * n_pre + row] : 0.0f;
          uint64_t m = bs_ballot(bx < batch && (all || xl != 0.0f));
          // kF values in flight (a row has a few active batch rows: one at a time, their
          // latencies add up); past the last one the lowest is read again and not added
          while (m) {
            constexpr int kF = 8;
            int at[kF];
            bool on[kF];
            float v[kF];
            const int first = __builtin_ctzll(m);
#pragma unroll
            for (int f = 0; f < kF; ++f) {
              on[f] = m != 0ull;
              at[f] = on[f] ? __builtin_ctzll(m) : first;
              m &= m - 1;
              v[f] = gj[b0 + at[f]];
            }
#pragma unroll
            for (int f = 0; f < kF; ++f) {
              const float xv =
                  __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(xl), at[f]));
              const float prod = xv * v[f];
              acc = on[f] ? acc + prod : acc;
            }
          }
        }
        if (s < end) gw[s] = acc;
      }
    }
  }
  if (!kHet && gw) {
#pragma unroll
    for (int o = BS_WAVE / 2; o > 0; o >>= 1) sw += __shfl_xor(sw, o);
    block_atomic_sum<kBlock / BS_WAVE>(sw, gw);
  }
}

// The transposed form of `batch` rows of n_post values: batch columns of gT (whole groups of
// `lanes`), tiles of the transposition and how many lie across the posts.
struct VjpBt {
  int32_t lanes, Bp;
  int64_t tj, tiles;
  int32_t wgs() const { return (int32_t)(tiles < kTrWgs ? tiles : kTrWgs); }
};

VjpBt vjp_bt(int32_t batch, int32_t n_post) {
  const int32_t lanes = batch <= 16 ? 16 : 64;
  const int64_t Bp = ((int64_t)batch + lanes - 1) / lanes * lanes;
  const int64_t tj = ((int64_t)n_post + kTr) / kTr;    // posts and the zero row
  return VjpBt{lanes, (int32_t)Bp, tj, tj * ((Bp + kTr - 1) / kTr)};
}

// Workspace the transposed form takes, 0 where it is never taken (vjp_bt_pays decides for a call).
size_t vjp_bt_bytes(int32_t batch, int32_t n_pre, int32_t n_post) {
  if (n_pre < 1 || n_post < 1 || batch < 3 || batch > (1 << 29)) return 0;
  if (batch < 8 && (int64_t)batch * n_pre < 20000) return 0;   // rarely pays: not worth the memory
  const VjpBt t = vjp_bt(batch, n_post);
  const int64_t n = ((int64_t)n_post + 1) * t.Bp;
  if (n >= (1LL << 30)) return 0;                      // 32-bit element offsets
  return (size_t)(n + t.wgs()) * 4;
}

// Whether the transposed form is the faster one, for rows of k synapses (their mean for CSR;
// unknown, k < 1: 64), from the costs of both in us.  Per-row kernel: a wave walks its rows'
// chunks of 64 synapses once per batch row, one after another, or the gathers of g are the
// limit (slower once g outgrows the L2).  Transposed: the transposition at 2 (16 lanes) or 4
// TB/s, then a chunk per lane group.  Measured (us per call, per-row / transposed, K
// synapses a row): 3 x (7000 -> 10k, K = 20) 6.3 / 11.2, the same -> 1M 12.5 / 48.9; 8 x (500 ->
// 400k, K = 20) 7.8 / 30.6; 17 x (500 -> 100k, K = 20) 15.0 / 21.4, 64 rows of it 70 / 25; 8 x
// (10k -> 500, K = 20) 15.2 / 12.3; 16 x (5000 -> 1M, K = 100) 205 / 69; 64 x (3200 -> 4000, K =
// 80) 95 / 23; 64 x (500 -> 10k, K = 1000) 509 / 72.
bool vjp_bt_pays(int32_t batch, int32_t n_pre, int32_t n_post, int32_t k) {
  const VjpBt t = vjp_bt(batch, n_post);
  const double kk = k > 0 ? k : 64, waves = 64.0 * bs_num_cus();
  const double rounds = std::ceil(n_pre / waves), chunks = std::ceil(kk / BS_WAVE);
  const double visit = (double)batch * n_post * 4 > 32e6 ? 2.4e-5 : 6e-6;
  const double row = 2.0 + std::fmax(rounds * batch * (0.45 + 0.4 * chunks),
                                     (double)batch * n_pre * kk * visit);
  const bool narrow = t.lanes == 16;
  const double move = ((double)batch + t.Bp) * n_post * 4 / (narrow ? 2e6 : 4e6);
  const double bt = 8.0 + move +
                    std::fmax(rounds * (t.Bp / t.lanes) * chunks * (narrow ? 1.7 : 3.4),
                              (double)t.Bp * n_pre * kk * 0.8e-6);
  return bt < row;
}

int grid_for(int64_t work_items_waves) {
  const int64_t cap = (int64_t)bs_num_cus() * 16;
  int64_t b = (work_items_waves + (kBlock / BS_WAVE) - 1) / (kBlock / BS_WAVE);
  if (b < 1) b = 1;
  if (b > cap) b = cap;
  return (int)b;
}

}  // namespace

int bs_fill_f32(float* p, int64_t n, float v, hipStream_t s) {
  if (n <= 0) return BS_OK;
  int64_t b = (n + kBlock - 1) / kBlock;
  const int64_t cap = (int64_t)bs_num_cus() * 8;
  if (b > cap) b = cap;
  k_fill_f32<<<(int)b, kBlock, 0, s>>>(p, n, v);
  BS_CHECK_LAUNCH();
  return BS_OK;
}

extern "C" int bs_event_scatter_f32(const int32_t* active, const int32_t* n_active, int32_t n_pre,
                                    const int32_t* indptr, const int32_t* indices, int32_t k,
                                    const float* w, float w_homo, int32_t n_post, float* out,
                                    int32_t accumulate, bs_stream_t stream) {
  bs_clear_error();
  BS_CHECK_ARG(n_pre >= 0 && n_post >= 0, "bs_event_scatter_f32: negative size");
  BS_CHECK_ARG(indptr != nullptr || k >= 0, "bs_event_scatter_f32: k=%d < 0", k);
  hipStream_t s = bs_stream(stream);
  if (n_post > 0) BS_CHECK_ARG(out != nullptr, "bs_event_scatter_f32: out is NULL");
  if (!accumulate) {
    int rc = bs_fill_f32(out, n_post, 0.0f, s);
    if (rc) return rc;
  }
  if (n_pre == 0 || n_post == 0 || (indptr == nullptr && k == 0)) return BS_OK;
  BS_CHECK_ARG(active && n_active && indices, "bs_event_scatter_f32: NULL pointer");
  const bool het = w != nullptr;
  if (indptr == nullptr) {
    const int64_t cpr = ((int64_t)k + BS_WAVE - 1) / BS_WAVE;
    const int g = grid_for((int64_t)n_pre * cpr);
    if (het)
      k_scatter<false, true><<<g, kBlock, 0, s>>>(active, n_active, n_pre, nullptr, indices, k,
                                                  w, w_homo, n_post, out);
    else
      k_scatter<false, false><<<g, kBlock, 0, s>>>(active, n_active, n_pre, nullptr, indices, k,
                                                   nullptr, w_homo, n_post, out);
  } else {
    const int g = grid_for(n_pre);
    if (het)
      k_scatter<true, true><<<g, kBlock, 0, s>>>(active, n_active, n_pre, indptr, indices, 0, w,
                                                 w_homo, n_post, out);
    else
      k_scatter<true, false><<<g, kBlock, 0, s>>>(active, n_active, n_pre, indptr, indices, 0,
                                                  nullptr, w_homo, n_post, out);
  }
  BS_CHECK_LAUNCH();
  return BS_OK;
}

extern "C" int bs_spike_pack(const void* spk, int32_t spk_dtype, int32_t n, uint32_t* bits,
                             bs_stream_t stream) {
  bs_clear_error();
  BS_CHECK_ARG(n >= 0, "bs_spike_pack: n=%d < 0", n);
  BS_CHECK_ARG(spk_dtype == BS_SPK_U8 || spk_dtype == BS_SPK_F32,
               "bs_spike_pack: unknown spike dtype %d", spk_dtype);
  if (n == 0) return BS_OK;
  BS_CHECK_ARG(spk && bits, "bs_spike_pack: NULL pointer");
  hipStream_t s = bs_stream(stream);
  const int g = grid_for(((int64_t)n + BS_WAVE - 1) / BS_WAVE);
  if (spk_dtype == BS_SPK_U8) k_pack<uint8_t><<<g, kBlock, 0, s>>>((const uint8_t*)spk, n, bits);
  else k_pack<float><<<g, kBlock, 0, s>>>((const float*)spk, n, bits);
  BS_CHECK_LAUNCH();
  return BS_OK;
}

extern "C" int bs_event_gather_f32(const uint32_t* spk_bits, int32_t n_pre,
                                   const int64_t* slice_ptr, const int32_t* sell_pre,
                                   const float* sell_w, float w_homo, int32_t n_post, float* out,
                                   bs_stream_t stream) {
  bs_clear_error();
  BS_CHECK_ARG(n_pre >= 0 && n_post >= 0, "bs_event_gather_f32: negative size");
  if (n_post == 0) return BS_OK;
  BS_CHECK_ARG(slice_ptr && sell_pre && out && (spk_bits || n_pre == 0),
               "bs_event_gather_f32: NULL pointer");
  BS_CHECK_ARG(((uintptr_t)sell_pre & 15) == 0 && ((uintptr_t)sell_w & 15) == 0,
               "bs_event_gather_f32: sell_pre / sell_w must be 16-byte aligned");
  hipStream_t s = bs_stream(stream);
  const int64_t n_slices = ((int64_t)n_post + BS_WAVE - 1) / BS_WAVE;
  const int g = (int)((n_slices + (kBlock / BS_WAVE) - 1) / (kBlock / BS_WAVE));
  const int64_t nwords = ((int64_t)n_pre + 31) / 32;
  const bool lds = nwords * 4 <= 64 * 1024;
  const size_t shm = lds ? (size_t)nwords * 4 : 0;
  const bool het = sell_w != nullptr;
  if (het && lds)
    k_gather<true, true><<<g, kBlock, shm, s>>>(spk_bits, n_pre, slice_ptr, sell_pre, sell_w,
                                                w_homo, n_post, out);
  else if (het)
    k_gather<true, false><<<g, kBlock, 0, s>>>(spk_bits, n_pre, slice_ptr, sell_pre, sell_w,
                                               w_homo, n_post, out);
  else if (lds)
    k_gather<false, true><<<g, kBlock, shm, s>>>(spk_bits, n_pre, slice_ptr, sell_pre, nullptr,
                                                 w_homo, n_post, out);
  else
    k_gather<false, false><<<g, kBlock, 0, s>>>(spk_bits, n_pre, slice_ptr, sell_pre, nullptr,
                                                w_homo, n_post, out);
  BS_CHECK_LAUNCH();
  return BS_OK;
}

namespace {

// Pre rows per workgroup of k_matvec and of k_mv_finish's atomics: enough workgroups (over all
// batch rows) to fill the chip, at most kRowsCap rows each.
int32_t matvec_rows(int32_t batch, int32_t n_pre) {
  const int64_t g = (int64_t)bs_num_cus() * 4;
  const int64_t rows = ((int64_t)n_pre * batch + g - 1) / g;
  return (int32_t)(rows < 64 ? 64 : (rows > kRowsCap ? kRowsCap : rows));
}

// Ranges and row groups of k_mv_lds; R = 0 where k_matvec is kept: below 2e7 synapses (5e7 events
// of a shared weight; 2e6 for batches of 8, or 32), where its two launches cost more than the
// atomics they save, past 8 ranges, and where the costs say that LDS would not win with a
// quarter of the rows active.  Elsewhere the estimate decides on the device.  A batch with one
// row group each and few spans takes no estimate: its single launch is the shorter way from
// p ~ 0.01 on, and must promise twice the atomics' speed.
// us per call, k_matvec / LDS always / as decided here, at p = 0.002, 0.01, 0.05:
//   100k x 100k, K = 1000          19.7/23/20   69/28/26    272/83/76
//   250k x 100k, K = 100            7.9/34/14   19/37/24     70/43/36
//   250k x 4000, K = 100            9.5/16/12   28/19/17    116/27/25
//   8 x (20k -> 20k, K = 100)       6.9/23/11   14/27/17     46/29/27
//   64 x (3200 -> 4000, K = 80)     6.8/9.7/9.4 13/13/13     43/18/17
//   128 x (200k -> 20k, K = 100)   249/322/240  1209/573/471 6035/1150/1026
//   16 x (2000 -> 128k, K = 20)     6.0/43/5.9  6.2/47/6.2   8.0/51/8.0
// The constants below are fits to such calls.
struct MvPlan {
  int32_t nr, len, R;
  int32_t sample;                      // threads per batch row of the estimate; 0: LDS always
  MvCost cost;
};

MvPlan mv_plan(int32_t batch, int32_t n_pre, int32_t k, int32_t n_post, bool csr, bool count,
               int32_t kE) {
  MvPlan p{};
  if (csr || batch < 1 || n_pre < 1 || n_post < 1 || k < 1 || k >= (1 << 30)) return p;
  const int32_t least = (n_post + kMvPosts - 1) / kMvPosts;
  if (least > 8) return p;
  const double syn = (double)n_pre * k * batch;
  if (syn < (batch >= (count ? 32 : 8) ? 2e6 : (count ? 5e7 : 2e7))) return p;
  int32_t nr = least, R = 1;
  if (batch >= 8) {
    const int32_t want = 512 / batch < 8 ? 512 / batch : 8;
    const int32_t most = (n_post + 255) / 256;
    nr = want > nr ? want : nr;
    nr = nr < most ? nr : (most > least ? most : least);
  }
  const int64_t wgs = (int64_t)batch * nr;
  if (wgs < 256) {
    const int64_t rows = ((int64_t)n_pre + 63) / 64;
    const int64_t g = 512 / wgs;
    R = (int32_t)(g < rows ? g : rows);
    if (R < 1) R = 1;
  }
  const int32_t spans = ((n_pre - 1) / R) / kMvSpan + 1;         // of each of R groups
  const double rounds = R > 1 ? 1.0 : std::ceil((double)wgs / 512);
  MvCost& c = p.cost;
  c.R = R;
  c.rs = (n_pre - 1) / kMvSpan + 1;
  const int32_t threads = kMvSample / kE, need = (n_pre - 1) / kE + 1;
  p.sample = threads / batch < 1 ? 1 : threads / batch;
  p.sample = p.sample < need ? p.sample : need;
  const int32_t rows = mv_sample_rows(p.sample, kE) < batch ? mv_sample_rows(p.sample, kE) : batch;
  const int64_t seen = (int64_t)p.sample * kE < n_pre ? (int64_t)p.sample * kE : n_pre;
  c.per = (float)((double)n_pre / (double)(seen * rows) * k);
  c.group = 1.0f / (float)(kMvSyn + n_post / 4);
  c.direct0 = 9.0f;
  // few pre rows leave few workgroups for the atomics, 5e-3 us an event each (4000 rows of
  // 10,000 synapses at p = 0.1 take 487 us in k_matvec, 70 here; 200 of 200,000 17 ms, 1.4 ms)
  const int32_t per_wg = matvec_rows(batch, n_pre);
  c.direct1 = (float)std::fmax(batch * 5.4e-5 + 0.16 / n_post,
                               5e-3 / ((n_pre - 1) / per_wg + 1));
  c.lds0 = batch > 1 ? 11.0f : 4.0f;
  c.span = (float)(5.5 * rounds);
  c.last = c.span * (float)spans;
  c.read = (float)(rounds * ((count ? 0.3e-3 : 1.4e-3) / nr +
                             (0.03 + 0.003 * ((k - 1) / BS_WAVE + 1)) / k));
  c.part = (float)((double)batch * n_post * 2.4e-6);
  if (R == 1 && rounds * spans < 9) p.sample = 0;
  const float dense = 0.25f * (float)n_pre * (float)k, most = c.lds_us(dense, c.groups(dense));
  if (c.direct_us(dense) < (p.sample ? 1.3f : 2.0f) * most) return MvPlan{};
  p.nr = nr;
  p.len = (n_post + nr - 1) / nr;
  p.R = R;
  return p;
}

size_t mv_ws_bytes(const MvPlan& p, int32_t batch, int32_t n_post) {
  return p.sample ? (size_t)batch * (kMvHdr + (p.R > 1 ? (size_t)p.R * n_post : 0)) * 4 : 0;
}

// Shared launcher of the fused mat-vec (event or value-weighted).
template <bool kVal>
int matvec_launch(const void* spk, int32_t spk_dtype, int32_t batch, int32_t n_pre,
                  const int32_t* indptr, const int32_t* indices, int32_t k, const float* w,
                  float w_homo, int32_t n_post, float* out, int32_t accumulate, void* ws,
                  size_t ws_bytes, hipStream_t s, const char* who) {
  BS_CHECK_ARG(n_pre >= 0 && n_post >= 0, "%s: negative size", who);
  BS_CHECK_ARG(batch >= 1 && batch <= 65535, "%s: batch %d outside [1, 65535]", who, batch);
  BS_CHECK_ARG(indptr != nullptr || k >= 0, "%s: k=%d < 0", who, k);
  BS_CHECK_ARG(spk_dtype == BS_SPK_U8 || spk_dtype == BS_SPK_F32, "%s: unknown spike dtype %d",
               who, spk_dtype);
  if (n_post > 0) BS_CHECK_ARG(out != nullptr, "%s: out is NULL", who);
  const MvPlan mp = mv_plan(batch, n_pre, k, n_post, indptr != nullptr, !kVal && w == nullptr,
                            spk_dtype == BS_SPK_U8 ? 16 : 4);
  const size_t mneed = mv_ws_bytes(mp, batch, n_post);
  if (mp.R > 0 && (mneed == 0 || ws != nullptr)) {
    BS_CHECK_ARG(spk && indices, "%s: NULL pointer", who);
    BS_CHECK_ARG(ws_bytes >= mneed, "%s: workspace of %zu bytes needed (got %zu)", who, mneed,
                 ws_bytes);
    const dim3 mg((unsigned)(mp.R == 1 ? mp.nr : (mp.R + 7) / 8 * 8 * mp.nr), (unsigned)batch);
    uint32_t* part = (uint32_t*)ws;
    const int32_t rows = matvec_rows(batch, n_pre);
    const int64_t gp = mp.R > 1 ? ((int64_t)n_post + BS_WAVE - 1) / BS_WAVE : 1;
    const int64_t gr = ((int64_t)n_pre + rows - 1) / rows;
    const dim3 fg((unsigned)(gp > gr ? gp : gr), (unsigned)batch);
#define BS_ML(T, H)                                                                        \
  do {                                                                                     \
    k_mv_lds<T, H, kVal><<<mg, kMvB, 0, s>>>((const T*)spk, n_pre, indices, k, w, w_homo,    \
                                             n_post, mp.nr, mp.len, mp.R, mp.sample, mp.cost, \
                                             accumulate, out, part);                       \
    BS_CHECK_LAUNCH();                                                                     \
    if (mp.sample)                                                                         \
      k_mv_finish<T, H, kVal><<<fg, kBlock, 0, s>>>((const T*)spk, n_pre, rows, indices, k, w, \
                                                    n_post, mp.R, w_homo, accumulate, part,  \
                                                    out);                                  \
  } while (0)
    if (spk_dtype == BS_SPK_U8) { if (w) BS_ML(uint8_t, true); else BS_ML(uint8_t, false); }
    else { if (w) BS_ML(float, true); else BS_ML(float, false); }
#undef BS_ML
    BS_CHECK_LAUNCH();
    return BS_OK;
  }
  if (!accumulate) {
    int rc = bs_fill_f32(out, (int64_t)batch * n_post, 0.0f, s);
    if (rc) return rc;
  }
  if (n_pre == 0 || n_post == 0 || (indptr == nullptr && k == 0)) return BS_OK;
  BS_CHECK_ARG(spk && indices, "%s: NULL pointer", who);
  const int32_t rows = matvec_rows(batch, n_pre);
  const int64_t g = ((int64_t)n_pre + rows - 1) / rows;
  const size_t shm = n_post <= kLdsPosts ? (size_t)n_post * sizeof(float) : 0;
  const bool het = w != nullptr, csr = indptr != nullptr;
#define BS_MV(T, C, H)                                                                \
  k_matvec<T, C, H, kVal><<<dim3((unsigned)g, (unsigned)batch), kBlock, shm, s>>>(       \
      (const T*)spk, n_pre, rows, indptr, indices, k, w, w_homo, n_post, out)
  if (spk_dtype == BS_SPK_U8) {
    if (csr) { if (het) BS_MV(uint8_t, true, true); else BS_MV(uint8_t, true, false); }
    else { if (het) BS_MV(uint8_t, false, true); else BS_MV(uint8_t, false, false); }
  } else {
    if (csr) { if (het) BS_MV(float, true, true); else BS_MV(float, true, false); }
    else { if (het) BS_MV(float, false, true); else BS_MV(float, false, false); }
  }
#undef BS_MV
  BS_CHECK_LAUNCH();
  return BS_OK;
}

}  // namespace

extern "C" int bs_event_matvec_f32(const void* spk, int32_t spk_dtype, int32_t n_pre,
                                   const int32_t* indptr, const int32_t* indices, int32_t k,
                                   const float* w, float w_homo, int32_t n_post, float* out,
                                   int32_t accumulate, bs_stream_t stream) {
  bs_clear_error();
  return matvec_launch<false>(spk, spk_dtype, 1, n_pre, indptr, indices, k, w, w_homo, n_post,
                              out, accumulate, nullptr, 0, bs_stream(stream), "bs_event_matvec_f32");
}

extern "C" int bs_event_matvec_batch_f32(const void* spk, int32_t spk_dtype, int32_t batch,
                                         int32_t n_pre, const int32_t* indptr,
                                         const int32_t* indices, int32_t k, const float* w,
                                         float w_homo, int32_t n_post, float* out,
                                         int32_t accumulate, bs_stream_t stream) {
  bs_clear_error();
  return matvec_launch<false>(spk, spk_dtype, batch, n_pre, indptr, indices, k, w, w_homo,
                              n_post, out, accumulate, nullptr, 0, bs_stream(stream),
                              "bs_event_matvec_batch_f32");
}

extern "C" int bs_value_matvec_f32(const float* x, int32_t n_pre, const int32_t* indptr,
                                   const int32_t* indices, int32_t k, const float* w,
                                   float w_homo, int32_t n_post, float* out, int32_t accumulate,
                                   bs_stream_t stream) {
  bs_clear_error();
  return matvec_launch<true>(x, BS_SPK_F32, 1, n_pre, indptr, indices, k, w, w_homo, n_post,
                             out, accumulate, nullptr, 0, bs_stream(stream), "bs_value_matvec_f32");
}

extern "C" int bs_value_matvec_batch_f32(const float* x, int32_t batch, int32_t n_pre,
                                         const int32_t* indptr, const int32_t* indices, int32_t k,
                                         const float* w, float w_homo, int32_t n_post,
                                         float* out, int32_t accumulate, bs_stream_t stream) {
  bs_clear_error();
  return matvec_launch<true>(x, BS_SPK_F32, batch, n_pre, indptr, indices, k, w, w_homo, n_post,
                             out, accumulate, nullptr, 0, bs_stream(stream),
                             "bs_value_matvec_batch_f32");
}

extern "C" size_t bs_matvec_workspace_size(int32_t batch, int32_t n_pre, int32_t k,
                                           int32_t n_post, int32_t count) {
  bs_clear_error();
  return mv_ws_bytes(mv_plan(batch, n_pre, k, n_post, false, count != 0, 4), batch, n_post);
}

extern "C" int bs_matvec_ws_f32(const void* spk, int32_t spk_dtype, int32_t value, int32_t batch,
                                int32_t n_pre, const int32_t* indices, int32_t k, const float* w,
                                float w_homo, int32_t n_post, float* out, int32_t accumulate,
                                void* workspace, size_t workspace_bytes, bs_stream_t stream) {
  bs_clear_error();
  hipStream_t s = bs_stream(stream);
  return value ? matvec_launch<true>(spk, spk_dtype, batch, n_pre, nullptr, indices, k, w, w_homo,
                                     n_post, out, accumulate, workspace, workspace_bytes, s,
                                     "bs_matvec_ws_f32")
               : matvec_launch<false>(spk, spk_dtype, batch, n_pre, nullptr, indices, k, w,
                                      w_homo, n_post, out, accumulate, workspace,
                                      workspace_bytes, s, "bs_matvec_ws_f32");
}

namespace {

int vjp_batch(const void* spk, int32_t spk_dtype, int32_t batch, int32_t n_pre,
              const int32_t* indptr, const int32_t* indices, int32_t k, const float* w,
              float w_homo, int32_t n_post, const float* grad_out, float* grad_spk,
              float* grad_w, void* ws, size_t ws_bytes, bs_stream_t stream) {
  BS_CHECK_ARG(batch >= 0 && n_pre >= 0 && n_post >= 0,
               "bs_event_matvec_vjp_batch_f32: negative size");
  BS_CHECK_ARG(indptr != nullptr || k >= 0, "bs_event_matvec_vjp_batch_f32: k=%d < 0", k);
  BS_CHECK_ARG(spk_dtype == BS_SPK_U8 || spk_dtype == BS_SPK_F32,
               "bs_event_matvec_vjp_batch_f32: unknown spike dtype %d", spk_dtype);
  hipStream_t s = bs_stream(stream);
  const bool het = w != nullptr, csr = indptr != nullptr;
  if (grad_w && !het) {  // homogeneous: one scalar, accumulated with atomics below
    int rc = bs_fill_f32(grad_w, 1, 0.0f, s);
    if (rc) return rc;
  }
  if (n_pre == 0 || (!grad_spk && !grad_w)) return BS_OK;
  BS_CHECK_ARG(spk && indices && (grad_out || n_post == 0 || batch == 0),
               "bs_event_matvec_vjp_batch_f32: NULL pointer");
  if (!csr && k == 0) {  // no synapse: grad_spk is zero, grad_w empty
    return grad_spk ? bs_fill_f32(grad_spk, (int64_t)batch * n_pre, 0.0f, s) : BS_OK;
  }
  const int g = grid_for(n_pre);
  const size_t need = vjp_bt_bytes(batch, n_pre, n_post);
  if (need > 0 && ws != nullptr && vjp_bt_pays(batch, n_pre, n_post, k)) {
    BS_CHECK_ARG(ws_bytes >= need, "bs_event_matvec_vjp_batch_ws_f32: workspace of %zu bytes "
                 "needed (got %zu)", need, ws_bytes);
    const VjpBt t = vjp_bt(batch, n_post);
    float* gT = (float*)ws;
    uint32_t* odd = (uint32_t*)(gT + ((int64_t)n_post + 1) * t.Bp);
    k_transpose_g<<<t.wgs(), kBlock, 0, s>>>(grad_out, batch, n_post, t.Bp, (int32_t)t.tj,
                                             (int32_t)t.tiles, gT, odd);
    BS_CHECK_LAUNCH();
#define BS_BT1(T, C, H, L)                                                                   \
  k_matvec_vjp_bt<T, C, H, L><<<g, kBlock, 0, s>>>((const T*)spk, batch, n_pre, indptr, indices, \
                                                   k, w, w_homo, n_post, gT, t.Bp, odd,       \
                                                   t.wgs(), grad_spk, grad_w)
#define BS_BT(T, C, H) do { if (t.lanes == 16) BS_BT1(T, C, H, 16); else BS_BT1(T, C, H, 64); } while (0)
    if (spk_dtype == BS_SPK_U8) {
      if (csr) { if (het) BS_BT(uint8_t, true, true); else BS_BT(uint8_t, true, false); }
      else { if (het) BS_BT(uint8_t, false, true); else BS_BT(uint8_t, false, false); }
    } else {
      if (csr) { if (het) BS_BT(float, true, true); else BS_BT(float, true, false); }
      else { if (het) BS_BT(float, false, true); else BS_BT(float, false, false); }
    }
#undef BS_BT
#undef BS_BT1
    BS_CHECK_LAUNCH();
    return BS_OK;
  }
  // batch == 0 or n_post == 0 go through the kernel: it writes grad_w = 0 (g never read)
#define BS_VJPB(T, C, H)                                                                    \
  k_matvec_vjp_batch<T, C, H><<<g, kBlock, 0, s>>>((const T*)spk, batch, n_pre, indptr,       \
                                                   indices, k, w, w_homo, n_post, grad_out,   \
                                                   grad_spk, grad_w)
  if (spk_dtype == BS_SPK_U8) {
    if (csr) { if (het) BS_VJPB(uint8_t, true, true); else BS_VJPB(uint8_t, true, false); }
    else { if (het) BS_VJPB(uint8_t, false, true); else BS_VJPB(uint8_t, false, false); }
  } else {
    if (csr) { if (het) BS_VJPB(float, true, true); else BS_VJPB(float, true, false); }
    else { if (het) BS_VJPB(float, false, true); else BS_VJPB(float, false, false); }
  }
#undef BS_VJPB
  BS_CHECK_LAUNCH();
  return BS_OK;
}

}  // namespace

extern "C" int bs_event_matvec_vjp_batch_f32(const void* spk, int32_t spk_dtype, int32_t batch,
                                             int32_t n_pre, const int32_t* indptr,
                                             const int32_t* indices, int32_t k, const float* w,
                                             float w_homo, int32_t n_post, const float* grad_out,
                                             float* grad_spk, float* grad_w,
                                             bs_stream_t stream) {
  bs_clear_error();
  return vjp_batch(spk, spk_dtype, batch, n_pre, indptr, indices, k, w, w_homo, n_post, grad_out,
                   grad_spk, grad_w, nullptr, 0, stream);
}

extern "C" size_t bs_event_matvec_vjp_batch_workspace_size(int32_t batch, int32_t n_pre,
                                                           int32_t n_post) {
  bs_clear_error();
  return vjp_bt_bytes(batch, n_pre, n_post);
}

extern "C" int bs_event_matvec_vjp_batch_ws_f32(const void* spk, int32_t spk_dtype,
                                                int32_t batch, int32_t n_pre,
                                                const int32_t* indptr, const int32_t* indices,
                                                int32_t k, const float* w, float w_homo,
                                                int32_t n_post, const float* grad_out,
                                                float* grad_spk, float* grad_w, void* workspace,
                                                size_t workspace_bytes, bs_stream_t stream) {
  bs_clear_error();
  return vjp_batch(spk, spk_dtype, batch, n_pre, indptr, indices, k, w, w_homo, n_post, grad_out,
                   grad_spk, grad_w, workspace, workspace_bytes, stream);
}

namespace {

// Whether k_matvec_vjp_lds is the faster of the two (kernel times, us; L2 gathers / LDS).
// With g resident (n_post <= 40,832) filling LDS costs ~9 us, the L2 kernel 5 us per 1e6
// synapses: 10k x 100 synapses 8.7 / 10.7, 2k x 1000 9.2 / 7.9, 20k x 200 19.1 / 12.3,
// 100k x 200 91 / 43.  With nr > 2 ranges a synapse slot (rows are padded to CP chunks) costs
// (2.0 + 0.28 nr) 1e-6 us, an L2 gather 4.9e-6, or 7e-6 when the synapses do not stay in the
// 256 MB memory-side cache: 100k posts, K = 100 (28 % padding) 51 / 54, K = 128 62 / 57,
// 5k x 1000 28 / 21, 100k x 1000 699 / 318; 400k posts (20 ranges) 359 / 456.
bool vjp_lds(int32_t n_pre, int32_t k, int32_t n_post, int bytes_per_syn) {
  const double syn = (double)n_pre * k;
  if (k >= (1 << 28)) return false;                   // 32-bit byte offsets inside a row
  const int32_t nr = (int32_t)(((int64_t)n_post + kLvR - 1) / kLvR);
  if (nr <= 2) return syn >= 1.5e6;
  if (syn < 3e6) return false;
  const int64_t cpr = ((int64_t)k + BS_WAVE - 1) / BS_WAVE;
  const int64_t slots = cpr <= 2 ? cpr : cpr <= 4 ? 4 : cpr <= 8 ? 8 : (cpr + 15) / 16 * 16;
  const double gather = syn * bytes_per_syn > 256e6 ? 7.0 : 4.9;
  return (2.0 + 0.28 * nr) * 1.15 * (double)(slots * BS_WAVE) < gather * k;
}

}  // namespace

extern "C" int bs_event_matvec_vjp_f32(const void* spk, int32_t spk_dtype, int32_t n_pre,
                                       const int32_t* indptr, const int32_t* indices, int32_t k,
                                       const float* w, float w_homo, int32_t n_post,
                                       const float* grad_out, float* grad_spk, float* grad_w,
                                       bs_stream_t stream) {
  bs_clear_error();
  BS_CHECK_ARG(n_pre >= 0 && n_post >= 0, "bs_event_matvec_vjp_f32: negative size");
  BS_CHECK_ARG(indptr != nullptr || k >= 0, "bs_event_matvec_vjp_f32: k=%d < 0", k);
  BS_CHECK_ARG(spk_dtype == BS_SPK_U8 || spk_dtype == BS_SPK_F32,
               "bs_event_matvec_vjp_f32: unknown spike dtype %d", spk_dtype);
  hipStream_t s = bs_stream(stream);
  const bool het = w != nullptr, csr = indptr != nullptr;
  if (grad_w && !het) {  // homogeneous: one scalar, accumulated with atomics below
    int rc = bs_fill_f32(grad_w, 1, 0.0f, s);
    if (rc) return rc;
  }
  if (n_pre == 0 || (!grad_spk && !grad_w)) return BS_OK;
  BS_CHECK_ARG(spk && indices && (grad_out || n_post == 0),
               "bs_event_matvec_vjp_f32: NULL pointer");
  if (n_post == 0 || (!csr && k == 0)) {  // no synapse: every gradient is zero
    if (grad_spk) {
      int rc = bs_fill_f32(grad_spk, n_pre, 0.0f, s);
      if (rc) return rc;
    }
    return BS_OK;
  }
  if (!csr && vjp_lds(n_pre, k, n_post, het ? (grad_w ? 12 : 8) : 4)) {
    const int cpr = (k + BS_WAVE - 1) / BS_WAVE;
    const int gl = bs_num_cus();
#define BS_VJPL(T, CP, H, G)                                                               \
  do {                                                                                     \
    if (n_post > 2 * kLvR)                                                                 \
      k_matvec_vjp_lds<T, CP, H, G, true><<<gl, kLvB, 0, s>>>(                             \
          (const T*)spk, n_pre, indices, k, w, w_homo, n_post, grad_out, grad_spk, grad_w);  \
    else                                                                                   \
      k_matvec_vjp_lds<T, CP, H, G, false><<<gl, kLvB, 0, s>>>(                            \
          (const T*)spk, n_pre, indices, k, w, w_homo, n_post, grad_out, grad_spk, grad_w);  \
  } while (0)
#define BS_VJPL2(T, CP)                                                 \
  do {                                                                  \
    if (!het) BS_VJPL(T, CP, false, false);                             \
    else if (grad_w) BS_VJPL(T, CP, true, true);                        \
    else BS_VJPL(T, CP, true, false);                                   \
  } while (0)
#define BS_VJPL3(T)                                                                         \
  do {                                                                                      \
    if (cpr == 1) BS_VJPL2(T, 1); else if (cpr == 2) BS_VJPL2(T, 2);                        \
    else if (cpr <= 4) BS_VJPL2(T, 4); else if (cpr <= 8) BS_VJPL2(T, 8);                   \
    else BS_VJPL2(T, 16);                                                                   \
  } while (0)
    if (spk_dtype == BS_SPK_U8) BS_VJPL3(uint8_t); else BS_VJPL3(float);
#undef BS_VJPL3
#undef BS_VJPL2
#undef BS_VJPL
    BS_CHECK_LAUNCH();
    return BS_OK;
  }
  const int g = grid_for(n_pre);
#define BS_VJP(T, C, H)                                                                   \
  k_matvec_vjp<T, C, H><<<g, kBlock, 0, s>>>((const T*)spk, n_pre, indptr, indices, k, w, \
                                             w_homo, n_post, grad_out, grad_spk, grad_w)
  if (spk_dtype == BS_SPK_U8) {
    if (csr) { if (het) BS_VJP(uint8_t, true, true); else BS_VJP(uint8_t, true, false); }
    else { if (het) BS_VJP(uint8_t, false, true); else BS_VJP(uint8_t, false, false); }
  } else {
    if (csr) { if (het) BS_VJP(float, true, true); else BS_VJP(float, true, false); }
    else { if (het) BS_VJP(float, false, true); else BS_VJP(float, false, false); }
  }
#undef BS_VJP
  BS_CHECK_LAUNCH();
  return BS_OK;
}
