// Connectivity construction on the device (brainstate/nn/_event_fixedprob.py:142-196).
//
// With replacement (allow_multi_conn=True) the reference draws
// numpy.random.RandomState(seed).randint(0, n_post, (n_pre, K)) on the host (:163-168), then,
// for afferent_ratio < 1, rng.random(n_pre) < afferent_ratio from the same stream (:186).
// That stream is reproduced here bit for bit:
//   * MT19937 (Matsumoto & Nishimura 1998) seeded with init_genrand(seed), state regenerated in
//     blocks of 624 words, outputs tempered;
//   * numpy's legacy bounded integers: draw = word & mask with mask the smallest 2^j - 1 >=
//     n_post - 1, redrawn while draw > n_post - 1 (no draw at all when n_post == 1);
//   * random(): (a * 2^26 + b) / 2^53 with a = word >> 5, b = next word >> 6.
// The twist is sequential from block to block, so the stream is cut into S segments of 2^m
// blocks and the state at the start of each is found by jump-ahead (mt_jump.h): a segment's 624
// state words are XORs of words that follow another segment's state, picked by the set bits
// of x^(jump) mod P.  k_mt_jump runs once per level, each quadrupling the segments whose
// state is known; k_mt_gen then twists all segments at once, tempering, writing the words and
// counting the accepted draws on the way (a word budget of expected draws + 12 standard
// deviations); k_mt_place ranks and places every accepted draw.  8e7 draws below 1e6 (135k
// blocks): one workgroup twisting every block, then passes to temper, count, scan and place,
// took 42.5 ms; this form 0.50 ms (263 segments: jumps 115 us, twists 189, placing 145 = 4.5 TB/s).
//
// Without replacement (allow_multi_conn=False) the reference uses its JAX generator
// (init_indices_without_replace, :39-62), which cannot be reproduced without JAX.  Here each
// row draws K values with Philox4x32-10 (Salmon et al. 2011, counter = (row, position,
// round, attempt), key = seed) and Lemire's unbiased bounded integers, then redraws the later
// copy of every repeated value until the row is duplicate-free; the row keeps draw order.
#include <cmath>
#include <type_traits>

#include "common.h"
#include "mt_jump.h"

namespace {

constexpr int kMtN = 624;
constexpr int kMtM = 397;
constexpr uint32_t kMtA = 0x9908b0dfu;
constexpr int kGen = 256;  // generator workgroup (one wave per quarter of a block)

__device__ __forceinline__ uint32_t mt_mix(uint32_t a, uint32_t b) {
  const uint32_t y = (a & 0x80000000u) | (b & 0x7fffffffu);
  return (y >> 1) ^ ((y & 1u) ? kMtA : 0u);
}

__device__ __forceinline__ uint32_t mt_temper(uint32_t y) {
  y ^= y >> 11;
  y ^= (y << 7) & 0x9d2c5680u;
  y ^= (y << 15) & 0xefc60000u;
  y ^= y >> 18;
  return y;
}

struct MtState {
  uint32_t x[kMtN];
};

// Segment 0's state; the states that k_mt_jump accumulates into cleared; info[0] = blocks,
// info[1] = 0 when nothing is drawn (else k_mt_place records the position, -1 until then).
__global__ __launch_bounds__(kGen) void k_mt_init(MtState s0, int32_t segs, int64_t blocks,
                                                  int64_t need, uint32_t* __restrict__ states,
                                                  int64_t* __restrict__ info) {
  for (int64_t i = (int64_t)blockIdx.x * kGen + threadIdx.x; i < (int64_t)segs * kMtN;
       i += (int64_t)gridDim.x * kGen)
    states[i] = i < kMtN ? s0.x[i] : 0u;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    info[0] = blocks;
    info[1] = need == 0 ? 0 : -1;
  }
}

// Words tid, tid + 227 and tid + 454 of the block that follows `o` (624 words in LDS), for
// tid < 227 (the third exists for tid < 170).  Word i needs new word i - 227, which the same
// thread has just formed, so a block needs no exchange but the old words; word 623's mix takes
// new word 0, which every thread forms for itself (three broadcast reads).
constexpr int kStep = kMtN - kMtM;          // 227
constexpr int kThird = kMtN - 2 * kStep;    // 170
__device__ __forceinline__ void mt_block(const uint32_t* o, int tid, uint32_t (&v)[3]) {
  const int t = tid < kStep ? tid : 0;
  const int t3 = tid < kThird ? tid : kThird - 1;
  const uint32_t a0 = o[t], a1 = o[t + 1], am = o[t + kMtM];
  const uint32_t b0 = o[t + kStep], b1 = o[t + kStep + 1];
  const uint32_t c0 = o[t3 + 2 * kStep], cn = o[t3 < kThird - 1 ? t3 + 2 * kStep + 1 : 0];
  const uint32_t z0 = o[0], z1 = o[1], zm = o[kMtM];
  const uint32_t c1 = t3 < kThird - 1 ? cn : zm ^ mt_mix(z0, z1);
  v[0] = am ^ mt_mix(a0, a1);
  v[1] = v[0] ^ mt_mix(b0, b1);
  v[2] = v[1] ^ mt_mix(c0, c1);
}

// Jump polynomials on the device, [e][r - 1] = x^(r * 624 * 2^e) mod P: constants of the
// generator, uploaded once per device and exponent (jump_table).
__device__ uint32_t d_jump[mt_jump::kMaxE + 1][3][mt_jump::kWords];

// One level: states of segments [nsrc, 4 nsrc) from those of [0, nsrc); segment r * nsrc + src
// is `src` advanced by r * nsrc segments, poly[r - 1].  Workgroup = (source, part of the
// polynomials): it regenerates the source's words x[0, hi) in LDS block by block, then each
// wave takes a run of 32-bit polynomial words: lane l holds the window of 41 words at i0 + 10 l
// and XORs the ones the three polynomials' 32 bits (wave-uniform) pick into its 3 x 10
// outputs, so a window word is read once from LDS for 96 bits instead of once per set bit
// (one target per workgroup: 69 us for the level from 64 to 256 segments).  The waves meet in
// LDS, the parts in `states`.  Bound by VALU and branch issue.
constexpr int kJumpB = 1024;
constexpr int kJumpW = kJumpB / BS_WAVE;
constexpr int kJumpT = 10;                       // outputs per lane: 63 lanes cover 624
constexpr int kJumpR = 3;                        // targets per source
constexpr int kJumpX = mt_jump::kDeg + kMtN;     // words any set bit can reach
constexpr int kJumpPad = 640;                    // window words past it are read, never used
__global__ __launch_bounds__(kJumpB) void k_mt_jump(uint32_t* __restrict__ states, int32_t nsrc,
                                                    int32_t segs, int32_t parts, int e) {
  __shared__ __align__(16) uint32_t x[kJumpX + kJumpPad];
  __shared__ uint32_t s_out[kJumpR][kMtN];
  const int tid = threadIdx.x;
  const int lane = bs_lane();
  const int wid = __builtin_amdgcn_readfirstlane(tid / BS_WAVE);
  const int32_t part = blockIdx.x % parts;
  const int32_t src = (int32_t)(blockIdx.x / parts);
  const uint32_t* poly = d_jump[e][0];
  const int32_t per = ((mt_jump::kWords + parts - 1) / parts + kJumpW - 1) / kJumpW;
  const int32_t w0 = (part * kJumpW + wid) * per;                      // this wave's words
  const int32_t w1 = w0 + per < mt_jump::kWords ? w0 + per : mt_jump::kWords;
  const int32_t last = (part + 1) * kJumpW * per * 32 + kMtN;          // words the part reads
  const int32_t hi = last < kJumpX ? last : kJumpX;
  for (int i = tid; i < kMtN; i += kJumpB) x[i] = states[(int64_t)src * kMtN + i];
  for (int i = tid; i < kJumpR * kMtN; i += kJumpB) s_out[0][i] = 0u;
  for (int i = kMtN + tid; i < kJumpX + kJumpPad; i += kJumpB) x[i] = 0u;
  __syncthreads();
  for (int32_t n0 = kMtN; n0 < hi; n0 += kMtN) {   // 33 blocks at most: within x's padding
    if (tid < kGen) {
      uint32_t v[3];
      mt_block(x + n0 - kMtN, tid, v);
      if (tid < kStep) {
        x[n0 + tid] = v[0];
        x[n0 + tid + kStep] = v[1];
      }
      if (tid < kThird) x[n0 + tid + 2 * kStep] = v[2];
    }
    __syncthreads();
  }
  uint32_t acc[kJumpR][kJumpT];
#pragma unroll
  for (int q = 0; q < kJumpR; ++q)
#pragma unroll
    for (int j = 0; j < kJumpT; ++j) acc[q][j] = 0u;
  for (int32_t w = w0; w < w1; ++w) {
    uint32_t bits[kJumpR];
#pragma unroll
    for (int q = 0; q < kJumpR; ++q)
      bits[q] = src + (q + 1) * nsrc < segs
                    ? __builtin_amdgcn_readfirstlane(poly[q * mt_jump::kWords + w]) : 0u;
    uint32_t r[31 + kJumpT];
    const uint32_t* p = x + w * 32 + lane * kJumpT;
#pragma unroll
    for (int k = 0; k < 31 + kJumpT; ++k) r[k] = p[k];
#pragma unroll
    for (int k = 0; k < 32; ++k) {
#pragma unroll
      for (int q = 0; q < kJumpR; ++q) {
        if ((bits[q] >> k) & 1u) {
#pragma unroll
          for (int j = 0; j < kJumpT; ++j) acc[q][j] ^= r[k + j];
        }
      }
    }
  }
#pragma unroll
  for (int q = 0; q < kJumpR; ++q)
#pragma unroll
    for (int j = 0; j < kJumpT; ++j)
      if (lane * kJumpT + j < kMtN) atomicXor(&s_out[q][lane * kJumpT + j], acc[q][j]);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kJumpR; ++q) {
    const int32_t tgt = src + (q + 1) * nsrc;
    if (tgt >= segs) break;
    for (int i = tid; i < kMtN; i += kJumpB) {
      uint32_t* d = states + (int64_t)tgt * kMtN + i;
      if (parts == 1) *d = s_out[q][i];
      else atomicXor(d, s_out[q][i]);
    }
  }
}

// Segment s: its 2^m blocks twisted one after another from its state, every word tempered and
// written; lofs[b] = draws accepted in the segment before block b, segtot[s] = in all of it.
// Waves 0-3 form block b from the old words while waves 4-7 temper, store and count block
// b - 1: one barrier per block, and the chain from block to block holds the twist alone (all
// in the same four waves: 0.36 us per block).
constexpr int kGenB = 2 * kGen;
__global__ __launch_bounds__(kGenB) void k_mt_gen(const uint32_t* __restrict__ states, int m,
                                                  int64_t blocks, uint32_t rng, uint32_t mask,
                                                  uint32_t* __restrict__ words,
                                                  uint32_t* __restrict__ lofs,
                                                  uint32_t* __restrict__ segtot) {
  __shared__ uint32_t st[2][kMtN];
  __shared__ uint32_t s_c[2][kGen / BS_WAVE];
  const bool twist = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kGen) == 0;
  const int tid = threadIdx.x % kGen;
  const int64_t b0 = (int64_t)blockIdx.x << m;
  const int32_t nb = (int32_t)((1LL << m) < blocks - b0 ? (1LL << m) : blocks - b0);
  for (int i = threadIdx.x; i < kMtN; i += kGenB)
    st[0][i] = states[(int64_t)blockIdx.x * kMtN + i];
  __syncthreads();
  uint32_t run = 0;
  // iteration b: block b from st[b & 1] into the other half, while st[b & 1] (block b - 1) is
  // written out; counts of block b - 1 are added up in iteration b + 1
  const bool third = tid < kMtN - 2 * kGen;
  const int t2 = third ? tid + 2 * kGen : kMtN - 1;
  auto step = [&](int32_t b, auto half) {
    constexpr int h = decltype(half)::value;
    const uint32_t* o = st[h];
    uint32_t* nw = st[h ^ 1];
    if (twist) {
      if (b < nb) {
        uint32_t v[3];
        mt_block(o, tid, v);
        if (tid < kStep) {
          nw[tid] = v[0];
          nw[tid + kStep] = v[1];
        }
        if (tid < kThird) nw[tid + 2 * kStep] = v[2];
      }
      if (tid == 0 && b >= 2 && b <= nb + 1) {
        lofs[b0 + b - 2] = run;
        run += s_c[h ^ 1][0] + s_c[h ^ 1][1] + s_c[h ^ 1][2] + s_c[h ^ 1][3];
      }
    } else if (b >= 1 && b <= nb) {
      const uint32_t x0 = mt_temper(o[tid]), x1 = mt_temper(o[tid + kGen]);
      const uint32_t x2 = mt_temper(o[t2]);
      uint32_t* dst = words + (b0 + b - 1) * kMtN;   // wave-uniform base
      dst[(uint32_t)tid] = x0;
      dst[(uint32_t)tid + kGen] = x1;
      if (third) dst[(uint32_t)tid + 2 * kGen] = x2;
      const uint32_t c = (uint32_t)(__popcll(bs_ballot((x0 & mask) <= rng)) +
                                    __popcll(bs_ballot((x1 & mask) <= rng)) +
                                    __popcll(bs_ballot(third && (x2 & mask) <= rng)));
      if (bs_lane() == 0) s_c[h][tid / BS_WAVE] = c;
    }
    __syncthreads();
  };
  for (int32_t b = 0; b <= nb + 1; b += 2) {
    step(b, std::integral_constant<int, 0>());
    step(b + 1, std::integral_constant<int, 1>());
  }
  if (threadIdx.x == 0) segtot[blockIdx.x] = run;
}

// Places accepted draws: out[rank] = word & mask for ranks below `need`; the draw of rank
// need - 1 records the stream position after it in info[1].  A workgroup takes 2^kPlaceM
// consecutive blocks of one segment (fewer when segments are shorter), each wave every fourth
// of them: ten ballots rank a block's words, with no barrier.
constexpr int kPlaceM = 5;
__global__ __launch_bounds__(kGen) void k_mt_place(const uint32_t* __restrict__ words,
                                                   const uint32_t* __restrict__ lofs,
                                                   const uint32_t* __restrict__ segtot, int m,
                                                   int64_t blocks, int64_t need, uint32_t rng,
                                                   uint32_t mask, int32_t* __restrict__ out,
                                                   int64_t* __restrict__ info) {
  __shared__ int64_t s_p[kGen / BS_WAVE];
  const int lane = bs_lane();
  const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / BS_WAVE));
  const int pm = m < kPlaceM ? m : kPlaceM;
  const int64_t bb = (int64_t)blockIdx.x << pm;
  const int32_t seg = (int32_t)(bb >> m);
  // accepted draws of the segments before this one
  int64_t c = 0;
  for (int32_t s = threadIdx.x; s < seg; s += kGen) c += segtot[s];
  for (int o = BS_WAVE / 2; o > 0; o >>= 1) c += __shfl_xor(c, o);
  if (lane == 0) s_p[wid] = c;
  __syncthreads();
  const int64_t base0 = s_p[0] + s_p[1] + s_p[2] + s_p[3];
  for (int k = wid; k < (1 << pm); k += kGen / BS_WAVE) {
    const int64_t b = bb + k;
    if (b >= blocks) break;
    int64_t r = base0 + lofs[b];
    if (r >= need) break;  // ranks only grow
    uint32_t w[10];
#pragma unroll
    for (int q = 0; q < 10; ++q) {
      const int i = q * BS_WAVE + lane;
      w[q] = i < kMtN ? words[b * kMtN + i] : 0xffffffffu;
    }
#pragma unroll
    for (int q = 0; q < 10; ++q) {
      const int i = q * BS_WAVE + lane;
      const bool ok = i < kMtN && (w[q] & mask) <= rng;
      const uint64_t bal = bs_ballot(ok);
      const int64_t x = r + bs_rank_below(bal);
      if (ok && x < need) {
        out[x] = (int32_t)(w[q] & mask);
        if (x == need - 1) info[1] = b * kMtN + i + 1;
      }
      r += __popcll(bal);
    }
  }
}

// sel[i] = random() < ratio for the 2 * n words starting after the last index draw.
__global__ void k_mt_select(const uint32_t* __restrict__ words, const int64_t* __restrict__ info,
                            int64_t n_words, int32_t n, double ratio,
                            uint8_t* __restrict__ sel) {
  const int64_t p = info[1];
  if (p < 0 || p + 2 * (int64_t)n > n_words) return;  // reported by the host check
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t a = words[p + 2 * i] >> 5;
    const uint32_t c = words[p + 2 * i + 1] >> 6;
    const double u = ((double)a * 67108864.0 + (double)c) / 9007199254740992.0;
    sel[i] = u < ratio ? 1 : 0;
  }
}

// indptr[i + 1] = k * (selected rows <= i), one workgroup; rows of selected pre neurons are
// copied to out (when given) at indptr[i].
__global__ __launch_bounds__(1024) void k_sel_indptr(const uint8_t* __restrict__ sel, int32_t n,
                                                     int32_t k, int32_t* __restrict__ indptr) {
  __shared__ int64_t part[1024];
  const int64_t per = ((int64_t)n + 1023) / 1024;
  const int64_t lo = threadIdx.x * per;
  const int64_t hi = lo + per < n ? lo + per : n;
  int64_t c = 0;
  for (int64_t i = lo; i < hi; ++i) c += sel[i] ? 1 : 0;
  part[threadIdx.x] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    int64_t s = 0;
    for (int t = 0; t < 1024; ++t) {
      const int64_t v = part[t];
      part[t] = s;
      s += v;
    }
    indptr[0] = 0;
  }
  __syncthreads();
  int64_t s = part[threadIdx.x];
  for (int64_t i = lo; i < hi; ++i) {
    s += sel[i] ? 1 : 0;
    indptr[i + 1] = (int32_t)(s * k);
  }
}

__global__ void k_sel_copy(const int32_t* __restrict__ idx, const uint8_t* __restrict__ sel,
                           const int32_t* __restrict__ indptr, int32_t n, int32_t k,
                           int32_t* __restrict__ out) {
  const int64_t total = (int64_t)n * k;
  for (int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; x < total;
       x += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i = x / k;
    if (sel[i]) out[indptr[i] + (x - i * k)] = idx[x];
  }
}

__global__ void k_fill_i32(int32_t* __restrict__ p, int64_t n, int32_t v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

// ---- Philox4x32-10 ----
struct U4 {
  uint32_t x, y, z, w;
};

__device__ __forceinline__ U4 philox(U4 c, uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const uint64_t p0 = (uint64_t)0xD2511F53u * c.x;
    const uint64_t p1 = (uint64_t)0xCD9E8D57u * c.z;
    c = U4{(uint32_t)(p1 >> 32) ^ c.y ^ k0, (uint32_t)p1, (uint32_t)(p0 >> 32) ^ c.w ^ k1,
           (uint32_t)p0};
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  return c;
}

// Uniform integer in [0, n) for draw (row, pos, round): Lemire's multiply-shift with exact
// rejection, the four Philox words of attempt a tried in order (each word is rejected with
// probability below 1/2, so 16 attempts fail with probability below 2^-64; the last word is
// then kept).
__device__ uint32_t bounded_draw(uint32_t k0, uint32_t k1, uint32_t row, uint32_t pos,
                                 uint32_t round, uint32_t n) {
  const uint32_t thr = (uint32_t)(-n) % n;  // 2^32 mod n
  uint64_t m = 0;
  for (uint32_t a = 0; a < 16; ++a) {
    const U4 r = philox(U4{row, pos, round, a}, k0, k1);
    const uint32_t v[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      m = (uint64_t)v[q] * n;
      if ((uint32_t)m >= thr) return (uint32_t)(m >> 32);
    }
  }
  return (uint32_t)(m >> 32);
}

constexpr int kUniqMax = 2048;     // K per row for the without-replacement sampler
constexpr int kUniqBlock = 256;
constexpr int kUniqRounds = 1 << 16;  // redraw rounds per row (a bound, never reached for K < n_post / 2)

// One workgroup per row: draw K values, sort (value, position) pairs, redraw every position
// holding a repeat of a value seen at an earlier position, until the row has no repeats.
__global__ __launch_bounds__(kUniqBlock) void k_unique_rows(uint32_t k0, uint32_t k1, int32_t n_pre,
                                                            int32_t k, int32_t n_post,
                                                            int32_t* __restrict__ out) {
  __shared__ uint64_t key[kUniqMax];
  __shared__ uint32_t val[kUniqMax];
  __shared__ uint32_t rnd[kUniqMax];
  __shared__ int s_any;
  int kp = 1;
  while (kp < k) kp <<= 1;
  for (int32_t row = blockIdx.x; row < n_pre; row += gridDim.x) {
    for (int p = threadIdx.x; p < k; p += kUniqBlock) {
      rnd[p] = 0;
      val[p] = bounded_draw(k0, k1, (uint32_t)row, (uint32_t)p, 0u, (uint32_t)n_post);
    }
    for (int round = 0; round < kUniqRounds; ++round) {
      for (int p = threadIdx.x; p < kp; p += kUniqBlock)
        key[p] = p < k ? (((uint64_t)val[p] << 32) | (uint32_t)p) : ~0ull;
      if (threadIdx.x == 0) s_any = 0;
      __syncthreads();
      for (int size = 2; size <= kp; size <<= 1) {  // bitonic sort, ascending
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
          for (int p = threadIdx.x; p < kp; p += kUniqBlock) {
            const int q = p ^ stride;
            if (q > p) {
              const bool up = (p & size) == 0;
              const uint64_t a = key[p], c = key[q];
              if ((a > c) == up) {
                key[p] = c;
                key[q] = a;
              }
            }
          }
          __syncthreads();
        }
      }
      for (int s = threadIdx.x + 1; s < k; s += kUniqBlock) {
        if ((key[s] >> 32) == (key[s - 1] >> 32)) {  // a later position repeats a value
          const uint32_t p = (uint32_t)key[s];
          rnd[p] += 1;
          val[p] = bounded_draw(k0, k1, (uint32_t)row, p, rnd[p], (uint32_t)n_post);
          s_any = 1;
        }
      }
      __syncthreads();
      const int any = s_any;
      __syncthreads();
      if (!any) break;
    }
    for (int p = threadIdx.x; p < k; p += kUniqBlock) out[(int64_t)row * k + p] = (int32_t)val[p];
    __syncthreads();
  }
}

uint32_t gen_mask(uint32_t rng) {
  uint32_t m = rng;
  m |= m >> 1;
  m |= m >> 2;
  m |= m >> 4;
  m |= m >> 8;
  m |= m >> 16;
  return m;
}

// Words the generator may need: expected draws + 12 standard deviations + a block of slack.
int64_t word_budget(int64_t need, uint32_t rng, int64_t extra) {
  if (need == 0) return extra + 2 * kMtN;
  const double p = ((double)rng + 1.0) / ((double)gen_mask(rng) + 1.0);
  const double mean = (double)need / p;
  const double sd = std::sqrt((double)need * (1.0 - p)) / p;
  return (int64_t)(mean + 12.0 * sd) + extra + 2 * kMtN;
}

// Workgroups per source of a level of jumps: levels with few sources split their polynomials
// (down to 2 or 3 32-bit words per wave) so that the level fills the chip.
int jump_parts(int64_t srcs) {
  const int64_t p = 256 / srcs;
  return (int)(p < 1 ? 1 : (p > 16 ? 16 : p));
}

// Segments of 2^m blocks.  Few long segments leave the chip idle while they twist, many
// short ones cost a jump each, and every level of jumps is a launch that regenerates 33 blocks:
// m minimises the sum, with costs fitted to kernel traces (a level 12.5 us and (34 + 25 per
// target of a source) / parts; twisting 0.32 / 0.385 / 0.485 / 0.61 us per block with 1 .. 4
// segments on a compute unit).  For 134k blocks m = 8 / 9 / 10 take 193 + 124 / 115 + 192 /
// 91 + 327 us of jumps + twists (508 / 491 / 597 us per call); short streams stay in one
// segment (below ~70 blocks) or few (430 blocks, 256k draws: 165 us in one, 80 in 14).
struct MtPlan {
  int m, levels;
  int32_t segs;
};

MtPlan mt_plan(int64_t blocks) {
  constexpr double kLevelUs = 12.5, kSourceUs = 34.0, kTargetUs = 25.0;
  constexpr double kTwistUs[] = {0.32, 0.385, 0.485, 0.61};
  constexpr int64_t kMaxSegs = 1024, kCus = 256;
  MtPlan best{0, 0, 0};
  double cost = 0.0;
  for (int m = 0; m <= 22; ++m) {
    const int64_t segs = (blocks + (1LL << m) - 1) >> m;
    if (segs > kMaxSegs) continue;
    int levels = 0;
    double c = (double)(segs > 1 ? 1LL << m : blocks) * kTwistUs[(segs - 1) / kCus];
    for (int64_t nsrc = 1; nsrc < segs; nsrc *= 4, ++levels) {
      const int64_t srcs = segs - nsrc < nsrc ? segs - nsrc : nsrc;
      const int64_t tgts = (segs < 4 * nsrc ? segs : 4 * nsrc) - nsrc;
      c += kLevelUs + (kSourceUs + kTargetUs * (double)((tgts + srcs - 1) / srcs)) /
                          jump_parts(srcs);
    }
    if (best.segs == 0 || c < cost) {
      best = MtPlan{m, levels, (int32_t)segs};
      cost = c;
    }
    if (segs == 1) break;
  }
  return best;
}

// Makes d_jump[e] valid on the current device: a synchronous copy the first time, so every
// stream sees it from then on.
int jump_table(int e) {
  constexpr int kDevs = 64;
  static std::mutex mu;
  static bool done[kDevs][mt_jump::kMaxE + 1];
  int dev = 0;
  BS_CHECK_HIP(hipGetDevice(&dev));
  BS_CHECK_ARG(e >= 0 && e <= mt_jump::kMaxE && dev < kDevs, "bs_conn_fixed_num: jump 2^%d on "
               "device %d out of range", e, dev);
  std::lock_guard<std::mutex> lock(mu);
  if (done[dev][e]) return BS_OK;
  constexpr size_t kBytes = 3 * sizeof(mt_jump::Poly);
  BS_CHECK_HIP(hipMemcpyToSymbol(HIP_SYMBOL(d_jump), mt_jump::powers(e), kBytes, kBytes * e,
                                 hipMemcpyHostToDevice));
  done[dev][e] = true;
  return BS_OK;
}

struct MtWs {
  int64_t blocks;
  MtPlan plan;
  size_t off_words, off_lofs, off_tot, off_states, off_info, bytes;
};

MtWs mt_ws(int64_t need, uint32_t rng, int64_t extra) {
  MtWs w;
  w.blocks = (word_budget(need, rng, extra) + kMtN - 1) / kMtN;
  w.plan = mt_plan(w.blocks);
  size_t o = 0;
  auto take = [&](size_t bytes) {
    const size_t at = o;
    o += (bytes + 255) & ~(size_t)255;
    return at;
  };
  w.off_words = take((size_t)w.blocks * kMtN * 4);
  w.off_lofs = take((size_t)w.blocks * 4);
  w.off_tot = take((size_t)w.plan.segs * 4);
  w.off_states = take((size_t)w.plan.segs * kMtN * 4);
  w.off_info = take(256);
  w.bytes = o;
  return w;
}

}  // namespace

extern "C" size_t bs_conn_fixed_num_workspace_size(int32_t n_pre, int32_t k, int32_t n_post,
                                                    int32_t with_selection) {
  bs_clear_error();
  if (n_pre < 0 || k < 0 || n_post < 1) {
    bs_set_error("bs_conn_fixed_num_workspace_size: bad sizes n_pre=%d k=%d n_post=%d", n_pre,
                 k, n_post);
    return 0;
  }
  const uint32_t rng = (uint32_t)(n_post - 1);
  const int64_t need = rng == 0 ? 0 : (int64_t)n_pre * k;
  return mt_ws(need, rng, with_selection ? 2 * (int64_t)n_pre : 0).bytes;
}

extern "C" int bs_conn_fixed_num(uint32_t seed, int32_t n_pre, int32_t k, int32_t n_post,
                                 int32_t* indices, double afferent_ratio, uint8_t* selected,
                                 void* workspace, size_t workspace_bytes, bs_stream_t stream) {
  bs_clear_error();
  BS_CHECK_ARG(n_pre >= 0 && k >= 0 && n_post >= 1, "bs_conn_fixed_num: bad sizes");
  BS_CHECK_ARG(indices || (int64_t)n_pre * k == 0, "bs_conn_fixed_num: indices is NULL");
  BS_CHECK_ARG(workspace, "bs_conn_fixed_num: workspace is NULL");
  const uint32_t rng = (uint32_t)(n_post - 1);
  const uint32_t mask = gen_mask(rng);
  const int64_t total = (int64_t)n_pre * k;
  const int64_t need = rng == 0 ? 0 : total;  // n_post == 1: numpy draws nothing
  const int64_t extra = selected ? 2 * (int64_t)n_pre : 0;
  const MtWs w = mt_ws(need, rng, extra);
  BS_CHECK_ARG(workspace_bytes >= w.bytes, "bs_conn_fixed_num: workspace %zu < %zu bytes",
               workspace_bytes, w.bytes);
  hipStream_t s = bs_stream(stream);
  char* ws = (char*)workspace;
  uint32_t* words = (uint32_t*)(ws + w.off_words);
  uint32_t* lofs = (uint32_t*)(ws + w.off_lofs);
  uint32_t* segtot = (uint32_t*)(ws + w.off_tot);
  uint32_t* states = (uint32_t*)(ws + w.off_states);
  int64_t* info = (int64_t*)(ws + w.off_info);
  const MtPlan& pl = w.plan;
  BS_CHECK_ARG(pl.segs > 0, "bs_conn_fixed_num: %lld blocks exceed the generator's reach",
               (long long)w.blocks);
  MtState s0;
  mt_jump::seed_state(seed, s0.x);
  k_mt_init<<<pl.segs < 256 ? pl.segs : 256, kGen, 0, s>>>(s0, pl.segs, w.blocks, need, states,
                                                           info);
  BS_CHECK_LAUNCH();
  for (int d = 0; d < pl.levels; ++d) {
    const int32_t nsrc = 1 << (2 * d);
    const int32_t srcs = pl.segs - nsrc < nsrc ? pl.segs - nsrc : nsrc;
    const int parts = jump_parts(srcs);
    const int rc = jump_table(pl.m + 2 * d);
    if (rc) return rc;
    k_mt_jump<<<srcs * parts, kJumpB, 0, s>>>(states, nsrc, pl.segs, parts, pl.m + 2 * d);
    BS_CHECK_LAUNCH();
  }
  k_mt_gen<<<pl.segs, kGenB, 0, s>>>(states, pl.m, w.blocks, rng, mask, words, lofs, segtot);
  BS_CHECK_LAUNCH();
  if (total > 0) {
    if (need == 0) {  // one target: every index is 0
      k_fill_i32<<<bs_num_cus() * 4, 256, 0, s>>>(indices, total, 0);
    } else {
      const int pm = pl.m < kPlaceM ? pl.m : kPlaceM;
      const int64_t g = (w.blocks + (1LL << pm) - 1) >> pm;
      BS_CHECK_ARG(g <= INT32_MAX, "bs_conn_fixed_num: too many draws");
      k_mt_place<<<(int)g, kGen, 0, s>>>(words, lofs, segtot, pl.m, w.blocks, need, rng, mask,
                                         indices, info);
    }
    BS_CHECK_LAUNCH();
  }
  if (selected && n_pre > 0) {
    k_mt_select<<<(n_pre + 255) / 256 < 4096 ? (n_pre + 255) / 256 : 4096, 256, 0, s>>>(
        words, info, w.blocks * kMtN, n_pre, afferent_ratio, selected);
    BS_CHECK_LAUNCH();
  }
  int64_t hinfo[2];
  BS_CHECK_HIP(hipMemcpyAsync(hinfo, info, sizeof(hinfo), hipMemcpyDeviceToHost, s));
  BS_CHECK_HIP(hipStreamSynchronize(s));
  if (hinfo[1] < 0 || hinfo[1] + extra > w.blocks * kMtN) {
    bs_set_error("bs_conn_fixed_num: word budget of %lld blocks exhausted",
                 (long long)w.blocks);
    return BS_ERR_LAUNCH;
  }
  return BS_OK;
}

extern "C" int bs_csr_from_selected(const int32_t* indices, int32_t n_pre, int32_t k,
                                    const uint8_t* selected, int32_t* indptr, int32_t* out,
                                    bs_stream_t stream) {
  bs_clear_error();
  BS_CHECK_ARG(n_pre >= 0 && k >= 0, "bs_csr_from_selected: bad sizes");
  BS_CHECK_ARG(selected && indptr, "bs_csr_from_selected: NULL pointer");
  BS_CHECK_ARG(!out || indices, "bs_csr_from_selected: indices is NULL");
  BS_CHECK_ARG((int64_t)n_pre * k < ((int64_t)1 << 31), "bs_csr_from_selected: %lld synapses "
               "exceed int32 offsets", (long long)n_pre * k);
  hipStream_t s = bs_stream(stream);
  k_sel_indptr<<<1, 1024, 0, s>>>(selected, n_pre, k, indptr);
  BS_CHECK_LAUNCH();
  if (out && (int64_t)n_pre * k > 0) {
    k_sel_copy<<<bs_num_cus() * 8, 256, 0, s>>>(indices, selected, indptr, n_pre, k, out);
    BS_CHECK_LAUNCH();
  }
  return BS_OK;
}

extern "C" int bs_conn_fixed_num_unique(uint64_t seed, int32_t n_pre, int32_t k, int32_t n_post,
                                        int32_t* indices, bs_stream_t stream) {
  bs_clear_error();
  BS_CHECK_ARG(n_pre >= 0 && k >= 0 && n_post >= 1, "bs_conn_fixed_num_unique: bad sizes");
  BS_CHECK_ARG(k <= n_post, "bs_conn_fixed_num_unique: K=%d distinct targets out of %d", k,
               n_post);
  BS_CHECK_ARG(k <= kUniqMax, "bs_conn_fixed_num_unique: K=%d above %d", k, kUniqMax);
  BS_CHECK_ARG(indices || (int64_t)n_pre * k == 0, "bs_conn_fixed_num_unique: indices is NULL");
  if ((int64_t)n_pre * k == 0) return BS_OK;
  int grid = bs_num_cus() * 8;
  if (grid > n_pre) grid = n_pre;
  k_unique_rows<<<grid, kUniqBlock, 0, bs_stream(stream)>>>(
      (uint32_t)seed, (uint32_t)(seed >> 32), n_pre, k, n_post, indices);
  BS_CHECK_LAUNCH();
  return BS_OK;
}
