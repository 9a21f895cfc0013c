// Jump-ahead polynomials of MT19937 (host code, no HIP): x^J mod P over GF(2), P the
// characteristic polynomial of the word recurrence x[n+624] = x[n+397] ^ f(x[n], x[n+1]).
//
// Every bit of the state words satisfies the linear recurrence whose characteristic
// polynomial is P (degree 19937), so x[n + J] = XOR of x[n + i] over the set bits i of
// x^J mod P, for whole words and any n >= 1 (Haramoto, Matsumoto, Nishimura, Panneton and
// L'Ecuyer, "Efficient jump ahead for F2-linear random number generators", 2008).  At n = 0
// only the top bit of x[0] takes part in the recurrence, and only the top bit of a window's
// first word is ever read again, so the window of 624 words that starts at J follows.
//
// P comes from the recurrence's own constants (Matsumoto and Nishimura 1998, appendix A):
// with T = t^624 + t^397, U = t^623 + t^396 and a_i bit i of the twist constant,
//   P = T (U^31 + a_0 U^30 + ... + a_30) + a_31,
// 135 terms, the second highest at 19314: a reduction may fold 64 bits at a time.
#pragma once

#include <stdint.h>
#include <string.h>

#include <mutex>

namespace mt_jump {

constexpr int kDeg = 19937;
constexpr int kW64 = 312;              // 64-bit words of a residue (31 spare bits, zero)
constexpr int kWords = 2 * kW64;       // the same in 32-bit words: 624
constexpr int kMaxE = 28;              // x^(624 * 2^e), e <= kMaxE
constexpr uint32_t kTwistA = 0x9908b0dfu;

struct Poly {
  uint64_t w[kW64];
};

// dst ^= v << bit (v 64 bits wide)
inline void xor_at(uint64_t* dst, uint64_t v, int bit) {
  const int q = bit >> 6, r = bit & 63;
  dst[q] ^= v << r;
  if (r) dst[q + 1] ^= v >> (64 - r);
}

// Exponents of P below kDeg.
struct Terms {
  int n = 0;
  int e[160];
  Terms() {
    uint64_t h[kW64 + 2] = {1}, t[kW64 + 2];
    for (int i = 0; i <= 31; ++i) {  // Horner in U, then one factor T
      const int s = i < 31 ? 1 : 0;
      memset(t, 0, sizeof(t));
      for (int w = 0; w < kW64 - 9; ++w)
        if (h[w]) {
          xor_at(t, h[w], 64 * w + 624 - s);
          xor_at(t, h[w], 64 * w + 397 - s);
        }
      t[0] ^= (kTwistA >> i) & 1u;
      memcpy(h, t, sizeof(h));
    }
    for (int b = 0; b < kDeg; ++b)
      if ((h[b >> 6] >> (b & 63)) & 1u) e[n++] = b;
  }
};

// v (2 * kW64 words) reduced mod P into out.
inline void reduce(const Terms& P, uint64_t* v, Poly* out) {
  for (int w = 2 * kW64 - 1; w >= kW64; --w) {
    const uint64_t hi = v[w];
    if (!hi) continue;
    v[w] = 0;
    for (int i = 0; i < P.n; ++i) xor_at(v, hi, 64 * w - kDeg + P.e[i]);
  }
  const int top = kDeg & 63;  // bits kDeg.. of the last word kept
  const uint64_t hi = v[kW64 - 1] >> top;
  if (hi) {
    v[kW64 - 1] &= (1ull << top) - 1;
    for (int i = 0; i < P.n; ++i) xor_at(v, hi, P.e[i]);
  }
  memcpy(out->w, v, sizeof(out->w));
}

inline uint64_t spread(uint32_t x) {  // bit i -> bit 2i
  uint64_t v = x;
  v = (v | (v << 16)) & 0x0000ffff0000ffffull;
  v = (v | (v << 8)) & 0x00ff00ff00ff00ffull;
  v = (v | (v << 4)) & 0x0f0f0f0f0f0f0f0full;
  v = (v | (v << 2)) & 0x3333333333333333ull;
  return (v | (v << 1)) & 0x5555555555555555ull;
}

inline void square(const Terms& P, const Poly& a, Poly* out) {
  uint64_t v[2 * kW64 + 1];
  for (int w = 0; w < kW64; ++w) {
    v[2 * w] = spread((uint32_t)a.w[w]);
    v[2 * w + 1] = spread((uint32_t)(a.w[w] >> 32));
  }
  v[2 * kW64] = 0;
  reduce(P, v, out);
}

// a * b mod P, four bits of a at a time.
inline void multiply(const Terms& P, const Poly& a, const Poly& b, Poly* out) {
  static thread_local uint64_t tab[16][kW64 + 1];
  memset(tab[0], 0, sizeof(tab[0]));
  memcpy(tab[1], b.w, sizeof(b.w));
  tab[1][kW64] = 0;
  for (int k = 2; k < 16; ++k)
    for (int w = 0; w <= kW64; ++w)
      tab[k][w] = k & 1 ? tab[k - 1][w] ^ tab[1][w]
                        : (tab[k / 2][w] << 1) | (w ? tab[k / 2][w - 1] >> 63 : 0);
  uint64_t v[2 * kW64 + 1];
  memset(v, 0, sizeof(v));
  for (int s = 60; s >= 0; s -= 4) {
    if (s != 60)
      for (int w = 2 * kW64; w >= 0; --w) v[w] = (v[w] << 4) | (w ? v[w - 1] >> 60 : 0);
    for (int w = 0; w < kW64; ++w) {
      const uint64_t* t = tab[(a.w[w] >> s) & 15];
      for (int j = 0; j <= kW64; ++j) v[w + j] ^= t[j];
    }
  }
  reduce(P, v, out);
}

// {x^J, x^2J, x^3J} mod P for J = 624 * 2^e; nullptr when e is out of range.  Constants of the
// generator, formed on first use (squares about 30 us each, x^3J 0.5 ms) and kept.
inline const Poly* powers(int e) {
  static Poly sq[kMaxE + 2];
  static Poly t[kMaxE + 1][3];
  static bool done[kMaxE + 1];
  static int have = 0;
  static std::mutex mu;
  static const Terms P;
  if (e < 0 || e > kMaxE) return nullptr;
  std::lock_guard<std::mutex> lock(mu);
  if (done[e]) return t[e];
  sq[0].w[624 >> 6] = 1ull << (624 & 63);
  for (; have < e + 1; ++have) square(P, sq[have], &sq[have + 1]);
  t[e][0] = sq[e];
  t[e][1] = sq[e + 1];
  multiply(P, sq[e], sq[e + 1], &t[e][2]);
  done[e] = true;
  return t[e];
}

// init_genrand: the 624 state words of a 32-bit seed.
inline void seed_state(uint32_t seed, uint32_t* x) {
  for (int i = 0; i < 624; ++i) {
    x[i] = seed;
    seed = 1812433253u * (seed ^ (seed >> 30)) + (uint32_t)(i + 1);
  }
}

}  // namespace mt_jump
