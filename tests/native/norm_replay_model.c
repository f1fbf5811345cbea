/*
 * CPU model of the library's replay of an fp32 fused-multiply-add chain s = fma(x, x, s), the
 * accumulation order of torch's CPU norm(2) (came_amd/csrc/came8_norm.h), written to check its
 * exactness argument against the serial chain on adversarial inputs.  Test infrastructure only.
 *
 * Segment records follow the kernel's rules: a segment holds 512 chain elements; lane l of `lanes` (64, or
 * the 16 of the kernel that takes several segments a wavefront) accounts elements lanes * q + l in two fp32
 * sums of fused multiply-adds, one started at 2^E (even mantissa) and one a unit 2^(E-23) above it (odd).  A
 * lane's value is the first sum less its start in units, or 2^24 when that is 2^23 or more (the sum left the
 * binade, or met a NaN or an infinity), when the sums are not one unit apart any more (a tie, which rounds to
 * the even side), or for E = 128, the binade above the largest; the segment's value is the lanes' integer
 * sum, at most 2^24.
 * The walk skips a segment whose record covers the chain's binade when m + value < 2^24 and replays
 * the others.  A replay (segment_replay) follows the kernel's wavefront form: lane l holds the chain
 * elements 8l .. 8l + 7 of the segment; each round takes every lane's increments under the chain's current
 * binade as prefixes from the same pair of sums (elements already applied count as 0), a saturating prefix of
 * the lanes' totals, and the first element where a lane's pair shows an exception or the prefix leaves the
 * binade; the elements before it are one integer add, that element is one fmaf, and the next round starts
 * after it.  A chain at zero takes its elements one by one.
 */
#include <math.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

static int binade(float s) {
  uint32_t b;
  memcpy(&b, &s, 4);
  int e = (int)(b >> 23);
  return e == 0 ? -126 : e - 127;
}
static int est_binade(double v) {
  if (!(v > 0x1p-125)) return -126;
  if (!(v <= 0x1.fffffep127)) return 127;
  return binade((float)v);
}
static float from_bits(uint32_t b) {
  float v;
  memcpy(&v, &b, 4);
  return v;
}
static uint32_t to_bits(float v) {
  uint32_t b;
  memcpy(&b, &v, 4);
  return b;
}
static uint32_t lane_value(float even, float odd, int E) {
  const uint32_t base = (uint32_t)(E + 127) << 23;
  const uint32_t n = to_bits(even) - base;
  return n < (1u << 23) && to_bits(odd) - base == n + 1u && E < 128 ? n : (1u << 24);
}
/* the record of cnt <= 512 chain elements x[0 .. cnt) under binade E (-126 .. 128) */
uint32_t seg_value(const float* x, int64_t cnt, int E, int lanes) {
  const uint32_t base = (uint32_t)(E + 127) << 23;
  uint64_t tot = 0;
  for (int lane = 0; lane < lanes; ++lane) {
    float even = from_bits(base), odd = from_bits(base + 1u);
    for (int64_t k = lane; k < 512; k += lanes) {
      const float v = k < cnt ? x[k] : 0.0f;
      even = fmaf(v, v, even);
      odd = fmaf(v, v, odd);
    }
    tot += lane_value(even, odd, E);
  }
  return tot > (1u << 24) ? (1u << 24) : (uint32_t)tot;
}

#define SAT (1u << 25)
static uint32_t sat_add(uint32_t a, uint32_t b) {
  uint32_t v = a + b;
  return v < SAT ? v : SAT;
}
static float value_of(uint32_t m, int E) { return from_bits(((uint32_t)(E + 126) << 23) + m); }

/* one segment of cnt <= 512 chain elements x[0 .. cnt) from s; *rounds counts the rounds */
float segment_replay(const float* x, int cnt, float s, int64_t* rounds) {
  if (s == 0.0f) {
    for (int k = 0; k < cnt; ++k) s = fmaf(x[k], x[k], s);
    return s;
  }
  int pos = 0;
  while (pos < cnt) {
    ++*rounds;
    if (!(s <= 0x1.fffffep127f)) { /* +inf or NaN: only a NaN element changes an infinite chain */
      if (s != s) break;
      int first = -1;
      for (int k = pos; k < cnt; ++k)
        if (x[k] != x[k]) { first = k; break; }
      if (first >= 0) s = fmaf(x[first], x[first], s);
      break;
    }
    const int E = binade(s);
    const uint32_t m = to_bits(s) - ((uint32_t)(E + 126) << 23);
    const uint32_t room = (1u << 24) - m;
    const uint32_t base = (uint32_t)(E + 127) << 23;
    uint32_t incl[512], excl[64], acc = 0;
    int event[512];
    for (int lane = 0; lane < 64; ++lane) {
      float even = from_bits(base), odd = from_bits(base + 1u);
      for (int j = 0; j < 8; ++j) {
        const int k = lane * 8 + j;
        const float v = k >= pos && k < cnt ? x[k] : 0.0f;
        even = fmaf(v, v, even);
        odd = fmaf(v, v, odd);
        incl[k] = to_bits(even) - base;
        event[k] = incl[k] >= (1u << 23) || to_bits(odd) - base != incl[k] + 1u;
      }
      excl[lane] = acc;
      acc = sat_add(acc, incl[lane * 8 + 7] < SAT ? incl[lane * 8 + 7] : SAT);
    }
    int ev = -1;
    for (int k = 0; k < 512 && ev < 0; ++k)
      if (event[k] || excl[k / 8] + (incl[k] < SAT ? incl[k] : SAT) >= room) ev = k;
    if (ev < 0) {
      s = value_of(m + acc, E);
      break;
    }
    const int lane = ev / 8, j = ev % 8;
    const uint32_t before = excl[lane] + (j > 0 ? incl[ev - 1] : 0u);
    s = value_of(m + before, E);
    s = fmaf(x[ev], x[ev], s);
    pos = ev + 1;
  }
  return s;
}

float chain_serial_from(const float* x, int64_t n, float s) {
  for (int64_t k = 0; k < n; ++k) s = fmaf(x[k], x[k], s);
  return s;
}

float chain_serial(const float* x, int64_t n) {
  float s = 0.0f;
  for (int64_t k = 0; k < n; ++k) s = fmaf(x[k], x[k], s);
  return s;
}

/* est[g]: estimated chain value at the start of segment g; lanes: of a segment's records; returns the chain,
   *replays the count of replayed segments (the first one always is) and *rounds the wavefront rounds they took */
float chain_replay_stats(const float* x, int64_t n, const double* est, int lanes, int64_t* replays, int64_t* rounds) {
  const int L = 512;
  int64_t nseg = (n + L - 1) / L;
  int* Ea = malloc(sizeof(int) * (nseg ? nseg : 1));
  int* two = malloc(sizeof(int) * (nseg ? nseg : 1));
  uint32_t* wa = malloc(sizeof(uint32_t) * (nseg ? nseg : 1));
  uint32_t* wb = malloc(sizeof(uint32_t) * (nseg ? nseg : 1));
  for (int64_t g = 0; g < nseg; ++g) {
    int64_t k0 = g * L, cnt = n - k0 < L ? n - k0 : L;
    Ea[g] = est_binade(est[g] * 0.875);
    two[g] = est_binade(est[g] * 1.015625) > Ea[g];
    wa[g] = seg_value(x + k0, cnt, Ea[g], lanes);
    wb[g] = two[g] ? seg_value(x + k0, cnt, Ea[g] + 1, lanes) : (1u << 24);
  }
  float s = 0.0f;
  *replays = 0;
  *rounds = 0;
  for (int64_t g = 0; g < nseg && s == s; ++g) {
    int64_t k0 = g * L, cnt = n - k0 < L ? n - k0 : L;
    int ok = 0;
    if (g == 0) {
      ok = 0; /* from zero, without its record */
    } else if (s <= 0x1.fffffep127f) {
      int E = binade(s);
      uint32_t b;
      memcpy(&b, &s, 4);
      uint32_t m = b - ((uint32_t)(E + 126) << 23);
      uint32_t add = E == Ea[g] ? wa[g] : ((two[g] && E == Ea[g] + 1) ? wb[g] : (1u << 25));
      if ((uint64_t)m + add < (1u << 24)) {
        uint32_t r = ((uint32_t)(E + 126) << 23) + m + add;
        memcpy(&s, &r, 4);
        ok = 1;
      }
    } else if (wa[g] < (1u << 24) || (two[g] && wb[g] < (1u << 24))) {
      ok = 1; /* s = +inf and no element of the segment can be NaN */
    }
    if (!ok) {
      ++*replays;
      s = segment_replay(x + k0, (int)cnt, s, rounds);
    }
  }
  free(Ea);
  free(two);
  free(wa);
  free(wb);
  return s;
}

float chain_replay(const float* x, int64_t n, const double* est, int lanes, int64_t* replays) {
  int64_t rounds = 0;
  return chain_replay_stats(x, n, est, lanes, replays, &rounds);
}
