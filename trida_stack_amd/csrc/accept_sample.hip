// Sampled self-spec acceptance (speculative rejection sampling with top-k / top-p truncation).
//
// Three launches on the caller's stream:
//   truncate (grid rows): one 512-thread block per verify row finds the truncated distribution's
//       statistics: m = max y (y = logit / T, the banned id at -inf), thr = the smallest kept y and
//       Zk = sum over kept y of exp(y - m), so that P(x) = [y_x >= thr] exp(y_x - m) / Zk.
//       An evenly spaced 2048-element sample of the row places a window that should hold the truncation
//       boundary; ONE streaming pass, in four segments spread over the row, then accumulates the row max, a
//       histogram of the values that can matter (the mass of the others, most of the row, stays in
//       registers) and collects the window's values into LDS, the window being placed anew from the
//       histogram after each segment. The boundary bin's values settle thr exactly. Segments whose window
//       missed are streamed again; rows out of the histogram's range (massive ties, |y| from 2^18
//       on) take an exact radix select over the order-preserving keys of
//       y, 8 bits per pass.
//       Bound by the instructions of 16 waves per CU beside the row's bytes (two rows per CU at a time). 512
//       rows of 248320, half of them peaked, against every element in the histogram: 231 -> 182 us at T = 0.7,
//       top_p = 0.95 (413 -> 123 at 0.5 / 0.8, 257 -> 250 at 1.2 / 0.98, where two thirds of a row are kept and the
//       boundary moves with each late token), 181 -> 113 with top_k = 50, 111 -> 94 (5.4 TB/s) untruncated; rows
//       of 248319, which scalar loads served: 572 -> 176. Widened bf16 rows take the same (177 at 0.7 / 0.95;
//       in the draft pass, behind the launch that has just written them, 210).
//   resid_sums (grid NC x B): every block re-derives its sequence's accepted length from the drafted
//       tokens' ratios P_i(d_i) / q_i(d_i), then sums the correction weights max(0, P_a - q_a) (P_K
//       when every draft is accepted) and P_a over its chunk of the vocabulary, in fp64.
//   resid_pick (grid B): inverse CDF in vocabulary order with one uniform: the chunk where the
//       cumulative weight first exceeds u * total, then the token inside it.
// Nothing allocates; scratch holds the per-row statistics and the chunk sums.
#include <limits.h>
#include <math.h>

#include <algorithm>

#include "common.h"

namespace trida {
namespace {

constexpr int kT = 512;  // threads of the truncation block
constexpr int kTW = kT / kWave;
constexpr int kSample = 2048;
constexpr int kCap = 12288;  // LDS collection capacity (values)
constexpr int kWaveCap = kCap / kTW;
constexpr int kSortCap = 8192;  // values sorted at a time (a power of two, <= kCap)
constexpr int kTopCount = 1024;  // entries at the top of a row that are always collected
constexpr int kU = 4;            // 16-byte loads in flight per thread
constexpr int kTileV = kT * kU;  // vectors per tile of the streaming pass
constexpr int kQueue = 384;      // a wave's queue: up to 127 waiting elements and 4 new ones per lane
constexpr int kSub = 1024;       // sub-bins of the boundary bin
constexpr int kBins = 256;  // digits of one radix pass
constexpr int kMaxTopK = 4096;
constexpr uint32_t kKeyLo = 0x00800000u;  // smallest finite key (key(-inf) + 1)
constexpr uint32_t kKeyHi = 0xff7fffffu;  // largest finite key (key(+inf) - 1)
constexpr int kRT = 256;                  // threads of the residual kernels

// Order-preserving map float -> uint32 (larger value, larger key) and its inverse.
__device__ __forceinline__ uint32_t fkey(float y) {
  const uint32_t u = __float_as_uint(y);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float kval(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// y = logit / T rounded to fp32 exactly as an IEEE fp32 division (the reference divides the fp32
// logits by the temperature), -0 folded into +0 so that equal values have equal keys, the banned id at
// -inf. rt = 1/T in fp64: the fp64 product is within 2^-52 (relative) of x/T, while x/T is never within
// 2^-48 of a midpoint between two floats unless it is one exactly, which needs T's odd significand
// times a 25-bit odd significand to fit 24 bits, i.e. T a power of two, where the product is exact.
// So rounding the fp64 product to fp32 gives the correctly rounded quotient, in three instructions.
template <bool kDiv>
__device__ __forceinline__ float exact_y(float x, double rt) {
  const float y = kDiv ? (float)((double)x * rt) : x;
  return y + 0.f;  // -0 + 0 = +0; every other value is unchanged
}
template <bool kDiv>
__device__ __forceinline__ float make_y(float x, int ix, double rt, int ban) {
  return (ix == ban) ? -INFINITY : exact_y<kDiv>(x, rt);
}

__device__ __forceinline__ int next_pow2(int n) {
  int p = 1;
  while (p < n) p <<= 1;
  return p;
}

// Value histogram of the streaming pass: 2048 bins of 1/32 nat over d = y - mref in (-24, 40]
// (mref = the sample max, rounded to a bin); bin 0 holds the largest values. Bin kNB is the spare bin: entries with d > 40, which are
// caught afterwards from the row max and send the row to the radix select, and a few at the lower end. The
// others with d <= -24, -inf entries, the banned id and padding lanes only add their mass to the total.
// Each bin is one 64-bit LDS word: the count in bits 46..63 and, below, the sum of r * 2^26 with
// r = exp(d - top of the bin) in (e^-1/32, 1]: one integer LDS atomic per element (fp64 and fp32 LDS
// atomics measured several times slower on gfx950). Rows need V < 2^18 for the count field.
constexpr int kNB = 2048;
constexpr float kTop = 40.f;
constexpr float kPerNat = 32.f;
constexpr double kBinRatio = 0x1.f03f56a88b5d8p-1;  // exp(-1 / kPerNat): the scale of bin b + 1 over bin b
constexpr int kSeg = 4;  // the streaming pass re-places its collection window between segments
constexpr int kCountShift = 46;
constexpr unsigned long long kMassMask = (1ull << kCountShift) - 1ull;
constexpr int kMaxPackedV = (1 << 18) - 1;

struct Shared {
  float coll[kCap];           // the streaming pass: kWaveCap slots per wave; afterwards packed at the front
  float queue[kTW][kQueue];  // each wave's elements above the floor, waiting to be folded 128 at a time
  unsigned long long hist[kNB + 1];
  unsigned cnt[kBins];  // radix-select digits
  double mass[kBins];
  double red[kTW];
  int n;
  int ipar[6];
  int wlo[kSeg], whi[kSeg];  // the window each segment collected (bins, inclusive)
  int top[kSeg];             // and the bins [0, top)
  int nseg[kSeg][kTW];       // each wave's collected values after each segment (past kWaveCap: some were dropped)
  double dpar[4];
  unsigned umax;
};
// The truncation block's LDS. Everything the kernel calls is inlined: with real functions for its rare steps it
// needs a stack, and every launch was 10 us longer.
__shared__ Shared sh;

// ---------------------------------------------------------------- block reductions (512 threads)
__device__ __forceinline__ double block_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
  __syncthreads();
  if (threadIdx.x % kWave == 0) sh.red[threadIdx.x / kWave] = v;
  __syncthreads();
  double t = 0.0;
#pragma unroll
  for (int w = 0; w < kTW; ++w) t += sh.red[w];
  return t;
}
__device__ __forceinline__ float block_max(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, kWave));
  __syncthreads();
  if (threadIdx.x % kWave == 0) sh.red[threadIdx.x / kWave] = v;
  __syncthreads();
  float t = -INFINITY;
#pragma unroll
  for (int w = 0; w < kTW; ++w) t = fmaxf(t, (float)sh.red[w]);
  return t;
}
__device__ __forceinline__ int block_isum(int v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
  __syncthreads();
  if (threadIdx.x % kWave == 0) sh.red[threadIdx.x / kWave] = (double)v;
  __syncthreads();
  int t = 0;
#pragma unroll
  for (int w = 0; w < kTW; ++w) t += (int)sh.red[w];
  return t;
}
// Exclusive prefix sum over the block in thread order; *total gets the block total.
__device__ __forceinline__ double block_excl_scan(double v, double* total) {
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
  double inc = v;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const double o = __shfl_up(inc, off, kWave);
    if (lane >= off) inc += o;
  }
  double ex = __shfl_up(inc, 1, kWave);
  if (lane == 0) ex = 0.0;
  __syncthreads();
  if (lane == kWave - 1) sh.red[w] = inc;
  __syncthreads();
  double base = 0.0, tot = 0.0;
#pragma unroll
  for (int i = 0; i < kTW; ++i) {
    base += (i < w) ? sh.red[i] : 0.0;
    tot += sh.red[i];
  }
  *total = tot;
  return base + ex;
}

// Bitonic sort, descending, of s[0..n) (n a power of two); starts and ends with a barrier.
__device__ void sort_desc(int n) {
  float* s = sh.coll;
  __syncthreads();
  if (n <= kT) {  // a few elements per lane of one wave, whose LDS operations complete in order: no barriers
    if (threadIdx.x < kWave) {
      for (int k = 2; k <= n; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
          for (int i = threadIdx.x; i < (n >> 1); i += kWave) {
            const int lo = ((i & ~(j - 1)) << 1) | (i & (j - 1));
            const int hi = lo + j;
            const float a = s[lo], b = s[hi];
            const bool sw = (lo & k) == 0 ? a < b : a > b;
            s[lo] = sw ? b : a;
            s[hi] = sw ? a : b;
          }
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          __builtin_amdgcn_wave_barrier();
        }
    }
    __syncthreads();
    return;
  }
  for (int k = 2; k <= n; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = threadIdx.x; i < (n >> 1); i += kT) {
        const int lo = ((i & ~(j - 1)) << 1) | (i & (j - 1));
        const int hi = lo + j;
        const float a = s[lo], b = s[hi];
        const bool desc = (lo & k) == 0;
        if (desc ? (a < b) : (a > b)) {
          s[lo] = b;
          s[hi] = a;
        }
      }
      __syncthreads();
    }
}

// Appends y (where pred) to s_coll through one LDS counter bump per wave; the counter keeps counting
// past kCap so that an overflow is visible. Called by every lane of the wave.
__device__ __forceinline__ void append(float y, bool pred) {
  const uint64_t bal = __ballot(pred);
  if (bal == 0) return;
  const int lane = threadIdx.x % kWave;
  int base = 0;
  if (lane == 0) base = atomicAdd(&sh.n, __popcll(bal));
  base = __shfl(base, 0, kWave);
  const int slot = base + __popcll(bal & ((1ull << lane) - 1ull));
  if (pred && slot < kCap) sh.coll[slot] = y;
}

// A row as its 16-byte aligned vectors [0, n4) and the <= 6 elements in front of and behind them (a row
// of an odd vocabulary starts anywhere in a 16-byte line).
struct RowView {
  const float* row;
  const u32x4* body;
  int pre, n4, V;
  __device__ RowView(const float* r, int v) : row(r), V(v) {
    pre = min((int)((0u - (unsigned)((uintptr_t)r >> 2)) & 3u), v);
    body = reinterpret_cast<const u32x4*>(r + pre);
    n4 = (v - pre) >> 2;
  }
  // id of edge element j (the elements outside the vectors, in order), V past the last one
  __device__ int edge(int j) const { return min(j < pre ? j : j + 4 * n4, V); }
};

// Calls f(y, ix, valid) for every element of a row; U 16-byte loads in flight per thread.
template <bool kDiv, int U = 4, typename F>
__device__ __forceinline__ void for_each_y(const RowView& rv, double rt, int ban, F&& f) {
  const int tid = threadIdx.x;
  for (int base = 0; base < rv.n4; base += kT * U) {
    u32x4 x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = rv.body[min(base + u * kT + tid, rv.n4 - 1)];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = base + u * kT + tid;
      const bool ok = j < rv.n4;
      const float xs[4] = {__uint_as_float(x[u].x), __uint_as_float(x[u].y), __uint_as_float(x[u].z),
                           __uint_as_float(x[u].w)};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int ix = rv.pre + 4 * j + e;
        f(make_y<kDiv>(xs[e], ix, rt, ban), ix, ok);
      }
    }
  }
  const int ix = rv.edge(tid);
  const bool ok = ix < rv.V;
  f(make_y<kDiv>(rv.row[ok ? ix : 0], ix, rt, ban), ix, ok);
}

struct TruncArgs {
  const float* logits;
  int64_t batch_stride, row_stride;  // elements
  int R, V;
  double rt;    // 1 / temperature
  int top_k;    // active when 0 < top_k < V
  float top_p;  // active when < 1
  int ban;      // banned id (-1: none)
  int flags;    // bit 0: skip the window pass (exact radix select only)
  int G, first;       // row group: block j of sequence b handles row first + j (rows >= R are skipped)
  const int* state;   // per sequence: -1 = every row so far accepted; >= 0 = decided (skip); null: none
  float* m_out;
  float* thr_out;
  double* zk_out;
  int* status_out;
  int* passes_out;
};

// Bin of an element from its raw logit x: t = 32 (40 - d) with d = x / T - mref, as one fma whose
// coefficients the block derives once (tA = -32 / T, tB = 32 (40 + mref)). Monotone in x.
__device__ __forceinline__ unsigned bin_of_t(float t) {
  return min((unsigned)(int)__builtin_amdgcn_fmed3f(t, -1.f, (float)kNB), (unsigned)kNB);
}
// exp(top of the bin) relative to exp(mref); consecutive bins scale by kBinRatio
__device__ __forceinline__ double bin_scale(int bin) { return exp((double)kTop - (double)bin / kPerNat); }
__device__ __forceinline__ double bin_mass(unsigned long long h, double scale) {  // relative to exp(mref)
  return ldexp((double)(h & kMassMask), -26) * scale;
}

struct BinMap {  // the per-row coefficients of the element -> bin / exponent maps
  float tA, tB;       // t = fma(x, tA, tB)
  float nm;           // -mref
  double rt;          // 1 / T
  float eA, eL, eB;   // exp(d) = exp2(cold_exp(x)) * cold_scale
  double cold_scale;  // what the rounding of eB took away
  __device__ unsigned bin(float x) const { return bin_of_t(fmaf(x, tA, tB)); }
  // an element's histogram entry: a count of one and its mass relative to its bin's upper edge
  __device__ unsigned long long packed(float x, unsigned bin) const {
    // y = x / T as the kept set and the probabilities round it (a likely token's y of 16..32 rounds by up to 1e-6,
    // which would be an error of its mass); mref and the edge are multiples of 2^-5, so that d is exact
    const float edge = fmaf((float)bin, -1.f / kPerNat, kTop);
    const float d = exact_y<true>(x, rt) + (nm - edge);
    const float r = __builtin_amdgcn_exp2f(d * 1.44269504f) * 0x1p26f;
    return (1ull << kCountShift) | (unsigned long long)(unsigned)r;
  }
  __device__ void set(double rt_, float mref) {
    rt = rt_;
    tA = -kPerNat * (float)rt;
    tB = kPerNat * (kTop + mref);
    nm = -mref;
    const double l2e = 1.4426950408889634, s = rt * l2e;
    // eA: the 16 leading bits of s less one unit of them; eL, the rest, is positive (x = -inf stays -inf) and never tiny
    eA = __uint_as_float((__float_as_uint((float)s) & 0xffffff00u) - 0x100u);
    eL = (float)(s - (double)eA);
    eB = (float)(-(double)mref * l2e);
    cold_scale = exp2(-(double)mref * l2e - (double)eB);
  }
  // log2(e) d + const in two products, the slope log2(e) / T held to 40 bits. With one fp32 slope every exponent was off
  // by up to 2^-24 |x / T|, the same way for the whole row; with eL at 2^-24 of eA its product, mostly less than half a
  // unit of the first sum, was rounded away for the whole row alike. As it is, the roundings of a row's entries are
  // independent. Normaliser error of untruncated rows at T = 1, one slope -> two: 5.6e-8 -> 3e-9 without a
  // shift, 1.4e-6 -> 3e-9 at logits of about 100, 1.3e-5 -> 5e-9 at 1000; 0.5 to 1 us of 96 per 512 rows.
  __device__ float cold_exp(float x) const { return fmaf(x, eL, fmaf(x, eA, eB)); }
};

// Count of j < lim with base + sum_{i<j} e_i < target, e_i = exp(s_i - m) in fp64 (a prefix, since
// the partial sums only grow); *tot = sum_{j<lim} e_j.
__device__ int count_below(int lim, double m, double base, double target, double* tot) {
  const float* s = sh.coll;
  const int L = (lim + kT - 1) / kT;
  const int j0 = min(lim, (int)threadIdx.x * L), j1 = min(lim, j0 + L);
  double loc = 0.0;
  for (int j = j0; j < j1; ++j) loc += exp((double)s[j] - m);
  const double ex = block_excl_scan(loc, tot);
  int c = 0;
  double run = base + ex;
  for (int j = j0; j < j1; ++j) {
    c += run < target;
    run += exp((double)s[j] - m);
  }
  return block_isum(c);
}

// sum over j < n with s_j >= thr of exp(s_j - m)
__device__ double mass_at_least(int n, float thr, double m) {
  const float* s = sh.coll;
  double loc = 0.0;
  for (int j = threadIdx.x; j < n; j += kT) loc += (s[j] >= thr) ? exp((double)s[j] - m) : 0.0;
  return block_sum(loc);
}

__device__ int count_cmp(int n, float v, bool strictly_greater) {
  const float* s = sh.coll;
  int c = 0;
  for (int j = threadIdx.x; j < n; j += kT) c += strictly_greater ? (s[j] > v) : (s[j] == v);
  return block_isum(c);
}

// Pads the collection to a power of two with -inf and sorts it (descending).
__device__ void sort_collection(int n) {
  const int np = next_pow2(max(n, 2));
  for (int j = n + threadIdx.x; j < np; j += kT) sh.coll[j] = -INFINITY;
  sort_desc(np);
}

// One fallback pass over the keys: counts/mass (relative to the exact max m) above khi, and either a
// histogram of [klo, khi] in digits of 2^shift keys or a collection of that range. On want_z it also
// sums the whole row's mass and counts its finite entries.
template <bool kDiv, bool kHist>
__device__ void range_pass(const RowView& rv, const TruncArgs& a, float m, uint32_t klo, uint32_t khi, int shift,
                           bool want_z, int* ca_out, double* ma_out, double* z_out, int* cf_out) {
  if (kHist)
    for (int j = threadIdx.x; j < kBins; j += kT) {
      sh.cnt[j] = 0u;
      sh.mass[j] = 0.0;
    }
  if (threadIdx.x == 0) sh.n = 0;
  __syncthreads();
  int ca = 0, cf = 0;
  double ma = 0.0, z = 0.0;
  for_each_y<kDiv, 2>(rv, a.rt, a.ban, [&](float y, int ix, bool ok) {
    const bool fin = ok && (y > -INFINITY);
    const uint32_t key = fkey(y);
    const float e = __expf(y - m);
    const bool above = fin && key > khi;
    const bool in = fin && key >= klo && key <= khi;
    ca += above;
    ma += above ? e : 0.f;
    if (want_z) {
      z += fin ? e : 0.f;
      cf += fin;
    }
    if (kHist) {
      if (in) {
        const int bin = (int)((key - klo) >> shift);
        atomicAdd(&sh.cnt[bin], 1u);
        atomicAdd(&sh.mass[bin], (double)e);
      }
    } else {
      append(y, in);
    }
  });
  *ca_out = block_isum(ca);
  *ma_out = block_sum(ma);
  if (want_z) {
    *z_out = block_sum(z);
    *cf_out = block_isum(cf);
  }
  __syncthreads();
}

// Exact radix select with the exact row max m. Count mode (use_k): the top_k-th largest value; mass
// mode: the smallest y whose strictly-greater mass is < top_p * Z. Writes thr / Zk (relative to m).
template <bool kDiv>
__device__ __forceinline__ void radix_resolve(const RowView& rv, const TruncArgs& a, float m, bool use_k, bool use_p,
                              float* thr_out, double* zk_out, int* passes) {
  const double md = (double)m;
  uint32_t klo = kKeyLo, khi = kKeyHi;
  int shift = 24;
  int ca = 0, cf = 0;
  double ma = 0.0, Z = 0.0, z = 0.0;
  bool count_mode = use_k;
  const int k = a.top_k;
  double tp = 0.0;
  // results of the select
  float v = -INFINITY;  // count mode: kth; mass mode: thr
  int c_gt = 0, c_eq = 0;
  double zk = 0.0;
  bool resolved = false;
  for (int it = 0; !resolved; ++it) {
    range_pass<kDiv, true>(rv, a, m, klo, khi, shift, it == 0, &ca, &ma, &z, &cf);
    ++*passes;
    if (it == 0) {
      Z = z;
      if (count_mode && cf <= k) count_mode = false;  // fewer finite entries than k: top-k keeps them all
      if (!count_mode && !use_p) {                    // nothing left to select
        *thr_out = -INFINITY;
        *zk_out = Z;
        return;
      }
      tp = (double)a.top_p * Z;
    }
    if (threadIdx.x == 0) {
      const int nb = (int)(((uint64_t)khi - klo) >> shift) + 1;
      double cum = count_mode ? (double)ca : ma;
      int pick = -1, last = -1;
      double cum_last = cum;
      for (int bin = nb - 1; bin >= 0; --bin) {
        if (sh.cnt[bin] == 0u) continue;
        const double add = count_mode ? (double)sh.cnt[bin] : sh.mass[bin];
        if ((count_mode && cum + add >= (double)k) || (!count_mode && cum + add >= tp)) {
          pick = bin;
          break;
        }
        last = bin;
        cum_last = cum;
        cum += add;
      }
      if (pick < 0) {  // mass mode: every entry qualifies, so the smallest one is the threshold
        pick = max(last, 0);
        cum = cum_last;
      }
      sh.ipar[0] = pick;
      sh.dpar[0] = cum;  // count or mass strictly above the picked digit
    }
    __syncthreads();
    const int pick = sh.ipar[0];
    const double cum = sh.dpar[0];
    const uint32_t nlo = klo + ((uint32_t)pick << shift);
    const uint32_t nhi = (uint32_t)min((uint64_t)khi, (uint64_t)nlo + (1ull << shift) - 1ull);
    const unsigned cnt = sh.cnt[pick];
    const double bmass = sh.mass[pick];
    __syncthreads();
    if (nlo == nhi) {  // one key: every entry of the digit has the same value
      v = kval(nlo);
      if (count_mode) {
        c_gt = (int)cum;
        c_eq = (int)cnt;
      } else {
        zk = cum + bmass;
      }
      resolved = true;
    } else if (cnt <= (unsigned)kSortCap) {
      klo = nlo;
      khi = nhi;
      int ca2 = 0, cf2 = 0;
      double ma2 = 0.0, z2 = 0.0;
      range_pass<kDiv, false>(rv, a, m, klo, khi, 0, false, &ca2, &ma2, &z2, &cf2);
      ++*passes;
      const int n = min(sh.n, kSortCap);
      sort_collection(n);
      if (count_mode) {
        v = sh.coll[min(max(k - 1 - ca2, 0), max(n - 1, 0))];
        c_gt = ca2 + count_cmp(n, v, true);
        c_eq = count_cmp(n, v, false);
      } else {
        double tot = 0.0;
        int nk = count_below(n, md, ma2, tp, &tot);
        nk = min(max(nk, 1), n);
        v = sh.coll[nk - 1];
        zk = ma2 + mass_at_least(n, v, md);
      }
      resolved = true;
    } else {
      klo = nlo;
      khi = nhi;
      shift = shift >= 8 ? shift - 8 : 0;
    }
  }
  if (!count_mode) {
    *thr_out = v;
    *zk_out = zk;
    return;
  }
  // top-k: the values above kth (fewer than k <= kMaxTopK, so they fit), then the nucleus over the
  // k-value list {values > kth} + (k - c_gt) copies of kth
  const float kth = v;
  int ca2 = 0, cf2 = 0;
  double ma2 = 0.0, z2 = 0.0;
  const uint32_t kk = fkey(kth);
  range_pass<kDiv, false>(rv, a, m, kk + 1u, kKeyHi, 0, false, &ca2, &ma2, &z2, &cf2);
  ++*passes;
  const int n = min(sh.n, kSortCap);
  sort_collection(n);
  const double e_k = exp((double)kth - md);
  double s_gt = 0.0;
  const double copies = (double)(k - c_gt);
  if (use_p) {
    double tot = 0.0;
    // total first: S = sum_{coll} e + copies * e_k
    (void)count_below(n, md, 0.0, -1.0, &tot);
    s_gt = tot;
    const double target = (double)a.top_p * (s_gt + copies * e_k);
    int nk = count_below(n, md, 0.0, target, &tot);
    int ncp = 0;
    for (int i = threadIdx.x; i < k - c_gt; i += kT) ncp += (s_gt + (double)i * e_k) < target;
    ncp = block_isum(ncp);
    nk = max(nk + ncp, 1);
    if (nk <= c_gt) {
      const float thr = sh.coll[nk - 1];
      *thr_out = thr;
      *zk_out = mass_at_least(n, thr, md);
      return;
    }
  } else {
    double tot = 0.0;
    (void)count_below(n, md, 0.0, -1.0, &tot);
    s_gt = tot;
  }
  *thr_out = kth;
  *zk_out = s_gt + (double)c_eq * e_k;
}

// Keeps the collected logits whose bin lies in [lo, hi] and that came from a segment in the bit set
// `segs` (entry j of wave w came from segment s when nseg[s-1][w] <= j < nseg[s][w]), packed at the front of
// sh.coll; returns how many.
__device__ __forceinline__ int compact_bins(const BinMap& bm, int lo, int hi, unsigned segs) {
  constexpr int kPer = kWaveCap / kT;  // steps per wave's slots
  static_assert(kWaveCap % kT == 0, "whole steps");
  float v[kTW * kPer];
  unsigned kp = 0u;
  const bool all = segs == (1u << kSeg) - 1u;
#pragma unroll
  for (int u = 0; u < kTW * kPer; ++u) {
    const int w = u / kPer, j = (u % kPer) * kT + (int)threadIdx.x, n = min(sh.nseg[kSeg - 1][w], kWaveCap);
    v[u] = -INFINITY;
    if ((u % kPer) * kT >= n) continue;  // block-uniform
    v[u] = j < n ? sh.coll[w * kWaveCap + j] : -INFINITY;
    const int bin = (int)bm.bin(v[u]);
    bool keep = j < n && bin >= lo && bin <= hi;
    if (!all) {
      int s = 0;
      while (s < kSeg - 1 && j >= sh.nseg[s][w]) ++s;
      keep = keep && ((segs >> s) & 1u);
    }
    kp |= (unsigned)keep << u;
  }
  double tot = 0.0;
  int at = (int)block_excl_scan((double)__popc(kp), &tot);  // every read of sh.coll precedes its barriers
#pragma unroll
  for (int u = 0; u < kTW * kPer; ++u)
    if ((kp >> u) & 1u) sh.coll[at++] = v[u];
  __syncthreads();
  return (int)tot;
}

// Segment s of the streaming pass: the row's tiles (kTileV vectors, the last one partial) number 0 mod 16;
// the other multiples of 4; the other even ones; the odd ones: 1/16, 3/16, 1/4 and 1/2 of the row, each
// spread over all of it (token ids are not exchangeable: a vocabulary's first ids are its frequent tokens).
// The edge elements belong to segment 0.
__device__ __forceinline__ int seg_tile(int s, int i) {
  if (s == 0) return 16 * i;
  if (s == 1) return 16 * (i / 3) + 4 * (i % 3 + 1);
  return s == 2 ? 4 * i + 2 : 2 * i + 1;
}
__device__ __forceinline__ int seg_size(const RowView& rv, int s) {
  const int nt = (rv.n4 + kTileV - 1) / kTileV, n16 = (nt + 15) / 16;
  const int cnt = s == 0 ? n16 : s == 1 ? (nt + 3) / 4 - n16 : s == 2 ? (nt + 1) / 4 : nt / 2;
  const int tl = nt - 1, sl = (tl & 1) ? 3 : (tl & 2) ? 2 : (tl & 15) ? 1 : 0;  // the last tile's segment
  int n = 4 * cnt * kTileV;
  if (nt > 0 && s == sl) n -= 4 * (nt * kTileV - rv.n4);
  return s == 0 ? n + rv.V - 4 * rv.n4 : n;
}

// The logit below which no element has a bin < b: bin b's lower edge, half a bin and the rounding of the
// element -> bin map further down.
__device__ __forceinline__ float below_bin(const BinMap& bm, int b) {
  return (bm.tB - ((float)b + 0.5f + 1e-6f * fabsf(bm.tB))) / -bm.tA;
}
// And above which no element has a bin >= b: bin b's upper edge, by the same margin further up.
__device__ __forceinline__ float above_bin(const BinMap& bm, int b) {
  return (bm.tB - ((float)b - 0.5f - 1e-6f * fabsf(bm.tB))) / -bm.tA;
}

// Streams a segment of the row in the logits' own units: the division by the temperature is folded into
// the bin / exponent maps, and the exact y = x / T is only formed for the few collected values.
// kHist: elements above x_lo (which lies below the floor, below_bin) wait in their wave's queue; each two
// full waves of 64 go to the histogram and, those with a bin in [wlo, whi] or below `top`, to the collection.
// The others only add their mass (relative to exp(mref), less the rounding of bm.eB) to `tail`: fp32 over a
// tile's 16 elements of a thread, fp64 across tiles. Without the queue every wave would run the 30 instructions of the
// histogram for each of its elements, as some lane always has one above the floor (the block issues 16 waves'
// instructions per CU, and the pass was bound by that: 33 a element, now 15 and 35 per element above the
// floor); and below the histogram's range its LDS atomics all met in one bin. A NaN makes `tail` NaN.
// Otherwise only the elements between x_lo and x_hi are looked at, and those of the bins [wlo, whi] collected.
template <bool kHist>
__device__ __forceinline__ void stream_segment(const RowView& rv, const TruncArgs& a, const BinMap& bm, int s, float x_lo,
                                               float x_hi, int top, int wlo, int whi, float& mx, double& tail,
                                               int& have) {
  const int tid = threadIdx.x, lane = tid % kWave;
  float* queue = sh.queue[tid / kWave];
  int fill = 0;  // wave-uniform
  const unsigned wspan = (unsigned)(whi - wlo);
  // folds the n (<= 128) elements at the end of the queue, two per lane. The collected values go to the wave's own
  // slots (kHist; `have` of them so far, wave-uniform), or behind a counter that the block shares.
  auto fold = [&](int n) {
    fill -= n;
    float x[2];
    uint64_t in[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int j = h * kWave + lane;
      x[h] = queue[fill + min(j, n - 1)];
      const unsigned bin = bm.bin(x[h]);
      bool keep = (unsigned)((int)bin - wlo) <= wspan;
      if (kHist) {
        keep = keep || (int)bin < top;
        if (j < n) atomicAdd(&sh.hist[bin], bm.packed(x[h], bin));
      }
      in[h] = __ballot(keep && j < n);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const bool mine = (in[h] >> lane) & 1ull;
      if (kHist) {
        const int at = have + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(in[h] >> 32),
                                                            __builtin_amdgcn_mbcnt_lo((uint32_t)in[h], 0u));
        if (mine && at < kWaveCap) sh.coll[(tid / kWave) * kWaveCap + at] = x[h];
        have += __popcll(in[h]);
      } else {
        append(x[h], mine);
      }
    }
  };
  auto push = [&](float x, bool hot) {
    const uint64_t bal = __ballot(hot);
    if (bal == 0) return;
    if (hot)
      queue[fill + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u))] = x;
    fill += __popcll(bal);
  };
  auto one = [&](float x, float& cold) {
    bool hot = x > x_lo;
    if (kHist) {
      mx = fmaxf(mx, x);
      const float e = __builtin_amdgcn_exp2f(bm.cold_exp(x));
      cold += hot ? 0.f : e;
    } else {
      hot = hot && x < x_hi;
    }
    push(x, hot);
  };
  // the next tile's loads are issued before the current tile is folded, so the fold hides their
  // latency; addresses are clamped to the last vector
  const int n4 = rv.n4;
  auto load = [&](u32x4 (&dst)[kU], int tile) {
#pragma unroll
    for (int u = 0; u < kU; ++u) dst[u] = rv.body[min(tile * kTileV + u * kT + tid, n4 - 1)];
  };
  const int nt = (n4 + kTileV - 1) / kTileV;
  u32x4 xn[kU];
  int tile = seg_tile(s, 0);
  if (tile < nt) load(xn, tile);
  for (int i = 0; tile < nt; ++i) {
    const int base = tile * kTileV;
    u32x4 x[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) x[u] = xn[u];
    tile = seg_tile(s, i + 1);
    if (tile < nt) load(xn, tile);
    // block-uniform: does this tile hold the banned id or padding lanes?
    const int e0 = rv.pre + 4 * base;
    const bool odd = base + kTileV > n4 || (unsigned)(a.ban - e0) < (unsigned)(4 * kTileV);
    float cold = 0.f;
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      float xv[4] = {__uint_as_float(x[u].x), __uint_as_float(x[u].y), __uint_as_float(x[u].z), __uint_as_float(x[u].w)};
      if (odd) {
        const int j = base + u * kT + tid;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (j >= n4 || rv.pre + 4 * j + e == a.ban) xv[e] = -INFINITY;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) one(xv[e], cold);
      while (fill >= 2 * kWave) fold(2 * kWave);
    }
    if (kHist) tail += (double)cold;
  }
  if (s == 0 && tid < kWave) {
    const int ix = rv.edge(tid);
    float cold = 0.f;
    one(ix < rv.V && ix != a.ban ? rv.row[ix] : -INFINITY, cold);
    if (kHist) tail += (double)cold;
  }
  while (fill > 0) fold(min(fill, 2 * kWave));
}

// ---------------------------------------------------------------- the histogram, read by one wave
// The steps between the segments run on the block's first wave: across all eight, the same few values computed
// by each, they cost the CU's two blocks 17k cycles apiece (7 us alone, 45 us beside a streaming block).
// Lane l holds the 32 bins [32 l, 32 l + 32) of the histogram: their mass (relative to exp(mref)) and count, and
// the inclusive sums over the lanes.
constexpr int kLB = kNB / kWave;
static_assert(kLB == 32, "a lane's bins are one nat");
struct LaneBins {
  double sc;        // bin_scale(32 l)
  double rk;        // kBinRatio^(l % 32)
  double im;        // inclusive mass
  unsigned ic;      // inclusive count
  double m;
  unsigned c;
  __device__ void init() {
    const int lane = threadIdx.x % kWave;
    sc = bin_scale(lane * kLB);
    rk = exp(-(double)(lane % kLB) / (double)kPerNat);
  }
  __device__ void load() {
    const int lane = threadIdx.x % kWave, k0 = lane % kLB;
    double ms = 0.0, r = sc * rk * 0x1p-26;
    unsigned cs = 0u;
    // bin (l + i) % 32 at step i: the lanes' reads fall on all banks
#pragma unroll 4
    for (int i = 0; i < kLB; ++i) {
      const int k = (k0 + i) % kLB;
      const unsigned long long h = sh.hist[lane * kLB + k];
      cs += (unsigned)(h >> kCountShift);
      ms += (double)(h & kMassMask) * r;
      r *= k == kLB - 1 ? kBinRatio * 0x1.5bf0a8b145769p+1 : kBinRatio;  // wraps by a factor of e
    }
    m = ms;
    c = cs;
    im = ms;
    ic = cs;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const double om = __shfl_up(im, off, kWave);
      const unsigned oc = (unsigned)__shfl_up((int)ic, off, kWave);
      im += lane >= off ? om : 0.0;
      ic += lane >= off ? oc : 0u;
    }
  }
  __device__ double mass() const { return __shfl(im, kWave - 1, kWave); }
  // the first bin at which the cumulative mass reaches tgt (> 0), -1 if none does; *before: the mass above it
  __device__ int find_mass(double tgt, double* before) const {
    const int lane = threadIdx.x % kWave;
    const uint64_t hit = __ballot(im >= tgt);
    if (hit == 0) return -1;
    const int L = __builtin_ctzll(hit);
    const double base = L > 0 ? __shfl(im, L - 1, kWave) : 0.0;
    const double sl = __shfl(sc, L, kWave) * rk * 0x1p-26;
    const double add = lane < kLB ? (double)(sh.hist[L * kLB + lane % kLB] & kMassMask) * sl : 0.0;
    double inc = add;
#pragma unroll
    for (int off = 1; off < kLB; off <<= 1) {
      const double o = __shfl_up(inc, off, kWave);
      inc += lane >= off ? o : 0.0;
    }
    uint64_t in = __ballot(lane < kLB && base + inc >= tgt);
    if (in == 0) in = 1ull << (63 - __builtin_clzll(__ballot(add > 0.0) | 1ull));  // lost to rounding: the last one
    const int k = __builtin_ctzll(in);
    *before = base + (k > 0 ? __shfl(inc, k - 1, kWave) : 0.0);
    return L * kLB + k;
  }
  // the first bin at which the cumulative count reaches tgt (>= 1), -1 if none does
  __device__ int find_count(unsigned tgt, unsigned* before) const {
    const int lane = threadIdx.x % kWave;
    const uint64_t hit = __ballot(ic >= tgt);
    if (hit == 0) return -1;
    const int L = __builtin_ctzll(hit);
    const unsigned base = L > 0 ? (unsigned)__shfl((int)ic, L - 1, kWave) : 0u;
    unsigned inc = lane < kLB ? (unsigned)(sh.hist[L * kLB + lane % kLB] >> kCountShift) : 0u;
#pragma unroll
    for (int off = 1; off < kLB; off <<= 1) {
      const unsigned o = (unsigned)__shfl_up((int)inc, off, kWave);
      inc += lane >= off ? o : 0u;
    }
    const int k = __builtin_ctzll(__ballot(lane < kLB && base + inc >= tgt));
    *before = base + (k > 0 ? (unsigned)__shfl((int)inc, k - 1, kWave) : 0u);
    return L * kLB + k;
  }
  __device__ unsigned count_above(int bin) const {  // entries of the bins < bin
    const int lane = threadIdx.x % kWave, L = bin / kLB;
    unsigned v = lane < bin % kLB ? (unsigned)(sh.hist[L * kLB + lane] >> kCountShift) : 0u;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += (unsigned)__shfl_xor((int)v, off, kWave);
    return v + (L > 0 ? (unsigned)__shfl((int)ic, L - 1, kWave) : 0u);
  }
};

// The block's sum of `tail` from its waves' partial sums (sh.red), after a barrier.
__device__ __forceinline__ void tail_partials(double tail) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) tail += __shfl_xor(tail, off, kWave);
  if (threadIdx.x % kWave == 0) sh.red[threadIdx.x / kWave] = tail;
}
__device__ __forceinline__ double tail_total() {
  double t = 0.0;
#pragma unroll
  for (int w = 0; w < kTW; ++w) t += sh.red[w];
  return t;
}

// One wave: places a collection window from a histogram of part of the row (the sample, or the segments seen
// so far): the bin where that histogram's own boundary falls (the k_seen-th largest for top-k, the
// top_p mass point for top-p), widened to about `budget` entries of the next segment; `scale` =
// entries of the next segment per counted entry. `tail`: the mass below the histogram.
// The floor (in: the bins below it are counted completely) moves up to just below where the boundary of the
// whole row can lie, with f = the share of the row seen: for top-k, past the bin by which the count seen exceeds
// k f by 5 standard deviations; for top-p, where the mass below (seen / f) has shrunk to 3/4 of (1 - top_p) Z for
// a low estimate of Z, each group of 32 bins scaled up from its count less 3 standard deviations, and below at
// least 64 counted entries: the few likely tokens of a peaked row lie anywhere above. A floor that proves too
// high costs the row a second pass. The top (top-p): the bins that hold the row's first kTopCount entries or so.
// Leaves wlo, whi, top and the floor in sh.ipar[0..3], the entries of the boundary bin and the next in sh.ipar[4].
__device__ __forceinline__ void place_window(LaneBins& lb, bool use_k, float top_p, int top_k, float f, double tail,
                                             float scale, float budget, int floor_bin) {
  lb.load();
  const float up = __builtin_amdgcn_rcpf(f);
  // a low estimate of the row's mass (no entry: 1 - 3 inf = -inf, so a factor of 1)
  double z_lo = lb.m * (double)fmaxf(1.f, up * (1.f - 3.f * __builtin_amdgcn_rsqf((float)lb.c)));
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) z_lo += __shfl_xor(z_lo, off, kWave);
  z_lo += tail * (double)fmaxf(1.f, 0.9f * up);
  const double zall = lb.mass() + tail;
  const float all = budget * __builtin_amdgcn_rcpf(scale), k_seen = (float)top_k * f;  // in counted entries
  unsigned before = 0u;
  double mb;
  int B, wlo = 0, top = 0, fl;
  float hi_c = all;
  if (use_k) {
    B = lb.find_count((unsigned)fmaxf(1.f, ceilf(k_seen)), &before);
    if (B < 0) B = kNB - 1;
    const int b = lb.find_count((unsigned)(k_seen + 5.f * __builtin_amdgcn_sqrtf(k_seen) + 12.f), &before);
    fl = b < 0 ? kNB : b + 3;
  } else {
    B = lb.find_mass((double)top_p * zall, &mb);
    if (B < 0) B = kNB - 1;
    const int b = lb.find_mass(zall - (double)(0.75f * f * (1.f - top_p)) * z_lo, &mb);
    const int sparse = lb.find_count((unsigned)(64.f + 512.f * f) + 1u, &before);
    fl = b < 0 || sparse < 0 ? kNB : max(b + 3, sparse + 1);
    top = max(lb.find_count((unsigned)((float)kTopCount * f) + 1u, &before), 0);
    const float cB = (float)lb.count_above(B), nB = (float)(sh.hist[B] >> kCountShift);
    if (cB - 0.5f * all >= 0.f) wlo = min(max(lb.find_count((unsigned)(cB - 0.5f * all) + 1u, &before), 0), B);
    hi_c = cB + nB + 0.5f * all;
  }
  int whi = lb.find_count((unsigned)fmaxf(1.f, ceilf(hi_c)), &before);
  if (whi < 0) whi = kNB - 1;
  if (threadIdx.x == 0) {
    sh.ipar[0] = wlo;
    sh.ipar[1] = min(max(whi, B) + 1, kNB - 1);  // one bin of slack below: values tied across a bin edge
    sh.ipar[2] = top;
    sh.ipar[3] = min(floor_bin, fl);
    sh.ipar[4] = (int)(sh.hist[B] >> kCountShift) + (int)(sh.hist[min(B + 1, kNB - 1)] >> kCountShift);
  }
}

// One wave: the mass of the whole row (sh.dpar[0]) and the bin that holds the k-th largest value (top-k) or
// the nucleus boundary (top-p): sh.ipar[0], -1 if it lies below the histogram; the entries of it and the next bin (top-k:
// and of all above), sh.ipar[1]; the mass above it, sh.dpar[1].
__device__ __forceinline__ void find_boundary(LaneBins& lb, bool use_k, float top_p, int top_k, double tail) {
  lb.load();
  const double Z = lb.mass() + tail + bin_mass(sh.hist[kNB], bin_scale(kNB));
  unsigned before = 0u;
  double mb = 0.0;
  const int B = use_k ? lb.find_count((unsigned)top_k, &before) : lb.find_mass((double)top_p * Z, &mb);
  if (threadIdx.x == 0) {
    unsigned need = before;
    if (B >= 0)
      for (int b = B; b <= min(B + 1, kNB - 1); ++b) need += (unsigned)(sh.hist[b] >> kCountShift);
    sh.ipar[0] = B;
    sh.ipar[1] = (int)need;
    sh.dpar[0] = Z;
    sh.dpar[1] = mb;
  }
}

// Exact y = x / T of the collected logits, in place.
template <bool kDiv>
__device__ void collected_to_y(int n, double rt) {
  for (int j = threadIdx.x; j < n; j += kT) sh.coll[j] = exact_y<kDiv>(sh.coll[j], rt);
  __syncthreads();
}

// Top-p candidates (the collected logits of the boundary bin B and of bin B + 1) to exact y, in place,
// packed at the front; returns how many, and the largest and smallest. Bins are monotone in the logit, so a value
// of bin B + 1 is <= every value of bin B in y and can only be kept when it ties with the smallest of them: the
// others are dropped, which about halves what is looked at.
template <bool kDiv>
__device__ __forceinline__ int boundary_to_y(const BinMap& bm, int n, int B, double rt, float* ytop, float* ylow) {
  constexpr int kPer = kCap / kT;
  float y[kPer];
  unsigned inb = 0u;  // bit u: entry u is in bin B (then: is kept)
  float ymin = INFINITY, ymax = -INFINITY;
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    if (u * kT >= n) break;  // block-uniform
    const int j = u * kT + (int)threadIdx.x;
    const float x = j < n ? sh.coll[j] : -INFINITY;
    const bool in = j < n && (int)bm.bin(x) == B;
    y[u] = j < n ? exact_y<kDiv>(x, rt) : -INFINITY;
    ymin = in ? fminf(ymin, y[u]) : ymin;
    ymax = in ? fmaxf(ymax, y[u]) : ymax;
    inb |= (unsigned)in << u;
  }
  ymin = -block_max(-ymin);
  ymax = block_max(ymax);
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    if (u * kT >= n) break;
    inb |= (unsigned)(u * kT + (int)threadIdx.x < n && y[u] == ymin) << u;
  }
  double tot = 0.0;
  int w = (int)block_excl_scan((double)__popc(inb), &tot);  // every read of sh.coll precedes its barriers
#pragma unroll
  for (int u = 0; u < kPer; ++u)
    if ((inb >> u) & 1u) sh.coll[w++] = y[u];
  __syncthreads();
  *ytop = ymax;
  *ylow = ymin;
  return (int)tot;
}

// The nucleus boundary among the n values y of sh.coll (ylow <= y <= ytop, within a bin): the smallest y whose
// strictly preceding mass (descending) is below tgt, masses exp(y - ytop). A histogram of kSub sub-bins finds the
// one that crosses tgt, and one wave ranks its few values against each other (a bitonic sort of all of
// them took a quarter of the kernel's instructions). *mass: the mass of every value >= thr. Masses are summed as
// integers, 46 bits below ytop's: the result does not depend on the order. False (nothing done to sh.coll) when
// the sub-bin holds more than a wave's values that are not all equal.
__device__ __forceinline__ bool sub_boundary(int n, float ytop, float ylow, double tgt, float* thr, double* mass) {
  const int tid = threadIdx.x;
  unsigned long long* sub = sh.hist;
  const double tq = tgt * 0x1p46;
  if (!(tq > 0.0) || !(ytop > ylow)) {  // the largest value alone, with its ties
    const float t = ytop > ylow ? ytop : ylow;
    double c = 0.0;
    for (int j = tid; j < n; j += kT) c += sh.coll[j] == t;
    *thr = t;
    *mass = block_sum(c);
    return true;
  }
  const float inv = (float)kSub / (ytop - ylow);
  auto sub_of = [&](float y) { return min(kSub - 1, (int)((ytop - y) * inv)); };
  auto mass_of = [&](float y) { return (unsigned long long)(exp((double)y - (double)ytop) * 0x1p46); };
  __syncthreads();  // the histogram has been read
  for (int j = tid; j < kSub; j += kT) sub[j] = 0ull;
  if (tid == 0) sh.n = 0;
  __syncthreads();
  for (int j = tid; j < n; j += kT) atomicAdd(&sub[sub_of(sh.coll[j])], mass_of(sh.coll[j]));
  __syncthreads();
  if (tid < kWave) {
    constexpr int kPL = kSub / kWave;
    unsigned long long s = 0ull;
#pragma unroll 4
    for (int i = 0; i < kPL; ++i) s += sub[tid * kPL + (tid + i) % kPL];
    unsigned long long inc = s;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const unsigned long long o = __shfl_up(inc, off, kWave);
      inc += tid >= off ? o : 0ull;
    }
    const uint64_t hit = __ballot((double)inc >= tq);
    if (hit == 0) {
      if (tid == 0) sh.ipar[0] = -1;
      if (tid == kWave - 1) sh.dpar[0] = (double)inc;
    } else if (tid == (int)__builtin_ctzll(hit)) {
      unsigned long long run = inc - s;
      int i = 0;
      while (i < kPL - 1 && (double)(run + sub[tid * kPL + i]) < tq) run += sub[tid * kPL + i++];
      sh.ipar[0] = tid * kPL + i;
      sh.dpar[0] = (double)run;
    }
  }
  __syncthreads();
  const int S = sh.ipar[0];
  const double above = sh.dpar[0];
  if (S < 0) {  // tgt exceeds the sum (by rounding): every value is kept
    *thr = ylow;
    *mass = above * 0x1p-46;
    return true;
  }
  float* list = sh.queue[0];
  float lo = INFINITY, hi = -INFINITY;
  for (int j = tid; j < n; j += kT) {
    const float y = sh.coll[j];
    if (sub_of(y) == S) {
      lo = fminf(lo, y);
      hi = fmaxf(hi, y);
      const int at = atomicAdd(&sh.n, 1);
      if (at < kWave) list[at] = y;
    }
  }
  __syncthreads();
  const int cnt = sh.n;
  if (cnt > kWave) {  // more than a wave's values, unless they are one: rows of widened bf16 logits hold hundreds of each
    lo = -block_max(-lo);
    hi = block_max(hi);
    if (lo != hi) return false;
    *thr = hi;
    *mass = (above + (double)sub[S]) * 0x1p-46;
    return true;
  }
  if (tid < kWave) {
    const float y = tid < cnt ? list[tid] : -INFINITY;
    const unsigned long long q = tid < cnt ? mass_of(y) : 0ull;
    unsigned long long prec = 0ull;  // the mass of the list's values before this one (ties in list order)
    for (int j = 0; j < cnt; ++j) {
      const float yj = __shfl(y, j, kWave);
      const unsigned long long qj = __shfl(q, j, kWave);
      prec += yj > y || (yj == y && j < tid) ? qj : 0ull;
    }
    const bool kept = tid < cnt && above + (double)prec < tq;
    float t = kept ? y : INFINITY;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) t = fminf(t, __shfl_xor(t, off, kWave));
    if (t == INFINITY) t = wave_max(y);  // (cannot be: the sub-bin's first value starts below tgt)
    unsigned long long at = tid < cnt && y >= t ? q : 0ull;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) at += __shfl_xor(at, off, kWave);
    if (tid == 0) {
      sh.dpar[1] = above + (double)at;
      sh.dpar[2] = (double)t;
    }
  }
  __syncthreads();
  *thr = (float)sh.dpar[2];
  *mass = sh.dpar[1] * 0x1p-46;
  return true;
}

template <bool kDiv>
__global__ __launch_bounds__(kT, 4) void truncate_kernel(TruncArgs a) {
  const int b = blockIdx.x / a.G, i = a.first + (int)(blockIdx.x % a.G);
  if (i >= a.R || (a.state && a.state[b] >= 0)) return;  // block-uniform: past the rows, or decided
  const int r = b * a.R + i;
  const int V = a.V, tid = threadIdx.x;
  const RowView rv(a.logits + (int64_t)b * a.batch_stride + (int64_t)i * a.row_stride, V);
  const bool use_k = a.top_k > 0 && a.top_k < V;
  const bool use_p = a.top_p < 1.f;
  const bool collect = use_k || use_p;
  bool window = !(a.flags & 1) && V <= kMaxPackedV && a.rt < 0x1p120;  // (1 / T and its multiples fit fp32)
  int passes = 0;  // segments streamed (kSeg = one pass over the row)

  float mx = -INFINITY;  // max logit (the banned id excluded)
  bool nan = false;
  double Z = 0.0, cum = 0.0;  // window path: the row's mass and the mass above the boundary bin
  int B = -1, need = 0;       // the boundary bin and the entries it takes to resolve it
  float mref = 0.f;
  BinMap bm{};
  const int ns = min(kSample, V);
  float xs[kSample / kT];
  if (window) {
    // ---- sample: evenly spaced entries; their max is the exponent reference of the pass, their
    // histogram places the first segment's window
    float smax = -INFINITY;
    if (rv.n4 >= kSample) {
      // kT evenly spaced 16-byte vectors of 4 adjacent entries each: a line per 4 entries (entries one
      // by one would fetch a line each, a quarter of the row's bytes at V = 248320)
      static_assert(kSample == 4 * kT, "one vector of the sample per thread");
      const int jv = (int)((int64_t)tid * rv.n4 / kT);
      const u32x4 w = rv.body[jv];
      const float x4[4] = {__uint_as_float(w.x), __uint_as_float(w.y), __uint_as_float(w.z), __uint_as_float(w.w)};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        xs[u] = (rv.pre + 4 * jv + u != a.ban && x4[u] == x4[u]) ? x4[u] : -INFINITY;
        smax = xs[u] < INFINITY ? fmaxf(smax, xs[u]) : smax;
      }
    } else {
#pragma unroll
      for (int u = 0; u < kSample / kT; ++u) {
        const int j = u * kT + tid;
        const int ix = (int)((int64_t)min(j, ns - 1) * V / ns);
        const float x = rv.row[ix];
        xs[u] = (j < ns && ix != a.ban && x == x) ? x : -INFINITY;
        smax = xs[u] < INFINITY ? fmaxf(smax, xs[u]) : smax;
      }
    }
    smax = block_max(smax);
    mref = smax > -INFINITY ? exact_y<kDiv>(smax, a.rt) : 0.f;
    // Past 2^18 an fp32 y no longer tells bins apart (half a bin to a unit), the bin map rounds by whole bins and, for rows
    // masked with the type's lowest value, overflows: such a row goes to the exact select.
    window = fabsf(mref) < 0x1p18f;
  }
  if (window) {
    mref = rintf(mref * kPerNat) / kPerNat;  // a whole bin: see BinMap::packed
    bm.set(a.rt, mref);
    for (int j = tid; j <= kNB; j += kT) sh.hist[j] = 0ull;
    __syncthreads();
    LaneBins lb;
    if (tid < kWave) lb.init();
    if (collect) {
#pragma unroll
      for (int u = 0; u < kSample / kT; ++u) {
        const float x = xs[u] < INFINITY ? xs[u] : -INFINITY;
        const unsigned bin = bm.bin(x);
        if (bin < (unsigned)kNB) atomicAdd(&sh.hist[bin], bm.packed(x, bin));
      }
    }
    __syncthreads();
    // ---- the streaming pass, kSeg segments: max, histogram down to the floor, collection of a window placed
    // from the sample's histogram and again from the row's own after every segment. Run again without
    // floors when the boundary turns out to lie below the last one. Without truncation only the few entries above the
    // sample's max, which may carry most of the mass, go to the histogram: its exponents are exact to 2^-26.
    int w_lo = kNB + 1, w_hi = kNB + 1, w_top = 0, floor_bin = collect ? kNB : (int)(kTop * kPerNat);
    int seen = 0, counted = ns;
    double tail = 0.0;
    bool floors = true;
    int have = 0;
    int s = collect ? -1 : 0;
    while (true) {
      if (s >= 0) {
        if (tid == 0) {
          sh.wlo[s] = w_lo;
          sh.whi[s] = min(w_hi, floor_bin - 1);
          sh.top[s] = min(w_top, floor_bin);
        }
        stream_segment<true>(rv, a, bm, s, below_bin(bm, floor_bin), 0.f, w_top, w_lo, w_hi, mx, tail, have);
        ++passes;
        seen += seg_size(rv, s);
        counted = seen;
        tail_partials(tail);
        if (tid % kWave == 0) sh.nseg[s][tid / kWave] = have;
        __syncthreads();
      }
      const int next = s + 1 < kSeg ? seg_size(rv, s + 1) : 0;
      if (s == kSeg - 1) {
        if (tid < kWave) find_boundary(lb, use_k, a.top_p, a.top_k, tail_total() * bm.cold_scale);
      } else if (collect && next > 0 && tid < kWave) {
        int got = 0;
        if (s >= 0)
          for (int w = 0; w < kTW; ++w) got += sh.nseg[s][w];
        const float room = fmaxf(0.75f * kCap - (float)got, 0.f);
        place_window(lb, use_k, a.top_p, a.top_k, (float)counted / (float)V, s < 0 ? 0.0 : tail_total() * bm.cold_scale,
                     (float)next / (float)counted, s < 0 ? 0.2f * kCap : room / (float)(kSeg - 1 - s), floor_bin);
      }
      __syncthreads();
      if (s == kSeg - 1) {
        B = sh.ipar[0];
        need = sh.ipar[1];
        Z = sh.dpar[0];
        cum = sh.dpar[1];
        // the boundary bin and the one below it have to lie above the floor
        if (!collect || floor_bin >= kNB || (B >= 0 && B + 1 < floor_bin)) break;
        floors = false;
        floor_bin = kNB;
        tail = 0.0;
        seen = 0;
        s = -1;  // the last window stands for the first segment
        __syncthreads();
        for (int j = tid; j <= kNB; j += kT) sh.hist[j] = 0ull;
        have = 0;
      } else if (collect && next > 0) {
        // A row so flat that its boundary bin will not fit the collection goes to the exact select after the first segment,
        // whose counts show kCap entries as 768 +- 28 (V = 248320). 512 rows, standard deviation of y 0.14, top_p = 0.95:
        // 873 -> 828 us, top_p = 0.8 at 0.2: 833 -> 758.
        if (s == 0 && !use_k && (float)sh.ipar[4] * ((float)V / (float)counted) > (float)kCap) {
          window = false;
          mx = -INFINITY;
          break;
        }
        w_lo = sh.ipar[0];
        w_hi = sh.ipar[1];
        w_top = sh.ipar[2];
        if (floors && s >= 0) floor_bin = sh.ipar[3];
        if (s < 0)
          for (int j = tid; j <= kNB; j += kT) sh.hist[j] = 0ull;
      }
      __syncthreads();
      ++s;
    }
    nan = tail != tail;
  }
  if (!window) {
    for_each_y<kDiv>(rv, a.rt, a.ban, [&](float y, int ix, bool ok) {
      mx = fmaxf(mx, ok ? y : -INFINITY);
      nan |= ok && y != y;
    });
    passes += kSeg;
  }
  mx = block_max(mx);
  if (tid == 0) sh.umax = 0u;
  __syncthreads();
  if (__ballot(nan) && tid % kWave == 0) atomicOr(&sh.umax, 1u);
  __syncthreads();
  const bool bad = sh.umax != 0u || mx == INFINITY;  // a NaN, or a +inf logit
  // the exact row max of y (the window path tracked the raw logits; y = x / T is monotone in x)
  const float ymax = window ? exact_y<kDiv>(mx, a.rt) : mx;
  float thr = -INFINITY;
  double zk = 0.0;
  int status = 0;
  if (bad) {
    status = 1;
  } else if (!(ymax > -INFINITY)) {
    status = 2;
  } else {
    const double md = (double)ymax;
    // the target must lie within the histogram, and what resolves it fit the collection
    bool ok = window && !(ymax - mref > kTop) && (!collect || (B >= 0 && need <= (use_k ? kSortCap : kCap)));
    if (ok && !collect) {
      zk = Z * exp((double)mref - md);
    } else if (ok) {
      // values tied in y may straddle a bin edge (the bins come from the logits), so the
      // candidate set takes one more bin below the boundary bin
      const int c_lo = use_k ? 0 : B, c_hi = min(B + 1, kNB - 1);
      // keep what the segments whose window held [c_lo, c_hi] collected (and that fit the
      // collection); stream the others again
      unsigned complete = 0u;
      for (int s = 0; s < kSeg; ++s) {
        int fill = 0;
        for (int w = 0; w < kTW; ++w) fill = max(fill, sh.nseg[s][w]);
        complete |= (unsigned)(((c_lo >= sh.wlo[s] && c_hi <= sh.whi[s]) || c_hi < sh.top[s]) && fill <= kWaveCap) << s;
      }
      int n2 = compact_bins(bm, c_lo, c_hi, complete);
      if (complete != (1u << kSeg) - 1u) {
        __syncthreads();
        if (tid == 0) sh.n = n2;
        __syncthreads();
        const float x_lo = below_bin(bm, c_hi + 1), x_hi = c_lo > 0 ? above_bin(bm, c_lo) : INFINITY;
        double none = 0.0;
        int unused = 0;
        for (int s = 0; s < kSeg; ++s) {
          if ((complete >> s) & 1u) continue;
          stream_segment<false>(rv, a, bm, s, x_lo, x_hi, 0, c_lo, c_hi, mx, none, unused);
          ++passes;
        }
        __syncthreads();
        n2 = min(sh.n, kCap);
      }
      ok = n2 == need;  // exactly the candidates that the histogram counted; else the exact select
      if (ok && use_k) {
        collected_to_y<kDiv>(n2, a.rt);
        sort_collection(n2);
        const int k = min(a.top_k, n2);
        thr = sh.coll[k - 1];
        if (use_p) {
          double Sk = 0.0, tot = 0.0;
          (void)count_below(k, md, 0.0, -1.0, &Sk);
          const int nk = max(count_below(k, md, 0.0, (double)a.top_p * Sk, &tot), 1);
          thr = sh.coll[nk - 1];
        }
        zk = mass_at_least(n2, thr, md);
      } else if (ok) {
        float ytop, ylow;
        n2 = boundary_to_y<kDiv>(bm, n2, B, a.rt, &ytop, &ylow);
        const double base = cum * exp((double)mref - md), target = (double)a.top_p * Z;
        const double et = exp((double)ytop - md);
        double mass;
        if (sub_boundary(n2, ytop, ylow, (target - cum) * exp((double)mref - (double)ytop), &thr, &mass)) {
          zk = base + mass * et;
        } else if ((ok = n2 <= kSortCap)) {
          sort_collection(n2);
          double tot = 0.0;
          const int nk = min(max(count_below(n2, md, base, target * exp((double)mref - md), &tot), 1), max(n2, 1));
          thr = sh.coll[nk - 1];
          zk = base + mass_at_least(n2, thr, md);
        }
      }
    }
    if (!ok) {
      int rp = 0;
      radix_resolve<kDiv>(rv, a, ymax, use_k, use_p, &thr, &zk, &rp);
      passes += rp * kSeg;
    }
  }
  if (tid == 0) {
    a.m_out[r] = ymax;
    a.thr_out[r] = thr;
    a.zk_out[r] = zk;
    a.status_out[r] = status;
    if (a.passes_out) a.passes_out[r] = passes;
  }
}

// ---------------------------------------------------------------- acceptance and correction
struct AcceptArgs {
  const float* p;
  int64_t p_bs, p_rs;
  const float* q;
  int64_t q_bs, q_rs;
  const int64_t* drafts;
  int64_t d_st;
  const int32_t* n_live;
  const float* u_acc;
  int64_t u_st;
  const float* u_samp;
  const int64_t* ctx;
  int B, V, K;
  double rt;  // 1 / temperature
  int ban;
  const float* m;  // [B * (K + 1)] row statistics
  const float* thr;
  const double* zk;
  const int* status;
  int* state;    // per sequence: -1 while every verified draft was accepted, else the accepted length
  int* rstatus;  // per sequence: OR of the row statuses seen
  int NC, chunk;
  double* sums;  // [B][NC][2]: correction weight, P
  int32_t* n_acc;
  int64_t* token;
  int64_t* crop;
  double* ratio;  // [B, K] or null
  int32_t* status_out;
};

// P_row(x) exactly (fp64 exponential) from the row statistics, 0 outside the kept set: the drafted
// tokens' probabilities in the accept test.
__device__ __forceinline__ double prob_exact(const AcceptArgs& a, int srow, float x, int ix) {
  const float y = make_y<true>(x, ix, a.rt, a.ban);  // the product with rt = 1 is exact
  if (!(y > -INFINITY) || !(y >= a.thr[srow])) return 0.0;
  return exp((double)y - (double)a.m[srow]) / a.zk[srow];
}

// The correction draw's weights over a row (fp32 exponential: a relative error of ~1e-7 per entry,
// so the cumulative weight is off by at most ~1e-7 in probability units).
struct RowW {
  const float* p;
  const float* q;  // null: weights are P_K itself
  float m, thr, inv_zk;
  double rt;
  int ban;
  __device__ __forceinline__ float prob(float x, int ix) const {
    const float y = make_y<true>(x, ix, rt, ban);
    return (y > -INFINITY && y >= thr) ? __expf(y - m) * inv_zk : 0.f;
  }
  __device__ __forceinline__ void at(int ix, float* w, float* pp) const {
    const float P = prob(p[ix], ix);
    *pp = P;
    *w = q ? fmaxf(P - q[ix], 0.f) : P;
  }
};
__device__ __forceinline__ RowW row_weights(const AcceptArgs& a, int b, int r) {
  const int srow = b * (a.K + 1) + r;
  RowW w;
  w.p = a.p + (int64_t)b * a.p_bs + (int64_t)r * a.p_rs;
  w.q = r < a.K ? a.q + (int64_t)b * a.q_bs + (int64_t)r * a.q_rs : nullptr;
  w.m = a.m[srow];
  w.thr = a.thr[srow];
  w.inv_zk = (float)(1.0 / a.zk[srow]);
  w.rt = a.rt;
  w.ban = a.ban;
  return w;
}

__device__ __forceinline__ double rblock_sum(double v, double* sh) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
  __syncthreads();
  if (threadIdx.x % kWave == 0) sh[threadIdx.x / kWave] = v;
  __syncthreads();
  double t = 0.0;
#pragma unroll
  for (int w = 0; w < kRT / kWave; ++w) t += sh[w];
  return t;
}

// The accept test of the row group [first, first + G) of sequence b, one wave: the drafted token's
// ratio P_i(d_i) / q_i(d_i) per row, accepted while ratio >= 1 or u_i < ratio (and i < n_live). Decides
// the sequence at its first rejection, or once row K (the bonus row) has been reached.
__global__ __launch_bounds__(kWave) void accept_scan_kernel(AcceptArgs a, int first, int G) {
  const int b = blockIdx.x, lane = threadIdx.x;
  if (first > 0 && a.state[b] >= 0) return;
  const int i = first + lane;
  const bool row_here = lane < G && i <= a.K;
  const bool draft_here = lane < G && i < a.K;
  const int live = a.n_live ? min(max((int)a.n_live[b], 0), a.K) : a.K;
  bool acc = false;
  double ratio = 0.0;
  if (draft_here) {
    const int64_t d = a.drafts[(int64_t)b * a.d_st + i];
    if (d >= 0 && d < a.V) {
      const int srow = b * (a.K + 1) + i;
      const double P = prob_exact(a, srow, a.p[(int64_t)b * a.p_bs + (int64_t)i * a.p_rs + d], (int)d);
      const double q = (double)a.q[(int64_t)b * a.q_bs + (int64_t)i * a.q_rs + d];
      ratio = q > 0.0 ? P / fmax(q, 1e-30) : 0.0;
      acc = (i < live) && (ratio >= 1.0 || (double)a.u_acc[(int64_t)b * a.u_st + i] < ratio);
    }
  }
  const uint64_t drafts = __ballot(draft_here);
  const uint64_t rej = drafts & ~__ballot(acc);
  int n = -1;  // still open
  if (rej) n = first + __builtin_ctzll(rej);
  else if (first + G > a.K) n = a.K;  // this group holds row K: every draft accepted
  int st = row_here ? a.status[b * (a.K + 1) + i] : 0;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) st |= __shfl_xor(st, off, kWave);
  if (a.ratio && draft_here && (n < 0 || i <= n)) a.ratio[(int64_t)b * a.K + i] = ratio;
  if (lane == 0) {
    a.state[b] = n;
    a.rstatus[b] = (first > 0 ? a.rstatus[b] : 0) | st;
  }
}

__global__ __launch_bounds__(kRT) void resid_sums_kernel(AcceptArgs a) {
  const int c = blockIdx.x, b = blockIdx.y;
  const int tid = threadIdx.x;
  __shared__ int s_nacc;
  __shared__ double s_red[kRT / kWave];
  if (tid == 0) s_nacc = min(max(a.state[b], 0), a.K);
  __syncthreads();
  if (c == 0) {  // the per-sequence outputs; ratios past the first rejection are 0
    const int n_acc = s_nacc;
    if (a.ratio)
      for (int i = n_acc + 1 + tid; i < a.K; i += kRT) a.ratio[(int64_t)b * a.K + i] = 0.0;
    if (tid == 0) {
      a.n_acc[b] = n_acc;
      a.crop[b] = (a.ctx ? a.ctx[b] : 0) + 1 + n_acc;
      a.status_out[b] = a.rstatus[b];
    }
  }
  __syncthreads();
  const RowW rw = row_weights(a, b, s_nacc);
  const int lo = c * a.chunk, hi = min(a.V, lo + a.chunk);
  double sw = 0.0, sp = 0.0;
  // Four 16-byte loads in flight per thread, the elements outside the chunk's aligned vectors (<= 6) one per thread.
  // One element per load and iteration left the pass waiting on memory: 512 rows of 248320 185 -> 97 us
  // (2.7 -> 5.2 TB/s). q is read by element where its rows are not aligned as p's.
  const float* pc = rw.p + lo;
  const int len = hi - lo, pre = min((int)((0u - (unsigned)((uintptr_t)pc >> 2)) & 3u), len), n4 = (len - pre) >> 2;
  const u32x4* p4 = reinterpret_cast<const u32x4*>(pc + pre);
  const float* qc = rw.q ? rw.q + lo : nullptr;
  const bool qvec = qc && ((uintptr_t)(qc + pre) & 15) == 0;
  auto add = [&](float x, float q, int ix) {
    const float P = rw.prob(x, ix);
    sp += P;
    if (qc) sw += fmaxf(P - q, 0.f);
  };
  constexpr int U = 4;
  for (int base = 0; base < n4; base += kRT * U) {
    u32x4 x[U], qv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = min(base + u * kRT + tid, n4 - 1);
      x[u] = p4[j];
      qv[u] = u32x4{0u, 0u, 0u, 0u};
      if (qvec) {
        qv[u] = *reinterpret_cast<const u32x4*>(qc + pre + 4 * j);
      } else if (qc) {
#pragma unroll
        for (int e = 0; e < 4; ++e) qv[u][e] = __float_as_uint(qc[pre + 4 * j + e]);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = base + u * kRT + tid;
      if (j >= n4) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e) add(__uint_as_float(x[u][e]), __uint_as_float(qv[u][e]), lo + pre + 4 * j + e);
    }
  }
  {
    const int j = tid < pre ? tid : tid + 4 * n4;
    if (j < len) add(pc[j], qc ? qc[j] : 0.f, lo + j);
  }
  if (!qc) sw = sp;
  sw = rblock_sum(sw, s_red);
  sp = rblock_sum(sp, s_red);
  if (tid == 0) {
    a.sums[((int64_t)b * a.NC + c) * 2 + 0] = sw;
    a.sums[((int64_t)b * a.NC + c) * 2 + 1] = sp;
  }
}

constexpr int kPickChunk = 4096;  // the largest chunk: its weights fit the pick kernel's LDS

__global__ __launch_bounds__(kRT) void resid_pick_kernel(AcceptArgs a) {
  const int b = blockIdx.x, tid = threadIdx.x;
  const int lane = tid % kWave, w = tid / kWave;
  __shared__ int s_chunk, s_last, s_tok, s_sel;
  __shared__ double s_t;
  __shared__ double s_red[kRT / kWave];
  __shared__ float s_w[kPickChunk];
  const int r = a.n_acc[b];
  // one wave finds the chunk, lane l holding the chunks [l L, l L + L): a serial walk over the chunk sums by one
  // thread was a memory latency per chunk (512 rows of 61 chunks: 25 -> 17 us)
  if (tid < kWave) {
    const double* s = a.sums + (int64_t)b * a.NC * 2;
    const int L = (a.NC + kWave - 1) / kWave, c0 = min(a.NC, lane * L), c1 = min(a.NC, c0 + L);
    double lw = 0.0, lp = 0.0;
    for (int c = c0; c < c1; ++c) {
      lw += s[2 * c];
      lp += s[2 * c + 1];
    }
    double tw = lw, tp = lp;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const double ow = __shfl_up(tw, off, kWave), op = __shfl_up(tp, off, kWave);
      tw += lane >= off ? ow : 0.0;
      tp += lane >= off ? op : 0.0;
    }
    const int sel = __shfl(tw, kWave - 1, kWave) > 0.0 ? 0 : 1;  // an empty residual draws from P itself
    const double own = sel ? lp : lw, inc = sel ? tp : tw;
    const double t = (double)a.u_samp[b] * __shfl(inc, kWave - 1, kWave);
    const uint64_t hit = __ballot(inc > t), some = __ballot(own > 0.0);
    // the first lane whose chunks carry the cumulative weight past t, else the last with any weight
    const int src = hit ? __builtin_ctzll(hit) : some ? 63 - __builtin_clzll(some) : 0;
    const double before = src > 0 ? __shfl(inc, src - 1, kWave) : 0.0;
    if (lane == src) {
      double cum = before;
      int pick = -1, lastpos = c0;
      for (int c = c0; c < c1; ++c) {
        const double v = s[2 * c + sel];
        if (v > 0.0) lastpos = c;
        if (hit && cum + v > t) {
          pick = c;
          break;
        }
        cum += v;
      }
      if (hit && pick < 0) {  // the lane's own sum rounds below the scan's: its last weighted chunk
        pick = lastpos;
        cum -= s[2 * pick + sel];
      }
      s_last = !hit;
      s_chunk = hit ? pick : lastpos;
      s_t = t - cum;
      s_sel = sel;
    }
    if (lane == 0) s_tok = INT_MAX;
  }
  __syncthreads();
  const int c = s_chunk, sel = s_sel;
  const bool last = s_last;
  const double t = s_t;
  const int lo = c * a.chunk, hi = min(a.V, lo + a.chunk), len = hi - lo;
  // stage the chunk's weights in LDS with coalesced loads, then scan contiguous runs per thread
  const RowW rw = row_weights(a, b, r);
#pragma unroll 4
  for (int j = tid; j < len; j += kRT) {
    float wt, pp;
    rw.at(lo + j, &wt, &pp);
    s_w[j] = sel ? pp : wt;
  }
  __syncthreads();
  const int L = (len + kRT - 1) / kRT;
  const int j0 = min(len, tid * L), j1 = min(len, j0 + L);
  double loc = 0.0;
  int lastpos = -1;
  for (int j = j0; j < j1; ++j) {
    loc += (double)s_w[j];
    if (s_w[j] > 0.f) lastpos = lo + j;
  }
  // exclusive scan over the block (thread order = vocabulary order)
  double inc = loc;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const double o = __shfl_up(inc, off, kWave);
    if (lane >= off) inc += o;
  }
  double ex = __shfl_up(inc, 1, kWave);
  if (lane == 0) ex = 0.0;
  if (lane == kWave - 1) s_red[w] = inc;
  __syncthreads();
  for (int i = 0; i < w; ++i) ex += s_red[i];
  int found = INT_MAX;
  if (!last && ex <= t && t < ex + loc) {
    double run = ex;
    for (int j = j0; j < j1; ++j) {
      run += (double)s_w[j];
      if (run > t) {
        found = lo + j;
        break;
      }
    }
  }
  if (found != INT_MAX) atomicMin(&s_tok, found);
  // the last positive-weight token of the chunk: used when u * total lands past the summed weight
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) lastpos = max(lastpos, __shfl_xor(lastpos, off, kWave));
  __syncthreads();
  if (lane == 0) s_red[w] = (double)lastpos;
  __syncthreads();
  if (tid == 0) {
    int lp = -1;
    for (int i = 0; i < kRT / kWave; ++i) lp = max(lp, (int)s_red[i]);
    const int tok = s_tok != INT_MAX ? s_tok : max(lp, 0);
    a.token[b] = tok;
  }
}

int ban_of(int64_t ban_id, int64_t V) { return (ban_id >= 0 && ban_id < V) ? (int)ban_id : -1; }

int launch_truncate(const TruncArgs& ta, int rows, hipStream_t st) {
  if (ta.rt != 1.0) hipLaunchKernelGGL((truncate_kernel<true>), dim3(rows), dim3(kT), 0, st, ta);
  else hipLaunchKernelGGL((truncate_kernel<false>), dim3(rows), dim3(kT), 0, st, ta);
  return launch_status("truncate_kernel");
}

int check_trunc_params(int64_t V, float temperature, int64_t top_k, float top_p) {
  TRIDA_CHECK(V > 0 && V < INT_MAX / 2, TRIDA_ERR_ARG, "V=%lld out of range", (long long)V);
  TRIDA_CHECK(temperature > 0.f && temperature < INFINITY, TRIDA_ERR_ARG,
              "temperature must be positive and finite (greedy decoding has its own entry point)");
  TRIDA_CHECK(top_p > 0.f && top_p <= 1.f, TRIDA_ERR_ARG, "top_p must lie in (0, 1]");
  TRIDA_CHECK(top_k >= 0, TRIDA_ERR_ARG, "top_k must be >= 0 (0 disables it)");
  TRIDA_CHECK(top_k == 0 || top_k >= V || top_k <= kMaxTopK, TRIDA_ERR_ARG, "top_k=%lld above the supported %d",
              (long long)top_k, kMaxTopK);
  return TRIDA_OK;
}

void plan_chunks(int64_t B, int64_t V, int* NC, int* chunk) {
  int64_t nc = std::min<int64_t>(64, std::max<int64_t>(1, cdiv(1024, B)));
  nc = std::min<int64_t>(nc, std::max<int64_t>(1, cdiv(V, 1024)));
  nc = std::max<int64_t>(nc, cdiv(V, kPickChunk));  // a chunk's weights fit the pick kernel's LDS
  *chunk = (int)cdiv(V, nc);
  *NC = (int)cdiv(V, *chunk);
}

struct ScratchLayout {
  int64_t m, thr, zk, status, state, rstatus, sums, total;
};
ScratchLayout layout(int64_t B, int64_t K, int64_t V) {
  int NC, chunk;
  plan_chunks(B, V, &NC, &chunk);
  const int64_t rows = B * (K + 1);
  ScratchLayout L;
  L.m = 0;
  L.thr = L.m + align_up(rows * 4, 256);
  L.zk = L.thr + align_up(rows * 4, 256);
  L.status = L.zk + align_up(rows * 8, 256);
  L.state = L.status + align_up(rows * 4, 256);
  L.rstatus = L.state + align_up(B * 4, 256);
  L.sums = L.rstatus + align_up(B * 4, 256);
  L.total = L.sums + align_up(B * NC * 2 * 8, 256);
  return L;
}

}  // namespace
}  // namespace trida

using namespace trida;

extern "C" int trida_truncate_stats(const float* logits, int64_t B, int64_t R, int64_t V, int64_t batch_stride,
                                    int64_t row_stride, float temperature, int64_t top_k, float top_p,
                                    int64_t ban_id, int flags, float* m_out, float* thr_out, double* zk_out,
                                    int32_t* status_out, int32_t* passes_out, void* stream) {
  TRIDA_CHECK(logits && m_out && thr_out && zk_out && status_out, TRIDA_ERR_NULL, "null pointer argument");
  TRIDA_CHECK(B > 0 && R > 0 && B * R < INT_MAX, TRIDA_ERR_ARG, "bad B=%lld R=%lld", (long long)B, (long long)R);
  const int rc = check_trunc_params(V, temperature, top_k, top_p);
  if (rc != TRIDA_OK) return rc;
  TRIDA_CHECK(row_stride >= V && (B == 1 || batch_stride >= (R - 1) * row_stride + V), TRIDA_ERR_ARG,
              "strides too small");
  TruncArgs ta{logits, batch_stride, row_stride, (int)R, (int)V, 1.0 / (double)temperature, (int)top_k, top_p,
               ban_of(ban_id, V), flags, (int)R, 0, nullptr,
               m_out, thr_out, zk_out, status_out, passes_out};
  return launch_truncate(ta, (int)(B * R), static_cast<hipStream_t>(stream));
}

extern "C" int64_t trida_sample_accept_scratch_bytes(int64_t B, int64_t R, int64_t V, int64_t K) {
  (void)R;
  if (B <= 0 || V <= 0 || K < 0) return -1;
  return layout(B, K, V).total;
}

extern "C" int trida_sample_accept(const float* p_logits, int64_t B, int64_t R, int64_t V, int64_t p_batch_stride,
                                   int64_t p_row_stride, const float* q_probs, int64_t q_batch_stride,
                                   int64_t q_row_stride, const int64_t* drafts, int64_t K, int64_t draft_stride,
                                   const int32_t* n_live, const float* u_accept, int64_t u_stride,
                                   const float* u_sample, const int64_t* ctx_len, float temperature, int64_t top_k,
                                   float top_p, int64_t ban_id, int32_t* n_acc, int64_t* token, int64_t* crop,
                                   double* ratio, int32_t* status, void* scratch, int64_t scratch_bytes,
                                   void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  TRIDA_CHECK(p_logits && u_sample && n_acc && token && crop && status && scratch, TRIDA_ERR_NULL,
              "null pointer argument");
  TRIDA_CHECK(K == 0 || (q_probs && drafts && u_accept), TRIDA_ERR_NULL, "q_probs, drafts and u_accept are needed when K > 0");
  TRIDA_CHECK(B > 0 && B <= 65535 && K >= 0 && K <= kWave && R >= K + 1, TRIDA_ERR_ARG,
              "need 0 < B <= 65535, 0 <= K <= 64 and R >= K + 1 (B=%lld K=%lld R=%lld)", (long long)B, (long long)K,
              (long long)R);
  const int rc = check_trunc_params(V, temperature, top_k, top_p);
  if (rc != TRIDA_OK) return rc;
  TRIDA_CHECK(p_row_stride >= V && (B == 1 || p_batch_stride >= (R - 1) * p_row_stride + V), TRIDA_ERR_ARG,
              "p strides too small");
  TRIDA_CHECK(K == 0 || (q_row_stride >= V && (B == 1 || (q_batch_stride >= (K - 1) * q_row_stride + V &&
                                                          draft_stride >= K && u_stride >= K))),
              TRIDA_ERR_ARG, "q / draft / uniform strides too small");
  const ScratchLayout L = layout(B, K, V);
  TRIDA_CHECK(scratch_bytes >= L.total, TRIDA_ERR_WORKSPACE, "scratch of %lld bytes, need %lld",
              (long long)scratch_bytes, (long long)L.total);
  TRIDA_CHECK((uintptr_t)scratch % 256 == 0, TRIDA_ERR_ALIGN, "scratch must be 256-byte aligned");
  char* s = static_cast<char*>(scratch);
  float* m = reinterpret_cast<float*>(s + L.m);
  float* thr = reinterpret_cast<float*>(s + L.thr);
  double* zk = reinterpret_cast<double*>(s + L.zk);
  int* st = reinterpret_cast<int*>(s + L.status);
  double* sums = reinterpret_cast<double*>(s + L.sums);

  int* state = reinterpret_cast<int*>(s + L.state);
  int* rstatus = reinterpret_cast<int*>(s + L.rstatus);
  int NC, chunk;
  plan_chunks(B, V, &NC, &chunk);
  AcceptArgs aa{p_logits, p_batch_stride, p_row_stride, q_probs, q_batch_stride, q_row_stride, drafts, draft_stride,
                n_live, u_accept, u_stride, u_sample, ctx_len, (int)B, (int)V, (int)K, 1.0 / (double)temperature,
                ban_of(ban_id, V), m, thr, zk, st, state, rstatus, NC, chunk, sums, n_acc, token, crop, ratio, status};

  // Only rows up to a sequence's first rejection decide anything. Rows 0..G0-1 of every sequence go
  // first (G0 sized so that this group alone fills the GPU, ~512 blocks, and a row per lane of the scan); a one-wave scan per
  // sequence then settles the sequences it can, and one more group evaluates all the remaining rows
  // of the rest at once (decided sequences' blocks exit at once), followed by the final scan.
  const int R1 = (int)K + 1;
  const int G0 = (int)std::min<int64_t>({R1, std::max<int64_t>(8, cdiv(512, B)), kWave});
  int r = TRIDA_OK;
  for (int g = 0; g < 2; ++g) {
    const int first = g == 0 ? 0 : G0, cnt = g == 0 ? G0 : R1 - G0;
    if (cnt <= 0) break;
    TruncArgs ta{p_logits, p_batch_stride, p_row_stride, R1, (int)V, 1.0 / (double)temperature, (int)top_k, top_p,
                 ban_of(ban_id, V), 0, cnt, first, g > 0 ? state : nullptr, m, thr, zk, st, nullptr};
    r = launch_truncate(ta, (int)(B * cnt), stream);
    if (r != TRIDA_OK) return r;
    hipLaunchKernelGGL(accept_scan_kernel, dim3(B), dim3(kWave), 0, stream, aa, first, cnt);
    r = launch_status("accept_scan_kernel");
    if (r != TRIDA_OK) return r;
  }
  hipLaunchKernelGGL(resid_sums_kernel, dim3(NC, B), dim3(kRT), 0, stream, aa);
  r = launch_status("resid_sums_kernel");
  if (r != TRIDA_OK) return r;
  hipLaunchKernelGGL(resid_pick_kernel, dim3(B), dim3(kRT), 0, stream, aa);
  return launch_status("resid_pick_kernel");
}

namespace trida {
namespace {
__global__ __launch_bounds__(256) void probs_kernel(const float* logits, int64_t bs, int64_t rs, int R, int V,
                                                    double rt, int ban, const float* m, const float* thr,
                                                    const double* zk, float* out, int64_t obs, int64_t ors) {
  const int r = blockIdx.y;
  const int b = r / R, i = r % R;
  const float* row = logits + (int64_t)b * bs + (int64_t)i * rs;
  float* o = out + (int64_t)b * obs + (int64_t)i * ors;
  const float mm = m[r], t = thr[r];
  const float inv = (float)(1.0 / zk[r]);
  for (int ix = blockIdx.x * 256 + threadIdx.x; ix < V; ix += gridDim.x * 256) {
    const float y = make_y<true>(row[ix], ix, rt, ban);
    o[ix] = (y > -INFINITY && y >= t) ? __expf(y - mm) * inv : 0.f;
  }
}
// 16-byte accesses at any element's address: the hardware takes them, and a row of an odd vocabulary starts anywhere
typedef u32x4 __attribute__((aligned(4))) u32x4_el4;
typedef u32x4 __attribute__((aligned(2))) u32x4_el2;

// Row-mapped form: out row out_rows[b K + j] of sequence b = P of logits row in_rows[b K + j] (whose
// statistics are at [b, in_rows[..]]). An index outside its range skips the row: the maps are device
// data the host cannot check. Four elements per thread per step, the last V % 4 one per thread.
__global__ __launch_bounds__(256) void probs_rows_kernel(const float* logits, int64_t bs, int64_t rs, int R, int V,
                                                         double rt, int ban, const float* m, const float* thr,
                                                         const double* zk, const int64_t* in_rows,
                                                         const int64_t* out_rows, int K, int Ro, float* out,
                                                         int64_t obs, int64_t ors) {
  const int r = blockIdx.y;
  const int b = r / K;
  const int64_t i = in_rows[r], o = out_rows[r];
  if (i < 0 || i >= R || o < 0 || o >= Ro) return;  // block-uniform
  const float* row = logits + (int64_t)b * bs + i * rs;
  float* dst = out + (int64_t)b * obs + o * ors;
  const int64_t si = (int64_t)b * R + i;
  const float mm = m[si], t = thr[si];
  const float inv = (float)(1.0 / zk[si]);
  auto p_of = [&](float x, int ix) {
    const float y = make_y<true>(x, ix, rt, ban);
    return (y > -INFINITY && y >= t) ? __expf(y - mm) * inv : 0.f;
  };
  const int n4 = V >> 2;
  for (int j = blockIdx.x * 256 + threadIdx.x; j < n4; j += gridDim.x * 256) {
    const u32x4 w = reinterpret_cast<const u32x4_el4*>(row)[j];
    u32x4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = __float_as_uint(p_of(__uint_as_float(w[e]), 4 * j + e));
    reinterpret_cast<u32x4_el4*>(dst)[j] = y;
  }
  const int ix = 4 * n4 + (int)threadIdx.x;
  if (blockIdx.x == 0 && ix < V) dst[ix] = p_of(row[ix], ix);
}

// dst[b, k, :] = fp32(src[b, rows[b, k], :]) for bf16 (kBf16) or fp32 sources; a row index outside
// [0, R) skips the row. 16-byte loads (8 bf16 or 4 fp32 elements), the last V % 8 / V % 4 one per thread.
template <bool kBf16>
__global__ __launch_bounds__(256) void gather_rows_kernel(const void* src, int64_t sbs, int64_t srs, int R, int V,
                                                          const int64_t* rows, int K, float* dst, int64_t dbs,
                                                          int64_t drs) {
  const int r = blockIdx.y;
  const int b = r / K, k = r % K;
  const int64_t i = rows[r];
  if (i < 0 || i >= R) return;  // block-uniform
  float* d = dst + (int64_t)b * dbs + (int64_t)k * drs;
  const int64_t off = (int64_t)b * sbs + i * srs;
  constexpr int E = kBf16 ? 8 : 4;
  const int nv = V / E, ix = nv * E + (int)threadIdx.x;
  if (kBf16) {
    const uint16_t* s = static_cast<const uint16_t*>(src) + off;
    for (int j = blockIdx.x * 256 + threadIdx.x; j < nv; j += gridDim.x * 256) {
      const u32x4 w = reinterpret_cast<const u32x4_el2*>(s)[j];
      u32x4 lo, hi;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        lo[2 * e] = w[e] << 16;
        lo[2 * e + 1] = w[e] & 0xffff0000u;
        hi[2 * e] = w[2 + e] << 16;
        hi[2 * e + 1] = w[2 + e] & 0xffff0000u;
      }
      reinterpret_cast<u32x4_el4*>(d)[2 * j] = lo;
      reinterpret_cast<u32x4_el4*>(d)[2 * j + 1] = hi;
    }
    if (blockIdx.x == 0 && ix < V) d[ix] = bf2f(s[ix]);
  } else {
    const float* s = static_cast<const float*>(src) + off;
    for (int j = blockIdx.x * 256 + threadIdx.x; j < nv; j += gridDim.x * 256)
      reinterpret_cast<u32x4_el4*>(d)[j] = reinterpret_cast<const u32x4_el4*>(s)[j];
    if (blockIdx.x == 0 && ix < V) d[ix] = s[ix];
  }
}
}  // namespace
}  // namespace trida

extern "C" int trida_truncated_probs_rows(const float* logits, int64_t B, int64_t R, int64_t V, int64_t batch_stride,
                                          int64_t row_stride, float temperature, int64_t ban_id, const float* m,
                                          const float* thr, const double* zk, const int64_t* in_rows,
                                          const int64_t* out_rows, int64_t K, float* probs, int64_t Ro,
                                          int64_t out_batch_stride, int64_t out_row_stride, void* stream) {
  TRIDA_CHECK(logits && m && thr && zk && in_rows && out_rows && probs, TRIDA_ERR_NULL, "null pointer argument");
  TRIDA_CHECK(B > 0 && R > 0 && K >= 0 && Ro > 0 && B * K <= 65535 && V > 0 && V < INT_MAX / 2, TRIDA_ERR_ARG,
              "bad shape");
  TRIDA_CHECK(temperature > 0.f && temperature < INFINITY, TRIDA_ERR_ARG, "temperature must be positive");
  TRIDA_CHECK(row_stride >= V && out_row_stride >= V &&
                  (B == 1 || (batch_stride >= (R - 1) * row_stride + V &&
                              out_batch_stride >= (Ro - 1) * out_row_stride + V)),
              TRIDA_ERR_ARG, "strides too small");
  if (K == 0) return TRIDA_OK;
  const int gx = (int)std::min<int64_t>(cdiv(V, 256 * 4), 256);
  hipLaunchKernelGGL(probs_rows_kernel, dim3(gx, (unsigned)(B * K)), dim3(256), 0, static_cast<hipStream_t>(stream), logits,
                     batch_stride, row_stride, (int)R, (int)V, 1.0 / (double)temperature, ban_of(ban_id, V), m, thr, zk,
                     in_rows, out_rows, (int)K, (int)Ro, probs, out_batch_stride, out_row_stride);
  return launch_status("probs_rows_kernel");
}

extern "C" int trida_gather_rows(const void* src, int dtype, int64_t B, int64_t R, int64_t V, int64_t batch_stride,
                                 int64_t row_stride, const int64_t* rows, int64_t K, float* dst,
                                 int64_t out_batch_stride, int64_t out_row_stride, void* stream) {
  TRIDA_CHECK(src && rows && dst, TRIDA_ERR_NULL, "null pointer argument");
  TRIDA_CHECK(dtype == 0 || dtype == 1, TRIDA_ERR_ARG, "dtype must be 0 (fp32) or 1 (bf16)");
  TRIDA_CHECK(B > 0 && R > 0 && K >= 0 && B * K <= 65535 && V > 0 && V < INT_MAX / 2, TRIDA_ERR_ARG, "bad shape");
  TRIDA_CHECK(row_stride >= V && out_row_stride >= V &&
                  (B == 1 || (batch_stride >= (R - 1) * row_stride + V &&
                              out_batch_stride >= (K - 1) * out_row_stride + V)),
              TRIDA_ERR_ARG, "strides too small");
  if (K == 0) return TRIDA_OK;
  const int gx = (int)std::min<int64_t>(cdiv(V, 256 * (dtype == 1 ? 8 : 4)), 256);
  const dim3 grid(gx, (unsigned)(B * K));
  const hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == 1)
    hipLaunchKernelGGL((gather_rows_kernel<true>), grid, dim3(256), 0, st, src, batch_stride, row_stride, (int)R, (int)V,
                       rows, (int)K, dst, out_batch_stride, out_row_stride);
  else
    hipLaunchKernelGGL((gather_rows_kernel<false>), grid, dim3(256), 0, st, src, batch_stride, row_stride, (int)R, (int)V,
                       rows, (int)K, dst, out_batch_stride, out_row_stride);
  return launch_status("gather_rows_kernel");
}

extern "C" int trida_truncated_probs(const float* logits, int64_t B, int64_t R, int64_t V, int64_t batch_stride,
                                     int64_t row_stride, float temperature, int64_t ban_id, const float* m,
                                     const float* thr, const double* zk, float* probs, int64_t out_batch_stride,
                                     int64_t out_row_stride, void* stream) {
  TRIDA_CHECK(logits && m && thr && zk && probs, TRIDA_ERR_NULL, "null pointer argument");
  TRIDA_CHECK(B > 0 && R > 0 && B * R <= 65535 && V > 0 && V < INT_MAX / 2, TRIDA_ERR_ARG, "bad shape");
  TRIDA_CHECK(temperature > 0.f && temperature < INFINITY, TRIDA_ERR_ARG, "temperature must be positive");
  TRIDA_CHECK(row_stride >= V && out_row_stride >= V &&
                  (B == 1 || (batch_stride >= (R - 1) * row_stride + V &&
                              out_batch_stride >= (R - 1) * out_row_stride + V)),
              TRIDA_ERR_ARG, "strides too small");
  const int gx = (int)std::min<int64_t>(cdiv(V, 256 * 8), 256);
  hipLaunchKernelGGL(probs_kernel, dim3(gx, B * R), dim3(256), 0, static_cast<hipStream_t>(stream), logits, batch_stride, row_stride, (int)R,
                     (int)V, 1.0 / (double)temperature, ban_of(ban_id, V), m, thr, zk, probs, out_batch_stride, out_row_stride);
  return launch_status("probs_kernel");
}

// ---------------------------------------------------------------- draws from given truncation statistics
// The residual kernels with no drafts: per row, the inverse CDF in vocabulary order of
// P(x) = [y_x >= thr] exp(y_x - m) / zk at one uniform. Scratch: the per-row bookkeeping those kernels
// read and write, then the chunk sums.
namespace trida {
namespace {
struct DrawScratch {
  int64_t state, rstatus, status, n_acc, crop, sums, total;
};
DrawScratch draw_layout(int64_t rows, int64_t V) {
  int NC, chunk;
  plan_chunks(rows, V, &NC, &chunk);
  DrawScratch L;
  L.state = 0;
  L.rstatus = L.state + align_up(rows * 4, 256);
  L.status = L.rstatus + align_up(rows * 4, 256);
  L.n_acc = L.status + align_up(rows * 4, 256);
  L.crop = L.n_acc + align_up(rows * 4, 256);
  L.sums = L.crop + align_up(rows * 8, 256);
  L.total = L.sums + align_up(rows * NC * 2 * 8, 256);
  return L;
}
}  // namespace
}  // namespace trida

extern "C" int64_t trida_sample_rows_scratch_bytes(int64_t rows, int64_t V) {
  if (rows <= 0 || V <= 0) return 0;
  return draw_layout(rows, V).total;
}

extern "C" int trida_sample_rows(const float* logits, int64_t rows, int64_t V, int64_t row_stride, float temperature,
                                 int64_t ban_id, const float* m, const float* thr, const double* zk, const float* u,
                                 int64_t* token, void* scratch, int64_t scratch_bytes, void* stream) {
  TRIDA_CHECK(logits && m && thr && zk && u && token && scratch, TRIDA_ERR_NULL, "null pointer argument");
  TRIDA_CHECK(rows > 0 && rows <= 65535 && V > 0 && V < INT_MAX / 2, TRIDA_ERR_ARG, "bad shape rows=%lld V=%lld",
              (long long)rows, (long long)V);
  TRIDA_CHECK(temperature > 0.f && temperature < INFINITY, TRIDA_ERR_ARG, "temperature must be positive");
  TRIDA_CHECK(row_stride >= V, TRIDA_ERR_ARG, "row_stride too small");
  const DrawScratch L = draw_layout(rows, V);
  TRIDA_CHECK(scratch_bytes >= L.total, TRIDA_ERR_WORKSPACE, "scratch of %lld bytes, need %lld",
              (long long)scratch_bytes, (long long)L.total);
  TRIDA_CHECK((uintptr_t)scratch % 256 == 0, TRIDA_ERR_ALIGN, "scratch must be 256-byte aligned");
  char* s = static_cast<char*>(scratch);
  int NC, chunk;
  plan_chunks(rows, V, &NC, &chunk);
  AcceptArgs aa{logits, row_stride, 0, nullptr, 0, 0, nullptr, 0, nullptr, nullptr, 0, u, nullptr, (int)rows, (int)V, 0,
                1.0 / (double)temperature, ban_of(ban_id, V), m, thr, zk, nullptr,
                reinterpret_cast<int*>(s + L.state), reinterpret_cast<int*>(s + L.rstatus), NC, chunk,
                reinterpret_cast<double*>(s + L.sums), reinterpret_cast<int32_t*>(s + L.n_acc), token,
                reinterpret_cast<int64_t*>(s + L.crop), nullptr, reinterpret_cast<int32_t*>(s + L.status)};
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(resid_sums_kernel, dim3(NC, rows), dim3(kRT), 0, st, aa);
  const int r = launch_status("resid_sums_kernel (draw)");
  if (r != TRIDA_OK) return r;
  hipLaunchKernelGGL(resid_pick_kernel, dim3(rows), dim3(kRT), 0, st, aa);
  return launch_status("resid_pick_kernel (draw)");
}
