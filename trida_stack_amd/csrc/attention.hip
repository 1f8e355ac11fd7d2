// Canvas attention over a bf16 KV cache (draft / verify / mixed masks), MFMA on gfx950.
//
// Query rows of one KV head are the pairs (canvas row t, GQA head g), row m = t * G + g, so the G query
// heads sharing a KV head form one [T*G, D] matrix. Keys p in [0, prefix + T) of the cache; row t sees
// key p when p < prefix (the committed prefix) or, inside the block (j = p - prefix):
//   mask 0 (verify, causal)       j <= t
//   mask 1 (draft, bidirectional) always
//   mask 2 (canvas, mixed)        j <= t for t < n_clean, always for t >= n_clean
//
// attn_partial: workgroup = (sequence, KV head, query tile of <= 128 rows, key split), 4 waves of 16 or 32
//   rows each. Per 64-key step, K and V are staged in one of two LDS buffers (swizzled, loaded to LDS directly while
//   the other is in use); every wave computes S^T = K Q^T for its rows with v_mfma_f32_16x16x32_bf16 (K fragments
//   from LDS, Q in registers), runs the online softmax within the wave, and accumulates O^T += V^T P^T
//   with the V^T fragments read by ds_read_b64_tr_b16.
//   Writes the unnormalised O (bf16), row max and row sum (fp32) of its split. A last tile of <= 16
//   rows can join the tile before it as its extra rows (a canvas of 33 rows x 4 heads = 128 + 4), so
//   the keys stream once for all rows.
// attn_combine: merges the splits per row (log-sum-exp weights), applies the optional output gate
//   sigmoid(gate) and writes bf16; attn_combine2 does the same for exactly two splits in one memory round
//   trip per row.
#include <math.h>

#include "common.h"

namespace trida {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr int kNW = 4;              // waves per workgroup
constexpr int kWR = 16;             // an MFMA row tile
constexpr int kMT = kNW * 2 * kWR;  // query rows per workgroup (two row tiles per wave), before extra rows
constexpr int kMTX = kMT + kWR;     // with a last tile's <= 16 extra rows
constexpr int kKB = 64;             // keys per step
constexpr float kLog2e = 1.4426950408889634f;
constexpr int kMaxLptSeqs = 256;  // batches up to this size are scheduled longest-first

// The max over the four lanes of a row (l, l ^ 16, l ^ 32, l ^ 48), without a trip through LDS: each swap leaves a
// lane's value and its partner's in the two results
__device__ __forceinline__ float row_max(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// 2^x with the hardware instruction: exact for the softmax's arguments x <= 0 down to -126, 0 below
// (where the library exp2f would return a denormal)
__device__ __forceinline__ float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 w) { return __builtin_bit_cast(bf16x8, w); }

struct AttnArgs {
  const uint16_t* q;        // [B, T, Hq, D]
  const uint16_t* k_cache;  // [B, Hkv, Lmax, D]
  const uint16_t* v_cache;
  const int32_t* prefix;    // [B]
  uint16_t* opart;          // [B, Hkv, QT, S, kMTX, D] bf16
  float* mpart;             // [B, Hkv, QT, S, kMTX]
  float* lpart;
  int T, Hq, Hkv, G, Lmax, S, QT, mask_mode, n_clean;
  float scale_log2;         // softmax scale * log2(e)
  // with one key split (S == 1) the partial kernel writes the final, gated output as the combine would
  const uint16_t* gate;     // row t, head h, dim d at gate + t * gate_st + h * gate_hs + d; or null
  int64_t gate_st, gate_hs;
  uint16_t* out;            // [B, T, Hq, D], or the weight-streaming GEMM's fragment order (frag)
  int frag;
};

// LDS tiles of one 64-key step, [key][D] with the pieces of a key XOR-swizzled so that the MFMA fragment reads
// touch distinct banks:
//   K  16-byte group g of key k at g ^ (k & 7) (16-byte fragment reads, 8 keys per 8 lanes)
//   V  32-byte unit u of key k at u ^ vswz(k): the V^T fragments of the P V^T product come from ds_read_b64_tr_b16
//      (8 bytes of one key per lane, handed out transposed), and the 32 lanes of a half-wave, 8 keys x 32 bytes,
//      then fall on distinct banks
// The tiles are written by global_load_lds: a wave's load fills 1 KB in lane order, so the swizzle is in the
// address that each lane loads from.
template <int D>
__device__ __forceinline__ int k_off(int key, int grp) { return key * D + ((grp ^ (key & 7)) << 3); }
template <int D>
__device__ __forceinline__ int vswz(int key) { return D >= 128 ? key & 7 : (key >> 1) & 3; }
template <int D>
__device__ __forceinline__ int v_off(int key, int unit) { return key * D + ((unit ^ vswz<D>(key)) << 4); }

// 64 lanes x 16 bytes from each lane's address to LDS at `lds` (bytes, wave-uniform) + 16 lane, asynchronously: counted by
// vmcnt, no register written. In asm because the compiler would wait for it before every later LDS read; nothing else in these
// kernels uses m0.
__device__ __forceinline__ void load_lds16(const uint16_t* src, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(src) : "memory", "m0");
}
__device__ __forceinline__ uint32_t lds_addr(const void* p) { return (uint32_t)(uintptr_t)p; }
// Every wave's loads to LDS have arrived and its LDS reads have returned: the other tile buffer may be overwritten.
__device__ __forceinline__ void step_barrier() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Fragment reads at an LDS byte address: a lane's addresses within a tile differ by constants (instruction
// offsets) from a few that depend on the swizzle, FragAt; left to the compiler, each of the step's fragments had
// an address register of its own.
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
// ds_read_b64_tr_b16 (gfx950): in each group of 16 lanes, lane 4 a + b receives element b of the 8-byte
// reads of lanes a, a + 4, a + 8 and a + 12 (in that order). A lane of group g reading key key0 + 4 g +
// (lane % 16) / 4 at columns d0 + 4 (lane % 4) .. + 3 thus receives V[key0 + 4 g + j][d0 + lane % 16] for
// j = 0..3: four keys of its V^T row, in the k slots of the MFMA's A operand.
template <int D>
struct FragAt {
  static constexpr int VU = D >= 128 ? 8 : 4;  // units of a key within the V swizzle's reach
  uint32_t k[2], v[VU];
  __device__ __forceinline__ FragAt(int l) {
    const int key = 4 * (l / 16) + (l % 16) / 4;
#pragma unroll
    for (int i = 0; i < 2; ++i) k[i] = 2 * k_off<D>(l % 16, 4 * i + l / 16);
#pragma unroll
    for (int u = 0; u < VU; ++u) v[u] = 2 * (v_off<D>(key, u) + 4 * (l % 4));
  }
  // K (or Q) row key0 + lane % 16, columns 32 kc + 8 (lane / 16) .. + 7; key0 a multiple of 16
  __device__ __forceinline__ bf16x8 row(uint32_t tile, int key0, int kc) const {
    return as_bf16x8(*(lds_u32x4*)(tile + k[kc % 2] + (uint32_t)(key0 * D * 2 + (kc / 2) * 128)));
  }
  // V^T row 16 ct + lane % 16, keys key0 + 4 (lane / 16) .. + 3
  __device__ __forceinline__ s16x4 col(uint32_t tile, int key0, int ct) const {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_s16x4*)(tile + v[ct % VU] + (uint32_t)(key0 * D * 2 + (ct / VU) * (VU * 32))));
  }
};

struct Tile {  // a workgroup's part, block-uniform
  int b, hk, m0, rows, nx;   // sequence, KV head, first query row, rows, those past kMT
  int prefix, nk, kb0, kb1;  // keys: the committed ones, all, the split's 64-key steps
  int64_t pbase;             // the split's slot of the partial results
};

// Workgroup = (sequence, KV head, query tile of kMT rows, key split); 4 waves, wave w owns RT row tiles of 16: rows
// [16 RT w, 16 RT (w + 1)) of the tile, their Q as B fragments in registers. Per 64-key step, K and V are staged
// in one of two LDS buffers while the next step's tiles stream into the other (global_load_lds), and the
// wave forms the transposed products S^T = K Q^T and O^T += V^T P^T on v_mfma_f32_16x16x32_bf16, so lane l holds
// 16 scores and 256 / 4 output values of one query row (l % 16) of each tile: the online softmax of a row is
// the lane's own, completed across its four lane groups by two lane swaps, and its probabilities are, as
// computed, the B operand of the product with V (a 32-key block takes slots 8 g + j = keys 32 kk + 4 g + j
// and 32 kk + 16 + 4 g + j - 4, which is where the two key tiles' accumulators put them). O is rescaled only
// when a row's running max moved. Writes the unnormalised O, the row max (log2 domain) and the row sum of its split.
// Each K and V fragment read feeds RT products: what bounds a step is LDS reads (each wave reads both tiles, 64
// KB at D = 256), so 32 rows per wave halve them against 16. RT = 1 serves tiles of <= 64 rows, whose waves
// would otherwise be idle.
// A call with its combine, against 8 waves of 16 rows, tiles staged through registers between two barriers and Q in LDS: 64
// sequences of 33 rows and 512-4096 keys 232 -> 205 us (head dim 256, nothing cached; 128: 131 -> 113.5), a 512-row
// chunk behind 3584 keys 73 -> 60.5, 33 rows over 8192 keys 32.9 -> 29.4, 50 sequences of 7 rows and 300 keys
// 39.2 -> 35.1. With one to three key steps per workgroup and more than one split it is up to 1 % slower (2 x 32
// rows over 5738 keys 38.7 -> 39.2). A step of 32 rows per wave takes about 3 us of MFMA, LDS reads and softmax one after
// the other, as 2 x 64 KB of tiles leave room for one workgroup per CU.
// Extra rows (EXTRA: the last tile's kMT .. kMT + 15): a third row tile of every wave, from the K fragments the wave
// reads for its own rows (Q from LDS); of their O^T, wave w accumulates the column tiles [XC w, XC (w + 1)).
template <int D, int RT, bool EXTRA>
__device__ __forceinline__ void attn_tile(const AttnArgs& a, const Tile& wt, uint16_t (*sKV)[2][kKB * D], uint16_t* sQx) {
  constexpr int KC = D / 32;         // 32-wide k-chunks of the head dim (QK^T)
  constexpr int CT = D / 16;         // 16-column tiles of O
  constexpr int GPR = D / 8;         // 16-byte groups per K row
  constexpr int NT = kNW * kWave;
  constexpr int KPL = kWave / GPR;          // keys per wave load (1 KB)
  constexpr int NL = kKB / (KPL * kNW);     // loads per wave of a tile
  constexpr int ST = RT + (EXTRA ? 1 : 0);  // row tiles that form scores: the extra rows are the last one
  constexpr int XC = CT / kNW;              // column tiles of the extra rows per wave
  constexpr int TILE = kKB * D;

  const int tid = threadIdx.x, w = tid / kWave, l = tid % kWave;
  const int b = wt.b, hk = wt.hk, m0 = wt.m0, rows = wt.rows, nx = wt.nx;
  const int prefix = wt.prefix, nk = wt.nk, kb0 = wt.kb0, kb1 = wt.kb1;
  const int64_t pbase = wt.pbase;
  const uint16_t* kh = a.k_cache + ((int64_t)b * a.Hkv + hk) * a.Lmax * D;
  const uint16_t* vh = a.v_cache + ((int64_t)b * a.Hkv + hk) * a.Lmax * D;

  // ---- the step's tiles, key KPL (w + 4 j) + l / GPR of each lane's load j (keys past the last one re-read it). The
  // swizzles depend on the key's low bits only, the same for every j.
  const int lkey = KPL * w + l / GPR, lg = l % GPR;
  const uint16_t* ksrc = kh + ((lg ^ (lkey & 7)) << 3);
  const uint16_t* vsrc = vh + ((((lg >> 1) ^ vswz<D>(lkey)) << 4) + ((lg & 1) << 3));
  auto load_step = [&](int kb, int buf) {
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      const int64_t row = (int64_t)min(kb * kKB + lkey + j * KPL * kNW, nk - 1) * D;
      const uint32_t at = lds_addr(&sKV[buf][0][0]) + (uint32_t)((w + j * kNW) * 1024);
      load_lds16(ksrc + row, __builtin_amdgcn_readfirstlane(at));
      load_lds16(vsrc + row, __builtin_amdgcn_readfirstlane(at + TILE * 2));
    }
  };
  load_step(kb0, 0);

  // ---- the Q rows as B fragments (rows past the tile zero)
  const int wr0 = w * RT * kWR;  // the wave's first row
  bf16x8 qf[RT][KC];
  {
    auto q_at = [&](int m, int kc) {
      const int t = m / a.G, g = m % a.G;
      return as_bf16x8(*reinterpret_cast<const u32x4*>(a.q + (((int64_t)b * a.T + t) * a.Hq + hk * a.G + g) * D + kc * 32 +
                                                       (l / 16) * 8));
    };
    const bf16x8 zero = as_bf16x8(u32x4{0u, 0u, 0u, 0u});
    // the softmax takes a scale >= 0: a negative one's sign goes to Q
    auto neg = [](bf16x8 v) { return as_bf16x8(__builtin_bit_cast(u32x4, v) ^ 0x80008000u); };
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int r = wr0 + rt * kWR + l % 16;
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
        qf[rt][kc] = q_at(m0 + min(r, rows - 1), kc);
        if (r >= rows) qf[rt][kc] = zero;
        else if (a.scale_log2 < 0.f) qf[rt][kc] = neg(qf[rt][kc]);
      }
    }
    if (EXTRA) {  // the first step's barrier publishes them
      for (int i = tid; i < kWR * GPR; i += NT) {
        const int r = i / GPR, m = m0 + kMT + min(r, nx - 1), t = m / a.G, g = m % a.G;
        const u32x4 v =
            *reinterpret_cast<const u32x4*>(a.q + (((int64_t)b * a.T + t) * a.Hq + hk * a.G + g) * D + (i % GPR) * 8);
        *reinterpret_cast<u32x4*>(&sQx[k_off<D>(r, i % GPR)]) =
            r < nx ? v ^ (a.scale_log2 < 0.f ? 0x80008000u : 0u) : u32x4{0u, 0u, 0u, 0u};
      }
    }
  }

  // o[rt][ct] holds O[row][16 ct + 4 (l / 16) + e] of this lane's query row of tile rt
  f32x4 o[RT][CT];
  f32x4 ox[EXTRA ? XC : 1];  // the extra rows' column tiles [XC w, XC (w + 1))
  float m_run[ST], l_run[ST];
  // the keys the lane's row sees are exactly [0, klim): the whole prefix, then the block keys its mask
  // allows (a prefix of the block for the causal rows, all of it for the others)
  int klim[ST];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) o[rt][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < (EXTRA ? XC : 1); ++c) ox[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int rt = 0; rt < ST; ++rt) {
    m_run[rt] = -INFINITY;
    l_run[rt] = 0.f;
    const int r = rt < RT ? wr0 + rt * kWR + l % 16 : kMT + min(l % 16, max(nx, 1) - 1);
    const int t = (m0 + r) / a.G;
    const bool all = a.mask_mode == 1 || (a.mask_mode == 2 && t >= a.n_clean);
    klim[rt] = all ? nk : min(nk, prefix + t + 1);
  }
  const int g4 = 4 * (l / 16);
  const float scale_log2 = fabsf(a.scale_log2);

  // ---- online softmax of one step's raw scores sc (keys 16 kt + g4 + e of the lane's row, which sees the keys
  // below lim) against the row's running max m (log2 units) and the lane's own part of the row sum, lsum; leaves the
  // probabilities as the B fragments of the two 32-key blocks in pb. The mask applies only on steps that reach the
  // block keys or the cache end (uniform); the exchange between a row's four lanes and `rescale` (of the row's O)
  // run only when a score passes the max. A max that moves only when passed by 2^8 saves most of the moves (205 instead of
  // 227 us on 64 ragged sequences, 62 instead of 67 on a 512-row chunk), but the largest probabilities are then no longer
  // just below 1, where bf16 is finest: 2.5 % more error against 64 bits.
  auto softmax_step = [&](f32x4 (&sc)[4], int key0, int lim, float& m, float& lsum, u32x4 (&pb)[2], auto&& rescale) {
    const bool edge = key0 + kKB > prefix || key0 + kKB > nk;
    if (edge) {
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int e = 0; e < 4; ++e) sc[kt][e] = key0 + 16 * kt + g4 + e < lim ? sc[kt][e] : -INFINITY;
    }
    float mx = fmaxf(fmaxf(sc[0][0], sc[0][1]), fmaxf(sc[0][2], sc[0][3]));
#pragma unroll
    for (int kt = 1; kt < 4; ++kt) mx = fmaxf(mx, fmaxf(fmaxf(sc[kt][0], sc[kt][1]), fmaxf(sc[kt][2], sc[kt][3])));
    mx *= scale_log2;
    if (__ballot(mx > m)) {
      const float m_new = fmaxf(m, row_max(mx));
      const float alpha = m_new > m ? exp2_hw(m - m_new) : 1.f;
      m = m_new;
      lsum *= alpha;
      rescale(alpha);
    }
    const float m_use = m == -INFINITY ? 0.f : m;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      float p[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        p[e] = fmaf(sc[2 * kk][e], scale_log2, -m_use);
        p[4 + e] = fmaf(sc[2 * kk + 1][e], scale_log2, -m_use);
      }
      if (edge && scale_log2 == 0.f) {  // 0 x -inf
#pragma unroll
        for (int e = 0; e < 8; ++e) p[e] = sc[2 * kk + e / 4][e % 4] == -INFINITY ? -INFINITY : p[e];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        p[e] = exp2_hw(p[e]);
        lsum += p[e];
      }
      pb[kk] = u32x4{f2bf2(p[0], p[1]), f2bf2(p[2], p[3]), f2bf2(p[4], p[5]), f2bf2(p[6], p[7])};
    }
  };

  const FragAt<D> at(l);
  uint32_t vx[EXTRA ? XC : 1];  // FragAt::v of the wave's extra column tiles
  if (EXTRA) {
#pragma unroll
    for (int c = 0; c < XC; ++c)
      vx[EXTRA ? c : 0] = 2 * (v_off<D>(4 * (l / 16) + (l % 16) / 4, w * XC + c) + 4 * (l % 4));
  }

  // a wave with no row of the tile (a last tile of fewer rows) only loads keys: its fragment
  // reads and MFMAs would be on padding
  if (!EXTRA && wr0 >= rows) {
    for (int kb = kb0; kb < kb1; ++kb) {
      step_barrier();
      if (kb + 1 < kb1) load_step(kb + 1, (kb - kb0 + 1) & 1);
    }
    return;
  }
  auto step = [&](int kb, bool last) {
    const int key0 = kb * kKB, buf = (kb - kb0) & 1;
    step_barrier();  // this step's tiles are in, the previous step's are consumed
    if (!last) load_step(kb + 1, buf ^ 1);  // in flight during this step's MFMAs
    const uint32_t tk = lds_addr(&sKV[0][0][0]) + (uint32_t)buf * (4 * TILE), tv = tk + 2 * TILE;
    FragAt<D> fk = at;  // this step's K and V addresses
#pragma unroll
    for (int i = 0; i < 2; ++i) fk.k[i] += tk;
#pragma unroll
    for (int u = 0; u < FragAt<D>::VU; ++u) fk.v[u] += tv;
    // ---- S^T = K Q^T: keys 16 kt + 4 (l / 16) + e of this lane's query rows (4 key tiles)
    f32x4 sacc[ST][4];
#pragma unroll
    for (int rt = 0; rt < ST; ++rt)
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) sacc[rt][kt] = f32x4{0.f, 0.f, 0.f, 0.f};
    // fragments are read two k-chunks ahead; the scheduling barriers keep the compiler from hoisting more of
    // them than there are registers
    bf16x8 kf[3][4], xf[3];
    auto read_k = [&](int kc) {
      if (EXTRA) xf[kc % 3] = at.row(lds_addr(sQx), 0, kc);
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) kf[kc % 3][kt] = fk.row(0, kt * 16, kc);
    };
    read_k(0);
    if (KC > 1) read_k(1);
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) {
      if (kc + 2 < KC) read_k(kc + 2);
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int rt = 0; rt < ST; ++rt)
          sacc[rt][kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[kc % 3][kt], rt < RT ? qf[rt < RT ? rt : 0][kc] : xf[kc % 3],
                                                                 sacc[rt][kt], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    // V^T fragments, groups of four column tiles, two groups ahead (the first two before the softmax)
    constexpr int VG = CT / 4, NV = (kKB / 32) * VG;  // groups per 32 keys, in all
    bf16x8 vf[3][4];
    auto read_v = [&](int i) {
      const int kk = i / VG;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int ct = (i % VG) * 4 + c;
        const s16x4 v0 = fk.col(0, 32 * kk, ct), v1 = fk.col(0, 32 * kk + 16, ct);
        const u32x2 w0 = __builtin_bit_cast(u32x2, v0), w1 = __builtin_bit_cast(u32x2, v1);
        vf[i % 3][c] = as_bf16x8(u32x4{w0.x, w0.y, w1.x, w1.y});
      }
    };
    read_v(0);
    read_v(1);
    __builtin_amdgcn_sched_barrier(0);
    u32x4 pb[ST][2];
#pragma unroll
    for (int rt = 0; rt < ST; ++rt) {
      softmax_step(sacc[rt], key0, klim[rt], m_run[rt], l_run[rt], pb[rt], [&](float alpha) {
        if (rt < RT) {
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[rt < RT ? rt : 0][ct][e] *= alpha;
        } else {
#pragma unroll
          for (int c = 0; c < (EXTRA ? XC : 1); ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) ox[c][e] *= alpha;
        }
      });
    }
    // ---- O^T += V^T P^T (V^T fragments by transposed LDS reads, in the slot order of the probabilities:
    // keys 32 kk + g4 .. + 3, then 32 kk + 16 + g4 .. + 3)
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      if (i + 2 < NV) read_v(i + 2);
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          const int ct = (i % VG) * 4 + c;
          o[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[i % 3][c], as_bf16x8(pb[rt][i / VG]), o[rt][ct], 0, 0, 0);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (EXTRA) {
#pragma unroll
      for (int kk = 0; kk < kKB / 32; ++kk)
#pragma unroll
        for (int c = 0; c < (EXTRA ? XC : 1); ++c) {
          const u32x2 w0 = __builtin_bit_cast(
              u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(tv + vx[c] + (uint32_t)(32 * kk * D * 2))));
          const u32x2 w1 = __builtin_bit_cast(
              u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(tv + vx[c] + (uint32_t)((32 * kk + 16) * D * 2))));
          ox[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(u32x4{w0.x, w0.y, w1.x, w1.y}), as_bf16x8(pb[ST - 1][kk]),
                                                          ox[c], 0, 0, 0);
        }
    }
  };
  // the last step, which loads nothing, apart: a conditional load in the loop left O's 128 registers moving
  // between its blocks
  for (int kb = kb0; kb + 1 < kb1; ++kb) step(kb, false);
  step(kb1 - 1, true);
#pragma unroll
  for (int rt = 0; rt < ST; ++rt) {  // the rows' sums
    l_run[rt] += __shfl_xor(l_run[rt], 16, kWave);
    l_run[rt] += __shfl_xor(l_run[rt], 32, kWave);
  }
  const int rx = kMT + (l % 16);  // the lane's extra row of the tile
  const bool extra = EXTRA && l % 16 < nx;
  if (a.S == 1) {
    // ---- the only split: O / l, rounded to bf16, then the gate, exactly as the combine computes it. The wave's gate
    // loads go out before its first store; one by one, each waited for memory behind the store before it, 32 in turn: with
    // nothing cached, 38 sequences of 32 rows and 188 keys took 45.4 instead of 38.7 us, 46 of 477 keys 61.6 instead of
    // 55.2, 64 of 33 rows and 512-4096 keys at head dim 256 208 instead of 205.
    auto gate_at = [&](int rr, int ct) {
      const int m = m0 + rr, t = m / a.G, hq = hk * a.G + m % a.G;
      return *reinterpret_cast<const u32x2*>(a.gate + ((int64_t)b * a.T + t) * a.gate_st + (int64_t)hq * a.gate_hs + ct * 16 + g4);
    };
    auto emit = [&](int rr, float lsum, const f32x4& v, u32x2 gw, int ct) {
      const int m = m0 + rr, t = m / a.G, hq = hk * a.G + m % a.G;
      const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
      const int c = ct * 16 + g4;
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = bf2f(f2bf(v[e])) * inv;
      if (a.gate) {
        const float gv[4] = {__uint_as_float(gw.x << 16), __uint_as_float(gw.x & 0xffff0000u),
                             __uint_as_float(gw.y << 16), __uint_as_float(gw.y & 0xffff0000u)};
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = bf2f(f2bf(y[e])) * (1.f / (1.f + __expf(-gv[e])));
      }
      uint16_t* dst = a.frag ? a.out + ws_frag_off(b * a.T + t, (int64_t)hq * D + c)
                             : a.out + (((int64_t)b * a.T + t) * a.Hq + hq) * D + c;
      *reinterpret_cast<u32x2*>(dst) = u32x2{f2bf2(y[0], y[1]), f2bf2(y[2], y[3])};
    };
    u32x2 gw[RT][CT], gx[EXTRA ? XC : 1];
    constexpr bool early = !(EXTRA && D == 128);  // there the registers (256) hold one row tile's
    auto load_gates = [&](int rt) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
        gw[rt][ct] = a.gate ? gate_at(min(wr0 + rt * kWR + (l % 16), rows - 1), ct) : u32x2{0u, 0u};
    };
    if (early) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) load_gates(rt);
    }
    if (EXTRA) {
#pragma unroll
      for (int c = 0; c < (EXTRA ? XC : 1); ++c)
        gx[c] = a.gate ? gate_at(kMT + min(l % 16, max(nx, 1) - 1), w * XC + c) : u32x2{0u, 0u};
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int r = wr0 + rt * kWR + (l % 16);
      if (r >= min(rows, kMT)) continue;
      if (!early) load_gates(rt);
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) emit(r, l_run[rt], o[rt][ct], gw[rt][ct], ct);
    }
    if (extra) {
#pragma unroll
      for (int c = 0; c < (EXTRA ? XC : 1); ++c) emit(rx, l_run[ST - 1], ox[c], gx[c], w * XC + c);
    }
    return;
  }
  // ---- write this split's unnormalised O (bf16: half the partial traffic; 8-byte row pieces) and row
  // stats (fp32)
  uint16_t* op = a.opart + pbase * kMTX * D;
  auto park = [&](int rr, const f32x4& v, int ct) {
    *reinterpret_cast<u32x2*>(&op[(int64_t)rr * D + ct * 16 + g4]) = u32x2{f2bf2(v[0], v[1]), f2bf2(v[2], v[3])};
  };
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int r = wr0 + rt * kWR + (l % 16);
    if (r >= min(rows, kMT)) continue;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) park(r, o[rt][ct], ct);
    if (l < 16) {
      a.mpart[pbase * kMTX + r] = m_run[rt];
      a.lpart[pbase * kMTX + r] = l_run[rt];
    }
  }
  if (extra) {
#pragma unroll
    for (int c = 0; c < (EXTRA ? XC : 1); ++c) park(rx, ox[c], w * XC + c);
    if (w == 0 && l < 16) {
      a.mpart[pbase * kMTX + rx] = m_run[ST - 1];
      a.lpart[pbase * kMTX + rx] = l_run[ST - 1];
    }
  }
}

// The launch: no extra rows, extra rows in every tile (the only one of its rows), or in the last of several, of which
// the others then form none. With the third row tile of zeros scored in all tiles, 64 sequences of 33 rows x 8 heads took 356
// instead of 344 us at head dim 256 (512-4096 keys), 32 of 67 x 4 177 instead of 171. At 64 and 128 both forms take the
// same (78, 154-155 us), and one tile in the launch of several is 1-2 % slower (its registers): those take kAll.
enum ExtraRows { kNone = 0, kAll = 1, kLast = 2 };
template <int D, int RT, int X>
__global__ __launch_bounds__(kNW* kWave, D == 256 ? 1 : 2) void attn_partial_kernel(AttnArgs a) {
  // [buffer][K, V] tiles
  __shared__ __align__(16) uint16_t sKV[2][2][kKB * D];
  __shared__ __align__(16) uint16_t sQx[X ? kWR * D : 8];  // the extra rows' Q, as K

  const int tid = threadIdx.x;
  const int per_pair = a.S * a.QT;                  // workgroups per (sequence, KV head)
  const int npair = (int)gridDim.x / per_pair, nseq = npair / a.Hkv;
  int b, hk, s, qt;
  if (nseq > 1 && nseq <= kMaxLptSeqs && npair % kXcds == 0) {
    // ragged batches: longest sequences first. Workgroups reach the XCDs round-robin in block order,
    // so (sequence, KV head) pairs are dealt to the XCDs in descending prefix length, each pair's
    // workgroups consecutive on one XCD (its query tiles share the keys in that L2); the longest pairs
    // start in the first wave of workgroups instead of wherever their batch index put them.
    __shared__ int s_len[kMaxLptSeqs];
    __shared__ int s_seq;
    const int x = (int)blockIdx.x % kXcds, j = (int)blockIdx.x / kXcds;
    const int pr = (j / per_pair) * kXcds + x;  // pair rank
    const int wi = j % per_pair;
    qt = wi % a.QT;
    s = wi / a.QT;
    hk = pr % a.Hkv;
    const int r = pr / a.Hkv;  // sequence rank: prefix length descending, batch index ascending
    for (int c = tid; c < nseq; c += kNW * kWave) s_len[c] = a.prefix[c];
    __syncthreads();
    for (int c = tid; c < nseq; c += kNW * kWave) {
      const int lc = s_len[c];
      int rank = 0;
      for (int o = 0; o < nseq; ++o) rank += (s_len[o] > lc) | ((s_len[o] == lc) & (o < c));
      if (rank == r) s_seq = c;
    }
    __syncthreads();
    b = s_seq;
  } else {
    // query tiles of one (split, kv head) read the same keys: innermost, and on one XCD
    int idx = xcd_major(blockIdx.x, gridDim.x);
    qt = idx % a.QT;
    idx /= a.QT;
    s = idx % a.S;
    idx /= a.S;
    hk = idx % a.Hkv;
    b = idx / a.Hkv;
  }
  const int M = a.T * a.G;
  const int m0 = qt * kMT;
  // the tile's rows: kMT, or for the last tile all that remain (<= kMTX: nx extra rows past kMT)
  const int rows = qt == a.QT - 1 ? M - m0 : kMT;
  const int nx = max(rows - kMT, 0);  // block-uniform
  // a prefix past the cache capacity (a caller's overlong decode) is clamped so that every key read
  // stays inside this sequence's [Lmax, D] rows
  const int prefix = min(max(a.prefix[b], 0), a.Lmax - a.T);
  const int nk = prefix + a.T;
  const int nblk = (nk + kKB - 1) / kKB;
  const int bps = (nblk + a.S - 1) / a.S;
  const int kb0 = s * bps;
  // the last query row of the tile bounds the keys any row can see under the causal masks
  const int t_last = (m0 + rows - 1) / a.G;
  const int kmax = (a.mask_mode == 1 || (a.mask_mode == 2 && t_last >= a.n_clean)) ? nk : min(nk, prefix + t_last + 1);
  const int kb1 = min(min(nblk, kb0 + bps), (kmax + kKB - 1) / kKB);

  const int64_t pbase = ((((int64_t)b * a.Hkv + hk) * a.QT + qt) * a.S + s);
  if (kb0 >= kb1) {
    // no key of this split is visible to the tile: only the (empty) row stats are written and the
    // combine skips the split without reading its O (never with one split: its keys start at 0 and every
    // row sees at least its own)
    for (int r = tid; r < rows; r += kNW * kWave) {
      a.mpart[pbase * kMTX + r] = -INFINITY;
      a.lpart[pbase * kMTX + r] = 0.f;
    }
    return;
  }
  const Tile wt{b, hk, m0, rows, nx, prefix, nk, kb0, kb1, pbase};
  if (X == kLast && nx == 0) attn_tile<D, RT, false>(a, wt, sKV, sQx);
  else attn_tile<D, RT, X != kNone>(a, wt, sKV, sQx);
}

struct CombineArgs {
  const uint16_t* opart;  // bf16
  const float* mpart;
  const float* lpart;
  const uint16_t* gate;  // row t, head h, dim d at gate + t * gate_st + h * gate_hs + d; or null
  uint16_t* out;         // [B, T, Hq, D], or the rows [B * T, Hq * D] in the weight-streaming GEMM's
                         // fragment order (frag)
  int T, Hq, Hkv, G, D, S, QT;
  int64_t gate_st, gate_hs;
  int frag;
};

// Block = a group of RB = 512 / D rows of one (sequence, KV head); thread = (row, 4 output columns).
// The split weights exp2(m_s - max) / sum of the group's rows are computed once into LDS; each thread
// then sums the O rows of the non-empty splits in split order. Every phase issues its loads together
// (clamped, unconditional): the listing's row statistics, a row's max and sum (one pass over m and l),
// 16 splits' O rows at a time, and the gate first of all, so the combine costs a few memory round trips
// instead of one per four splits.
constexpr int kMaxSplits = 256;
constexpr int kOB = 16;  // O rows in flight per thread

constexpr int kCT = 128;  // combine threads per block (2 waves): 2 rows of d 256 per block, so a
                          // batch-1 canvas (132 rows per KV head) spreads over the CUs
template <int D>
__global__ __launch_bounds__(kCT) void attn_combine_kernel(CombineArgs a) {
  constexpr int PER_ROW = D / 4;
  constexpr int RB = kCT / PER_ROW;  // rows per block: 2 (D=256), 4 (D=128), 8 (D=64)
  constexpr int NWV = kCT / kWave;
  constexpr int LP = kMaxSplits / kCT;  // splits per thread in the listing
  __shared__ float s_w[RB][kMaxSplits];  // rows of the group x listed splits
  __shared__ float s_inv[RB];
  __shared__ int s_list[kMaxSplits];
  __shared__ int s_cnt[LP][NWV];
  const int M = a.T * a.G;
  const int b = blockIdx.y / a.Hkv, hk = blockIdx.y % a.Hkv;
  const int m0 = blockIdx.x * RB;
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
  const int64_t pair = (int64_t)b * a.Hkv + hk;
  // this thread's output element group (rows past M compute on row M - 1 and store nothing)
  const int i = tid / PER_ROW;
  const int m = m0 + i;
  const int mc = min(m, M - 1);
  const int c = (tid % PER_ROW) * 4;
  const int t = mc / a.G, g = mc % a.G, hq = hk * a.G + g;
  u32x2 gw = {0u, 0u};
  if (a.gate)
    gw = *reinterpret_cast<const u32x2*>(a.gate + ((int64_t)b * a.T + t) * a.gate_st + (int64_t)hq * a.gate_hs + c);
  // list, in split order, the splits with a visible key for some row of the group (splits tid and
  // tid + kCT of each thread, S <= 256; wave ballots give each listed split its position)
  bool any[LP];
  {
    float mv[LP][RB];
#pragma unroll
    for (int q = 0; q < LP; ++q) {
      const int sp = min(tid + q * kCT, a.S - 1);
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        const int mr = min(m0 + r, M - 1);
        const int tq = min(mr / kMT, a.QT - 1);
        mv[q][r] = a.mpart[((pair * a.QT + tq) * a.S + sp) * kMTX + (mr - tq * kMT)];
      }
    }
#pragma unroll
    for (int q = 0; q < LP; ++q) {
      any[q] = false;
#pragma unroll
      for (int r = 0; r < RB; ++r) any[q] |= m0 + r < M && mv[q][r] != -INFINITY;
      any[q] &= tid + q * kCT < a.S;
    }
  }
  unsigned long long mask[LP];
#pragma unroll
  for (int q = 0; q < LP; ++q) {
    mask[q] = __ballot(any[q]);
    if (lane == 0) s_cnt[q][wave] = __popcll(mask[q]);
  }
  __syncthreads();
  int ns = 0;
#pragma unroll
  for (int q = 0; q < LP; ++q) {
    int off = ns;
    for (int w = 0; w < wave; ++w) off += s_cnt[q][w];
    if (any[q]) s_list[off + __popcll(mask[q] & ((1ull << lane) - 1ull))] = tid + q * kCT;
    for (int w = 0; w < NWV; ++w) ns += s_cnt[q][w];
  }
  __syncthreads();
  // per row: max, weights and 1 / sum (one wave per row, lanes over the listed splits; m and l of a
  // lane's splits loaded together)
  for (int ri = wave; ri < RB; ri += NWV) {
    const int mr = min(m0 + ri, M - 1);
    const int tq = min(mr / kMT, a.QT - 1);  // the last tile holds its extra rows past kMT
    const int64_t bs = (pair * a.QT + tq) * a.S;
    const int r = mr - tq * kMT;
    constexpr int JU = kMaxSplits / kWave;  // listed splits per lane, at most
    float mj[JU], lj[JU];
#pragma unroll
    for (int u = 0; u < JU; ++u) {
      const int j = lane + u * kWave;
      if (u * kWave < ns) {  // uniform
        const int sj = s_list[min(j, ns - 1)];
        mj[u] = a.mpart[(bs + sj) * kMTX + r];
        lj[u] = a.lpart[(bs + sj) * kMTX + r];
      }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int u = 0; u < JU; ++u)
      if (u * kWave < ns && lane + u * kWave < ns) mx = fmaxf(mx, mj[u]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, kWave));
    const float m_use = mx == -INFINITY ? 0.f : mx;
    float lsum = 0.f;
#pragma unroll
    for (int u = 0; u < JU; ++u) {
      const int j = lane + u * kWave;
      if (u * kWave < ns && j < ns) {
        const float w = exp2f(mj[u] - m_use);
        s_w[ri][j] = w;
        lsum += w * lj[u];
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) lsum += __shfl_xor(lsum, o, kWave);
    if (lane == 0) s_inv[ri] = lsum > 0.f ? 1.f / lsum : 0.f;
  }
  __syncthreads();
  const int tqc = min(mc / kMT, a.QT - 1);
  const int64_t bs = (pair * a.QT + tqc) * a.S;
  const uint16_t* obase = a.opart + (int64_t)(mc - tqc * kMT) * D + c;
  const int64_t sstride = (int64_t)kMTX * D;  // elements between consecutive splits
  auto ld4 = [](const uint16_t* p) {  // 4 bf16 -> fp32
    const u32x2 w = *reinterpret_cast<const u32x2*>(p);
    return f32x4{__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u), __uint_as_float(w.y << 16),
                 __uint_as_float(w.y & 0xffff0000u)};
  };
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int j0 = 0; j0 < ns; j0 += kOB) {
    f32x4 x[kOB];
#pragma unroll
    for (int u = 0; u < kOB; ++u) x[u] = ld4(obase + (bs + s_list[min(j0 + u, ns - 1)]) * sstride);
#pragma unroll
    for (int u = 0; u < kOB; ++u)
      if (j0 + u < ns) acc += s_w[i < RB ? i : 0][j0 + u] * x[u];  // uniform bound; split order kept
  }
  if (i >= RB || m >= M) return;
  const float inv = s_inv[i];
  float y[4] = {acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv};
  if (a.gate) {
    const float gv[4] = {__uint_as_float(gw.x << 16), __uint_as_float(gw.x & 0xffff0000u), __uint_as_float(gw.y << 16),
                         __uint_as_float(gw.y & 0xffff0000u)};
#pragma unroll
    for (int u = 0; u < 4; ++u)  // the attention output is rounded to bf16 before the gate, as torch does
      y[u] = bf2f(f2bf(y[u])) * (1.f / (1.f + __expf(-gv[u])));
  }
  uint16_t* dst = a.frag ? a.out + ws_frag_off(b * a.T + t, (int64_t)hq * D + c)
                         : a.out + (((int64_t)b * a.T + t) * a.Hq + hq) * D + c;
  *reinterpret_cast<u32x2*>(dst) = u32x2{f2bf2(y[0], y[1]), f2bf2(y[2], y[3])};
}

// Two splits (batches of sequences): thread = (row, 4 output columns), 256 threads = 1024 / D rows. Every
// load of a row -- both splits' statistics and O pieces, the gate -- is issued at once, so the combine is
// one memory round trip. The arithmetic is attn_combine_kernel's: a split whose row sees no key (m = -inf)
// adds nothing (and its O, which an empty split never wrote, is not used); with two terms the order of the
// sums cannot differ, so the results are bitwise equal.
constexpr int kC2T = 256;
bool combine_general = false;  // trida_attn_set_combine_general: the general combine for two splits too
template <int D>
__global__ __launch_bounds__(kC2T) void attn_combine2_kernel(CombineArgs a) {
  constexpr int PER_ROW = D / 4;
  constexpr int RB = kC2T / PER_ROW;
  const int M = a.T * a.G;
  const int b = blockIdx.y / a.Hkv, hk = blockIdx.y % a.Hkv;
  const int tid = threadIdx.x, i = tid / PER_ROW, c = (tid % PER_ROW) * 4;
  const int m = blockIdx.x * RB + i;
  if (m >= M) return;  // no barrier in this kernel
  const int t = m / a.G, g = m % a.G, hq = hk * a.G + g;
  const int64_t pair = (int64_t)b * a.Hkv + hk;
  const int tq = min(m / kMT, a.QT - 1);  // the last tile holds its extra rows past kMT
  const int64_t bs = (pair * a.QT + tq) * 2;
  const int r = m - tq * kMT;
  u32x2 gw = {0u, 0u};
  if (a.gate)
    gw = *reinterpret_cast<const u32x2*>(a.gate + ((int64_t)b * a.T + t) * a.gate_st + (int64_t)hq * a.gate_hs + c);
  const float m0 = a.mpart[bs * kMTX + r], m1 = a.mpart[(bs + 1) * kMTX + r];
  const float l0 = a.lpart[bs * kMTX + r], l1 = a.lpart[(bs + 1) * kMTX + r];
  const uint16_t* o0 = a.opart + (bs * kMTX + r) * D + c;
  const u32x2 x0w = *reinterpret_cast<const u32x2*>(o0);
  const u32x2 x1w = *reinterpret_cast<const u32x2*>(o0 + (int64_t)kMTX * D);
  const float mx = fmaxf(m0, m1);
  const float m_use = mx == -INFINITY ? 0.f : mx;
  const bool u0 = m0 != -INFINITY, u1 = m1 != -INFINITY;
  const float w0 = u0 ? exp2f(m0 - m_use) : 0.f, w1 = u1 ? exp2f(m1 - m_use) : 0.f;
  float lsum;
  {
#pragma clang fp contract(off)
    lsum = w0 * l0 + w1 * l1;  // each product rounded, as the lanes of the general combine's sum hold them
  }
  const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
  const float x0[4] = {__uint_as_float(x0w.x << 16), __uint_as_float(x0w.x & 0xffff0000u), __uint_as_float(x0w.y << 16),
                       __uint_as_float(x0w.y & 0xffff0000u)};
  const float x1[4] = {__uint_as_float(x1w.x << 16), __uint_as_float(x1w.x & 0xffff0000u), __uint_as_float(x1w.y << 16),
                       __uint_as_float(x1w.y & 0xffff0000u)};
  float y[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float acc = 0.f;
    if (u0) acc = fmaf(w0, x0[e], acc);
    if (u1) acc = fmaf(w1, x1[e], acc);
    y[e] = acc * inv;
  }
  if (a.gate) {
    const float gv[4] = {__uint_as_float(gw.x << 16), __uint_as_float(gw.x & 0xffff0000u), __uint_as_float(gw.y << 16),
                         __uint_as_float(gw.y & 0xffff0000u)};
#pragma unroll
    for (int e = 0; e < 4; ++e)  // the attention output is rounded to bf16 before the gate, as torch does
      y[e] = bf2f(f2bf(y[e])) * (1.f / (1.f + __expf(-gv[e])));
  }
  uint16_t* dst = a.frag ? a.out + ws_frag_off(b * a.T + t, (int64_t)hq * D + c)
                         : a.out + (((int64_t)b * a.T + t) * a.Hq + hq) * D + c;
  *reinterpret_cast<u32x2*>(dst) = u32x2{f2bf2(y[0], y[1]), f2bf2(y[2], y[3])};
}

// Splits per (sequence, KV head, query tile): as many as keep the grid within one workgroup per CU
// (a workgroup holds a CU's LDS), at least one key block each. Measured at batch 1 (33 canvas rows, 16 / 4 heads,
// d 256, us by splits, 32 being the plan): 8192 keys 8: 54.6, 16: 36.9, 28: 29.4, 32: 29.9; 2048 keys 8: 26.5, 21: 21.7,
// 32: 22.5; a grid just past the CU count (36 splits) runs a ragged second round, 44.4 at 8192 keys.
// When the query tiles alone fill the CUs (a batch of sequences), two splits per tile, so that the
// longest sequences of a ragged batch are not one workgroup's serial walk over their keys (64 sequences
// of 512-4096 keys, 33 rows x 4 heads, one query tile each: 1 split 245 us, 2: 189, 3: 212, 4: 226; 128 of them are even,
// 329 and 364). Between half of the CUs and all of them the first rule leaves one split, which is not the
// best there: 48 such sequences 232 us, with two splits 157; 24 of two tiles each 163, with two 102.
constexpr int64_t kCUs = 256;
int64_t plan_splits(int64_t B, int64_t Hkv, int64_t QT, int64_t max_keys, int64_t splits) {
  if (splits > 0) return splits;
  const int64_t nblk = cdiv(max_keys, kKB);
  if (B * Hkv * QT >= kCUs) return std::max<int64_t>(1, std::min<int64_t>(2, nblk));
  int64_t s = kCUs / (B * Hkv * QT);
  if (s > nblk) s = nblk;
  if (s > kMaxSplits) s = kMaxSplits;
  return s < 1 ? 1 : s;
}

// Query tiles of M rows per (sequence, KV head): kMT rows each. A last one of <= 16 rows joins the tile
// before it as its extra rows when its own workgroups would not fit beside the others on the CUs (a batch
// of sequences; 64 x 33 rows x 4 heads, 512-4096 keys: 237 us apart, 188 joined). Where they fit (batch 1) they run
// on otherwise idle CUs and the extra rows' work would only lengthen the full tile's (8192 keys 29.9 us apart, 32.0 joined;
// 2048 keys 22.5 and 24.8; 2 sequences 26.7 and 30.5). The two meet before the CUs are full: 8 sequences 49.2 and 45.8,
// 16 89 and 77, and 32 130 and 120 with three splits (135 with the planned two).
int64_t query_tiles(int64_t B, int64_t Hkv, int64_t M) {
  const int64_t qt = cdiv(M, kMT);
  return qt > 1 && M - (qt - 1) * kMT <= kWR && B * Hkv * qt > kCUs ? qt - 1 : qt;
}

}  // namespace
}  // namespace trida

using namespace trida;

extern "C" int64_t trida_attn_canvas_scratch_bytes(int64_t B, int64_t T, int64_t Hq, int64_t Hkv, int64_t D,
                                                   int64_t max_keys, int64_t splits) {
  if (B <= 0 || T <= 0 || Hkv <= 0 || Hq % Hkv || D <= 0) return 0;
  const int64_t QT = query_tiles(B, Hkv, T * (Hq / Hkv));
  const int64_t S = plan_splits(B, Hkv, QT, max_keys, splits);
  const int64_t slots = B * Hkv * QT * S;
  return align_up(slots * kMTX * D * 2, 256) + 2 * align_up(slots * kMTX * 4, 256);
}

namespace {
int attn_canvas_run(const uint16_t* q, const uint16_t* k_cache, const uint16_t* v_cache, const int32_t* prefix_len,
                    const uint16_t* gate, int64_t gate_row_stride, int64_t gate_head_stride, uint16_t* out, bool frag,
                    int64_t B, int64_t T, int64_t Hq, int64_t Hkv, int64_t D, int64_t Lmax, int mask_mode,
                    int64_t n_clean, float scale, int64_t max_keys, int64_t splits, void* scratch,
                    int64_t scratch_bytes, void* stream) {
  TRIDA_CHECK(q && k_cache && v_cache && prefix_len && out && scratch, TRIDA_ERR_NULL,
              "attn_canvas: q, k_cache, v_cache, prefix_len, out and scratch are required");
  TRIDA_CHECK(B > 0 && T > 0 && Hq > 0 && Hkv > 0 && Hq % Hkv == 0 && Lmax >= T, TRIDA_ERR_ARG,
              "attn_canvas: bad sizes B=%lld T=%lld Hq=%lld Hkv=%lld Lmax=%lld", (long long)B, (long long)T,
              (long long)Hq, (long long)Hkv, (long long)Lmax);
  TRIDA_CHECK(D == 64 || D == 128 || D == 256, TRIDA_ERR_ARG, "attn_canvas: head dim must be 64, 128 or 256");
  TRIDA_CHECK(mask_mode >= 0 && mask_mode <= 2, TRIDA_ERR_ARG, "attn_canvas: mask_mode is 0, 1 or 2");
  TRIDA_CHECK(((((uintptr_t)q) | (uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)out) & 15) == 0,
              TRIDA_ERR_ALIGN, "attn_canvas: q, caches and out must be 16-byte aligned");
  TRIDA_CHECK(gate == nullptr || (gate_head_stride >= D && gate_row_stride >= Hq * gate_head_stride - (gate_head_stride - D)),
              TRIDA_ERR_ARG, "attn_canvas: gate strides");
  const int64_t G = Hq / Hkv;
  const int64_t QT = query_tiles(B, Hkv, T * G);
  const int64_t S = plan_splits(B, Hkv, QT, max_keys > 0 ? max_keys : Lmax, splits);
  TRIDA_CHECK(S >= 1 && S <= kMaxSplits, TRIDA_ERR_ARG, "attn_canvas: 1..%d key splits", kMaxSplits);
  const int64_t need = trida_attn_canvas_scratch_bytes(B, T, Hq, Hkv, D, max_keys > 0 ? max_keys : Lmax, S);
  TRIDA_CHECK(scratch_bytes >= need, TRIDA_ERR_WORKSPACE, "attn_canvas: scratch %lld < %lld bytes",
              (long long)scratch_bytes, (long long)need);
  const int64_t slots = B * Hkv * QT * S;
  TRIDA_CHECK(slots < INT32_MAX && B * Hkv < 65535, TRIDA_ERR_ARG, "attn_canvas: grid too large");
  char* ws = static_cast<char*>(scratch);
  uint16_t* opart = reinterpret_cast<uint16_t*>(ws);
  float* mpart = reinterpret_cast<float*>(ws + align_up(slots * kMTX * D * 2, 256));
  float* lpart = reinterpret_cast<float*>(ws + align_up(slots * kMTX * D * 2, 256) + align_up(slots * kMTX * 4, 256));
  hipStream_t st = static_cast<hipStream_t>(stream);
  TRIDA_CHECK(!frag || B * T <= 48, TRIDA_ERR_ARG, "attn_canvas_frag: the fragment order holds at most 48 rows");
  AttnArgs a{q,           k_cache,         v_cache,          prefix_len, opart, mpart, lpart, (int)T, (int)Hq, (int)Hkv,
             (int)G,      (int)Lmax,       (int)S,           (int)QT,    mask_mode, (int)n_clean, scale * kLog2e, gate,
             gate_row_stride, gate_head_stride, out,         frag ? 1 : 0};
  const dim3 grid((unsigned)slots);
  // one row tile per wave where that covers the query rows
  const bool one = T * G <= kNW * kWR;
  const bool extra = T * G > QT * kMT;
#define TRIDA_ATTN_PARTIAL(DD)                                                                                   \
  if (one) hipLaunchKernelGGL((attn_partial_kernel<DD, 1, kNone>), grid, dim3(kNW * kWave), 0, st, a);           \
  else if (extra && QT > 1)                                                                                      \
    hipLaunchKernelGGL((attn_partial_kernel<DD, 2, DD == 256 ? kLast : kAll>), grid, dim3(kNW * kWave), 0, st, a); \
  else if (extra) hipLaunchKernelGGL((attn_partial_kernel<DD, 2, kAll>), grid, dim3(kNW * kWave), 0, st, a);     \
  else hipLaunchKernelGGL((attn_partial_kernel<DD, 2, kNone>), grid, dim3(kNW * kWave), 0, st, a);
  switch (D) {
    case 64: TRIDA_ATTN_PARTIAL(64) break;
    case 128: TRIDA_ATTN_PARTIAL(128) break;
    default: TRIDA_ATTN_PARTIAL(256) break;
  }
#undef TRIDA_ATTN_PARTIAL
  int rc = launch_status("attn_canvas/partial");
  if (rc || S == 1) return rc;  // one split: the partial kernel wrote the output
  CombineArgs c{opart, mpart, lpart, gate, out, (int)T, (int)Hq, (int)Hkv, (int)G, (int)D, (int)S, (int)QT,
                gate_row_stride, gate_head_stride, frag ? 1 : 0};
  if (S == 2 && !combine_general) {
    const dim3 cgrid((unsigned)cdiv(T * G, kC2T / (D / 4)), (unsigned)(B * Hkv));
    switch (D) {
      case 64: hipLaunchKernelGGL(attn_combine2_kernel<64>, cgrid, dim3(kC2T), 0, st, c); break;
      case 128: hipLaunchKernelGGL(attn_combine2_kernel<128>, cgrid, dim3(kC2T), 0, st, c); break;
      default: hipLaunchKernelGGL(attn_combine2_kernel<256>, cgrid, dim3(kC2T), 0, st, c); break;
    }
    return launch_status("attn_canvas/combine2");
  }
  const int64_t rows_per_block = kCT / (D / 4);
  const dim3 cgrid((unsigned)cdiv(T * G, rows_per_block), (unsigned)(B * Hkv));
  switch (D) {
    case 64: hipLaunchKernelGGL(attn_combine_kernel<64>, cgrid, dim3(kCT), 0, st, c); break;
    case 128: hipLaunchKernelGGL(attn_combine_kernel<128>, cgrid, dim3(kCT), 0, st, c); break;
    default: hipLaunchKernelGGL(attn_combine_kernel<256>, cgrid, dim3(kCT), 0, st, c); break;
  }
  return launch_status("attn_canvas/combine");
}
}  // namespace

extern "C" int trida_attn_set_combine_general(int on) {
  combine_general = on != 0;
  return TRIDA_OK;
}

extern "C" int trida_attn_canvas(const uint16_t* q, const uint16_t* k_cache, const uint16_t* v_cache,
                                 const int32_t* prefix_len, const uint16_t* gate, int64_t gate_row_stride,
                                 int64_t gate_head_stride, uint16_t* out, int64_t B, int64_t T, int64_t Hq, int64_t Hkv, int64_t D,
                                 int64_t Lmax, int mask_mode, int64_t n_clean, float scale, int64_t max_keys,
                                 int64_t splits, void* scratch, int64_t scratch_bytes, void* stream) {
  return attn_canvas_run(q, k_cache, v_cache, prefix_len, gate, gate_row_stride, gate_head_stride, out, false, B, T, Hq,
                         Hkv, D, Lmax, mask_mode, n_clean, scale, max_keys, splits, scratch, scratch_bytes, stream);
}

extern "C" int trida_attn_canvas_frag(const uint16_t* q, const uint16_t* k_cache, const uint16_t* v_cache,
                                      const int32_t* prefix_len, const uint16_t* gate, int64_t gate_row_stride,
                                      int64_t gate_head_stride, uint16_t* out_frag, int64_t B, int64_t T, int64_t Hq,
                                      int64_t Hkv, int64_t D, int64_t Lmax, int mask_mode, int64_t n_clean, float scale,
                                      int64_t max_keys, int64_t splits, void* scratch, int64_t scratch_bytes,
                                      void* stream) {
  return attn_canvas_run(q, k_cache, v_cache, prefix_len, gate, gate_row_stride, gate_head_stride, out_frag, true, B,
                         T, Hq, Hkv, D, Lmax, mask_mode, n_clean, scale, max_keys, splits, scratch, scratch_bytes,
                         stream);
}
