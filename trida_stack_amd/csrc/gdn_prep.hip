// GDN layer front half, fused: depthwise causal conv (width Kc) over [window ++ x] + SiLU, split
// into q / k / v, l2norm of q and k per head, and the gates g = -exp(A_log) softplus(a + dt_bias),
// beta = sigmoid(b).
//
// Launch: a thread owns 8 consecutive channels (one 16-byte piece); the Dk/8 threads of a q or k head reduce
// its sum of squares with a row-local reduction. Small grids take a grid of (sequence, row) x channel slices of 128
// pieces (the C = conv_dim channels of a row spread over several CUs). From 512 rows on, a block takes up to 16
// consecutive rows of a sequence: its thread keeps the conv weights and the last Kc - 1 source rows in registers,
// so a row is loaded once (and its chunk's Kc - 1 predecessors) instead of by each of the Kc rows that
// read it, and the weights (48 KB at C = 6144, as much as the row's four source rows) once per chunk.
// Rounding follows the CPU oracle: conv and SiLU in fp32, rounded to bf16, then l2norm in fp32 of the
// rounded values, rounded to bf16 again.
#include <algorithm>

#include "common.h"

namespace trida {
namespace {

constexpr int kMaxKc = 4;
constexpr int kNT = 128;  // threads, i.e. pieces, per block

template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
  // update_dpp with a defined old value and bound_ctrl: folds into the consuming add / max
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, true));
}
// Sum over aligned groups of W lanes (W = 4, 8 or 16); every lane receives its group's total.
template <int W>
__device__ __forceinline__ float lane_group_sum(float v) {
  if (W == 16) {
    v += dpp<0x128>(v);
    v += dpp<0x124>(v);
  } else if (W == 8) {
    v += __shfl_xor(v, 4, kWave);
  }
  v += dpp<0x4E>(v);
  v += dpp<0xB1>(v);
  return v;
}

struct PrepArgs {
  const uint16_t* x;  // [B, T, C] (batch stride x_sb, row stride x_st)
  const uint16_t* window;  // [B, Kc-1, C]
  const uint16_t* conv_w;  // [C, Kc]
  const uint16_t* a_in;    // [B, T, Hv] (batch stride ab_sb, row stride ab_st)
  const uint16_t* b_in;
  const float* A_log;  // [Hv]
  const float* dt_bias;
  uint16_t* q;  // [B, T, Hk, Dk]
  uint16_t* k;
  uint16_t* v;  // [B, T, Hv, Dv]
  float* g;     // [B, T, Hv]
  float* beta;
  uint16_t* window_out;  // [B, Kc-1, C] or null
  uint16_t* pre_out;     // [B, T, C] copy of the pre-conv rows x, or null
  const uint16_t* conv_bias;   // [C] or null
  const int32_t* win_idx;      // [B] window / window_out row of sequence b, or null (row b)
  const int32_t* pre_idx;      // [B] pre_out slot of sequence b, or null (slot b)
  const int32_t* cu_seqlens;   // [B + 1] packed ragged rows, or null (B x T rows)
  int T, C, Kc, Hk, Hv, Dk, Dv;
  int64_t x_sb, x_st, ab_sb, ab_st;
  int rows, chunks;  // rows per block and blocks per sequence (of T rows)
};

// Rows of sequence b: [row0, row0 + n) of the packed arrays. Contiguous form: n = T, row0 = b T (x and
// a / b rows then also move by their batch strides). Packed form: rows cu[b] .. cu[b + 1] - 1, at most T.
struct SeqRows {
  int64_t row0;
  int n;
};
__device__ __forceinline__ SeqRows seq_rows(const int32_t* cu_seqlens, int T, int b) {
  if (!cu_seqlens) return {(int64_t)b * T, T};
  const int lo = cu_seqlens[b];
  return {lo, max(0, min(cu_seqlens[b + 1] - lo, T))};
}

__device__ __forceinline__ void unpack8(const u32x4 w, float* f) {
  f[0] = bf2f((uint16_t)(w.x & 0xffff));
  f[1] = bf2f((uint16_t)(w.x >> 16));
  f[2] = bf2f((uint16_t)(w.y & 0xffff));
  f[3] = bf2f((uint16_t)(w.y >> 16));
  f[4] = bf2f((uint16_t)(w.z & 0xffff));
  f[5] = bf2f((uint16_t)(w.z >> 16));
  f[6] = bf2f((uint16_t)(w.w & 0xffff));
  f[7] = bf2f((uint16_t)(w.w >> 16));
}
__device__ __forceinline__ u32x4 pack8(const float* f) {
  u32x4 w;
  w.x = f2bf2(f[0], f[1]);
  w.y = f2bf2(f[2], f[3]);
  w.z = f2bf2(f[4], f[5]);
  w.w = f2bf2(f[6], f[7]);
  return w;
}

__device__ __forceinline__ float silu(float x) { return x / (1.f + __expf(-x)); }
// torch.nn.functional.softplus with beta 1 and threshold 20
__device__ __forceinline__ float softplus(float x) { return x > 20.f ? x : log1pf(__expf(x)); }

// IDX: the pool / packed forms (slot indices, cu_seqlens) may be in use; without it those pointers are ignored
// (null) and the plain form compiles without their loads and branches.
// MULTI: blocks of `a.rows` rows, four at a time: the next four rows' loads go out before the current ones are
// convolved. Otherwise one row per block.
// 4096 rows of 6144 channels: 48 -> 36 us; 8 x 1024 rows of 8192 137 -> 74; 64 x 33 rows with pre_out 31 -> 23.
template <int GW, int KC, bool MULTI, bool IDX>  // lanes per q/k head = Dk / 8; conv width
__global__ __launch_bounds__(kNT) void gdn_prep_kernel(PrepArgs a) {
  constexpr int G = MULTI ? 4 : 1;  // rows per step
  const int32_t* cu_seqlens = IDX ? a.cu_seqlens : nullptr;
  const int32_t* win_idx = IDX ? a.win_idx : nullptr;
  const int32_t* pre_idx = IDX ? a.pre_idx : nullptr;
  const int t0 = (int)(blockIdx.x % a.chunks) * (MULTI ? a.rows : 1);
  const int b = blockIdx.x / a.chunks;
  const SeqRows sr = seq_rows(cu_seqlens, a.T, b);
  if (t0 >= sr.n) return;  // past a packed sequence's rows (block-uniform)
  const int T = sr.n;
  const int t1 = MULTI ? min(T, t0 + a.rows) : t0 + 1;  // the block's rows [t0, t1)
  const int tid = threadIdx.x;
  const int key_dim = a.Hk * a.Dk;
  const int pieces = a.C / 8;
  const int p0 = blockIdx.y * kNT, p = p0 + tid;  // the block's first piece: a multiple of GW
  const bool live = p < pieces;                   // lanes past the last piece load it and store nothing
  const int c = min(p, pieces - 1) * 8;
  // the sequence's source rows (packed: row r of x at r x_st) and its window row
  const uint16_t* xb = cu_seqlens ? a.x + sr.row0 * a.x_st : a.x + (int64_t)b * a.x_sb;
  const int64_t ab0 = cu_seqlens ? sr.row0 * a.ab_st : (int64_t)b * a.ab_sb;
  const int wrow = win_idx ? win_idx[b] : b;
  const int prow_b = pre_idx ? pre_idx[b] : b;  // pre_out slot
  const uint16_t* wb = a.window + (int64_t)wrow * (a.Kc - 1) * a.C;
  auto src = [&](int tau) {  // source row tau; negative rows come from the window
    return *reinterpret_cast<const u32x4*>(tau >= 0 ? xb + (int64_t)tau * a.x_st + c : wb + (int64_t)(KC - 1 + tau) * a.C + c);
  };

  // every load of the first step first (one memory round trip): the gate inputs, the source rows of the thread's 8
  // channels, their conv weights (8 channels x KC taps, contiguous: KC 16-byte pieces) and bias. The loads
  // are unconditional (the gate inputs of blocks that do not write the gates, the bias from the conv
  // weights when there is none: in bounds, unused), so that no branch splits the round trip.
  const bool gates = blockIdx.y == 0;  // block-uniform
  const int hg = min(tid, a.Hv - 1);
  const uint16_t ar = a.a_in[ab0 + (int64_t)t0 * a.ab_st + hg];
  const uint16_t br = a.b_in[ab0 + (int64_t)t0 * a.ab_st + hg];
  const float alog = a.A_log[hg], dtb = a.dt_bias[hg];
  const uint16_t* cbias = a.conv_bias ? a.conv_bias : a.conv_w;
  u32x4 xs[KC - 1 + G], wsv[KC];
#pragma unroll
  for (int j = 0; j < KC - 1 + G; ++j) xs[j] = src(min(t0 - (KC - 1) + j, t1 - 1));
#pragma unroll
  for (int j = 0; j < KC; ++j) wsv[j] = reinterpret_cast<const u32x4*>(a.conv_w + (int64_t)c * KC)[j];
  const u32x4 bsv = *reinterpret_cast<const u32x4*>(cbias + c);
  float w[8][KC], bias[8];
#pragma unroll
  for (int ch = 0; ch < 8; ++ch)
#pragma unroll
    for (int j = 0; j < KC; ++j) {
      const int e = ch * KC + j;  // element of the 8 x KC weight block
      const uint32_t word = wsv[e / 8][(e % 8) / 2];
      w[ch][j] = __uint_as_float((e & 1) ? (word & 0xffff0000u) : (word << 16));
    }
  unpack8(bsv, bias);
#pragma unroll
  for (int ch = 0; ch < 8; ++ch) bias[ch] = a.conv_bias ? bias[ch] : 0.f;

  for (int t = t0; t < t1; t += G) {
    u32x4 xn[G];
    if (MULTI && t + G < t1) {
#pragma unroll
      for (int i = 0; i < G; ++i) xn[i] = src(min(t + G + i, t1 - 1));
    }
#pragma unroll
    for (int i = 0; i < G; ++i) {
      if (i > 0 && t + i >= t1) break;  // block-uniform
      // the pre-conv rows a rollback rebuilds the window from: the row itself is its last source row
      if (a.pre_out && live)
        *reinterpret_cast<u32x4*>(a.pre_out + ((int64_t)prow_b * a.T + t + i) * a.C + c) = xs[i + KC - 1];
      float acc[8];
#pragma unroll
      for (int ch = 0; ch < 8; ++ch) acc[ch] = bias[ch];
#pragma unroll
      for (int j = 0; j < KC; ++j) {
        float f[8];
        unpack8(xs[i + j], f);
#pragma unroll
        for (int ch = 0; ch < 8; ++ch) acc[ch] = fmaf(w[ch][j], f[ch], acc[ch]);
      }
#pragma unroll
      for (int ch = 0; ch < 8; ++ch) acc[ch] = bf2f(f2bf(silu(acc[ch])));
      // the q/k pieces come first (2 * key_dim / 8 of them, a multiple of GW) and are all live, so every
      // group of GW lanes belongs to one head
      if (p0 < 2 * key_dim / 8) {  // block-uniform: per-head l2norm (all lanes take part in the reduction)
        const bool is_qk = c < 2 * key_dim;  // uniform across a GW-lane group
        float ss = 0.f;
#pragma unroll
        for (int ch = 0; ch < 8; ++ch) ss = fmaf(acc[ch], acc[ch], ss);
        ss = lane_group_sum<GW>(ss);
        if (is_qk) {
          const float inv = rsqrtf(ss + 1e-6f);
#pragma unroll
          for (int ch = 0; ch < 8; ++ch) acc[ch] *= inv;
        }
      }
      if (live) {
        const u32x4 o = pack8(acc);
        const int64_t row = sr.row0 + t + i;  // output row (q, k, v, g, beta)
        if (c < key_dim)
          *reinterpret_cast<u32x4*>(a.q + row * key_dim + c) = o;
        else if (c < 2 * key_dim)
          *reinterpret_cast<u32x4*>(a.k + row * key_dim + (c - key_dim)) = o;
        else
          *reinterpret_cast<u32x4*>(a.v + row * (int64_t)a.Hv * a.Dv + (c - 2 * key_dim)) = o;
      }
    }
    if (MULTI) {
#pragma unroll
      for (int j = 0; j < KC - 1; ++j) xs[j] = xs[j + G];
#pragma unroll
      for (int i = 0; i < G; ++i) xs[KC - 1 + i] = xn[i];
    }
  }
  // the new conv window (last Kc-1 rows of [window ++ x]): the last row's blocks, each its own pieces
  if (a.window_out && t1 == T && live) {
    for (int wr = 0; wr < a.Kc - 1; ++wr)
      *reinterpret_cast<u32x4*>(a.window_out + ((int64_t)wrow * (a.Kc - 1) + wr) * a.C + c) = src(T - (a.Kc - 1) + wr);
  }
  if (gates) {
    for (int i = tid; i < (t1 - t0) * a.Hv; i += kNT) {
      const int t = t0 + i / a.Hv, hh = i % a.Hv;
      float av = bf2f(ar), bv = bf2f(br), al = alog, dt = dtb;
      if (i != tid || i != hg) {  // past the first row's heads: the inputs are loaded here
        const int64_t at = ab0 + (int64_t)t * a.ab_st + hh;
        av = bf2f(a.a_in[at]);
        bv = bf2f(a.b_in[at]);
        al = a.A_log[hh];
        dt = a.dt_bias[hh];
      }
      const int64_t o = (sr.row0 + t) * a.Hv + hh;
      a.g[o] = -__expf(al) * softplus(av + dt);
      a.beta[o] = 1.f / (1.f + __expf(-bv));
    }
  }
}

}  // namespace
}  // namespace trida

using namespace trida;

extern "C" int trida_gdn_prep(const uint16_t* x, const uint16_t* window, const uint16_t* conv_w,
                              const uint16_t* a_in, const uint16_t* b_in, const float* A_log,
                              const float* dt_bias, uint16_t* q, uint16_t* k, uint16_t* v, float* g,
                              float* beta, uint16_t* window_out, uint16_t* pre_out, int64_t B, int64_t T, int64_t Kc,
                              int64_t Hk, int64_t Hv, int64_t Dk, int64_t Dv, int64_t x_sb, int64_t x_st,
                              int64_t ab_sb, int64_t ab_st, const uint16_t* conv_bias, const int32_t* win_idx,
                              const int32_t* pre_idx, const int32_t* cu_seqlens, void* stream) {
  TRIDA_CHECK(x && window && conv_w && a_in && b_in && A_log && dt_bias && q && k && v && g && beta,
              TRIDA_ERR_NULL, "gdn_prep: a required pointer is NULL");
  TRIDA_CHECK(B > 0 && T > 0 && Hk > 0 && Hv > 0 && Hv % Hk == 0 && Kc >= 2 && Kc <= kMaxKc, TRIDA_ERR_ARG,
              "gdn_prep: bad sizes B=%lld T=%lld Hk=%lld Hv=%lld Kc=%lld", (long long)B, (long long)T,
              (long long)Hk, (long long)Hv, (long long)Kc);
  TRIDA_CHECK(Dk == 32 || Dk == 64 || Dk == 128, TRIDA_ERR_ARG, "gdn_prep: Dk must be 32, 64 or 128");
  TRIDA_CHECK(Dv % 8 == 0, TRIDA_ERR_ARG, "gdn_prep: Dv %% 8 == 0 required");
  const int64_t C = 2 * Hk * Dk + Hv * Dv;
  TRIDA_CHECK(x_st % 8 == 0 && x_sb % 8 == 0 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)window & 15) == 0,
              TRIDA_ERR_ALIGN, "gdn_prep: x / window must be 16-byte aligned with strides in multiples of 8");
  TRIDA_CHECK(x_st >= C, TRIDA_ERR_ARG, "gdn_prep: row stride of x smaller than conv_dim");
  TRIDA_CHECK(((uintptr_t)conv_w & 15) == 0, TRIDA_ERR_ALIGN, "gdn_prep: conv_w must be 16-byte aligned");
  TRIDA_CHECK(window_out == nullptr || window_out != window, TRIDA_ERR_ARG,
              "gdn_prep: window_out must not alias window");
  TRIDA_CHECK(pre_out == nullptr || (((uintptr_t)pre_out & 15) == 0 && pre_out != x), TRIDA_ERR_ARG,
              "gdn_prep: pre_out must be 16-byte aligned and not alias x");
  TRIDA_CHECK(conv_bias == nullptr || ((uintptr_t)conv_bias & 15) == 0, TRIDA_ERR_ALIGN,
              "gdn_prep: conv_bias must be 16-byte aligned");
  TRIDA_CHECK(B * T < INT32_MAX, TRIDA_ERR_ARG, "gdn_prep: too many rows");
  PrepArgs a{x, window, conv_w, a_in, b_in, A_log, dt_bias, q, k, v, g, beta, window_out, pre_out,
             conv_bias, win_idx, pre_idx, cu_seqlens,
             (int)T, (int)C, (int)Kc, (int)Hk, (int)Hv, (int)Dk, (int)Dv, x_sb, x_st, ab_sb, ab_st, 1, (int)T};
  hipStream_t st = static_cast<hipStream_t>(stream);
  // From 512 rows on a block takes several rows: as many as leave about 1536 blocks (12 waves per CU in flight), 4 to
  // 16, in chunks of equal length: 9.6 -> 7.6 us at 512 rows (4 per block), 12.2 -> 8.3 at 16 x 33 with pre_out. 300
  // rows take 5.3 us one per block, their launch and one memory round trip.
  const bool multi = B * T >= 512;
  // part of the entry point's contract, not of this launch: wider rows are refused here as they always were
  constexpr int kMaxWideC = 8192;
  TRIDA_CHECK(!multi || C <= kMaxWideC, TRIDA_ERR_ARG, "gdn_prep: conv_dim %lld above %d", (long long)C, kMaxWideC);
  const int64_t slices = cdiv(C / 8, kNT);
  const int64_t most = multi ? std::max<int64_t>(4, std::min<int64_t>(16, B * T * slices / 1536)) : 1;
  a.chunks = (int)cdiv(T, most);
  a.rows = (int)cdiv(T, a.chunks);
  TRIDA_CHECK(B * a.chunks < INT32_MAX, TRIDA_ERR_ARG, "gdn_prep: too many rows");
  const dim3 grid((unsigned)(B * a.chunks), (unsigned)slices);
  const bool idx = cu_seqlens || win_idx || pre_idx;
#define TRIDA_PREP_KC(GW, MU, IX)                                                                        \
  switch (Kc) {                                                                                          \
    case 2: hipLaunchKernelGGL((gdn_prep_kernel<GW, 2, MU, IX>), grid, dim3(kNT), 0, st, a); break;      \
    case 3: hipLaunchKernelGGL((gdn_prep_kernel<GW, 3, MU, IX>), grid, dim3(kNT), 0, st, a); break;      \
    default: hipLaunchKernelGGL((gdn_prep_kernel<GW, 4, MU, IX>), grid, dim3(kNT), 0, st, a); break;     \
  }
#define TRIDA_PREP_LAUNCH(GW)                        \
  if (multi && idx) { TRIDA_PREP_KC(GW, true, true) }     \
  else if (multi) { TRIDA_PREP_KC(GW, true, false) }      \
  else if (idx) { TRIDA_PREP_KC(GW, false, true) }        \
  else { TRIDA_PREP_KC(GW, false, false) }
  switch (Dk) {
    case 32: TRIDA_PREP_LAUNCH(4) break;
    case 64: TRIDA_PREP_LAUNCH(8) break;
    default: TRIDA_PREP_LAUNCH(16) break;
  }
#undef TRIDA_PREP_LAUNCH
#undef TRIDA_PREP_KC
  return launch_status("gdn_prep");
}
