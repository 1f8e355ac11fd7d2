// Weight-streaming bf16 GEMM for mid-size row counts: Y[M, N] = X[M, K] W[N, K]^T with 49 <= M <= 512 (the canvases of
// a small batch, a prefill chunk), fp32 accumulation, over the pre-shuffled weights of gemm.hip (tile t of 16
// rows, k-step s of 32 columns: 1 KB, lane 16 g + r holding W[16 t + r][32 s + 8 g .. + 8]) and with its epilogues
// (bf16 store, fp32 partial planes, SwiGLU; the first and last optionally scaled per row by the RMSNorm).
//
// A workgroup of 8 waves takes T column tiles and all rows, so that the weights are read once:
//   - the weights stream through LDS in stages of 8 k-steps, three buffers, loaded straight to LDS two stages
//     ahead (8 T KB each: what is in flight covers the memory latency); every wave reads each fragment once;
//   - the row tiles are dealt to the waves, tile w, w + 8, ...: up to 4 per wave. A wave loads their X fragments
//     from L2 into a register ring, D k-steps ahead, and no wave loads another's. X is in fragment order (mid_off:
//     every load 1 KB of consecutive bytes). Row-major, the 16 rows x 64 B of a load lie a row apart and meet in a few L2
//     channels, all workgroups at about the same columns: 264 x 19456 x 2560 took 64 instead of 43 us, 264 x 2560 x 4096
//     26 instead of 15. The producers write that order (trida_residual_mid, this kernel's SwiGLU epilogue);
//   - fragment by fragment the products are v_mfma_f32_16x16x32_bf16 with W as the A operand, as in gemm.hip.
// K may be split over kg groups of workgroups that write partial planes (summed in plane order by the consumer).
// Bound at 64 rows by the weights' stream (4.2 TB/s), from 264 rows on by the workgroup's own k-steps. Gate / up with X
// read from one k-step only, W from one 4 KB only, both: 64 rows 23.9 -> 23.5, 14.3, 13.8 us; 264 rows 42.7 -> 38.9,
// 31.6, 30.1; 512 rows 59.1 -> 55.7, 49.8, 47.5. What is left at 264 rows is 0.34 us a k-step: 0.2 of matrix instructions
// on the busiest SIMD, the rest LDS reads of the fragments (each wave reads all of the stage) that they do not cover;
// the memory latency of W adds a third. Every workgroup reads all of X from L2 (in all, with W, 10-12 TB/s). Measured beside the library's GEMM (gate / up with its SwiGLU pass;
// MI355X, cold weights): gate / up 19456 x 2560 30 -> 25 us at 64 rows, 42 -> 32 at 132, 51 -> 43 at 264, 64 -> 59 at
// 512; down 2560 x 9728 25 -> 14, 27 -> 20, 34 -> 25, 50 -> 35. Whole-K bf16 outputs of narrower weights are
// no faster (8224 x 2560: 15 -> 13, 19 -> 17, 22 -> 23, 32 -> 35), so those projections stay with the library.
#include <algorithm>

#include "common.h"

namespace trida {
namespace {

constexpr int kNW = 8;        // waves per workgroup
constexpr int kStage = 8;     // k-steps per stage
constexpr int kBufs = 3;
constexpr int kMaxT = 5;      // column tiles per workgroup: 3 x 8 x 5 KB of LDS
constexpr int kMaxMTW = 4;    // row tiles per wave
constexpr int kMinM = 49, kMaxM = kMaxMTW * kNW * 16;
constexpr int kCUs = 256;
enum Epilogue { kStore = 0, kParts = 1, kSilu = 2 };

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ bf16x8 as_bf(u32x4 w) { return __builtin_bit_cast(bf16x8, w); }
__device__ __forceinline__ float silu(float x) { return x / (1.f + __expf(-x)); }
__host__ __device__ constexpr int ss_chunks(int dim) { return (dim + 255) / 256; }

struct MidArgs {
  const uint16_t* X;  // fragment order
  const u32x4* Wp;
  void* out;  // bf16 rows (o_st; fragment order: of), or fp32 planes [kg][M][N]
  int64_t o_st;
  int M, N, K, epi, of;
  const float* ss;  // [M][ss_chunks(K)] sums of squares of X's 256-column chunks, or null: no RMSNorm
  float eps;
};

// Element offset of X[m][k] in the fragment order of mt row tiles: per k-step of 32 columns and row tile, 64 lanes x 16
// bytes, lane 16 g + r holding X[16 tile + r][32 step + 8 g .. + 8] (ws_frag_off with mt tiles per k-step).
__device__ __forceinline__ int64_t mid_off(int m, int k, int mt) {
  return (((int64_t)(k / 32) * mt + m / 16) * 64 + ((k % 32) / 8) * 16 + m % 16) * 8 + k % 8;
}

// 64 lanes x 16 bytes to LDS at `lds` (bytes, wave-uniform) + 16 lane, asynchronously: counted by vmcnt, no register
// written. In asm because the compiler would wait for it before every later LDS read; nothing else in these
// kernels uses m0.
__device__ __forceinline__ void load_lds16(const u32x4* src, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(src) : "memory", "m0");
}

// All of a wave's work with MY row tiles (0: it only loads weights).
template <int T, int MY, int D>
__device__ __forceinline__ void run(const MidArgs& a, u32x4 (*sW)[kStage][T][kWave], int w, int l) {
  const int tiles = a.N / 16, nsteps = a.K / 32;
  const int t0 = blockIdx.x * T, nt = min(T, tiles - t0);
  const int s0 = (int)((int64_t)nsteps * blockIdx.y / gridDim.y), s1 = (int)((int64_t)nsteps * (blockIdx.y + 1) / gridDim.y);
  const int n = s1 - s0, nst = (n + kStage - 1) / kStage;

  // the wave's T pieces of stage st: piece c = w + 8 i is k-step c / T of tile c % T (clamped: pieces past the end
  // of K or N are loaded again and not used)
  auto load_stage = [&](int st) {
    const uint32_t lds = (uint32_t)(uintptr_t)&sW[st % kBufs][0][0][0];
#pragma unroll
    for (int i = 0; i < T; ++i) {
      const int c = w + kNW * i, s = min(s0 + st * kStage + c / T, s1 - 1), t = t0 + min(c % T, nt - 1);
      load_lds16(a.Wp + ((int64_t)t * nsteps + s) * kWave + l, __builtin_amdgcn_readfirstlane(lds + (uint32_t)c * 1024u));
    }
  };
  load_stage(0);
  if (nst > 1) load_stage(1);

  constexpr int M1 = MY > 0 ? MY : 1;
  const int mt = (a.M + 15) / 16;
  const int64_t xstep = (int64_t)mt * kWave * 8;  // elements per k-step
  const uint16_t* xp[M1];
  u32x4 xr[D][M1];
  f32x4 acc[M1][T];
#pragma unroll
  for (int i = 0; i < M1; ++i) {
    xp[i] = a.X + (((int64_t)s0 * mt + w + kNW * i) * kWave + l) * 8;
#pragma unroll
    for (int t = 0; t < T; ++t) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  if (MY > 0) {
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
      for (int i = 0; i < MY; ++i) xr[d][i] = *reinterpret_cast<const u32x4*>(xp[i] + (int64_t)min(d, n - 1) * xstep);
  }

  for (int st = 0; st < nst; ++st) {
    // This stage's weights: loaded two stages ago (or before the ring). Younger than them are at least the X loads
    // of the stages between, (kStage + D) MY (the ring's first D and stage 0's for stage 1, more later): that
    // many may stay in flight. Stage 0 waits for all.
    if (st == 0 || MY == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(MY * (kStage + D) < 63 ? MY * (kStage + D) : 63) : "memory");
    // every wave's part is in, and the buffer that stage st + 2 overwrites has been read (by stage st - 1)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (st + 2 < nst) load_stage(st + 2);
    if (MY == 0) continue;
    const u32x4(*buf)[T][kWave] = sW[st % kBufs];
    u32x4 wf[2][T];
#pragma unroll
    for (int t = 0; t < T; ++t) wf[0][t] = buf[0][t][l];
#pragma unroll
    for (int j = 0; j < kStage; ++j) {
      const int ks = st * kStage + j;
      if (ks >= n) break;  // uniform
      if (j + 1 < kStage) {
#pragma unroll
        for (int t = 0; t < T; ++t) wf[(j + 1) & 1][t] = buf[j + 1][t][l];
      }
#pragma unroll
      for (int i = 0; i < M1; ++i) {
#pragma unroll
        for (int t = 0; t < T; ++t)
          acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf(wf[j & 1][t]), as_bf(xr[j % D][i]), acc[i][t], 0, 0, 0);
      }
      const int kn = min(ks + D, n - 1);
#pragma unroll
      for (int i = 0; i < M1; ++i) xr[j % D][i] = *reinterpret_cast<const u32x4*>(xp[i] + (int64_t)kn * xstep);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (MY == 0) return;

  // ---- epilogue: lane l holds Y[16 mt + l % 16][16 t + 4 (l / 16) + e]
#pragma unroll
  for (int i = 0; i < M1; ++i) {
    const int m = (w + kNW * i) * 16 + l % 16;
    float inv = 1.f;
    if (a.ss) {  // a lane group sums every fourth chunk
      const int C = ss_chunks(a.K);
      const float* row = a.ss + (int64_t)min(m, a.M - 1) * C;
      float q = 0.f;
      for (int c = l / 16; c < C; c += 4) q += row[c];
      q += __shfl_xor(q, 16, kWave);
      q += __shfl_xor(q, 32, kWave);
      inv = rsqrtf(q / (float)a.K + a.eps);
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
      f32x4 v = acc[i][t] * inv;
      if (a.epi == kSilu) {
        // lanes 0..31 hold the tile's rows 0..7 (gate), lanes 32..63 its rows 8..15 (the matching up)
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float up = __shfl_xor(v[e], 32, kWave);
          y[e] = silu(bf2f(f2bf(v[e]))) * bf2f(f2bf(up));
        }
        const int f = (t0 + t) * 8 + (l / 16) * 4;
        if (m < a.M && t < nt && l < 32)
          *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(a.out) + (a.of ? mid_off(m, f, mt) : (int64_t)m * a.o_st + f)) =
              u32x2{f2bf2(y[0], y[1]), f2bf2(y[2], y[3])};
      } else if (m < a.M && t < nt) {
        const int c = (t0 + t) * 16 + (l / 16) * 4;
        if (a.epi == kStore)
          *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(a.out) + (a.of ? mid_off(m, c, mt) : (int64_t)m * a.o_st + c)) =
              u32x2{f2bf2(v[0], v[1]), f2bf2(v[2], v[3])};
        else
          *reinterpret_cast<f32x4*>(static_cast<float*>(a.out) + ((int64_t)blockIdx.y * a.M + m) * a.N + c) = v;
      }
    }
  }
}

template <int T, int MTW>
__global__ __launch_bounds__(kNW* kWave) void wsmid_kernel(MidArgs a) {
  __shared__ __align__(16) u32x4 sW[kBufs][kStage][T][kWave];
  constexpr int D = MTW == 4 ? 4 : 8;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave), l = threadIdx.x % kWave;
  const int mt = (a.M + 15) / 16, my = (mt - w + kNW - 1) / kNW;  // MTW or one less; the waves meet at the same barriers
  if (my == MTW) run<T, MTW, D>(a, sW, w, l);
  else run<T, MTW - 1, D>(a, sW, w, l);
}

struct Plan {
  int T, kg;
};
// Column tiles per workgroup and K splits by the cycles of the busiest CU: per k-step the largest of the matrix work
// (the row tiles of one SIMD's two waves, 16 cycles a tile), the loads (64 B per cycle of X and weights) and the
// LDS reads (8 waves, 128 B per cycle); 6000 for a workgroup's first loads and its epilogue; partial planes at the
// memory's 2 KB per cycle, written and read. Against T = 2..5 and 1 to 8 splits at 64, 132, 264 and 512 rows the plan is
// the fastest or within 1 us of it: gate / up at 264 rows T = 2: 69, 3: 55, 4: 63, 5: 41 us (planned); down there T = 3 in
// 4 splits 27.1, 4 in 6 25.5 (planned), 5 in 8 24.9, 4 in 1 82; at 132 rows 3 in 4 20.4 (planned), 4 in 6 19.5.
Plan plan_mid(int64_t M, int64_t N, int64_t K, int epi) {
  const int64_t tiles = N / 16, nsteps = K / 32, mt = cdiv(M, 16);
  Plan best{0, 0};
  double best_cost = 0;
  for (int T = 2; T <= kMaxT; ++T) {
    const double step = std::max<double>({(double)(cdiv(mt, 4) * T * 16), (double)((mt + T) * 16), (double)(std::min<int64_t>(mt, kNW) * T * 8)});
    for (int kg = 1; kg <= (epi == kParts ? 16 : 1); ++kg) {
      if (kg > 1 && nsteps / kg < kStage) break;
      const int64_t rounds = cdiv(cdiv(tiles, T) * kg, kCUs);
      const double cost = (double)rounds * ((double)cdiv(nsteps, kg) * step + 6000.0) +
                          (epi == kParts ? (double)kg * (double)(M * N) * 8.0 / 2048.0 : 0.0);
      if (!best.T || cost < best_cost) {
        best_cost = cost;
        best = {T, kg};
      }
    }
  }
  return best;
}

template <int T>
void launch(const MidArgs& a, int kg, hipStream_t st) {
  const dim3 grid((unsigned)cdiv(a.N / 16, T), (unsigned)kg);
  switch ((a.M + 127) / 128) {
    case 1: hipLaunchKernelGGL((wsmid_kernel<T, 1>), grid, dim3(kNW * kWave), 0, st, a); break;
    case 2: hipLaunchKernelGGL((wsmid_kernel<T, 2>), grid, dim3(kNW * kWave), 0, st, a); break;
    case 3: hipLaunchKernelGGL((wsmid_kernel<T, 3>), grid, dim3(kNW * kWave), 0, st, a); break;
    default: hipLaunchKernelGGL((wsmid_kernel<T, 4>), grid, dim3(kNW * kWave), 0, st, a); break;
  }
}

// h += r (bf16 rows, the residual stream) in place, ss[row][chunk] = the sum of h^2 over each 256 columns (one wave
// each), and hf = h once more in the fragment order of mt row tiles
__global__ __launch_bounds__(kWave) void residual_mid_kernel(uint16_t* h, int64_t h_st, const uint16_t* r, int64_t r_st,
                                                             int dim, float* ss, uint16_t* hf, int mt) {
  const int row = blockIdx.x, c = blockIdx.y, l = threadIdx.x, e = c * 256 + l * 4;
  float q = 0.f;
  if (e < dim) {
    uint16_t* hp = h + (int64_t)row * h_st + e;
    const u32x2 hv = *reinterpret_cast<const u32x2*>(hp), rv = *reinterpret_cast<const u32x2*>(r + (int64_t)row * r_st + e);
    u32x2 o;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      o[i] = f2bf2(__uint_as_float(hv[i] << 16) + __uint_as_float(rv[i] << 16),
                   __uint_as_float(hv[i] & 0xffff0000u) + __uint_as_float(rv[i] & 0xffff0000u));
      const float lo = __uint_as_float(o[i] << 16), hi = __uint_as_float(o[i] & 0xffff0000u);
      q = fmaf(hi, hi, fmaf(lo, lo, q));
    }
    *reinterpret_cast<u32x2*>(hp) = o;
    *reinterpret_cast<u32x2*>(hf + mid_off(row, e, mt)) = o;
  }
  q = wave_sum(q);
  if (l == 0) ss[(int64_t)row * ss_chunks(dim) + c] = q;
}

bool shape_ok(int64_t M, int64_t N, int64_t K) {
  return M >= kMinM && M <= kMaxM && N > 0 && K > 0 && N % 16 == 0 && K % 32 == 0 && N < INT32_MAX && K < INT32_MAX;
}

}  // namespace
}  // namespace trida

using namespace trida;

extern "C" int trida_wsgemm_mid_plan(int64_t M, int64_t N, int64_t K, int epilogue, int32_t* kgroups) {
  TRIDA_CHECK(kgroups, TRIDA_ERR_NULL, "wsgemm_mid_plan: kgroups is required");
  TRIDA_CHECK(shape_ok(M, N, K) && epilogue >= kStore && epilogue <= kSilu, TRIDA_ERR_ARG,
              "wsgemm_mid_plan: need %d <= M <= %d, N %% 16 == 0, K %% 32 == 0 and epilogue 0..2", kMinM, kMaxM);
  *kgroups = plan_mid(M, N, K, epilogue).kg;
  return TRIDA_OK;
}

extern "C" int64_t trida_ws_mid_elems(int64_t M, int64_t K) {
  return M >= kMinM && M <= kMaxM && K > 0 && K % 32 == 0 ? cdiv(M, 16) * 16 * K : 0;
}

extern "C" int trida_residual_mid(uint16_t* h, int64_t h_row_stride, const uint16_t* r, int64_t r_row_stride, int64_t rows,
                                  int64_t dim, float* ss, uint16_t* h_frag, void* stream) {
  TRIDA_CHECK(h && r && ss && h_frag, TRIDA_ERR_NULL, "residual_mid: h, r, ss and h_frag are required");
  TRIDA_CHECK(rows >= kMinM && rows <= kMaxM && dim > 0 && dim % 32 == 0 && dim < INT32_MAX && h_row_stride >= dim &&
                  r_row_stride >= dim && h_row_stride % 4 == 0 && r_row_stride % 4 == 0,
              TRIDA_ERR_ARG, "residual_mid: need %d <= rows <= %d, dim %% 32 == 0 and row strides of at least dim, in fours",
              kMinM, kMaxM);
  TRIDA_CHECK((((uintptr_t)h | (uintptr_t)r) & 7) == 0 && ((uintptr_t)h_frag & 15) == 0 && ((uintptr_t)ss & 3) == 0,
              TRIDA_ERR_ALIGN, "residual_mid: h and r 8-byte, h_frag 16-byte aligned");
  hipLaunchKernelGGL(residual_mid_kernel, dim3((unsigned)rows, (unsigned)ss_chunks((int)dim)), dim3(kWave), 0,
                     static_cast<hipStream_t>(stream), h, h_row_stride, r, r_row_stride, (int)dim, ss, h_frag,
                     (int)cdiv(rows, 16));
  return launch_status("residual_mid");
}

extern "C" int trida_wsgemm_mid(const uint16_t* X, const float* ss, float eps, const uint16_t* Wp, int64_t M, int64_t N,
                                int64_t K, int epilogue, void* out, int64_t out_row_stride, int flags, void* stream) {
  TRIDA_CHECK(X && Wp && out, TRIDA_ERR_NULL, "wsgemm_mid: X, Wp and out are required");
  TRIDA_CHECK(shape_ok(M, N, K) && epilogue >= kStore && epilogue <= kSilu, TRIDA_ERR_ARG,
              "wsgemm_mid: need %d <= M <= %d, N %% 16 == 0, K %% 32 == 0 and epilogue 0..2 (M=%lld N=%lld K=%lld)", kMinM,
              kMaxM, (long long)M, (long long)N, (long long)K);
  TRIDA_CHECK(!ss || epilogue != kParts, TRIDA_ERR_ARG, "wsgemm_mid: the RMSNorm takes the bf16 (0) or SwiGLU (2) epilogue");
  const bool of = flags & TRIDA_WS_OUT_FRAG;
  TRIDA_CHECK((flags & ~TRIDA_WS_OUT_FRAG) == 0 && (!of || (epilogue != kParts && (epilogue == kSilu ? N / 2 : N) % 32 == 0)),
              TRIDA_ERR_ARG, "wsgemm_mid: a fragment-order output needs the bf16 or SwiGLU epilogue and a width of 32s");
  TRIDA_CHECK(epilogue == kParts || of || (out_row_stride >= (epilogue == kSilu ? N / 2 : N) && out_row_stride % 4 == 0),
              TRIDA_ERR_ARG, "wsgemm_mid: bad output row stride");
  TRIDA_CHECK(((((uintptr_t)X) | (uintptr_t)Wp | (uintptr_t)out) & 15) == 0 && ((uintptr_t)ss & 3) == 0, TRIDA_ERR_ALIGN,
              "wsgemm_mid: X, Wp and out must be 16-byte aligned");
  const Plan p = plan_mid(M, N, K, epilogue);
  const MidArgs a{X, reinterpret_cast<const u32x4*>(Wp), out, out_row_stride, (int)M, (int)N, (int)K, epilogue,
                  of ? 1 : 0, ss, eps};
  hipStream_t st = static_cast<hipStream_t>(stream);
  switch (p.T) {
    case 2: launch<2>(a, p.kg, st); break;
    case 3: launch<3>(a, p.kg, st); break;
    case 4: launch<4>(a, p.kg, st); break;
    default: launch<5>(a, p.kg, st); break;
  }
  return launch_status("wsgemm_mid");
}
