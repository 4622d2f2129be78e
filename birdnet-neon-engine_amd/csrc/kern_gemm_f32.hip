// fp32 1x1 convolution / GEMM of the registry's PW op (src/rt_ops_f32.c:129-212, gemm_f32 / gemm_f32_range_gate
// src/gemm_f32.c:141-197), bit-identical: every output (m, n), n < Np, is one fp32 FMA chain over k < Kp from +0 in
// k order (the 8 x 8 register tile's chains, src/gemm_f32_kblock.h), + b[n], the activation (the NEON SiLU / max 0),
// + residual, stored at its padded row; a gated A is the fp32 product A[m][k] gate[k] (the value an in-place gating
// multiply stores).
//
// The chains run on the matrix cores: v_mfma_f32_16x16x4_f32 adds its four products to each accumulator one after
// the other in k order, each a fused multiply-add rounded to nearest even with denormals kept, so a row of them is
// the FMA chain (compared with fmaf chains on 20 million sums: normal, wide-range, denormal and arbitrary bit
// patterns, infinities, NaNs and signed zeros; tests/test_gpu_f32pw.py holds it). 64 multiply-adds a clock and SIMD
// against 16 on the vector unit, which bounded the kernel before.
//
// Tiling: the rows of all windows in one list; a wave owns TM x 16 rows by 16 channels, the block's 4 waves lie WM
// down the rows and 4 / WM across the channels. Rows go through LDS in chunks of 32 k (each wave of a row group reads
// them), a chunk ahead in registers; a row's k are stored by k % 4, the instruction's operand lane, so that a lane
// reads its four steps of 16 k at once. A wave's weights go from the package panels [Np/8][Kp][8] straight to
// registers (four k of two panels are 256 contiguous bytes a load), also a chunk ahead. Weights are the instruction's
// rows, so a lane ends with four neighbouring channels of a row, one 16-byte store.
#include <type_traits>

#include "bnh_internal.h"
#include "bnh_num.h"

#define GF_KC 32
#define GF_RS (GF_KC + 4)  // LDS row stride in floats: neighbouring rows four banks apart

typedef float gf_f4 __attribute__((ext_vector_type(4)));

// GATE: there is a gate; V: A, gate, output and residual rows are 16-byte aligned
template <int TM, int WM, bool GATE, bool V>
__global__ __launch_bounds__(256, WM == 1 ? 6 : 4) void k_gemm_f32(const float *__restrict__ A, long long a_ws, int lda, int M,
                                                  int rows, int Kp, const float *__restrict__ gate,
                                                  long long g_ws, const float *__restrict__ w,
                                                  const float *__restrict__ bias, int Np, bnh_epi32 e,
                                                  double i_m, double i_ow, double i_rw) {
  constexpr int BM = 16 * TM * WM, WN = 4 / WM, NL = (BM + 31) / 32;
  __shared__ __attribute__((aligned(16))) float As[2][BM * GF_RS];
  __shared__ uint32_t tbl[256];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, c16 = lane & 15, h = lane >> 4;
  const int wm = wv / WN, wn = wv % WN;
  const int m0 = (int)blockIdx.x * BM;
  const int n0 = (blockIdx.y * WN + wn) * 16;  // this wave's channels
  const bool live = n0 < Np;
  if (e.act == 1) bnh_silu_table(tbl);
  // loader: 4 k of a row each, 16 rows x 16 k a wave (their LDS writes fall into 64 banks); rows past the end repeat
  // the last one, unused
  const float *arow[NL], *grow[GATE ? NL : 1];
  int lk[NL], ls[NL];
#pragma unroll
  for (int j = 0; j < NL; j++) {
    const int i = tid + 256 * j, row = i % (4 * BM) >> 2, q = i / (4 * BM) * 4 + (i & 3);
    int r = m0 + row;
    r = r < rows ? r : rows - 1;
    const int win = bnh_div(r, M, i_m);
    arow[j] = A + win * a_ws + (long long)(r - win * M) * lda;
    if (GATE) grow[j] = gate + win * g_ws;
    lk[j] = 4 * q;
    ls[j] = row * GF_RS + q;
  }
  // weights: lane (c16, h) holds channel n0 + c16 at k = 4 s + h (channels past Np repeat the last, unused)
  const int wc = n0 + c16 < Np ? n0 + c16 : Np - 1;
  const float *wl = w + (long long)(wc >> 3) * Kp * 8 + (wc & 7);
  float4 ra[NL], rg[GATE ? NL : 1];
  float wr[2][8];
  auto fetch = [&](int k0, float *wd) {
#pragma unroll
    for (int j = 0; j < NL; j++) {
      const int k = k0 + lk[j] < Kp ? k0 + lk[j] : Kp - 4;  // past Kp: in bounds, unused
      const float *a = arow[j] + k;
      if (V) ra[j] = *(const float4 *)a;
      else ra[j] = make_float4(a[0], a[1], a[2], a[3]);
      if (GATE) {
        const float *g = grow[j] + k;
        if (V) rg[j] = *(const float4 *)g;
        else rg[j] = make_float4(g[0], g[1], g[2], g[3]);
      }
    }
    if (k0 + GF_KC <= Kp) {
#pragma unroll
      for (int s = 0; s < 8; s++) wd[s] = wl[(k0 + 4 * s + h) * 8];
    } else {
#pragma unroll
      for (int s = 0; s < 8; s++) wd[s] = wl[(k0 + 4 * s + h < Kp ? k0 + 4 * s + h : Kp - 1) * 8];
    }
  };
  auto commit = [&](int buf) {
#pragma unroll
    for (int j = 0; j < NL; j++)
      if (BM >= 32 || tid < 8 * BM) {
        float4 v = ra[j];
        if (GATE) v.x *= rg[j].x, v.y *= rg[j].y, v.z *= rg[j].z, v.w *= rg[j].w;
        float *d = &As[buf][ls[j]];
        d[0] = v.x, d[8] = v.y, d[16] = v.z, d[24] = v.w;
      }
  };
  gf_f4 acc[TM];
#pragma unroll
  for (int i = 0; i < TM; i++) acc[i] = (gf_f4){0.f, 0.f, 0.f, 0.f};
  // the chunk at k0 in LDS buffer buf: all of its 8 steps, or those before Kp (a multiple of 4)
  auto chunk = [&](auto whole, int buf, int k0, const float *wk) {
    const float *ap = &As[buf][(wm * TM * 16 + c16) * GF_RS + 8 * h];
#pragma unroll
    for (int g = 0; g < 2; g++) {  // 16 k at a time
      gf_f4 av[TM];
#pragma unroll
      for (int i = 0; i < TM; i++) av[i] = *(const gf_f4 *)(ap + i * 16 * GF_RS + 4 * g);
#pragma unroll
      for (int s = 0; s < 4; s++)
        if (decltype(whole)::value || k0 + 16 * g + 4 * s < Kp) {
#pragma unroll
          for (int i = 0; i < TM; i++)
            acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wk[4 * g + s], av[i][s], acc[i], 0, 0, 0);
        }
    }
  };
  fetch(0, wr[0]);
  commit(0);
  __syncthreads();
  int k0 = 0;
  for (; Kp - k0 >= 2 * GF_KC; k0 += 2 * GF_KC) {
    fetch(k0 + GF_KC, wr[1]);
    if (live) chunk(std::true_type{}, 0, k0, wr[0]);
    commit(1);
    __syncthreads();
    fetch(k0 + 2 * GF_KC, wr[0]);  // past Kp after the last chunk: in bounds, unused
    if (live) chunk(std::true_type{}, 1, k0 + GF_KC, wr[1]);
    commit(0);
    __syncthreads();
  }
  if (Kp - k0 > GF_KC) {  // a whole chunk and part of one
    fetch(k0 + GF_KC, wr[1]);
    if (live) chunk(std::true_type{}, 0, k0, wr[0]);
    commit(1);
    __syncthreads();
    if (live) chunk(std::false_type{}, 1, k0 + GF_KC, wr[1]);
  } else if (k0 < Kp) {
    if (live) chunk(std::false_type{}, 0, k0, wr[0]);
  }
  // epilogue: + b, activation, + residual, padded store of channels n .. n + 3
  const int n = n0 + 4 * h;
  if (n >= Np) return;
  const float bv[4] = {bias[n], bias[n + 1], bias[n + 2], bias[n + 3]};
#pragma unroll
  for (int i = 0; i < TM; i++) {
    const int r = m0 + (wm * TM + i) * 16 + c16;
    if (r >= rows) continue;
    const int win = bnh_div(r, M, i_m), m = r - win * M;
    // row m of an image of ow columns with p pixels of halo: (m / ow + p) (ow + 2 p) + m % ow + p
    const long long orow = e.opad ? m + (long long)e.opad * (2 * bnh_div(m, e.ow, i_ow) + e.ow + 2 * e.opad + 1) : m;
    float *o = e.out + win * e.out_ws + orow * e.ldo + n;
    float y[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      y[j] = acc[i][j] + bv[j];
      if (e.act == 1) y[j] = bnh_silu_f32_t(y[j], tbl);
      else if (e.act == 2) y[j] = bnh_relu_f32(y[j]);
    }
    if (e.res) {
      const long long rrow = e.rpad ? m + (long long)e.rpad * (2 * bnh_div(m, e.rw, i_rw) + e.rw + 2 * e.rpad + 1) : m;
      const float *q = e.res + win * e.res_ws + rrow * e.ldr + n;
      if (V) {
        const float4 v = *(const float4 *)q;
        y[0] += v.x, y[1] += v.y, y[2] += v.z, y[3] += v.w;
      } else {
#pragma unroll
        for (int j = 0; j < 4; j++) y[j] += q[j];
      }
    }
    if (V) {
      *(float4 *)o = make_float4(y[0], y[1], y[2], y[3]);
    } else {
#pragma unroll
      for (int j = 0; j < 4; j++) o[j] = y[j];
    }
  }
}

template <int TM, int WM>
static void gf_launch(bool vec, int rows, int Np, hipStream_t st, const float *A, long long a_ws, int lda, int M,
                      int Kp, const float *gate, long long g_ws, const float *w, const float *bias,
                      const bnh_epi32 &e) {
  const dim3 grid((unsigned)bnh_ceil_div(rows, 16 * TM * WM), (unsigned)bnh_ceil_div(Np, 64 / WM));
#define GF_L(G, V)                                                                                                     \
  hipLaunchKernelGGL((k_gemm_f32<TM, WM, G, V>), grid, dim3(256), 0, st, A, a_ws, lda, M, rows, Kp, gate, g_ws, w,    \
                     bias, Np, e, 1.0 / M, 1.0 / (e.ow > 0 ? e.ow : 1), 1.0 / (e.rw > 0 ? e.rw : 1))
  if (gate && vec) GF_L(true, true);
  else if (gate) GF_L(true, false);
  else if (vec) GF_L(false, true);
  else GF_L(false, false);
#undef GF_L
}

extern "C" int bnh_gemm_f32(const float *A, long long a_ws, int lda, int M, const float *gate, long long g_ws,
                            const float *w, const float *bias, int Kp, int Np, const bnh_epi32 *e, int B,
                            void *stream) {
  BNH_REQ(A && w && bias && e && e->out && M > 0 && B > 0 && B <= 65535);
  BNH_REQ(Kp > 0 && Kp % 4 == 0 && Np > 0 && Np % 8 == 0 && lda >= Kp && e->ldo >= Np);
  BNH_REQ(e->act >= 0 && e->act <= 2 && e->opad >= 0 && e->opad <= 3 && (!e->opad || (e->ow > 0 && M % e->ow == 0)));
  BNH_REQ(!e->res || (e->ldr >= Np && (!e->rpad || (e->rw > 0 && M % e->rw == 0))));
  BNH_REQ(((uintptr_t)w & 15) == 0);
  BNH_REQ(B == 1 || (a_ws >= (long long)M * lda && (!gate || g_ws >= Kp)));
  // 16-byte accesses where the rows' addresses allow them
  auto rows16 = [&](const void *p, int ld, long long ws) {
    return ((uintptr_t)p & 15) == 0 && ld % 4 == 0 && (B == 1 || ws % 4 == 0);
  };
  const bool vec = rows16(A, lda, a_ws) && (!gate || rows16(gate, 0, g_ws)) && rows16(e->out, e->ldo, e->out_ws) &&
                   (!e->res || rows16(e->res, e->ldr, e->res_ws));
  // The split with the least work on the fullest CU: its blocks there times a wave's step (TM matrix instructions and
  // about half of one for its LDS reads and weights). Against 64 x 64 tiles on the
  // vector unit: 48 windows of 256 px, 136 -> 816 with SiLU 64 -> 39 us, 816 -> 136 gated 140 -> 53; one such window
  // 92 -> 13; 64 windows of 4000 px, 144 -> 24 100 -> 43; 256 windows of 64 px, 1392 -> 384 334 -> 204 (86 TFLOP/s).
  struct { int tm, wm; } best = {4, 1};
  double least = 0;
  static const struct { int tm, wm; } plan[] = {{4, 1}, {4, 2}, {2, 4}, {2, 1}, {2, 2}, {1, 4}, {1, 1}, {1, 2}};
  const long long all = (long long)M * B;
  // An output over its input or gate: a row has to be read before anything is stored over it, which holds for blocks of
  // 64 whole rows (Np <= 64; past its last barrier a block has read all it reads). Where each output row lies on its own
  // input row they can all run at once; else the windows run one after the other, each its own block or blocks.
  const bool rows_match = e->ldo == lda && !e->opad && (B == 1 || e->out_ws == a_ws);
  const bnh_region so = bnh_windows(e->out, e->out_ws, bnh_rows_span(M, e->ldo, e->ow, e->opad));
  const bool over_gate = gate && bnh_overlap(so, bnh_windows(gate, g_ws, Kp), B);
  const bool over = over_gate || (bnh_overlap(so, bnh_windows(A, a_ws, bnh_rows_span(M, lda, 0, 0)), B) &&
                                  !(rows_match && bnh_beside(A, Kp, (const float *)e->out, Np, lda)));
  const bool at_once = !over || (!over_gate && rows_match && e->out == A);
  for (const auto &p : plan) {
    if (over && least) break;  // the first of the list, 64 rows x 64 channels
    if (bnh_ceil_div(Np, 64 / p.wm) > 65535) continue;
    const long long blocks = bnh_ceil_div(all, 16 * p.tm * p.wm) * bnh_ceil_div(Np, 64 / p.wm);
    const double cost = (double)bnh_ceil_div(blocks, 256) * (p.tm + 0.5);
    if (least == 0 || cost < least) least = cost, best = {p.tm, p.wm};
  }
  // a launch takes at most 2^27 rows (a grid dimension is limited in threads)
  const int most = !at_once || (1 << 27) / M < 1 ? 1 : (1 << 27) / M;
  for (int b0 = 0; b0 < B; b0 += most) {
    const int nb = B - b0 < most ? B - b0 : most;
    bnh_epi32 f = *e;
    f.out += b0 * e->out_ws;
    if (f.res) f.res += b0 * e->res_ws;
    const float *a = A + b0 * a_ws, *g = gate ? gate + b0 * g_ws : nullptr;
    const int rows = M * nb;
    hipStream_t st = bnh_stream(stream);
#define GF_P(TM, WM)                                                                                                   \
  if (best.tm == TM && best.wm == WM) gf_launch<TM, WM>(vec, rows, Np, st, a, a_ws, lda, M, Kp, g, g_ws, w, bias, f)
    GF_P(4, 1);
    GF_P(4, 2);
    GF_P(2, 4);
    GF_P(2, 1);
    GF_P(2, 2);
    GF_P(1, 4);
    GF_P(1, 1);
    GF_P(1, 2);
#undef GF_P
    BNH_HIP(hipGetLastError());
  }
  return 0;
}
