// The fp32 and fp16 prototype heads of libbnneon on gfx950: PROTO variant 0 (fp32 cells and prototypes,
// src/rt_ops_f32.c:548-570), PROTO_F32H (fp16-stored prototypes, fp32 arithmetic, src/rt_ops_f32.c:572-591) and
// PROTO variant 1 (fp16, src/rt_ops_f16.c:227-250). Each is the L2 normalisation of the cells (pc_l2norm_f32 /
// pc_l2norm_f16), the cells x prototypes product of which only the column maxima over a window's cells are kept
// (gemm_f32_colmax, pc_proto_colmax_f32h, gemm_f16_colmax), then the class logits (bnh_proto_logits, kern_proto.hip).
//
// Bit-identical to the reference. Every product sum is one fused multiply-add chain in the reference's order: fp32
// from +0 over k; fp16 from +0 over each K block (the fp16 GEMM's balanced blocks of at most 128 steps), the blocks'
// widened results summed in fp32 from +0. The maximum over cells is exact and order-free (NaN-propagating FMAX).
//
// The fp32 chains run on the matrix cores: v_mfma_f32_16x16x4_f32 adds its four products one after the other in k
// order, each a fused multiply-add rounded to nearest even, denormals kept (compared bit for bit with fmaf chains).
// fp16 matrix instructions accumulate in fp32, so the fp16 chains run on the VALU: a thread owns 8 cells x 8
// prototypes (32 packed fp16 pairs), its operands two 16-byte LDS reads per k step each.
//
// Prototypes are repacked at load: kinds 0 and 1 into tiles of 16 prototypes x 16 k in the matrix instruction's
// operand order (lane (c, h) of a wave reads prototype c at k = h, 4 + h, 8 + h, 12 + h as one 16- or 8-byte word,
// zeros past Np and K); kind 2 into k-major rows [K][Npt] (Npt = Np rounded up to 256, zeros past Np), a block's 256
// prototypes at one k one contiguous 512 B run.
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include <type_traits>

#include "bnh_cells.h"
#include "bnh_f16.h"
#include "bnh_internal.h"
#include "bnh_num.h"

struct bnh_fproto {
  int kind;     // 0 fp32 (PROTO variant 0), 1 fp16-stored / fp32 math (PROTO_F32H), 2 fp16 (PROTO variant 1)
  int Np, K, Npt;
  int nblk, bs;  // kind 2: the fp16 GEMM's K blocks
  void *w;       // kinds 0, 1: [Np/16][K/16][64 lanes][4] (fp32, fp16 bit patterns); kind 2: k-major [K][Npt] fp16
};

// ------------------------------------------------------------------ L2 normalisation of the cells
// One wave per cell (bnh_cells.h). den = sqrtf(sum) + eps, a = x / den (correctly rounded division); F16: fp16 cells
// widened, a rounded to fp16 (nearest even). vec, avec: the rows of x and of a are 16-byte (fp16: 8-byte) aligned.
template <bool F16, int NV>
__global__ __launch_bounds__(256) void k_l2norm(const void *__restrict__ xv, long long x_ws, int P, int C, int ld,
                                                float eps, void *__restrict__ av, long long a_ws, long long cells,
                                                bool vec, bool avec) {
  __shared__ __attribute__((aligned(16))) float stage[4][8 * Cell<NV>::LS];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  long long cell = (long long)blockIdx.x * 4 + wv;
  const bool live = cell < cells;
  if (!live) cell = cells - 1;
  const long long w = cell / P;
  const int p = (int)(cell - w * P);
  const void *r = (const char *)xv + (w * x_ws + (long long)p * ld) * (F16 ? 2 : 4);
  constexpr int CH = Cell<NV>::CH;
  Cell<NV> x;
  float chain = 0.f;
  for (int c0 = 0; c0 < C; c0 += CH) {
    x.template load<F16>(r, c0, C, vec, lane);
    chain = x.squares(chain, C - c0 < CH ? C - c0 : CH, stage[wv], lane);
  }
  if (!live) return;
  const float den = cell_norm(chain, lane) + eps;
  const long long at = w * a_ws + (long long)p * C;
  for (int c0 = 0; c0 < C; c0 += CH) {
    if (C > CH) x.template load<F16>(r, c0, C, vec, lane);
#pragma unroll
    for (int j = 0; j < NV; j++) {
      const int c = c0 + 256 * j + 4 * lane;
      if (c >= C) continue;
      const float4 y = make_float4(x.v[j].x / den, x.v[j].y / den, x.v[j].z / den, x.v[j].w / den);
      if (F16) {
        uint16_t *a = (uint16_t *)av + at + c;
        const uint16_t e[4] = {hbits(f2h(y.x)), hbits(f2h(y.y)), hbits(f2h(y.z)), hbits(f2h(y.w))};
        if (avec) {
          *(uint2 *)a = make_uint2(e[0] | (uint32_t)e[1] << 16, e[2] | (uint32_t)e[3] << 16);
        } else {
          a[0] = e[0], a[1] = e[1], a[2] = e[2], a[3] = e[3];
        }
      } else {
        float *a = (float *)av + at + c;
        if (avec) {
          *(float4 *)a = y;
        } else {
          a[0] = y.x, a[1] = y.y, a[2] = y.z, a[3] = y.w;
        }
      }
    }
  }
}

#define FP_BM 64   // cells per tile of the fp16 kernel
#define FP_BN 256  // prototypes per block of the fp16 kernel

// ------------------------------------------------------------------ fp32 column maxima (kinds 0 and 1)
#define FF_KC 64           // k steps per LDS stage
#define FF_RS (FF_KC + 4)  // LDS row stride in floats: neighbouring cells four banks apart
typedef float fp_f4 __attribute__((ext_vector_type(4)));
// A wave owns TC x 16 cells by TN x 16 prototypes of one window and walks the window's cells 16 TC WC at a time; the
// block's 4 waves lie WC down the cells and 4 / WC across the prototypes. Cells go through LDS (every wave of a cell
// group reads them), a cell's k stored by k % 4, the instruction's operand lane, so that a lane reads its four steps of
// 16 k at once; prototypes go straight to registers; both are fetched a chunk ahead. WH: prototypes stored as fp16, widened
// exactly (PROTO_F32H). Bound by the matrix cores' 64 fp32 multiply-adds a clock and SIMD; the vector unit's 16 and
// an LDS read per 4 of them bounded the kernel before.
template <bool WH, int TC, int WC, int TN>
__global__ __launch_bounds__(256) void k_colmax_f32(const float *__restrict__ a, long long a_ws, int P, int K,
                                                    const void *__restrict__ wv, int Np, float *__restrict__ colmax,
                                                    long long cm_ws, int B) {
  constexpr int WN = 4 / WC, BM = 16 * TC * WC, NL = BM / 16;
  __shared__ __attribute__((aligned(16))) float As[2][BM * FF_RS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c16 = lane & 15, h = lane >> 4;
  const int wc = wave / WN, wn = wave % WN;
  // windows fastest, and neighbouring blocks under one L2: they read the same prototypes
  const unsigned blk = bnh_xcd_block(blockIdx.x, gridDim.x);
  const int win = (int)(blk % (unsigned)B);
  const int t0 = ((int)(blk / (unsigned)B) * WN + wn) * TN;  // this wave's first prototype tile
  const int K16 = (K + 15) / 16, ntile = (Np + 15) / 16;
  const float *aw = a + win * a_ws;
  // loader: 4 k of a cell each, 16 cells x 16 k a wave (their LDS writes fall into 64 banks)
  auto cell_of = [&](int j) { return (tid + 256 * j) % (4 * BM) >> 2; };
  auto quad_of = [&](int j) { return (tid + 256 * j) / (4 * BM) * 4 + (tid & 3); };
  size_t wt[TN];  // tiles past the last repeat it, unused
#pragma unroll
  for (int t = 0; t < TN; t++) wt[t] = (size_t)(t0 + t < ntile ? t0 + t : ntile - 1) * K16 * 64 + lane;
  float4 ra[NL];
  // this wave's prototypes of an even and an odd chunk: each 16 k reloaded for two chunks on as soon as they are used
  using wq = std::conditional_t<WH, uint2, float4>;
  wq w[2][TN][4];
  float mx[TN];
#pragma unroll
  for (int t = 0; t < TN; t++) mx[t] = -INFINITY;
  for (int m0 = 0; m0 < P; m0 += BM) {
    auto fetch_a = [&](int k0) {  // rows past P repeat the last cell; k past K: in bounds, unused
#pragma unroll
      for (int j = 0; j < NL; j++) {
        const int k = k0 + 4 * quad_of(j) < K ? k0 + 4 * quad_of(j) : K - 4;
        const int r = m0 + cell_of(j) < P ? m0 + cell_of(j) : P - 1;
        ra[j] = *(const float4 *)(aw + (long long)r * K + k);
      }
    };
    auto commit_a = [&](int buf) {
#pragma unroll
      for (int j = 0; j < NL; j++) {
        float *d = &As[buf][cell_of(j) * FF_RS + quad_of(j)];
        d[0] = ra[j].x, d[16] = ra[j].y, d[32] = ra[j].z, d[48] = ra[j].w;
      }
    };
    auto fetch_w = [&](int set, int g, int k0) {
      const int kt = k0 / 16 + g < K16 ? k0 / 16 + g : K16 - 1;
#pragma unroll
      for (int t = 0; t < TN; t++) w[set][t][g] = ((const wq *)wv)[wt[t] + (size_t)kt * 64];
    };
    fp_f4 acc[TC][TN];
#pragma unroll
    for (int i = 0; i < TC; i++)
#pragma unroll
      for (int t = 0; t < TN; t++) acc[i][t] = (fp_f4){0.f, 0.f, 0.f, 0.f};
    // the chunk at k0 in LDS buffer buf: all of its 16 steps, or the first n
    auto steps = [&](auto whole, auto buf_c, int k0, int n) {
      constexpr int buf = decltype(buf_c)::value;
      const float *ap = &As[buf][(wc * TC * 16 + c16) * FF_RS + 16 * h];
      fp_f4 av[2][TC];  // the operands of this and the next 16 k
#pragma unroll
      for (int i = 0; i < TC; i++) av[0][i] = *(const fp_f4 *)(ap + i * 16 * FF_RS);
#pragma unroll
      for (int g = 0; g < 4; g++) {
        if (g < 3) {
#pragma unroll
          for (int i = 0; i < TC; i++) av[(g + 1) & 1][i] = *(const fp_f4 *)(ap + i * 16 * FF_RS + 4 * (g + 1));
        }
        float wk[TN][4];
#pragma unroll
        for (int t = 0; t < TN; t++) {
          if constexpr (WH) {
            const h2 lo = __builtin_bit_cast(h2, w[buf][t][g].x), hi = __builtin_bit_cast(h2, w[buf][t][g].y);
            wk[t][0] = (float)lo.x, wk[t][1] = (float)lo.y, wk[t][2] = (float)hi.x, wk[t][3] = (float)hi.y;
          } else {
            wk[t][0] = w[buf][t][g].x, wk[t][1] = w[buf][t][g].y, wk[t][2] = w[buf][t][g].z, wk[t][3] = w[buf][t][g].w;
          }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 4; s++)
          if (decltype(whole)::value || 4 * g + s < n) {
#pragma unroll
            for (int i = 0; i < TC; i++)
#pragma unroll
              for (int t = 0; t < TN; t++)
                acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[g & 1][i][s], wk[t][s], acc[i][t], 0, 0, 0);
          }
        if (decltype(whole)::value) fetch_w(buf, g, k0 + 2 * FF_KC);
      }
    };
    std::integral_constant<int, 0> b0;
    std::integral_constant<int, 1> b1;
    __syncthreads();  // the previous cells' last reads of the buffers are done
    fetch_a(0);
#pragma unroll
    for (int g = 0; g < 4; g++) fetch_w(0, g, 0);
#pragma unroll
    for (int g = 0; g < 4; g++) fetch_w(1, g, FF_KC);
    commit_a(0);
    __syncthreads();
    int k0 = 0;
    for (; K - k0 >= 2 * FF_KC; k0 += 2 * FF_KC) {
      fetch_a(k0 + FF_KC);
      steps(std::true_type{}, b0, k0, 16);
      commit_a(1);
      __syncthreads();
      fetch_a(k0 + 2 * FF_KC);
      steps(std::true_type{}, b1, k0 + FF_KC, 16);
      commit_a(0);
      __syncthreads();
    }
    // the chains stop at K (a multiple of 8)
    if (K - k0 > FF_KC) {
      fetch_a(k0 + FF_KC);
      steps(std::true_type{}, b0, k0, 16);
      commit_a(1);
      __syncthreads();
      steps(std::false_type{}, b1, 0, (K - k0 - FF_KC) / 4);
    } else if (k0 < K) {
      steps(std::false_type{}, b0, 0, (K - k0) / 4);
    }
#pragma unroll
    for (int i = 0; i < TC; i++)
#pragma unroll
      for (int t = 0; t < TN; t++)
#pragma unroll
        for (int j = 0; j < 4; j++) mx[t] = bnh_fmax(mx[t], acc[i][t][j]);
  }
  // lane (c, h) holds prototype c over a quarter of the cells of its wave
#pragma unroll
  for (int t = 0; t < TN; t++) {
    mx[t] = bnh_fmax(mx[t], __shfl_xor(mx[t], 16));
    mx[t] = bnh_fmax(mx[t], __shfl_xor(mx[t], 32));
  }
  if (WC > 1) {
    __syncthreads();  // the last cells' reads are done
    float *red = &As[0][0];  // [TN][WC][WN][16]
    if (h == 0)
#pragma unroll
      for (int t = 0; t < TN; t++) red[((t * WC + wc) * WN + wn) * 16 + c16] = mx[t];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < TN; t++)
#pragma unroll
      for (int q = 0; q < WC; q++) mx[t] = bnh_fmax(mx[t], red[((t * WC + q) * WN + wn) * 16 + c16]);
  }
#pragma unroll
  for (int t = 0; t < TN; t++) {
    const int n = (t0 + t) * 16 + c16;
    if (wc == 0 && h == 0 && n < Np) colmax[win * cm_ws + n] = mx[t];
  }
}

template <bool WH>
static void ff_launch(const float *a, long long a_ws, int P, const bnh_fproto *W, float *colmax, long long cm_ws, int B,
                      bool over, hipStream_t st) {
  // The split with the least work on the fullest CU: its blocks there times the passes over the cells times a wave's
  // step (TC TN matrix instructions and about half of one for its operands). 64 cells x 1536 against 5000 prototypes:
  // 3 windows 4 cell tiles a wave 38 us, 2 by 2 waves 39, 1 by 4 waves 47 (281 us on the vector unit); one window 34, 23
  // and 25; 4 windows 57, 51 and 52; 16 windows against 12,000 321, 351 and 435.
  struct { int tc, wc, tn; } best = {4, 1, 1};
  static const struct { int tc, wc, tn; } plan[] = {{4, 1, 2}, {3, 1, 2}, {2, 1, 2}, {4, 1, 1}, {3, 1, 1},
                                                    {2, 1, 1}, {3, 2, 1}, {2, 2, 1}, {1, 2, 1}, {1, 4, 1}};
  double least = 0;
  for (const auto &p : plan) {
    if (over) {  // the first of the list: one block a window
      best = {p.tc, p.wc, p.tn};
      break;
    }
    const long long blocks = B * bnh_ceil_div(W->Np, 16 * p.tn * (4 / p.wc));
    // with four and more blocks a CU the registers of 6 and 8 tiles a wave leave too few waves to cover a block's start:
    // 64 windows of 64 cells against 20,000 fp32 prototypes, 2 x 2 tiles a wave for 4 x 2, K 64 251 -> 177 us, 200 441 -> 360,
    // 20 windows of K 1536 718 -> 666; fp16-stored ones, whose operands are half as wide, below K 256 only. What is left
    // to the vector unit's kernel before: K 64 160 us, K 8 73 against 122.
    if (blocks >= 1024 && (WH ? p.tc * p.tn == 8 && W->K <= 256 : p.tc * p.tn > 4)) continue;
    const double cost = (double)bnh_ceil_div(blocks, 256) * bnh_ceil_div(P, 16 * p.tc * p.wc) * (p.tc * p.tn + 0.5);
    if (least == 0 || cost < least) least = cost, best = {p.tc, p.wc, p.tn};
  }
#define FF_P(TC, WC, TN)                                                                                               \
  if (best.tc == TC && best.wc == WC && best.tn == TN)                                                                 \
  hipLaunchKernelGGL((k_colmax_f32<WH, TC, WC, TN>), dim3((unsigned)(B * bnh_ceil_div(W->Np, 16 * TN * (4 / WC)))),   \
                     dim3(256), 0, st, a, a_ws, P, W->K, (const void *)W->w, W->Np, colmax, cm_ws, B)
  FF_P(4, 1, 2);
  FF_P(3, 1, 2);
  FF_P(2, 1, 2);
  FF_P(4, 1, 1);
  FF_P(3, 1, 1);
  FF_P(2, 1, 1);
  FF_P(3, 2, 1);
  FF_P(2, 2, 1);
  FF_P(1, 2, 1);
  FF_P(1, 4, 1);
#undef FF_P
}

// ------------------------------------------------------------------ fp16 column maxima (kind 2)
#define HP_KC 32  // k steps per LDS stage
#define HP_AS 72  // As row stride in halves ([k][cell]; 16-byte aligned rows)
__global__ __launch_bounds__(256) void k_colmax_f16(const uint16_t *__restrict__ a, long long a_ws, int P, int K,
                                                    const uint16_t *__restrict__ w, int Npt, int Np, int bs, int nblk,
                                                    float *__restrict__ colmax, long long cm_ws, int B) {
  __shared__ __attribute__((aligned(16))) uint16_t As[2][HP_KC][HP_AS];
  __shared__ __attribute__((aligned(16))) uint4 Ws[2][HP_KC][FP_BN / 8];
  const int tid = threadIdx.x, cg = tid & 7, pg = tid >> 3;
  const int win = (int)(blockIdx.x % (unsigned)B), n0 = (int)(blockIdx.x / (unsigned)B) * FP_BN;
  const uint16_t *aw = a + win * a_ws;
  // loader roles: A, cell tid / 4 and k 8 (tid % 4) .. + 7; W rows (tid + 256 j) / 32, 8 prototypes each
  const int la_c = tid >> 2, la_k = 8 * (tid & 3);
  uint4 ra, rw[4];
  float mx[8];
#pragma unroll
  for (int j = 0; j < 8; j++) mx[j] = -INFINITY;
  for (int m0 = 0; m0 < P; m0 += FP_BM) {
    const int crow = m0 + la_c < P ? m0 + la_c : P - 1;
    const uint16_t *arow = aw + (long long)crow * K;
    auto load = [&](int k0) {
      ra = k0 + la_k < K ? *(const uint4 *)(arow + k0 + la_k) : make_uint4(0, 0, 0, 0);
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int i = tid + 256 * j, row = i >> 5, c8 = i & 31;
        rw[j] = k0 + row < K ? *(const uint4 *)(w + (long long)(k0 + row) * Npt + n0 + 8 * c8) : make_uint4(0, 0, 0, 0);
      }
    };
    auto store = [&](int buf) {
      const uint32_t v[4] = {ra.x, ra.y, ra.z, ra.w};
#pragma unroll
      for (int u = 0; u < 4; u++) {
        As[buf][la_k + 2 * u][la_c] = (uint16_t)(v[u] & 0xffffu);
        As[buf][la_k + 2 * u + 1][la_c] = (uint16_t)(v[u] >> 16);
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int i = tid + 256 * j, row = i >> 5, c8 = i & 31;
        Ws[buf][row][c8] = rw[j];
      }
    };
    h2 acc[8][4];
    float fb[8][8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
#pragma unroll
      for (int q = 0; q < 4; q++) acc[i][q] = (h2){(h16)0.0f, (h16)0.0f};
#pragma unroll
      for (int j = 0; j < 8; j++) fb[i][j] = 0.f;
    }
    __syncthreads();
    load(0);
    store(0);
    __syncthreads();
    int kend = bs < K ? bs : K;  // the end of the current K block
    for (int k0 = 0, cur = 0; k0 < K; k0 += HP_KC, cur ^= 1) {
      const bool more = k0 + HP_KC < K;
      if (more) load(k0 + HP_KC);
      const int kn = K - k0 < HP_KC ? K - k0 : HP_KC;  // a multiple of 8
      for (int kk = 0; kk < kn; kk += 8) {
#pragma unroll
        for (int k = kk; k < kk + 8; k++) {
          const uint4 av4 = *(const uint4 *)&As[cur][k][8 * cg];
          const uint4 wv4 = Ws[cur][k][pg];
          const h2 ap[4] = {__builtin_bit_cast(h2, av4.x), __builtin_bit_cast(h2, av4.y), __builtin_bit_cast(h2, av4.z),
                            __builtin_bit_cast(h2, av4.w)};
          const h2 wp[4] = {__builtin_bit_cast(h2, wv4.x), __builtin_bit_cast(h2, wv4.y), __builtin_bit_cast(h2, wv4.z),
                            __builtin_bit_cast(h2, wv4.w)};
#pragma unroll
          for (int i = 0; i < 8; i++) {
            const h16 ai = (i & 1) ? ap[i >> 1].y : ap[i >> 1].x;
            const h2 as = (h2){ai, ai};
#pragma unroll
            for (int q = 0; q < 4; q++) acc[i][q] = __builtin_elementwise_fma(wp[q], as, acc[i][q]);
          }
        }
        if (k0 + kk + 8 == kend) {  // a K block ends
          if (nblk > 1) {
#pragma unroll
            for (int i = 0; i < 8; i++)
#pragma unroll
              for (int q = 0; q < 4; q++) {
                fb[i][2 * q] = fb[i][2 * q] + (float)acc[i][q].x;
                fb[i][2 * q + 1] = fb[i][2 * q + 1] + (float)acc[i][q].y;
                acc[i][q] = (h2){(h16)0.0f, (h16)0.0f};
              }
          }
          kend = kend + bs < K ? kend + bs : K;
        }
      }
      if (more) store(cur ^ 1);
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 8; i++)
      if (m0 + 8 * cg + i < P)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const float lo = nblk > 1 ? fb[i][2 * q] : (float)acc[i][q].x;
          const float hi = nblk > 1 ? fb[i][2 * q + 1] : (float)acc[i][q].y;
          mx[2 * q] = bnh_fmax(mx[2 * q], lo);
          mx[2 * q + 1] = bnh_fmax(mx[2 * q + 1], hi);
        }
  }
#pragma unroll
  for (int j = 0; j < 8; j++) {
    mx[j] = bnh_fmax(mx[j], __shfl_xor(mx[j], 1));
    mx[j] = bnh_fmax(mx[j], __shfl_xor(mx[j], 2));
    mx[j] = bnh_fmax(mx[j], __shfl_xor(mx[j], 4));
  }
  float v = mx[0];
#pragma unroll
  for (int j = 1; j < 8; j++)
    if (cg == j) v = mx[j];
  const int n = n0 + 8 * pg + cg;
  if (n < Np) colmax[win * cm_ws + n] = v;
}

// ================================================================== host side
extern "C" {

bnh_fproto *bnh_fproto_new(int kind, int Np, int K, const void *w) {
  if (kind < 0 || kind > 2 || Np <= 0 || Np % 8 || K <= 0 || K % 8 || K > (1 << 20) || !w) {
    bnh_fail("bnh_fproto_new: kind %d Np %d K %d: expected kind 0..2, Np and K positive multiples of 8, K <= 2^20 and "
             "the prototype tensor", kind, Np, K);
    return nullptr;
  }
  const int Npt = (int)bnh_round_up(Np, FP_BN);
  const int K16 = (K + 15) / 16;
  const size_t esz = kind == 0 ? 4 : 2;
  const size_t bytes = (kind == 2 ? (size_t)K * Npt : (size_t)bnh_ceil_div(Np, 16) * K16 * 256) * esz;
  void *h = calloc(bytes, 1);
  bnh_fproto *W = (bnh_fproto *)calloc(1, sizeof *W);
  if (!h || !W) {
    free(h); free(W);
    bnh_fail("bnh_fproto_new: out of host memory");
    return nullptr;
  }
  const int n16 = Np / 16;
  for (int n = 0; n < Np; n++) {
    // the package panel holding prototype n and its column in the panel
    size_t base, step;
    if (kind < 2) {
      base = (size_t)(n / 8) * K * 8 + n % 8;  // [Np/8][K][8]
      step = 8;
    } else if (n / 16 < n16) {
      base = (size_t)(n / 16) * K * 16 + n % 16;  // [Np/16][K][16]
      step = 16;
    } else {
      base = (size_t)n16 * K * 16 + (n - 16 * n16);  // the tail panel [K][8]
      step = 8;
    }
    for (int k = 0; k < K; k++) {
      const size_t src = base + (size_t)k * step;
      const size_t dst = kind == 2 ? (size_t)k * Npt + n
                                   : (((size_t)(n / 16) * K16 + k / 16) * 64 + k % 4 * 16 + n % 16) * 4 + k % 16 / 4;
      if (esz == 4) ((float *)h)[dst] = ((const float *)w)[src];
      else ((uint16_t *)h)[dst] = ((const uint16_t *)w)[src];
    }
  }
  W->kind = kind; W->Np = Np; W->K = K; W->Npt = Npt;
  W->nblk = (K + 127) / 128;
  W->bs = ((K + W->nblk - 1) / W->nblk + 7) & ~7;
  const bool ok = (W->w = bnh_malloc(bytes)) && !bnh_memcpy_h2d(W->w, h, bytes);
  free(h);
  if (!ok) { bnh_fproto_free(W); return nullptr; }
  return W;
}

void bnh_fproto_free(bnh_fproto *W) {
  if (!W) return;
  if (W->w) (void)hipFree(W->w);
  free(W);
}

int bnh_l2norm_cells(const void *x, long long x_ws, int P, int C, int ld, float eps, int f16, void *a, long long a_ws,
                     int B, void *stream) {
  BNH_REQ(x && a && P > 0 && C > 0 && B > 0);
  BNH_REQ(C % 8 == 0 && ld >= C);
  BNH_REQ(B == 1 || (x_ws >= (long long)(P - 1) * ld + C && a_ws >= (long long)P * C));
  const long long cells = (long long)P * B;
  const uintptr_t mask = f16 ? 7 : 15;
  const bool vec = ((uintptr_t)x & mask) == 0 && ld % 4 == 0 && (B == 1 || x_ws % 4 == 0);
  const bool avec = ((uintptr_t)a & mask) == 0 && (B == 1 || a_ws % 4 == 0);
  auto launch = [&](auto nv) {
    constexpr int NV = decltype(nv)::value;
    hipLaunchKernelGGL((f16 ? k_l2norm<true, NV> : k_l2norm<false, NV>), dim3((unsigned)bnh_ceil_div(cells, 4)), dim3(256),
                       0, bnh_stream(stream), x, x_ws, P, C, ld, eps, a, a_ws, cells, vec, avec);
  };
  switch (cell_nv(C)) {
    case 1: launch(std::integral_constant<int, 1>{}); break;
    case 2: launch(std::integral_constant<int, 2>{}); break;
    case 4: launch(std::integral_constant<int, 4>{}); break;
    default: launch(std::integral_constant<int, 8>{});
  }
  BNH_HIP(hipGetLastError());
  return 0;
}

int bnh_fproto_colmax(const void *a, long long a_ws, int P, const bnh_fproto *W, float *colmax, long long cm_ws, int B,
                      void *stream) {
  BNH_REQ(a && W && colmax && P > 0 && B > 0);
  BNH_REQ(((uintptr_t)a & 15) == 0 && (B == 1 || a_ws % 8 == 0));
  BNH_REQ(B == 1 || (a_ws >= (long long)P * W->K && cm_ws >= W->Np));
  const long long blocks = (long long)B * (W->Npt / FP_BN);
  BNH_REQ(blocks < (1LL << 31));
  if (B == 1) a_ws = cm_ws = 0;
  if (W->kind == 2) {
    hipLaunchKernelGGL(k_colmax_f16, dim3((unsigned)blocks), dim3(256), 0, bnh_stream(stream), (const uint16_t *)a, a_ws,
                       P, W->K, (const uint16_t *)W->w, W->Npt, W->Np, W->bs, W->nblk, colmax, cm_ws, B);
  } else {
    // maxima over their cells: with one block a window, which has read all of them when it has passed its last barrier
    const bool over = bnh_overlap(bnh_windows(colmax, cm_ws, W->Np),
                                  bnh_windows((const float *)a, a_ws, (long long)P * W->K), B);
    BNH_REQ(!over || W->Np <= 128);
    // windows per launch such that its tiles of 16 prototypes stay under 2^23 (a grid dimension is limited in threads)
    const long long fit = (1LL << 23) / bnh_ceil_div(W->Np, 16);
    const int most = fit < 1 ? 1 : fit > B ? B : (int)fit;
    for (int b0 = 0; b0 < B; b0 += most) {
      const int nb = B - b0 < most ? B - b0 : most;
      const float *ab = (const float *)a + b0 * a_ws;
      if (W->kind == 1) ff_launch<true>(ab, a_ws, P, W, colmax + b0 * cm_ws, cm_ws, nb, over, bnh_stream(stream));
      else ff_launch<false>(ab, a_ws, P, W, colmax + b0 * cm_ws, cm_ws, nb, over, bnh_stream(stream));
      BNH_HIP(hipGetLastError());
    }
  }
  BNH_HIP(hipGetLastError());
  return 0;
}

}  // extern "C"
