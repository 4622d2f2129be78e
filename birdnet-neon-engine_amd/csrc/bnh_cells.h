// A wave's pass over one cell of a prototype head: its C values (fp32, or fp16 widened; C % 8 == 0) and the sum of
// their squares as libbnneon's kernels form it (pc_quant_cells_f32, pc_l2norm_f32): 8 fused chains, channel c in chain
// c % 8 in order of c, combined as ((t0 + t1) + (t2 + t3)) with t_j = chain_j + chain_{j + 4}.
//
// A cell is a memory round trip and a serial chain of C / 8 steps, nothing else: 256 NV values are fetched at once into
// registers (lane l holds values 4 l .. 4 l + 3 of each 256), laid out chain by chain in LDS, and lanes 0..7 read four
// steps of their chains at a time. Fetched 64 at a time with an LDS read per step, 1280 cells x 1536 took 26.7 us and
// 192 cells 22.5; the whole head of one window (64 cells, 59,180 int8 prototypes) went from 50.9 to 36.3 us, the fp32
// head of 3 windows against 5000 from 57.5 to 45.5. NV as C needs it, at most 8: the registers, LDS and code for 2048
// values cost cells of fewer their occupancy (16,384 cells x 64 to int8 11.0 us fetched 64 at a time, 25.3 with NV 8,
// 10.3 with NV 1; 8192 x 360 11.4, 16.4, 9.7 with NV 2).
#ifndef BNH_CELLS_H
#define BNH_CELLS_H
#include "bnh_f16.h"
#include "bnh_num.h"

// NV for cells of C values
static inline int cell_nv(int C) { return C <= 256 ? 1 : C <= 512 ? 2 : C <= 1024 ? 4 : 8; }

template <int NV>
struct Cell {
  static constexpr int CH = 256 * NV;    // values in registers at a time
  static constexpr int LS = CH / 8 + 4;  // floats of a chain in LDS
  float4 v[NV];
  // values c0 .. c0 + CH - 1 of row x, zeros past C; vec: the row is 16-byte (fp16: 8-byte) aligned
  template <bool F16>
  BNH_DEV void load(const void *x, int c0, int C, bool vec, int lane) {
#pragma unroll
    for (int j = 0; j < NV; j++) {
      const int c = c0 + 256 * j + 4 * lane;
      v[j] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (c >= C) continue;
      if (F16) {
        const uint16_t *r = (const uint16_t *)x + c;
        uint2 u;
        if (vec) u = *(const uint2 *)r;
        else u = make_uint2(r[0] | (uint32_t)r[1] << 16, r[2] | (uint32_t)r[3] << 16);
        v[j] = make_float4((float)hfrom((uint16_t)(u.x & 0xffffu)), (float)hfrom((uint16_t)(u.x >> 16)),
                           (float)hfrom((uint16_t)(u.y & 0xffffu)), (float)hfrom((uint16_t)(u.y >> 16)));
      } else {
        const float *r = (const float *)x + c;
        if (vec) v[j] = *(const float4 *)r;
        else v[j] = make_float4(r[0], r[1], r[2], r[3]);
      }
    }
  }
  // lane l < 8: chain l continued over the n values held; the whole block calls it (s: 8 LS floats a wave)
  BNH_DEV float squares(float chain, int n, float *s, int lane) const {
#pragma unroll
    for (int j = 0; j < NV; j++) {
      float *d = s + 4 * (lane & 1) * LS + 32 * j + (lane >> 1);
      d[0] = v[j].x, d[LS] = v[j].y, d[2 * LS] = v[j].z, d[3 * LS] = v[j].w;
    }
    __syncthreads();
    if (lane < 8) {
      const float *r = s + lane * LS;
      const int steps = n / 8;
      int i = 0;
      for (; i + 32 <= steps; i += 32) {
        float4 q[8];
#pragma unroll
        for (int u = 0; u < 8; u++) q[u] = *(const float4 *)(r + i + 4 * u);
#pragma unroll
        for (int u = 0; u < 8; u++) {
          chain = __builtin_fmaf(q[u].x, q[u].x, chain);
          chain = __builtin_fmaf(q[u].y, q[u].y, chain);
          chain = __builtin_fmaf(q[u].z, q[u].z, chain);
          chain = __builtin_fmaf(q[u].w, q[u].w, chain);
        }
      }
      for (; i < steps; i++) chain = __builtin_fmaf(r[i], r[i], chain);
    }
    __syncthreads();
    return chain;
  }
};
// sqrtf of the sum the chains of lanes 0..7 combine to
BNH_DEV float cell_norm(float chain, int lane) {
  const float s1 = __shfl(chain, (lane & 3) + 4);
  const float t = chain + s1;  // t_j in lanes 0..3
  const float t0 = __shfl(t, 0), t1 = __shfl(t, 1), t2 = __shfl(t, 2), t3 = __shfl(t, 3);
  return __builtin_sqrtf((t0 + t1) + (t2 + t3));
}
#endif
