// Host-side tests for buffers of one call that share memory, for entry points whose blocks may run in any order.
#ifndef BNH_REGION_H
#define BNH_REGION_H
#include <stdint.h>

// a buffer's windows: n bytes each at a stride of ws bytes from p
struct bnh_region {
  long long p, ws, n;
};
template <typename T>
static inline bnh_region bnh_windows(const T *p, long long ws, long long per) {
  return {(long long)(uintptr_t)p, ws * (long long)sizeof(T), per * (long long)sizeof(T)};
}
// whether B windows of two buffers share a byte. Equal strides (each window's buffers side by side) are told apart
// window by window, unequal ones by the buffers' whole extents.
static inline bool bnh_overlap(const bnh_region &a, const bnh_region &b, int B) {
  if (B > 1 && a.ws == b.ws && a.ws > 0) {
    // some window k, |k| < B, of b relative to a: a - b - b.n < k ws < a - b + a.n
    const long long lo = a.p - b.p - b.n, hi = a.p - b.p + a.n;
    long long k = lo / a.ws - (lo % a.ws < 0) + 1;  // the first one above lo
    if (k <= -B) k = 1 - B;
    return k < B && k * a.ws < hi;
  }
  auto lo = [B](const bnh_region &r) { return r.p + (r.ws < 0 ? (B - 1) * r.ws : 0); };
  auto hi = [B](const bnh_region &r) { return r.p + (r.ws > 0 ? (B - 1) * r.ws : 0) + r.n; };
  return lo(a) < hi(b) && lo(b) < hi(a);
}
// elements of one window of an image or list of M pixel rows of ld elements, w pixels an image row, `pad` of halo
static inline long long bnh_rows_span(int M, int ld, int w, int pad) {
  return (pad ? (long long)(M / w + 2 * pad) * (w + 2 * pad) : M) * ld;
}
// whether two column ranges, na and nb elements wide, lie beside each other in rows of ld elements, a and b being
// theirs in the first row: with the same window stride they share nothing
template <typename T>
static inline bool bnh_beside(const T *a, long long na, const T *b, long long nb, long long ld) {
  const long long d = (long long)((intptr_t)b - (intptr_t)a) / (long long)sizeof(T);
  return (d >= na && d + nb <= ld) || (-d >= nb && -d + na <= ld);
}
#endif
