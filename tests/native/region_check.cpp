// bnh_overlap and bnh_beside (csrc/bnh_region.h) against the bytes themselves: two buffers of B windows, every pair of
// small strides, lengths and offsets, marked byte by byte; the exact answer where the strides are equal or there is one
// window, and no overlap missed where they differ.
#include <stdio.h>
#include <string.h>

#include "bnh_region.h"

static int bytes_shared(long long pa, long long wa, long long na, long long pb, long long wb, long long nb, int B) {
  static char mark[512];
  memset(mark, 0, sizeof mark);
  for (int w = 0; w < B; w++)
    for (long long i = 0; i < na; i++) mark[128 + pa + w * wa + i] = 1;
  for (int w = 0; w < B; w++)
    for (long long i = 0; i < nb; i++)
      if (mark[128 + pb + w * wb + i]) return 1;
  return 0;
}

int main() {
  long long checked = 0, wrong = 0;
  for (int B = 1; B <= 4; B++)
    for (int wa = -3; wa <= 9; wa++)
      for (int wb = -3; wb <= 9; wb++)
        for (int na = 1; na <= 8; na++)
          for (int nb = 1; nb <= 8; nb++)
            for (int d = -40; d <= 40; d++) {
              const char *p = (const char *)4096;
              const bool got = bnh_overlap(bnh_windows(p, wa, na), bnh_windows(p + d, wb, nb), B);
              const int is = bytes_shared(0, wa, na, d, wb, nb, B);
              const bool exact = B == 1 || (wa == wb && wa > 0);
              wrong += exact ? got != (is != 0) : is && !got;
              checked++;
            }
  // columns of the same rows: M rows of ld, one window
  for (int ld = 1; ld <= 8; ld++)
    for (int na = 1; na <= ld; na++)
      for (int nb = 1; nb <= ld; nb++)
        for (int d = -12; d <= 12; d++)
          for (int M = 1; M <= 3; M++) {
            const float *p = (const float *)4096;
            const int is = bytes_shared(0, ld, na, d, ld, nb, M);
            wrong += bnh_beside(p, na, p + d, nb, ld) && is;          // never where they share
            wrong += !bnh_beside(p, na, p + d, nb, ld) && !is && M > 1 && d > -ld && d < ld;  // always where they lie so
            checked++;
          }
  printf("checked %lld mismatches %lld\n", checked, wrong);
  return wrong != 0;
}
