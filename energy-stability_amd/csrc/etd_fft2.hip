// etd_fft2.hip -- the two-stage line FFT (etd_fft.h) for elastic grids whose
// edge is no 16 R2: N = R1 R2 with R1 and R2 as near as they go (R2 <= R1 <=
// 15), which leaves few idle threads and few registers.  The radix passes
// (k_fft_axis) take one LDS round trip and barrier per radix and, for x, y
// and z alike, separate pack and unpack kernels; they stay for edges with no
// such pair (16, 125, 162, 200 and the smallest).
#include "etd_fft.h"

#define FFT2_EDGES(X)                                                                                             \
  X(18, 6, 3) X(20, 5, 4) X(24, 6, 4) X(25, 5, 5) X(27, 9, 3) X(30, 6, 5) X(36, 6, 6) X(40, 8, 5) X(45, 9, 5)     \
  X(50, 10, 5) X(54, 9, 6) X(60, 10, 6) X(72, 9, 8) X(75, 15, 5) X(81, 9, 9) X(90, 10, 9) X(100, 10, 10)          \
  X(108, 12, 9) X(120, 12, 10) X(135, 15, 9) X(150, 15, 10) X(180, 15, 12)

// N has a two-stage transform, here or with R1 = 16
bool fft2_supported(int N) {
  switch (N) {
#define X(E, A, B) case E:
    FFT2_EDGES(X)
#undef X
    return true;
    default: return fft16_supported(N);
  }
}

template <int SGN, typename T2, int IO>
bool launch_fft2(etd_ctx *c, T2 *data, int npair, int axis, fft_io io) {
  const unsigned groups = (unsigned)(((size_t)c->Ne * c->Ne + 15) / 16);
  const dim3 grid = IO == 3 ? dim3(3 * ((groups + 7) / 8 * 8)) : dim3(groups, npair);  // IO 3: npair is 3
  const double2 *tw = (const double2 *)c->tw;
  switch (c->Ne) {
#define X(E, A, B)                                                                                                 \
  case E:                                                                                                          \
    k_fft2<SGN, A, B, T2, IO><<<grid, 16 * (A > B ? A : B), 0, c->stream>>>(data, c->Ne3, axis, tw, io);           \
    return true;
    FFT2_EDGES(X)
#undef X
    default: return false;
  }
}

#define INST(T2)                                                          \
  template bool launch_fft2<1, T2, 0>(etd_ctx *, T2 *, int, int, fft_io); \
  template bool launch_fft2<1, T2, 1>(etd_ctx *, T2 *, int, int, fft_io); \
  template bool launch_fft2<1, T2, 3>(etd_ctx *, T2 *, int, int, fft_io); \
  template bool launch_fft2<-1, T2, 0>(etd_ctx *, T2 *, int, int, fft_io); \
  template bool launch_fft2<-1, T2, 2>(etd_ctx *, T2 *, int, int, fft_io); \
  template bool launch_fft2<-1, T2, 4>(etd_ctx *, T2 *, int, int, fft_io);
INST(float2)
INST(double2)
