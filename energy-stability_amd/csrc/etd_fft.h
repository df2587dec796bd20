// etd_fft.h -- the line FFT of the elastic path: register DFTs and the
// two-stage kernel, instantiated in etd_kernels.hip and etd_fft2.hip.
#ifndef ETD_FFT_H
#define ETD_FFT_H

#include <hip/hip_runtime.h>
#include <type_traits>

#include "etd_internal.h"

__device__ __forceinline__ size_t IDX(int n, int k, int j, int i) { return ((size_t)k * n + j) * n + i; }

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
// multiply by -i (sgn = +1, forward) or +i (sgn = -1, inverse)
__device__ __forceinline__ double2 cmi(double2 a, int sgn) {
  return sgn > 0 ? make_double2(a.y, -a.x) : make_double2(-a.y, a.x);
}

template <int R, int SGN>
__device__ __forceinline__ void dft_r(double2 *a) {
  if constexpr (R == 2) {
    double2 y0 = cadd(a[0], a[1]), y1 = csub(a[0], a[1]);
    a[0] = y0;
    a[1] = y1;
  } else if constexpr (R == 4) {
    double2 s02 = cadd(a[0], a[2]), d02 = csub(a[0], a[2]);
    double2 s13 = cadd(a[1], a[3]), d13 = cmi(csub(a[1], a[3]), SGN);
    a[0] = cadd(s02, s13);
    a[1] = cadd(d02, d13);
    a[2] = csub(s02, s13);
    a[3] = csub(d02, d13);
  } else if constexpr (R == 3) {
    const double h = 0.86602540378443864676;  // sin(2 pi / 3)
    double2 s = cadd(a[1], a[2]), d = csub(a[1], a[2]);
    double2 y0 = cadd(a[0], s);
    double2 t = make_double2(a[0].x - 0.5 * s.x, a[0].y - 0.5 * s.y);
    double2 id = cmi(make_double2(h * d.x, h * d.y), SGN);  // -i h d (forward)
    a[0] = y0;
    a[1] = cadd(t, id);
    a[2] = csub(t, id);
  } else {  // 5
    const double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;
    const double s1 = 0.95105651629515357212, s2 = 0.58778525229247312917;
    double2 b1 = cadd(a[1], a[4]), d1 = csub(a[1], a[4]);
    double2 b2 = cadd(a[2], a[3]), d2 = csub(a[2], a[3]);
    double2 y0 = cadd(a[0], cadd(b1, b2));
    double2 t1 = make_double2(a[0].x + c1 * b1.x + c2 * b2.x, a[0].y + c1 * b1.y + c2 * b2.y);
    double2 t2 = make_double2(a[0].x + c2 * b1.x + c1 * b2.x, a[0].y + c2 * b1.y + c1 * b2.y);
    // forward: y1 = t1 - i (s1 d1 + s2 d2), y4 = t1 + i(...); y2 = t2 - i (s2 d1 - s1 d2), y3 = t2 + i(...)
    double2 e1 = cmi(make_double2(s1 * d1.x + s2 * d2.x, s1 * d1.y + s2 * d2.y), SGN);
    double2 e2 = cmi(make_double2(s2 * d1.x - s1 * d2.x, s2 * d1.y - s1 * d2.y), SGN);
    a[0] = y0;
    a[1] = cadd(t1, e1);
    a[4] = csub(t1, e1);
    a[2] = cadd(t2, e2);
    a[3] = csub(t2, e2);
  }
}

// ---- two-stage line FFT for N = R1 R2 (R1, R2 <= 16 with factors 2, 3, 4, 5)
// x[n], n = n1 + R1 n2; Y[n1][k2] = sum_n2 x[n1 + R1 n2] W_R2^(n2 k2),
// times W_N^(n1 k2); X[k2 + R2 k1] = sum_n1 Y[n1][k2] W_R1^(n1 k1).  Both
// stages are DFTs in registers (composite sizes by one more split); the only
// LDS trip is the transpose between them, stored [line][k2][n1] with a
// one-element pad per k2 row and per line so that neither stage conflicts.
// A workgroup transforms 16 lines with max(R1, R2) threads each; lanes run
// along the line for the x axis and across lines (consecutive x) for y and z,
// so that global accesses cover whole 128-byte segments (for R1 = 16).
// R1 = 16 (N = 32 .. 256) is instantiated in etd_kernels.hip, the other edges
// in etd_fft2.hip.
template <int R, int SGN>
__device__ __forceinline__ void dft_any(double2 *a);

// (cos, sin) of 2 pi m / N, rounded once; a constant after unrolling.  The
// angle is taken within an eighth of a turn and in two parts: formed in one,
// 2 pi m / N is off by up to 4e-16, which every transform of that length then
// repeats (cos of a sixth of a turn came out as 0.5 + 1.1e-16).
template <int N>
__device__ __forceinline__ double2 turn(int m) {
  const double pi = 3.14159265358979323846, pi_lo = 1.22464679914735317723e-16;
  const int q = 4 * m / N % 4, r = 4 * m % N;  // quarter turns, and r / N of one
  double c, s;
  if (3 * r == N || 3 * r == 2 * N) {
    c = 0.86602540378443864676, s = 0.5;
  } else {
    const int k = 2 * r <= N ? r : N - r;
    const double p = pi * k, a = p / (2 * N);
    const double lo = (fma(-a, (double)(2 * N), p) + fma(pi, (double)k, -p) + pi_lo * k) / (2 * N);
    c = fma(-lo, sin(a), cos(a)), s = fma(lo, cos(a), sin(a));
  }
  if (2 * r > N) {
    const double t = c;
    c = s, s = t;
  }
  return q == 0 ? make_double2(c, s) : q == 1 ? make_double2(-s, c) : q == 2 ? make_double2(-c, -s) : make_double2(s, -c);
}

template <int A, int B, int SGN>
__device__ __forceinline__ void dft_split(double2 *x) {  // size A B, in place, natural order
  double2 y[A][B];
#pragma unroll
  for (int n1 = 0; n1 < A; n1++) {
    double2 t[B];
#pragma unroll
    for (int n2 = 0; n2 < B; n2++) t[n2] = x[n1 + A * n2];
    dft_any<B, SGN>(t);
#pragma unroll
    for (int k2 = 0; k2 < B; k2++) {
      if (n1 * k2 == 0) {
        y[n1][k2] = t[k2];
      } else {
        const double2 w = turn<A * B>(n1 * k2);
        y[n1][k2] = cmul(t[k2], make_double2(w.x, -SGN * w.y));
      }
    }
  }
#pragma unroll
  for (int k2 = 0; k2 < B; k2++) {
    double2 s[A];
#pragma unroll
    for (int n1 = 0; n1 < A; n1++) s[n1] = y[n1][k2];
    dft_any<A, SGN>(s);
#pragma unroll
    for (int k1 = 0; k1 < A; k1++) x[k2 + B * k1] = s[k1];
  }
}

template <int R, int SGN>
__device__ __forceinline__ void dft_any(double2 *a) {
  if constexpr (R == 1) {
  } else if constexpr (R == 2 || R == 3 || R == 4 || R == 5) {
    dft_r<R, SGN>(a);
  } else if constexpr (R == 16) {
    dft_split<4, 4, SGN>(a);
  } else if constexpr (R % 4 == 0) {
    dft_split<4, R / 4, SGN>(a);
  } else if constexpr (R % 3 == 0) {
    dft_split<3, R / 3, SGN>(a);
  } else if constexpr (R % 2 == 0) {
    dft_split<2, R / 2, SGN>(a);
  } else if constexpr (R % 5 == 0) {
    dft_split<5, R / 5, SGN>(a);
  }
}

constexpr int fft2_tpl(int R1, int R2) { return R1 > R2 ? R1 : R2; }
template <int R1, int R2>
struct fft2_cfg {
  static constexpr int N = R1 * R2;
  static constexpr int TPL = fft2_tpl(R1, R2);  // threads per line
  static constexpr int ROW = R1 + 1;          // one k2 row of Y (R1 n1 values + pad)
  static constexpr int LINE = R2 * ROW + 1;   // one line (+ pad)
  static constexpr int LDS = 16 * LINE * 16;  // bytes (double2)
};

// IO = 0: in place on data.  IO = 1 (forward x pass of an elastic
// evaluation): the input is read from the fields, eta_2r + i eta_2r+1 on the
// interior of the extended layout (the pack).  IO = 2 (inverse z pass): the
// output goes to the felas ring, real and imaginary parts to the slots of
// fields 2r and 2r+1, times 1/N^3 (the unpack); each value is rounded as the
// separate pack / unpack kernels round it.
// IO = 3, 4: the same with el_mix.  The pack forms the strain components
// 2r, 2r + 1 from every field; the three pairs of a group of lines go to one
// XCD one after another, so that the fields are read from HBM once (18 field
// passes of bytes for 12 fields: 250 us FP64, 159 us FP32 at N = 192, 4.1
// and 3.2 TB/s).  The unpack
// keeps what it overwrites on the box edges (edge_cell) for the next
// evaluation's lagged ghost cells.
struct fft_io {
  const void *u;
  void *E;
  int n, g, nac, ring, slot0;
  const double *ev;
};
// two or three coordinates of interior cell (x, y, z) lie within g of the box of edge N
__device__ __forceinline__ bool edge_cell(int x, int y, int z, int N, int g) {
  return (x < g || x >= N - g) + (y < g || y >= N - g) + (z < g || z >= N - g) >= 2;
}

template <int SGN, int R1, int R2, typename T2, int IO = 0>
__global__ __launch_bounds__(16 * fft2_tpl(R1, R2)) void k_fft2(T2 *data, size_t fs, int axis,
                                                                const double2 *__restrict__ tw, fft_io io) {
  using T = decltype(T2{}.x);
  using CF = fft2_cfg<R1, R2>;
  constexpr int N = CF::N, TPL = CF::TPL, ME = CF::N / CF::TPL;  // ME: elements per thread
  constexpr bool WHOLE = N * N % 128 == 0;  // groups of 16 lines are full and come in eights
  // the transpose between the stages holds FP32 pairs for FP32 data and R1 =
  // 16 (one rounding of the intermediate, within the FP32 transform's
  // accuracy; half the LDS, so twice the workgroups per CU) and FP64 pairs
  // otherwise
  using LT = typename std::conditional<sizeof(T2) == 8 && R1 == 16, float2, double2>::type;
  __shared__ LT buf[16 * CF::LINE];
  unsigned pr = blockIdx.y, bx = blockIdx.x;
  if constexpr (IO == 3) {  // gridDim.x = 3 groups, the groups rounded up to a multiple of 8
    const unsigned t = blockIdx.x >> 3;
    pr = t % 3;
    bx = t / 3 * 8 + (blockIdx.x & 7);
  }
  T2 *d = data + fs * pr;
  const int tid = threadIdx.x;
  const int ll = axis == 0 ? tid / TPL : tid & 15;  // line within the group
  const int j = axis == 0 ? tid % TPL : tid >> 4;   // thread within the line
  // The FP32 unpack writes each real field's row segment of 16 x as 64 bytes,
  // half a 128-byte line whose other half the next group of 16 lines writes.
  // Workgroups go to the 8 XCDs in turn and each XCD has its own L2, so there
  // each XCD takes a contiguous range of line groups (where gridDim.x = N^2 / 16
  // is a multiple of 8): both halves of a line meet in one L2.
  if constexpr ((IO == 2 || IO == 4) && sizeof(T2) == 8 && WHOLE) bx = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const unsigned L0 = bx * 16 + ll;
  const bool live = WHOLE || L0 < (unsigned)(N * N);  // the last group may be short
  const unsigned L = live ? L0 : 0;
  const unsigned x = L % N, o = L / N;
  const size_t base = axis == 0 ? (size_t)L * N : (axis == 1 ? x + (size_t)N * N * o : x + (size_t)N * o);
  const size_t stride = axis == 0 ? 1 : (axis == 1 ? (size_t)N : (size_t)N * N);
  LT *bl = buf + ll * CF::LINE;
  if (R1 == TPL || IO == 1 || IO == 3 || j < R1) {  // stage 1: thread n1 = j, DFT over n2 of x[n1 + R1 n2], twiddle, to LDS [k2][n1]
    const int n1 = j;
    double2 a[R2];
    if constexpr (IO == 1 || IO == 3) {
      // axis 0, pack: the group's 16 x rows of fields 2r and 2r+1 go to LDS
      // with consecutive threads on consecutive x (coalesced; the rows of the
      // extended layout start two ghost cells in), padded so that the strided
      // reads below take no extra bank passes
      constexpr int SP = N + R2;  // fits: the buffer holds 16 (N + R2 + 1) pairs
      static_assert(16 * SP * sizeof(T2) <= sizeof(buf), "staging fits the transpose buffer");
      T2 *stg = reinterpret_cast<T2 *>(buf);
      const T *u = (const T *)io.u;
      const size_t n3 = (size_t)io.n * io.n * io.n;
      const int pa = 2 * (int)pr, pb = pa + 1;
      // ME elements per thread, all loads issued before any store (the loop
      // is unrolled); a line past the last re-reads line 0
      T va[ME], vb[ME];
      if constexpr (IO == 3) {
        unsigned src[ME];
        double sa[ME], sb[ME];
#pragma unroll
        for (int k = 0; k < ME; k++) {
          const int e = tid + 16 * TPL * k, l2 = e / N, xx = e - l2 * N;
          const unsigned Lh = bx * 16 + l2, Lg = WHOLE || Lh < (unsigned)(N * N) ? Lh : 0;
          src[k] = (unsigned)IDX(io.n, (int)(Lg / N) + io.g, (int)(Lg % N) + io.g, xx + io.g);
          sa[k] = sb[k] = 0.0;
        }
        for (int q = 0; q < io.nac; q++) {
          const T *uq = u + n3 * q;
          const double ea = io.ev[6 * q + pa], eb = io.ev[6 * q + pb];
          T v[ME];
#pragma unroll
          for (int k = 0; k < ME; k++) v[k] = uq[src[k]];
#pragma unroll
          for (int k = 0; k < ME; k++) {
            sa[k] += ea * (double)v[k];
            sb[k] += eb * (double)v[k];
          }
        }
#pragma unroll
        for (int k = 0; k < ME; k++) {
          va[k] = (T)sa[k];
          vb[k] = (T)sb[k];
        }
      } else {
#pragma unroll
        for (int k = 0; k < ME; k++) {
          const int e = tid + 16 * TPL * k, l2 = e / N, xx = e - l2 * N;
          const unsigned Lh = bx * 16 + l2, Lg = WHOLE || Lh < (unsigned)(N * N) ? Lh : 0;
          const size_t src = IDX(io.n, (int)(Lg / N) + io.g, (int)(Lg % N) + io.g, xx + io.g);
          va[k] = u[n3 * pa + src];
          vb[k] = pb < io.nac ? u[n3 * pb + src] : (T)0;
        }
      }
#pragma unroll
      for (int k = 0; k < ME; k++) {
        const int e = tid + 16 * TPL * k, l2 = e / N, xx = e - l2 * N;
        T2 v;
        v.x = va[k];
        v.y = vb[k];
        stg[l2 * SP + xx] = v;
      }
      __syncthreads();
#pragma unroll
      for (int n2 = 0; n2 < R2; n2++) {
        const T2 v = stg[ll * SP + (R1 == TPL || n1 < R1 ? n1 : 0) + R1 * n2];
        a[n2] = make_double2(v.x, v.y);
      }
      __syncthreads();  // the transpose below reuses the buffer
    } else {
#pragma unroll
      for (int n2 = 0; n2 < R2; n2++) {
        const T2 v = d[base + (size_t)(n1 + R1 * n2) * stride];
        a[n2] = make_double2(v.x, v.y);
      }
    }
    dft_any<R2, SGN>(a);
    if (R1 == TPL || j < R1)
#pragma unroll
    for (int k2 = 0; k2 < R2; k2++) {
      double2 w = tw[(n1 * k2) % N];  // exp(-2 pi i n1 k2 / N)
      if (SGN < 0) w.y = -w.y;
      const double2 y = (n1 * k2 == 0) ? a[k2] : cmul(a[k2], w);
      LT v;
      v.x = y.x;
      v.y = y.y;
      bl[k2 * CF::ROW + n1] = v;
    }
  }
  __syncthreads();
  if ((R2 == TPL || j < R2) && live) {  // stage 2: thread k2 = j, DFT over n1, out X[k2 + R2 k1]
    const int k2 = j;
    double2 b[R1];
#pragma unroll
    for (int n1 = 0; n1 < R1; n1++) {
      const LT v = bl[k2 * CF::ROW + n1];
      b[n1] = make_double2(v.x, v.y);
    }
    dft_any<R1, SGN>(b);
#pragma unroll
    for (int k1 = 0; k1 < R1; k1++) {
      T2 v;
      v.x = b[k1].x;
      v.y = b[k1].y;
      const size_t m = base + (size_t)(k2 + R2 * k1) * stride;
      if constexpr (IO == 4) {
        const size_t N3 = (size_t)N * N * N;
        const double inv = 1.0 / ((double)N * N * N);
        T *E = (T *)io.E + (size_t)(2 * pr) * N3 + m;
        if (edge_cell((int)x, (int)o, k2 + R2 * k1, N, io.g)) {
          E[6 * N3] = E[0];
          E[7 * N3] = E[N3];
        }
        E[0] = (T)((double)v.x * inv);
        E[N3] = (T)((double)v.y * inv);
      } else if constexpr (IO == 2) {
        T *E = (T *)io.E;
        const size_t N3 = (size_t)N * N * N;
        const double inv = 1.0 / ((double)N * N * N);
        const int r = (int)pr;
        int sa = io.slot0 + 2 * r, sb = sa + 1;  // (slot0 + p) mod ring, p < nac < ring
        if (sa >= io.ring) sa -= io.ring;
        if (sb >= io.ring) sb -= io.ring;
        E[(size_t)sa * N3 + m] = (T)((double)v.x * inv);
        if (2 * r + 1 < io.nac) E[(size_t)sb * N3 + m] = (T)((double)v.y * inv);
      } else {
        d[m] = v;
      }
    }
  }
}

// edges with R1 < 16 (etd_fft2.hip); false where none is instantiated
template <int SGN, typename T2, int IO>
bool launch_fft2(etd_ctx *c, T2 *data, int npair, int axis, fft_io io);

#endif
