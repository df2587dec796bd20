// etd_fold.hip -- FP64 mode products of a basis whose modes are even or odd
// about the middle of the axis.
//
// The eigenvectors of the truncated second difference with the same kind of
// side at both ends (boundary ids 3 and 0) alternate in parity:
// V(n-1-i, m) = +-V(i, m), the sign changing from one mode to the next.  So
// with h = ceil(n / 2)
//   forward   out(m)     = sum_{k < h} A(m, k) (x(k) +- x(n-1-k))
//   backward  out(i)     = E(i) + O(i),  out(n-1-i) = E(i) - O(i),
//             E, O the sums of A(i, m) x(m) over the even and the odd modes:
// two half-size products in place of one, 2 n^4 -> n^4 flop per field pass.
// The full product is FP64-MFMA bound (n / 8 = 24.5 flop per byte at n = 196
// against a ridge of about 17 for what the copy kernel moves); the folded one
// sits at the ridge.  Measured, full against folded: n = 196, 13.5 fields a
// launch, 836 -> 521 us (38 TFLOP/s of the n^4 flop, 3.1 TB/s); n = 260, 4
// fields, 978 -> 442 us; n = 68, 4 fields, 12.0 -> 9.3 us; odd n = 49, 4
// fields, 18.6 -> 6.4 us.  Error against the exact product: 2.1e-16 to
// 3.1e-16 rms over n = 36 .. 100, 3.4e-16 to 4.5e-16 for the full one (half
// the terms).  Persistent workgroups (the next tile's first loads ahead of
// this tile's stores) spilled registers: 565 us at n = 196.
#include <hip/hip_runtime.h>
#include <float.h>
#include <math.h>
#include <string.h>

#include <type_traits>
#include <utility>

#include "etd_internal.h"

// ---- the rule
// forward: rows of A have alternating parity along k; backward: columns of A
// along the rows.  *first: the index of the first even mode (0 or 1).  The
// bound is what rounding leaves of the symmetry in a computed basis (angles
// up to 2 pi, an inversion: 6 eps for id 3, 67 eps for id 0 up to n = 272);
// bases read from files are symmetric to 1e-12 only and keep the full product.
// Even edges up to 32 keep the full product too: a launch is all it costs
// there (4 and 8 fields: 2.9 us full, 2.8 to 3.0 us folded at n = 12, 3.8
// against 3.2 to 3.4 us at n = 20; from n = 36 on 5.6 against 4.7 us and
// more).  The full product of an odd edge is the slow one at any size.
int fold_parity(int n, const double *A, int forward, int *first) {
  if (n < 8 || (n % 2 == 0 && n <= 32)) return 0;
  double big = 0.0;
  for (size_t l = 0; l < (size_t)n * n; l++) {
    if (!(fabs(A[l]) <= DBL_MAX)) return 0;
    big = fmax(big, fabs(A[l]));
  }
  const double tol = 128 * DBL_EPSILON * big;
  for (int e0 = 0; e0 < ((n & 1) ? 1 : 2); e0++) {
    int ok = 1;
    for (int m = 0; m < n && ok; m++) {
      const double s = (m & 1) == e0 ? 1.0 : -1.0;
      for (int k = 0; k < (n + 1) / 2 && ok; k++) {
        const double a = forward ? A[m + (size_t)n * k] : A[k + (size_t)n * m];
        const double b = forward ? A[m + (size_t)n * (n - 1 - k)] : A[n - 1 - k + (size_t)n * m];
        if (fabs(a - s * b) > tol) ok = 0;
      }
    }
    if (ok) {
      *first = e0;
      return 1;
    }
  }
  return 0;
}

// rows and K steps per parity: h of them, rows in two halves of RT tiles of 4
static int fold_rt(int n) { return ((n + 1) / 2 + 7) / 8; }
static int fold_chunks(int n) { return ((n + 1) / 2 + 15) / 16; }
// doubles of one chunk: 2 parities x 16 k x 8 RT rows, rounded up to whole 16-byte pieces for 256 threads
static constexpr int fold_chunk(int RT) { return (256 * RT + 511) / 512 * 512; }
size_t fold_A_doubles(int n) { return (size_t)fold_chunks(n) * fold_chunk(fold_rt(n)); }

// Af[kc][parity][k % 16][row], zero outside h x h; each entry the mean of the
// two it stands for
void arrange_fold_A(int n, const double *A, int forward, int e0, double *Af) {
  const int R = 8 * fold_rt(n), h = (n + 1) / 2;
  memset(Af, 0, sizeof(double) * fold_A_doubles(n));
  for (int par = 0; par < 2; par++) {
    const double s = par ? -1.0 : 1.0;
    for (int j = 0; j < h; j++) {
      const int m = (par ? 1 - e0 : e0) + 2 * j;
      if (m >= n) continue;
      for (int i = 0; i < h; i++) {
        if (2 * i + 1 == n && par) continue;  // an odd mode vanishes on the middle
        const double a = forward ? A[m + (size_t)n * i] : A[i + (size_t)n * m];
        const double b = forward ? A[m + (size_t)n * (n - 1 - i)] : A[n - 1 - i + (size_t)n * m];
        const int k = forward ? i : j, row = forward ? j : i;
        Af[(size_t)(k / 16) * fold_chunk(R / 8) + (par * 16 + k % 16) * R + row] = 0.5 * (a + s * b);
      }
    }
  }
}

// ---- the kernel
// A workgroup owns 64 columns and every row; wave w takes parity w % 2 and
// the row half w / 2, RT tiles of 4 rows by 4 tiles of 16 columns.
// v_mfma_f64_4x4x4f64 (1.5x the rate of the 16x16x4 form here) holds four
// 4x4x4 products; they are stacked along the columns, so that rows come in
// fours and little is padded: lane = x + 4 blk + 16 y holds A(row x, k y),
// B(k y, column 4 blk + x) and D(row y, column 4 blk + x).
//
// Chunks of 16 k pass through registers on their way to LDS: the fold (or,
// backward, the sorting by parity) happens once per element there, and the
// next chunk's loads fly during this chunk's products.  One LDS stage and two
// workgroups per CU, so one's barriers and epilogue hide behind the other's
// products; a second stage would leave room for one workgroup only.
// LDS row pads: columns 64 + 2 keeps the staging writes off each other's
// banks, both operands are then read as 16-byte pairs without conflicts
// (the A pair is two row tiles' rows, the B pair two column tiles' columns).
#define FOLD_COLS 64
#define FOLD_BROW (FOLD_COLS + 2)

template <int RT>
struct fold_cfg {
  static constexpr int R = 8 * RT;                     // rows per parity
  static constexpr int A_DBL = fold_chunk(RT);         // A chunk
  static constexpr int B_DBL = 2 * 16 * FOLD_BROW;     // folded columns of a chunk
  static constexpr int X_DBL = 2 * RT * 2 * 64 * 2;    // one round of the backward exchange (two row halves)
  static constexpr int LDS = 8 * (A_DBL + B_DBL);
  static constexpr int APT = A_DBL / 512;              // 16-byte A pieces per thread and chunk
};

template <int RT, bool EVEN, bool FWD>
__global__ __launch_bounds__(256, 2) void k_modeprod_fold(const double *__restrict__ Af, const double *__restrict__ in,
                                                          size_t in_fs, double *__restrict__ out, size_t out_fs, int n,
                                                          int e0, int accumulate) {
  using CF = fold_cfg<RT>;
  extern __shared__ __attribute__((aligned(16))) double sm[];
  double *sA = sm, *sB = sm + CF::A_DBL;
  const int tid = threadIdx.x, lane = tid & 63;
  const int par = (tid >> 6) & 1, half = tid >> 7;
  const double *src = in + in_fs * blockIdx.y;
  double *dst = out + out_fs * blockIdx.y;
  const int n2 = n * n, h = (n + 1) >> 1;
  const int nkc = (h + 15) >> 4;
  const int col0 = blockIdx.x * FOLD_COLS;

  // staging: this thread's column and its group of 4 k of each chunk
  const int scol = tid >> 2, kq = tid & 3;
  const bool colok = col0 + scol < n2;
  const double *sp = src + (size_t)n * (colok ? col0 + scol : 0);
  // what the loads of a chunk bring, in one vector register tuple each (an
  // array is kept in scratch memory): every load is unconditional, from a
  // clamped address, and what lies outside is zeroed on the way to LDS, so
  // nothing waits for the loads before the products
  typedef double v8d __attribute__((ext_vector_type(8)));
  v8d xr;
  typedef double stage_t __attribute__((ext_vector_type(2 * CF::APT)));
  stage_t ap;
  constexpr auto AIDX = std::make_index_sequence<CF::APT>{};
  auto fetch_a = [&](int kc, auto seq) {
    const double2 *g = reinterpret_cast<const double2 *>(Af) + (size_t)kc * (CF::A_DBL / 2) + tid;
    [&]<size_t... I>(std::index_sequence<I...>) {
      ((ap[2 * I] = g[256 * I].x, ap[2 * I + 1] = g[256 * I].y), ...);
    }(seq);
  };
  auto store_a = [&](auto seq) {
    [&]<size_t... I>(std::index_sequence<I...>) {
      ((reinterpret_cast<double2 *>(sA)[tid + 256 * I] = make_double2(ap[2 * I], ap[2 * I + 1])), ...);
    }(seq);
  };
  auto fetch = [&](int kc) {
    fetch_a(kc, AIDX);
    const int k0 = 16 * kc + 4 * kq;
    if constexpr (FWD) {  // x(k0 .. k0+3), then x(n-4-k0 .. n-1-k0); inside the column for k0 < h, n >= 8
      const int kk = k0 < h ? k0 : 0;
      const double *a = sp + kk, *b = sp + (n - 4 - kk);
      if constexpr (EVEN) {
        const double2 a0 = *(const double2 *)a, a1 = *(const double2 *)(a + 2);
        const double2 b0 = *(const double2 *)b, b1 = *(const double2 *)(b + 2);
        xr = (v8d){a0.x, a0.y, a1.x, a1.y, b0.x, b0.y, b1.x, b1.y};
      } else {
        xr = (v8d){a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
      }
    } else {  // modes 2 k0 .. 2 k0 + 7
      const int m = 2 * k0;
      if constexpr (EVEN) {
        const double2 t0 = *(const double2 *)(sp + (m < n ? m : 0)), t1 = *(const double2 *)(sp + (m + 2 < n ? m + 2 : 0));
        const double2 t2 = *(const double2 *)(sp + (m + 4 < n ? m + 4 : 0)),
                      t3 = *(const double2 *)(sp + (m + 6 < n ? m + 6 : 0));
        xr = (v8d){t0.x, t0.y, t1.x, t1.y, t2.x, t2.y, t3.x, t3.y};
      } else {
        auto at = [&](int i) { return sp[m + i < n ? m + i : 0]; };
        xr = (v8d){at(0), at(1), at(2), at(3), at(4), at(5), at(6), at(7)};
      }
    }
  };
  auto store = [&](int kc) {
    store_a(AIDX);
    double *w = sB + 4 * kq * FOLD_BROW + scol;
    auto one = [&](auto ic) {
      constexpr int i = decltype(ic)::value;
      const int k = 16 * kc + 4 * kq + i;
      double ev, od;
      if constexpr (FWD) {
        const double a = xr[i], b = xr[7 - i];
        const bool ok = colok && k < h;
        ev = ok ? (!EVEN && 2 * k + 1 == n ? a : a + b) : 0.0;  // the middle stands for itself
        od = ok ? a - b : 0.0;
      } else {
        const double p0 = colok && 2 * k < n ? xr[2 * i] : 0.0, p1 = colok && 2 * k + 1 < n ? xr[2 * i + 1] : 0.0;
        ev = e0 ? p1 : p0;
        od = e0 ? p0 : p1;
      }
      w[i * FOLD_BROW] = ev;
      w[(16 + i) * FOLD_BROW] = od;
    };
    one(std::integral_constant<int, 0>{});
    one(std::integral_constant<int, 1>{});
    one(std::integral_constant<int, 2>{});
    one(std::integral_constant<int, 3>{});
  };

  const int x = lane & 3, y = lane >> 4, c16 = lane & 15;
  const double *ra = sA + (par * 16 + y) * CF::R + half * 4 * RT + 2 * x;
  const double *rb = sB + (par * 16 + y) * FOLD_BROW + 2 * c16;

  double acc[RT][4];
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int u = 0; u < 4; u++) acc[t][u] = 0.0;
  fetch(0);
  for (int kc = 0; kc < nkc; kc++) {
    if (kc) __syncthreads();  // every wave is done with the stage
    store(kc);
    __syncthreads();
    if (kc + 1 < nkc) fetch(kc + 1);
    const int left = (h - 16 * kc + 3) >> 2;  // K steps of 4 in this chunk
#pragma unroll
    for (int s = 0; s < 4; s++) {
      if (s >= left) break;
      double a[RT], b[4];
#pragma unroll
      for (int t = 0; t + 1 < RT; t += 2) {
        const double2 v = *(const double2 *)(ra + 4 * s * CF::R + 4 * t);
        a[t] = v.x, a[t + 1] = v.y;
      }
      if constexpr (RT & 1) a[RT - 1] = *(ra + 4 * s * CF::R + 4 * (RT - 1) - x);
#pragma unroll
      for (int u = 0; u < 4; u += 2) {
        const double2 v = *(const double2 *)(rb + 4 * s * FOLD_BROW + 16 * u);
        b[u] = v.x, b[u + 1] = v.y;
      }
#pragma unroll
      for (int t = 0; t < RT; t++)
#pragma unroll
        for (int u = 0; u < 4; u++) acc[t][u] = __builtin_amdgcn_mfma_f64_4x4x4f64(a[t], b[u], acc[t][u], 0, 0, 0);
    }
  }

  // row of tile t in this lane (pairs of tiles interleave their rows), and
  // the first of its two columns of column tiles u, u + 1
  auto row_of = [&](int t) { return half * 4 * RT + ((RT & 1) && t == RT - 1 ? 4 * t + y : 4 * (t & ~1) + 2 * y + (t & 1)); };
  auto put = [&](int r, int u, double v0, double v1) {
    const int col = col0 + 16 * u + 2 * c16;
    double *o = dst + (size_t)n2 * r + col;
    if constexpr (EVEN) {  // n^2 even: both columns or none, 16-byte aligned
      if (col < n2) {
        double2 v = make_double2(v0, v1);
        if (accumulate) {
          const double2 w = *(const double2 *)o;
          v.x += w.x, v.y += w.y;
        }
        *(double2 *)o = v;
      }
    } else {
      if (col < n2) o[0] = accumulate ? o[0] + v0 : v0;
      if (col + 1 < n2) o[1] = accumulate ? o[1] + v1 : v1;
    }
  };
  if constexpr (FWD) {
    const int m0 = par ? 1 - e0 : e0;
#pragma unroll
    for (int t = 0; t < RT; t++) {
      const int m = m0 + 2 * row_of(t);
      if (m < n)
#pragma unroll
        for (int u = 0; u < 4; u += 2) put(m, u, acc[t][u], acc[t][u + 1]);
    }
  } else {
    // The even and the odd wave of a row half hold E and O of the same
    // elements: each hands the other half of its column tiles over and
    // writes both rows of the ones it keeps.  One LDS round of X_DBL doubles
    // when that fits the stage, else two.
    constexpr int ROUNDS = CF::X_DBL <= CF::A_DBL + CF::B_DBL ? 1 : 2;
    constexpr int TR = (RT + ROUNDS - 1) / ROUNDS;  // row tiles per round
    static_assert(2 * 2 * TR * 2 * 64 <= CF::A_DBL + CF::B_DBL, "exchange");
    double *mine = sm + (size_t)(half * 2 + par) * (TR * 2 * 64) + lane * 2;
    const double *theirs = sm + (size_t)(half * 2 + (par ^ 1)) * (TR * 2 * 64) + lane * 2;
#pragma unroll
    for (int r = 0; r < ROUNDS; r++) {
      __syncthreads();
#pragma unroll
      for (int t = r * TR; t < RT && t < (r + 1) * TR; t++) {
        const double2 give = par ? make_double2(acc[t][0], acc[t][1]) : make_double2(acc[t][2], acc[t][3]);
        *(double2 *)(mine + (t - r * TR) * 128) = give;
      }
      __syncthreads();
#pragma unroll
      for (int t = r * TR; t < RT && t < (r + 1) * TR; t++) {
        const double2 o = *(const double2 *)(theirs + (t - r * TR) * 128);
        // par 0 keeps tiles 0, 1 (its E, the other's O); par 1 keeps tiles 2, 3
        const double E0 = par ? o.x : acc[t][0], E1 = par ? o.y : acc[t][1];
        const double O0 = par ? acc[t][2] : o.x, O1 = par ? acc[t][3] : o.y;
        const int i = row_of(t), u = par ? 2 : 0;
        if (i < h) {
          put(i, u, E0 + O0, E1 + O1);
          if (EVEN || 2 * i + 1 != n) put(n - 1 - i, u, E0 - O0, E1 - O1);
        }
      }
    }
  }
}

template <int RT, bool EVEN, bool FWD>
static void fold_go(etd_ctx *c, const double *Af, const double *in, size_t in_fs, double *out, size_t out_fs,
                    int nfields, int e0, int accumulate) {
  using CF = fold_cfg<RT>;
  // two workgroups per CU, and what a launch may ask for without an attribute set on every device first
  static_assert(2 * CF::LDS <= 160 * 1024 && CF::LDS <= 64 * 1024, "LDS");
  const dim3 grid((unsigned)((c->n * c->n + FOLD_COLS - 1) / FOLD_COLS), nfields);
  k_modeprod_fold<RT, EVEN, FWD><<<grid, 256, CF::LDS, c->stream>>>(Af, in, in_fs, out, out_fs, c->n, e0, accumulate);
}

void launch_modeprod_fold(etd_ctx *c, const double *Af, int forward, int e0, const double *in, size_t in_fs,
                          double *out, size_t out_fs, int nfields, int accumulate) {
  etd_prof_begin(c, PC_MODEPROD);
  auto go = [&](auto rt) {
    constexpr int RT = decltype(rt)::value;
    if (c->n % 2 == 0) {
      if (forward) fold_go<RT, true, true>(c, Af, in, in_fs, out, out_fs, nfields, e0, accumulate);
      else fold_go<RT, true, false>(c, Af, in, in_fs, out, out_fs, nfields, e0, accumulate);
    } else {
      if (forward) fold_go<RT, false, true>(c, Af, in, in_fs, out, out_fs, nfields, e0, accumulate);
      else fold_go<RT, false, false>(c, Af, in, in_fs, out, out_fs, nfields, e0, accumulate);
    }
  };
  switch (fold_rt(c->n)) {
#define RTC(X) case X: go(std::integral_constant<int, X>{}); break;
    RTC(1) RTC(2) RTC(3) RTC(4) RTC(5) RTC(6) RTC(7) RTC(8) RTC(9) RTC(10) RTC(11) RTC(12) RTC(13) RTC(14) RTC(15)
    RTC(16) RTC(17)
#undef RTC
    default: break;
  }
  etd_prof_end(c, PC_MODEPROD);
}
