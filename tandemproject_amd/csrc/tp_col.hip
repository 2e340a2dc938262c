// tp_col.hip -- compact line solves with one lane per line and one wave per
// chunk of the line.
//
// Arithmetic of src/Subroutines3D.f90:84-141 (deriv) and :145-206 (filte):
// pentadiagonal RHS, forward substitution with the factors xl (penta,
// src/Subroutineso.f90), backward substitution with xu, in the reference's
// operation order.
//
// Layout of the work: a workgroup owns 64 adjacent lines (one per lane) of one
// sub-block; its P waves own consecutive chunks of ceil(L/P) points of those
// lines.  For eta and zeta lines the 64 lanes read and write 64 consecutive
// doubles of each row (the lines are adjacent in xi), so no staging is needed;
// xi lines are contiguous rows: their windows come through a small per-wave
// LDS transpose in pieces of 8 points, and their results are gathered in LDS
// and stored by the whole workgroup as contiguous runs of rows.  The factors
// of a row are the same for every lane and are read from LDS as broadcasts.
//
// Each wave keeps its chunk in registers and runs:
//   forward sweep from zero carries -> the pair (y[e-1], y[e]) that is an
//     affine function of the true incoming pair (its 2x2 matrix depends on
//     the factors only: tabulated per block, direction, kind and P);
//   composition of those maps over the preceding chunks -> the true carries;
//   forward sweep from the true carries (the reference's recurrence), and the
//   same three steps backwards.
// The carries come out of the composition rounded differently from the
// sequential sweep (~1 ulp).  Inside a chunk that difference decays by ~0.74
// per point, but the two roundings re-synchronise only by chance, and the
// last rows of a one-sided closure amplify whatever ulp difference is left
// (|l2| ~ 72 in the last row, |u2|, |u3| ~ 6 in the first rows).  So near such
// an end the chunks take their carries in a chain instead: each from the
// sweep its neighbour just finished, over at least COL_DECAY points, which
// in practice brings the end rows back to the sequential sweep's bits.
#include "tp_internal.hpp"

namespace tp {

template <int D>
__device__ inline void col_line(const Block &b, int q, int &base, int &jk) {
  if (D == 0) {            // q = zeta*ny + eta
    base = q * b.nx; jk = q;
  } else if (D == 1) {     // q = zeta*nx + xi, face index xi*nz + zeta
    const int xi = q % b.nx, ze = q / b.nx;
    base = ze * b.ny * b.nx + xi; jk = xi * b.nz + ze;
  } else {                 // q = eta*nx + xi
    base = q; jk = q;
  }
}

// element at a 32-bit byte offset from a wave-uniform base: lets the loads and
// stores use the scalar-base + 32-bit vector-offset addressing form
__device__ inline const double &at(const double *base, unsigned off) {
  return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(base) + off);
}
__device__ inline double &at(double *base, unsigned off) {
  return *reinterpret_cast<double *>(reinterpret_cast<char *>(base) + off);
}
// a xi output value, stored with the streaming hint
__device__ inline void st(double *base, unsigned off, double v) { st_stream(&at(base, off), v); }

// strided view of one line in global memory (boundary rows)
struct GLine {
  const double *p;
  int s;
  __device__ double operator()(int i) const { return p[(size_t)i * s]; }
};

// closure sums r0, r1, r2 of one face: read from the exchange's recv slots
// where they are used, or held as values
struct RcvFace {
  const double *rcv;
  int F, jk, ip;
  __device__ double operator()(int q) const { return rcv[(ip * 3 + q) * F + jk]; }
};
struct ValFace {
  double r[3];
  // a select, not an index: q may be known only at run time, and an indexed
  // register array would go to scratch memory
  __device__ double operator()(int q) const { return q == 0 ? r[0] : q == 1 ? r[1] : r[2]; }
};

// boundary rows of the derivative RHS (rows 0..2 and L-3..L-1); fs, fe: the
// closure sums received at the start and end faces
template <class SA, class FA>
__device__ inline double deriv_bnd_row(const Block &b, const CaseCoef &c, int D, int i, int L, const SA &sa,
                                       const FA &fs, const FA &fe) {
  const double aa = 0.6431406736919156, ab = 0.2586011023495066, ac = 0.007140953479797375;
  const int ie = L - 1;
  if (i <= 2) {
    if (b.ndf[D][0] == 0) {
      const double s0 = sa(0), s1 = sa(1), s2 = sa(2), s3 = sa(3), s4 = sa(4), s5 = sa(5), s6 = sa(6);
      double r = 0;
      if (i == 0) {
        r = r + c.abc[0][0] * (s1 - s0); r = r + c.abc[0][1] * (s2 - s0); r = r + c.abc[0][2] * (s3 - s0);
        r = r + c.abc[0][3] * (s4 - s0); r = r + c.abc[0][4] * (s5 - s0); r = r + c.abc[0][5] * (s6 - s0);
      } else if (i == 1) {
        r = r + c.abc[1][0] * (s0 - s1); r = r + c.abc[1][1] * (s2 - s1); r = r + c.abc[1][2] * (s3 - s1);
        r = r + c.abc[1][3] * (s4 - s1); r = r + c.abc[1][4] * (s5 - s1); r = r + c.abc[1][5] * (s6 - s1);
      } else {
        r = r + c.abc[2][0] * (s0 - s2); r = r + c.abc[2][1] * (s1 - s2); r = r + c.abc[2][2] * (s3 - s2);
        r = r + c.abc[2][3] * (s4 - s2); r = r + c.abc[2][4] * (s5 - s2); r = r + c.abc[2][5] * (s6 - s2);
      }
      return r;
    }
    if (i <= 1) {
      double t = 0;
      for (int q = 0; q <= LMD; q++) t = t + c.pbci[0][i][q] * sa(q);
      return t + fs(i);
    }
    return aa * (sa(3) - sa(1)) + ab * (sa(4) - sa(0)) + ac * (sa(5) - fs(2));
  }
  const int row = ie - i;  // 0: last row
  if (b.ndf[D][1] == 0) {
    const double e0 = sa(ie), e1 = sa(ie - 1), e2 = sa(ie - 2), e3 = sa(ie - 3), e4 = sa(ie - 4),
                 e5 = sa(ie - 5), e6 = sa(ie - 6);
    double r = 0;
    if (row == 0) {
      r = r + c.abc[0][0] * (e0 - e1); r = r + c.abc[0][1] * (e0 - e2); r = r + c.abc[0][2] * (e0 - e3);
      r = r + c.abc[0][3] * (e0 - e4); r = r + c.abc[0][4] * (e0 - e5); r = r + c.abc[0][5] * (e0 - e6);
    } else if (row == 1) {
      r = r + c.abc[1][0] * (e1 - e0); r = r + c.abc[1][1] * (e1 - e2); r = r + c.abc[1][2] * (e1 - e3);
      r = r + c.abc[1][3] * (e1 - e4); r = r + c.abc[1][4] * (e1 - e5); r = r + c.abc[1][5] * (e1 - e6);
    } else {
      r = r + c.abc[2][0] * (e2 - e0); r = r + c.abc[2][1] * (e2 - e1); r = r + c.abc[2][2] * (e2 - e3);
      r = r + c.abc[2][3] * (e2 - e4); r = r + c.abc[2][4] * (e2 - e5); r = r + c.abc[2][5] * (e2 - e6);
    }
    return r;
  }
  if (row <= 1) {
    double t = 0;
    for (int q = 0; q <= LMD; q++) t = t + c.pbci[0][row][q] * sa(ie - q);
    return -t - fe(row);
  }
  return aa * (sa(ie - 1) - sa(ie - 3)) + ab * (sa(ie) - sa(ie - 4)) + ac * (fe(2) - sa(ie - 5));
}

// boundary rows of the filter RHS
template <class SA, class FA>
__device__ inline double filter_bnd_row(const Block &b, const CaseCoef &c, int D, int i, int L, const SA &sa,
                                        const FA &fs, const FA &fe) {
  const int ie = L - 1;
  const double fa = c.fa, fb = c.fb, fc = c.fc;
  if (i <= 2) {
    if (b.ndf[D][0] == 0) {
      const double s0 = sa(0), s1 = sa(1), s2 = sa(2), s3 = sa(3), s4 = sa(4), s5 = sa(5);
      double res = 0;
      res = res + c.fex[0] * (s1 - s0); res = res + c.fex[1] * (s2 - s0); res = res + c.fex[2] * (s3 - s0);
      const double rv0 = s0 - res * c.ffx[0], rv1 = s0 - res * c.ffx[1], rv2 = s0 - res * c.ffx[2];
      if (i == 0) {
        const double ra0 = 2.0 * s0;
        return c.fam[0] * (rv0 + s1 - ra0) + c.fbm[0] * (rv1 + s2 - ra0) + c.fcm[0] * (rv2 + s3 - ra0);
      } else if (i == 1) {
        const double ra1 = 2.0 * s1;
        return c.fam[1] * (s0 + s2 - ra1) + c.fbm[1] * (rv0 + s3 - ra1) + c.fcm[1] * (rv1 + s4 - ra1);
      }
      const double ra2 = 2.0 * s2;
      return c.fam[2] * (s1 + s3 - ra2) + c.fbm[2] * (s0 + s4 - ra2) + c.fcm[2] * (rv0 + s5 - ra2);
    }
    if (i <= 1) {
      double t = 0;
      for (int q = 0; q <= LMF; q++) t = t + c.pbci[1][i][q] * sa(q);
      return t + fs(i);
    }
    const double ra2 = 2.0 * sa(2);
    return fa * (sa(1) + sa(3) - ra2) + fb * (sa(0) + sa(4) - ra2) + fc * (fs(2) + sa(5) - ra2);
  }
  const int row = ie - i;
  if (b.ndf[D][1] == 0) {
    const double e0 = sa(ie), e1 = sa(ie - 1), e2 = sa(ie - 2), e3 = sa(ie - 3), e4 = sa(ie - 4), e5 = sa(ie - 5);
    double res = 0;
    res = res + c.fex[0] * (e0 - e1); res = res + c.fex[1] * (e0 - e2); res = res + c.fex[2] * (e0 - e3);
    const double rv0 = e0 + res * c.ffx[0], rv1 = e0 + res * c.ffx[1], rv2 = e0 + res * c.ffx[2];
    if (row == 0) {
      const double ra0 = 2.0 * e0;
      return c.fam[0] * (e1 + rv0 - ra0) + c.fbm[0] * (e2 + rv1 - ra0) + c.fcm[0] * (e3 + rv2 - ra0);
    } else if (row == 1) {
      const double ra1 = 2.0 * e1;
      return c.fam[1] * (e2 + e0 - ra1) + c.fbm[1] * (e3 + rv0 - ra1) + c.fcm[1] * (e4 + rv1 - ra1);
    }
    const double ra2 = 2.0 * e2;
    return c.fam[2] * (e3 + e1 - ra2) + c.fbm[2] * (e4 + e0 - ra2) + c.fcm[2] * (e5 + rv0 - ra2);
  }
  if (row <= 1) {
    double t = 0;
    for (int q = 0; q <= LMF; q++) t = t + c.pbci[1][row][q] * sa(ie - q);
    return t + fe(row);
  }
  const double ra2 = 2.0 * sa(ie - 2);
  return fa * (sa(ie - 3) + sa(ie - 1) - ra2) + fb * (sa(ie - 4) + sa(ie) - ra2) +
         fc * (sa(ie - 5) + fe(2) - ra2);
}


constexpr int COL_TR = 65;   // row pitch (doubles) of the xi transpose buffer
constexpr int COL_DECAY = 48;  // points a carry travels sequentially before an amplifying closure

// doubles of one chunk's factors in LDS: the table's own [6][32], or a long
// line's five runs
__host__ __device__ constexpr int col_fac(int G) { return G == 1 ? 192 : COL_LONG_F; }

// dynamic LDS of a k_col launch, in doubles: carry pairs [2][P][64] (double2),
// chunk factors, and for xi the transposes [P][8][COL_TR]
__host__ __device__ constexpr int col_lds_doubles(int d, int P, int G) {
  return 2 * P * 64 * 2 + P * G * col_fac(G) + (d == 0 ? P * 8 * COL_TR : 0);
}

// a zero the optimiser cannot see through: offsetting the factor pointer by
// it at each sweep keeps the factor loads inside the sweep instead of being
// hoisted out of the chain-round loops and held in registers throughout
__device__ inline int opaque_zero() {
  int z;
  asm volatile("s_mov_b32 %0, 0" : "=s"(z));
  return z;
}

// Orders the LDS accesses of one wave around a transpose step.  The LDS
// instructions of a wave execute in issue order, so no memory fence (which
// would also wait for the wave's outstanding global loads) is needed; this
// only keeps the compiler from moving memory operations across.
__device__ inline void wave_sync() { __builtin_amdgcn_wave_barrier(); }

// value of a double held in lane l (wave-uniform result)
__device__ inline double lane_val(double v, int l) {
  const long long b = __builtin_bit_cast(long long, v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), l);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}

// Factors of the chunk's rows, copied to the wave's LDS slice:
// F[k] = l1, F[S+k] = l2, F[2S+k] = u1, F[3S+k] = u2, F[4S+k] = u3 of row
// k.  Every lane of the chunk reads the same address (an LDS broadcast).
template <int S>
struct ChunkLU {
  const double *F;
};

// Forward substitution over the chunk rows from the carry (ym2, ym1), in
// place when store is set.  Rows k >= n are capacity padding: their factors
// (l1 = -1, l2 = 0) and zero right-hand side make each of them swap the
// carried pair exactly (y = 0 + ym2 - 0), so after them the pair is the one
// of row n-1, swapped once more if their count is odd.  The opaque offset
// keeps each sweep's factor loads inside the sweep.
template <int C, int S>
__device__ inline void fwd_sweep(double (&r)[C], int n, const ChunkLU<S> &f, double &ym2, double &ym1,
                                 bool store) {
  const double *F = f.F + opaque_zero();
#pragma unroll
  for (int k = 0; k < C; k++) {
    const double f1 = F[k];
    const double f2 = F[S + k];
    const double y = r[k] - f1 * ym2 - f2 * ym1;
    if (store) r[k] = y;
    ym2 = ym1;
    ym1 = y;
  }
  if ((C - n) & 1) {
    const double t = ym2;
    ym2 = ym1;
    ym1 = t;
  }
}

// backward substitution from the carry (xp1, xp2) = (x[e+1], x[e+2]): the
// padding rows k >= n come first, each swapping the pair (u1 = u2 = 0,
// u3 = -1), so the carry enters them pre-swapped when their count is odd
template <int C, int S>
__device__ inline void bwd_sweep(double (&r)[C], int n, const ChunkLU<S> &f, double &xp1, double &xp2,
                                 bool store) {
  const double *F = f.F + opaque_zero();
  if ((C - n) & 1) {
    const double t = xp1;
    xp1 = xp2;
    xp2 = t;
  }
#pragma unroll
  for (int k = C - 1; k >= 0; k--) {
    const double g1 = F[2 * S + k];
    const double g2 = F[3 * S + k];
    const double g3 = F[4 * S + k];
    const double x = g1 * r[k] - g2 * xp1 - g3 * xp2;
    if (store) r[k] = x;
    xp2 = xp1;
    xp1 = x;
  }
}

// DIRECT: the launch forms the closure sums itself (a.direct) instead of
// reading the exchange's recv slots
// G: chunks side by side in a wave.  1: the wave's 64 lanes are 64 lines.
// COL_LONG_G, for lines longer than 16 waves of the largest chunks hold: 64 / G
// lines in G lane groups, each group the next chunk of the same lines, so that
// P waves hold G P chunks and the windows of a line still fit the registers.
template <int D, int KIND, int C, bool DIRECT, int G>
__global__ void __launch_bounds__(1024) k_col(LineArgs a) {
  extern __shared__ double lds[];
  const Work w = a.work[xcd_item(blockIdx.x, gridDim.x)];
  constexpr int d_col = 0;
#include "tp_col_body.hpp"
}

// The derivatives of the same fields along all three directions in one launch
// (the gradients of a stage), direction d of a work item into column out_col + d:
// three independent solves, each of which leaves most of a launch of its own
// idle on a small case.
// The zeta solves form their closure sums themselves, the others have none; up to
// 8 waves, so that the registers of the three together need not be spilled.
template <int C>
__global__ void __launch_bounds__(512) k_col_dirs(LineArgs a) {
  extern __shared__ double lds[];
  const Work w = a.work[xcd_item(blockIdx.x, gridDim.x)];
  constexpr int KIND = 0, G = 1;
  if (w.d == 0) {
    constexpr int D = 0, d_col = 0;
    constexpr bool DIRECT = false;
#include "tp_col_body.hpp"
  } else if (w.d == 1) {
    constexpr int D = 1, d_col = 1;
    constexpr bool DIRECT = false;
#include "tp_col_body.hpp"
  } else {
    constexpr int D = 2, d_col = 2;
    constexpr bool DIRECT = true;
#include "tp_col_body.hpp"
  }
}

size_t col_lds_bytes(int d, int P, int G) { return (size_t)col_lds_doubles(d, P, G) * sizeof(double); }

template <int D, int KIND>
static void launch_long(int P, int nwg, int nf, hipStream_t st, const LineArgs &a, hipEvent_t e0, hipEvent_t e1) {
  const size_t lds = col_lds_bytes(D, P, COL_LONG_G);
  if (KIND == 0 && a.direct)
    TP_LAUNCH_EV((k_col<D, KIND, COL_LONG_C, KIND == 0, COL_LONG_G>), dim3(nwg, nf), dim3(64 * P), lds, st, e0, e1, a);
  else
    TP_LAUNCH_EV((k_col<D, KIND, COL_LONG_C, false, COL_LONG_G>), dim3(nwg, nf), dim3(64 * P), lds, st, e0, e1, a);
}

template <int D, int KIND>
static void launch_col_c(int C, int P, int nwg, int nf, hipStream_t st, const LineArgs &a, hipEvent_t e0,
                         hipEvent_t e1) {
  const size_t lds = col_lds_bytes(D, P, 1);
  switch (C) {
#define CASE_C(CV)                                                                                     \
  case CV:                                                                                           \
    if (KIND == 0 && a.direct)                                                                       \
      TP_LAUNCH_EV((k_col<D, KIND, CV, KIND == 0, 1>), dim3(nwg, nf), dim3(64 * P), lds, st, e0, e1, a); \
    else                                                                                             \
      TP_LAUNCH_EV((k_col<D, KIND, CV, false, 1>), dim3(nwg, nf), dim3(64 * P), lds, st, e0, e1, a);    \
    break;
    CASE_C(8) CASE_C(12) CASE_C(16) CASE_C(20) CASE_C(24) CASE_C(28) CASE_C(32)
#undef CASE_C
  }
}

// register capacity of a chunk of `chunk` points: the next multiple of 4 from
// 8 (rows past the chunk are padding the sweeps run over)
int col_capacity(int chunk) {
  if (chunk > 32) return 0;
  return chunk <= 8 ? 8 : (chunk + 3) / 4 * 4;
}

// capacity of a launch of all three directions, at least C
int dirs_capacity(int C) { return C <= 12 ? 12 : C <= 16 ? 16 : C <= 24 ? 24 : 32; }

void launch_col_dirs(int C, int P, int nwg, int nf, hipStream_t st, const LineArgs &a) {
  const size_t lds = col_lds_bytes(0, P, 1);
  switch (C) {
#define CASE_C(CV) \
  case CV: hipLaunchKernelGGL(k_col_dirs<CV>, dim3(nwg, nf), dim3(64 * P), lds, st, a); break;
    CASE_C(12) CASE_C(16) CASE_C(24) CASE_C(32)
#undef CASE_C
  }
}

void launch_col(int d, int kind, int C, int P, int G, int nwg, int nf, hipStream_t st, const LineArgs &a,
                hipEvent_t e0, hipEvent_t e1) {
#define BY_KIND(D)                                                       \
  if (G == 1) {                                                          \
    if (kind == 0) launch_col_c<D, 0>(C, P, nwg, nf, st, a, e0, e1);     \
    else launch_col_c<D, 1>(C, P, nwg, nf, st, a, e0, e1);               \
  } else {                                                               \
    if (kind == 0) launch_long<D, 0>(P, nwg, nf, st, a, e0, e1);    \
    else launch_long<D, 1>(P, nwg, nf, st, a, e0, e1);              \
  }
  if (d == 0) { BY_KIND(0) }
  else if (d == 1) { BY_KIND(1) }
  else { BY_KIND(2) }
#undef BY_KIND
}

}  // namespace tp
