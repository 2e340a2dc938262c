// tp_col_body.hpp -- the body of the line-solve kernels (tp_col.hip), included
// inside each: as a function it would take the kernel's argument block by
// reference, and the compiler then no longer knows its pointers as global
// memory (flat accesses: the launches 2 to 4 % slower).
//
// In scope: LineArgs a, Work w, double *lds, and the constants D, KIND, C,
// DIRECT, G and d_col (added to the output column).
  const Block &b = a.blocks[w.blk];
  const CaseCoef &c = a.coef[b.cs];
  const int L = b.L[D];
  constexpr int NL = 64 / G, FS = G == 1 ? 32 : C, FC = col_fac(G);
  const int P = G * b.colP[D][KIND];              // chunks of this block's lines
  const int PL = blockDim.x >> 6;                 // waves of the launch, G of them hold at least P chunks
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int p = G == 1 ? wv : wv * G + lane / NL; // this lane's chunk
  const int li = lane % NL;                       // and line
  const int Cl = (L + P - 1) / P;
  const int Pe = (L + Cl - 1) / Cl;               // chunks holding points
  const int s0 = p * Cl;
  const int n = p < Pe ? min(Cl, L - s0) : 0;     // points of this lane's chunk
  const int nl = w.n;
  const bool act = li < nl;
  const int stride = D == 0 ? 1 : D == 1 ? b.nx : b.nx * b.ny;
  int base, jk;
  col_line<D>(b, w.a + (act ? li : 0), base, jk);
  const int fi = blockIdx.y;   // field of a merged launch
  const double *src = field_ptr(b, a.in_arr, a.in_col + fi * a.in_step);
  double *dst = field_ptr(b, a.out_arr, a.out_col + fi * a.out_step + d_col);
  const double *rcv = b.recv[D] + (size_t)fi * 6 * b.F[D];
  const int mcap = a.m > 0 ? a.m + fi : 0;
  double2 *pairA = reinterpret_cast<double2 *>(lds);      // [chunk][NL] carry-map inputs
  double2 *pairB = pairA + PL * 64;                       // [chunk][NL] pairs handed along a chain
  double *fw = reinterpret_cast<double *>(pairB + PL * 64) + wv * G * FC;   // the wave's chunk factors
  double *tr = reinterpret_cast<double *>(pairB + PL * 64) + PL * G * FC + wv * (8 * COL_TR);
  const double *T = b.col[D][KIND];
  // carry maps: of all chunks (G = 1), or of the window of chunks that this
  // wave composes: what comes from further away has died out (long_reach forms
  // the distance from the block's own factors; it depends on the filter's cut-off)
  const int reach = G == 1 ? 0 : b.colR[D][KIND];
  const int qf0 = G == 1 ? 0 : max(0, wv * G - reach), qb0 = G == 1 ? 0 : wv * G;
  double mapf[G == 1 ? 1 : 2], mapb[G == 1 ? 1 : 2];
  if (G == 1) {
    mapf[0] = T[lane];
    mapb[0] = T[64 + lane];
  } else {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      mapf[G == 1 ? 0 : h] = T[4 * qf0 + 64 * h + lane];
      mapb[G == 1 ? 0 : h] = T[4 * COL_LONG_Q + 4 * qb0 + 64 * h + lane];
    }
  }
  ChunkLU<FS> f;
  if (G == 1) {
    const double *F = T + 128 + 192 * min(p, Pe - 1);
    fw[lane] = F[lane]; fw[64 + lane] = F[64 + lane]; fw[128 + lane] = F[128 + lane];
    f.F = fw;
  } else {
    // the tables' chunks are laid out as the LDS holds them
    for (int g = 0; g < G; g++) {
      const double *F = T + 8 * COL_LONG_Q + (size_t)FC * min(wv * G + g, Pe - 1);
      for (int k = lane; k < 5 * C; k += 64) fw[g * FC + k] = F[k];
    }
    f.F = fw + (lane / NL) * FC;
  }
  wave_sync();   // the wave's own LDS writes precede its reads in issue order

  // Chains at one-sided closures.  End: the last Rhi chunks take their
  // forward carry from the chunk before them, one after the other.  Start:
  // the first Rlo chunks take their backward carry from the chunk after
  // them, which needs exact forward values there, so chunks 2..Rlo take
  // their forward carry from their predecessor too (chunk 1's carry, the
  // first chunk's zero-carry result, is exact already).
  const int Rc = (COL_DECAY + Cl - 1) / Cl;
  const int Rhi = b.ndf[D][1] == 0 ? min(Rc, Pe - 1) : 0;
  const int Rlo = b.ndf[D][0] == 0 ? min(Rc, Pe - 1) : 0;
  int tf = 0, Tf = 0, tb = 0, Tb = 0;   // chain round of this wave, rounds in all
  {
    int t = 0;
    for (int q = 0; q < Pe; q++) {
      const bool ch = (q >= 2 && q <= Rlo) || (Rhi > 0 && q >= Pe - Rhi);
      t = ch ? t + 1 : 0;
      if (q == p) tf = t;
      Tf = max(Tf, t);
    }
    t = 0;
    for (int q = Pe - 1; q >= 0; q--) {
      t = q < Rlo ? t + 1 : 0;
      if (q == p) tb = t;
      Tb = max(Tb, t);
    }
  }

  // DIRECT: the closure sums of the faces this wave's boundary rows need,
  // formed from the neighbour's field (its lines on the far side of the
  // face: the other end of the same lines for a periodic block, the partner
  // block's lines -- whose work items run beside these -- otherwise), as the
  // exchange forms them.  First, so that only the three sums per face stay
  // live while the window is loaded.
  ValFace fsum[2] = {{{0.0, 0.0, 0.0}}, {{0.0, 0.0, 0.0}}};
  if (DIRECT) {
#pragma unroll
    for (int ip = 0; ip < 2; ip++) {
      const bool need = ip == 0 ? n > 0 && s0 <= 2 : n > 0 && s0 + n - 1 >= L - 3;
      if (!need || !b.ndf[D][ip]) continue;
      const Block &nb = a.blocks[b.ncd[D][ip]];
      closure_sums<KIND>(b, nb, c, field_ptr(nb, a.in_arr, a.in_col + fi * a.in_step), src, D, ip, jk, a.n45,
                         fsum[ip].r[0], fsum[ip].r[1], fsum[ip].r[2]);
    }
  }

  // ---- window rows s0-3 .. s0+n+2, clamped to the line; the rows of the
  // capacity padding past them are not read (zero) ----
  double v[C + 6];
  const int nw = (D == 0 && G > 1 ? Cl : n) + 6;   // window rows in use
  if (D == 0) {
    // all global loads of the window first (8 lines x 8 consecutive points per
    // instruction), then the transposes through LDS piece by piece
    constexpr int NPC = (C + 6 + 7) / 8;
    double tmp[NPC][8];
#pragma unroll
    for (int t = 0; t < NPC; t++) {
#pragma unroll
      for (int j = 0; j < 8; j++) {
        // the (chunk, line) of lane 8j + lane / 8
        const int q = (lane >> 3) + 8 * j;
        const int sq = G == 1 ? s0 : (wv * G + q / NL) * Cl;
        const int row = min(max(sq - 3 + 8 * t + (lane & 7), 0), L - 1);
        const int rl = min(q % NL, nl - 1);
        tmp[t][j] = 8 * t < nw ? at(src, 8u * (unsigned)((w.a + rl) * b.nx + row)) : 0.0;
      }
    }
#pragma unroll
    for (int t = 0; t < NPC; t++) {
      if (8 * t < nw) {
#pragma unroll
        for (int j = 0; j < 8; j++) tr[(lane & 7) * COL_TR + (lane >> 3) + 8 * j] = tmp[t][j];
        wave_sync();
#pragma unroll
        for (int rr = 0; rr < 8; rr++)
          if (8 * t + rr < C + 6) v[8 * t + rr] = tr[rr * COL_TR + lane];
        wave_sync();
      } else {
#pragma unroll
        for (int rr = 0; rr < 8; rr++)
          if (8 * t + rr < C + 6) v[8 * t + rr] = 0.0;
      }
    }
  } else {
    const unsigned b8 = 8u * (unsigned)base, st8 = 8u * (unsigned)stride;
#pragma unroll
    for (int k = 0; k < C + 6; k++) {
      const int row = min(max(s0 - 3 + k, 0), L - 1);
      v[k] = k < nw ? at(src, b8 + (unsigned)row * st8) : 0.0;
    }
  }

  // ---- right-hand side ----
  // rows 0..2 and L-3..L-1 use the closure formulas, evaluated once, outside
  // the unrolled loop, by the (at most two) chunks that hold them
  // the closure rows at the line ends, with the closure sums formed above
  // (DIRECT) or read from the exchange's recv slots
  double rb0 = 0.0, rb1 = 0.0, rb2 = 0.0, re2 = 0.0, re1 = 0.0, re0 = 0.0;
  {
    const GLine g{src + base, stride};
    auto rows = [&](const auto &fs, const auto &fe) {
      if (n > 0 && s0 <= 2) {
        if (KIND == 0) {
          rb0 = deriv_bnd_row(b, c, D, 0, L, g, fs, fe);
          rb1 = deriv_bnd_row(b, c, D, 1, L, g, fs, fe);
          rb2 = deriv_bnd_row(b, c, D, 2, L, g, fs, fe);
        } else {
          rb0 = filter_bnd_row(b, c, D, 0, L, g, fs, fe);
          rb1 = filter_bnd_row(b, c, D, 1, L, g, fs, fe);
          rb2 = filter_bnd_row(b, c, D, 2, L, g, fs, fe);
        }
      }
      if (n > 0 && s0 + n - 1 >= L - 3) {
        if (KIND == 0) {
          re2 = deriv_bnd_row(b, c, D, L - 3, L, g, fs, fe);
          re1 = deriv_bnd_row(b, c, D, L - 2, L, g, fs, fe);
          re0 = deriv_bnd_row(b, c, D, L - 1, L, g, fs, fe);
        } else {
          re2 = filter_bnd_row(b, c, D, L - 3, L, g, fs, fe);
          re1 = filter_bnd_row(b, c, D, L - 2, L, g, fs, fe);
          re0 = filter_bnd_row(b, c, D, L - 1, L, g, fs, fe);
        }
      }
    };
    if (DIRECT) rows(fsum[0], fsum[1]);
    else rows(RcvFace{rcv, b.F[D], jk, 0}, RcvFace{rcv, b.F[D], jk, 1});
  }
  // derivative: interior stencil on every row, then the closure rows patched
  // in by the (at most two) chunks at each end that hold them; then the
  // padding rows zeroed
  double r[C];
  if (KIND == 1 && G > 1) {
    // long lines: the increment, added to the input at the store, as the
    // sequential kernel forms it.  A out = R + A in (below) reads the input
    // once, but its rounding grows with A's condition: 3.5e-14 of the field
    // at a cut-off of 0.85 pi, 1.6e-12 at 0.95, where the increment keeps
    // 1.1e-16 and 1.2e-16
#pragma unroll
    for (int k = 0; k < C; k++) {
      const double res = 2.0 * v[k + 3];
      r[k] = c.fa * (v[k + 2] + v[k + 4] - res) + c.fb * (v[k + 1] + v[k + 5] - res) +
             c.fc * (v[k] + v[k + 6] - res);
    }
  } else if (KIND == 1) {
    // filter: the solve yields the filtered field itself, A out = R + A in
    // (A the filter's left-hand side: interior rows (fbe, fal, 1, fal, fbe),
    // closure rows of each end from flhs, mirrored at the far end), rather
    // than the increment A^-1 R added to a second read of the input.  The
    // closure rows' A in is formed first, from the window (its rows found by
    // selects, not by indexing the register array), then every row's
    // R + A in with the window dying row by row.
    if (n > 0 && s0 <= 2) {
      const double *hd = &c.flhs[b.ndf[D][0]][0][0];
      double ah[3] = {0.0, 0.0, 0.0};
#pragma unroll
      for (int k = 0; k < 3 && k < C; k++) {
        const int i = s0 + k;   // row i sits at k; entries at columns i-2 .. i+2
        if (i <= 2) {
          const double *e = hd + 5 * i;
          const double s = e[0] * v[k + 1] + e[1] * v[k + 2] + v[k + 3] + e[3] * v[k + 4] + e[4] * v[k + 5];
          ah[0] = i == 0 ? s : ah[0]; ah[1] = i == 1 ? s : ah[1]; ah[2] = i == 2 ? s : ah[2];
        }
      }
      rb0 = rb0 + ah[0]; rb1 = rb1 + ah[1]; rb2 = rb2 + ah[2];
    }
    if (n > 0 && s0 + n - 1 >= L - 3) {
      const double *tl = &c.flhs[b.ndf[D][1]][0][0];
      double at0 = 0.0, at1 = 0.0, at2 = 0.0;
#pragma unroll
      for (int k = 0; k < C; k++) {
        const int i = s0 + k;   // mirrored: entry 4-q at column i+q-2
        if (i >= L - 3 && i <= L - 1) {
          const double *e = tl + 5 * (L - 1 - i);
          const double s = e[4] * v[k + 1] + e[3] * v[k + 2] + v[k + 3] + e[1] * v[k + 4] + e[0] * v[k + 5];
          at0 = i == L - 1 ? s : at0; at1 = i == L - 2 ? s : at1; at2 = i == L - 3 ? s : at2;
        }
      }
      re0 = re0 + at0; re1 = re1 + at1; re2 = re2 + at2;
    }
#pragma unroll
    for (int k = 0; k < C; k++) {
      const double res = 2.0 * v[k + 3];
      r[k] = c.fa * (v[k + 2] + v[k + 4] - res) + c.fb * (v[k + 1] + v[k + 5] - res) +
             c.fc * (v[k] + v[k + 6] - res) + (v[k + 3] + c.fal * (v[k + 2] + v[k + 4]) + c.fbe * (v[k + 1] + v[k + 5]));
    }
  } else {
#pragma unroll
    for (int k = 0; k < C; k++) {
      const double aa = 0.6431406736919156, ab = 0.2586011023495066, ac = 0.007140953479797375;
      r[k] = aa * (v[k + 4] - v[k + 2]) + ab * (v[k + 5] - v[k + 1]) + ac * (v[k + 6] - v[k]);
    }
  }
  // the closure rows patched in by the (at most two) chunks at each end that
  // hold them
  {
    if (n > 0 && s0 <= 2) {
#pragma unroll
      for (int k = 0; k < 3 && k < C; k++) {
        const int i = s0 + k;
        r[k] = i == 0 ? rb0 : i == 1 ? rb1 : i == 2 ? rb2 : r[k];
      }
    }
    if (n > 0 && s0 + n - 1 >= L - 3) {
#pragma unroll
      for (int k = 0; k < C; k++) {
        const int i = s0 + k;
        r[k] = i == L - 1 ? re0 : i == L - 2 ? re1 : i == L - 3 ? re2 : r[k];
      }
    }
  }
  if (n < C) {
#pragma unroll
    for (int k = 0; k < C; k++) r[k] = k < n ? r[k] : 0.0;   // padding rows carry a zero right-hand side
  }

  // ---- forward substitution ----
  double ym2 = 0.0, ym1 = 0.0;
  fwd_sweep<C>(r, n, f, ym2, ym1, false);
  pairA[p * NL + li] = make_double2(ym2, ym1);
  __syncthreads();
  double c0 = 0.0, c1 = 0.0;
  const int qfe = min(G == 1 ? p : wv * G + G - 1, Pe);
  for (int q = qf0; q < qfe; q++) {
    const double mq = G == 1 || q - qf0 < 16 ? mapf[0] : mapf[G == 1 ? 0 : 1];
    const int at = 4 * (G == 1 ? q : (q - qf0) & 15);
    const double m0 = lane_val(mq, at), m1 = lane_val(mq, at + 1);
    const double m2 = lane_val(mq, at + 2), m3 = lane_val(mq, at + 3);
    const double2 e = pairA[q * NL + li];
    const double t0 = m0 * c0 + m1 * c1 + e.x;
    const double t1 = m2 * c0 + m3 * c1 + e.y;
    if (G == 1 || q < p) { c0 = t0; c1 = t1; }
  }
  for (int t = 0; t <= Tf; t++) {
    if (t > 0) __syncthreads();
    if (tf == t) {
      if (t > 0) {
        const double2 e = pairB[(p - 1) * NL + li];
        c0 = e.x; c1 = e.y;
      }
      ym2 = c0; ym1 = c1;
      fwd_sweep<C>(r, n, f, ym2, ym1, true);
      pairB[p * NL + li] = make_double2(ym2, ym1);
    }
  }
  __syncthreads();   // every wave has read pairA and pairB before they are reused

  // ---- backward substitution ----
  double xp1 = 0.0, xp2 = 0.0;
  bwd_sweep<C>(r, n, f, xp1, xp2, false);
  pairA[p * NL + li] = make_double2(xp1, xp2);
  __syncthreads();
  double d0 = 0.0, d1 = 0.0;
  const int qbe = G == 1 ? p : qb0;
  for (int q = G == 1 ? Pe - 1 : min(Pe - 1, qb0 + G - 1 + reach); q > qbe; q--) {
    const double mq = G == 1 || q - qb0 < 16 ? mapb[0] : mapb[G == 1 ? 0 : 1];
    const int at = 4 * (G == 1 ? q : (q - qb0) & 15);
    const double m0 = lane_val(mq, at), m1 = lane_val(mq, at + 1);
    const double m2 = lane_val(mq, at + 2), m3 = lane_val(mq, at + 3);
    const double2 e = pairA[q * NL + li];
    const double t0 = m0 * d0 + m1 * d1 + e.x;
    const double t1 = m2 * d0 + m3 * d1 + e.y;
    if (G == 1 || q > p) { d0 = t0; d1 = t1; }
  }
  for (int t = 0; t <= Tb; t++) {
    if (t > 0) __syncthreads();
    if (tb == t) {
      if (t > 0) {
        const double2 e = pairB[(p + 1) * NL + li];
        d0 = e.x; d1 = e.y;
      }
      xp1 = d0; xp2 = d1;
      bwd_sweep<C>(r, n, f, xp1, xp2, true);
      pairB[p * NL + li] = make_double2(xp1, xp2);
    }
  }

  // ---- boundary derivatives kept for the characteristic conditions ----
  if (KIND == 0 && mcap > 0 && act && n > 0) {
    const int F = b.F[D];
    if (p == 0) b.drva[D][(0 * 5 + mcap - 1) * F + jk] = r[0];
    if (p == Pe - 1) {
      double xe = r[0];
#pragma unroll
      for (int k = 1; k < C; k++) xe = k == n - 1 ? r[k] : xe;
      b.drva[D][(1 * 5 + mcap - 1) * F + jk] = xe;
    }
  }

  // ---- store: the filtered field (on long lines the input and its increment),
  // or the derivative (which may accumulate) ----
  const bool add = KIND == 0 ? a.acc : G > 1;
  const double *ob = KIND == 0 ? dst : src;
  double *cpy = KIND == 1 && a.copy_arr >= 0 ? field_ptr(b, a.copy_arr, a.copy_col + fi * a.out_step) : nullptr;
  // xi: the work item's lines are consecutive rows of the block, one
  // contiguous span of nl * L doubles.  Once every wave is done with the
  // carry, factor and transpose areas, the whole LDS holds R of these rows at
  // a time (R the largest power of two that fits, at least 8), and the
  // workgroup stores them as one run of whole cache lines: a wave's own
  // pieces (8 rows x 8 points) would straddle 64-byte write granules.
  const int pitch = L + 1;
  int R = NL;
  while (R >= (G == 1 ? 8 : 2) && R * pitch > col_lds_doubles(0, PL, G)) R >>= 1;
  if (D == 0 && (G > 1 || R >= 8)) {
    double *tile = lds;
    __syncthreads();
    for (int h = 0; h * R < nl; h++) {
      if (act && li >= h * R && li < (h + 1) * R) {
        double *trow = tile + (li - h * R) * pitch + s0;
#pragma unroll
        for (int k = 0; k < C; k++)
          if (k < n) trow[k] = r[k];
      }
      __syncthreads();
      const int rows = min(R, nl - h * R);
      const int tot = rows * L;
      const unsigned base0 = (unsigned)(w.a + h * R) * (unsigned)b.nx;
      // element idx of the run sits at (row, col) = (idx / L, idx % L) of the
      // tile; each thread steps by blockDim.x = dq L + dr elements, so
      // (row, col) advance without a division, four elements at a time
      const int dq = (int)blockDim.x / L, dr = (int)blockDim.x - dq * L;
      int row = (int)threadIdx.x / L, col = (int)threadIdx.x - row * L;
      for (int i0 = threadIdx.x; i0 < tot; i0 += 4 * (int)blockDim.x) {
        double x4[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          x4[u] = i0 + u * (int)blockDim.x < tot ? tile[row * pitch + col] : 0.0;
          col += dr;
          row += dq;
          if (col >= L) { col -= L; row++; }
        }
        double o4[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int idx = i0 + u * (int)blockDim.x;
          o4[u] = add && idx < tot ? ld_stream(&at(ob, 8u * (base0 + (unsigned)idx))) : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int idx = i0 + u * (int)blockDim.x;
          if (idx < tot) {
            const unsigned o = 8u * (base0 + (unsigned)idx);
            const double y = add ? o4[u] + x4[u] : x4[u];
            st(dst, o, y);
            if (KIND == 1 && cpy) st(cpy, o, y);
          }
        }
      }
      __syncthreads();   // the tile is read before the next rows overwrite it
    }
  } else if (D == 0) {
#pragma unroll
    for (int t = 0; t < (C + 7) / 8; t++) {
      if (8 * t >= n) break;   // pieces past the chunk hold no rows of it
#pragma unroll
      for (int rr = 0; rr < 8; rr++)
        if (8 * t + rr < C) tr[rr * COL_TR + lane] = r[8 * t + rr];
      wave_sync();
      const int k = 8 * t + (lane & 7);
      const int row = min(s0 + k, L - 1);
      double xv[8], ov[8];
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const int rl = (lane >> 3) + 8 * j;
        xv[j] = tr[(lane & 7) * COL_TR + rl];
        ov[j] = add ? at(ob, 8u * (unsigned)((w.a + min(rl, nl - 1)) * b.nx + row)) : 0.0;
      }
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const int rl = (lane >> 3) + 8 * j;
        if (k < n && rl < nl) {
          const unsigned o = 8u * (unsigned)((w.a + rl) * b.nx + s0 + k);
          const double y = add ? ov[j] + xv[j] : xv[j];
          st(dst, o, y);
          if (KIND == 1 && cpy) st(cpy, o, y);
        }
      }
      wave_sync();
    }
  } else {
    const unsigned b8 = 8u * (unsigned)base, st8 = 8u * (unsigned)stride;
    double ov[C];
#pragma unroll
    for (int k = 0; k < C; k++)
      ov[k] = add && k < n ? at(ob, b8 + (unsigned)min(s0 + k, L - 1) * st8) : 0.0;
    if (act) {
#pragma unroll
      for (int k = 0; k < C; k++)
        if (k < n) {
          const unsigned o = b8 + (unsigned)(s0 + k) * st8;
          const double y = add ? ov[k] + r[k] : r[k];
          // the default policy: a row's 512 bytes start anywhere in a cache
          // line, and the neighbouring work item writes the rest of its edge
          // lines; the streaming hint evicts them half-written
          at(dst, o) = y;
          if (KIND == 1 && cpy) at(cpy, o) = y;
        }
    }
  }
