// condense_tile.h -- blocked elimination of one cell system per workgroup (small
// ones: per wavefront) with the interior factors in LDS and every product on FP64 MFMA tiles (family 11;
// also the elimination of the flux families' reduced systems).  Included by
// hdg_kernels.hip.
#pragma once

// The cell system [A_ii A_ib b_i; A_bi A_bb b_b] is condensed as
//   P A_ii = L U                    (partial pivoting, getrf's choice)
//   Y  = L^-1 P [A_ib b_i]          forward substitution, NT x 16-row tiles
//   Z  = U^-T A_bi^T                the boundary rows of the LU, transposed
//   S  = A_bb - Z^T Y,  g = b_b - Z^T y
// which is what the elimination of the whole system computes, with only A_ii
// (NI <= 16 NT rows) inside the sequential part.
//  - A_ii sits in LDS (column-major, leading dimension 16 NT + 8: the four
//    16-row groups of an MFMA operand then cover every bank twice) and is
//    factored by panels of 16 columns: one wavefront holds the panel one row per
//    lane (two rows for NT > 4), so a pivot step is a DPP maximum, a row
//    broadcast through SGPRs and one FMA per panel column, without a barrier.
//    The rows of an eliminated pivot keep taking part with the columns already
//    eliminated, which leaves the inverse of the panel's unit-lower block in
//    place of its multipliers.  The wavefronts then permute their
//    16-column strips, form U12 with that inverse and apply the rank-16 update.
//  - the columns of [A_ib b_i] and the rows of A_bi are independent: a
//    wavefront takes 16 of each as NT accumulator tiles, whose layout is both
//    an A and a B operand of the next product, so the substitutions and S run
//    from registers.  Only Y is exchanged between wavefronts, through LDS,
//    `chunk` strips at a time.
// What bounds it, in cycles per cell of one workgroup or wavefront (Darcy 24^3
// k=3, 339,000, two workgroups on a CU): panels 79,500 (the pivot chain, some
// 130 instructions a column for one wavefront), Y 61,000 and Z 47,000 (entries
// from the tables, then chains of dependent MFMA), S with its staging 69,000,
// A_ii 32,000, the inverse 21,000; MFMA issue itself is about a fifth.
// Measured, condensation kernels in all, against the kernels they replace
// (register-grid, workspace-panel and blocked eliminations, the reduced systems
// formed by kernels of their own and written to memory, the inverses by another):
//   map level, 4,096 cells of 108 + 54, both maps   17.1 -> 5.1 ms
//   Darcy 64^3 k=2 (27 + 54 of 108 + 54)            25.2 -> 9.2 ms
//   Darcy 24^3 k=3 (64 + 96 of 256 + 96)            17.6 -> 3.3 ms
//   elasticity 5,814 cells k=2 (60 + 108)            9.4 -> 1.5 ms
//   elasticity 1,728 cells k=3 (105 + 180)          12.1 -> 2.1 ms
// The symmetry of the reduced systems (half of S formed, both halves stored; a
// column's weights looked up once) and no scratch memory gave 11.9 -> 9.7, 6.2 ->
// 3.5, 2.8 -> 1.6 and 3.3 -> 2.2 ms of the last four; not storing U, which no
// recovery of theirs reads, the rest.  No instance uses scratch memory: the
// addresses of a generator's tables, hoisted out of the cell loop, had cost the
// wavefront kernels of two row tiles 36 to 64 bytes a lane, and those of one tile
// the fourth wavefront a SIMD (RefGen::begin; 64^3 k=2 9.43 -> 9.24 ms, 2D k=3,
// 16,247 cells, 161 -> 141 us, 3D k=1, 13,547 cells, 127 -> 115 us).

// c ? a : b and c ? a : 0 by masks.  The compiler turns a conditional of loaded
// values into branches around the loads, one latency after the other; through
// these every load of a tile is in flight at once.
__device__ inline int lane_mask(bool c) {
  int m = c ? -1 : 0;
  asm("" : "+v"(m));  // (or it is recognised as the conditional it came from)
  return m;
}
__device__ inline double pick(bool c, double a, double b) {
  const int m = lane_mask(c);
  return __hiloint2double((__double2hiint(a) & m) | (__double2hiint(b) & ~m),
                          (__double2loint(a) & m) | (__double2loint(b) & ~m));
}
__device__ inline double keep_if(bool c, double a) {
  const int m = lane_mask(c);
  return __hiloint2double(__double2hiint(a) & m, __double2loint(a) & m);
}

// A copy of v the compiler cannot see through: what is built on it (bounds,
// masks, addresses) stays in the loop or phase that uses it, where hoisted out
// of the cell loop it spills.
__device__ inline int opaque_v(int v) {
  asm volatile("" : "+v"(v));
  return v;
}
__device__ inline int opaque_s(int v) {
  asm volatile("" : "+s"(v));
  return v;
}

// Where a generator's entries go: rows and columns of the four blocks, and the
// right-hand side.  (RefGen below has forms of its own for each.)
template <class G>
struct TileSrc {
  using Sh = typename G::Shared;
  static constexpr bool kSym = false;  // A_bi^T = +-A_ib, A_ii, A_bb and so S symmetric
  struct Col {  // a boundary unknown: a column of A_ib (nb: b_i), a row of A_bi
    int c;
  };
  __device__ static Col col(const G&, const Sh&, int c, int) { return {c}; }
  __device__ static double ii(const G& g, const Sh& sh, int r, int c, int64_t cell, double*) {
    return GenCall<G>::entry(g, sh, r, c, cell);
  }
  __device__ static double ib(const G& g, const Sh& sh, const Col& b, int r, int ni, int nb,
                              int64_t cell) {
    return GenCall<G>::entry(g, sh, r, ni + min(b.c, nb), cell);
  }
  __device__ static double bi(const G& g, const Sh& sh, const Col& b, int k, int ni, int nb,
                              int64_t cell) {
    return GenCall<G>::entry(g, sh, ni + min(b.c, nb - 1), k, cell);
  }
  __device__ static double bb(const G& g, const Sh& sh, const Col& r, int c, int ni, int nb,
                              int64_t cell) {
    return GenCall<G>::entry(g, sh, ni + min(r.c, nb - 1), ni + min(c, nb), cell);
  }
};

// What a generator sets up once per workgroup (nothing, by default).
template <class G>
__device__ inline void tile_start(const G&, typename G::Shared&, int, int) {}

// A table entry at a wave-uniform base and a lane's 32-bit byte offset (one
// address register per lane).
__device__ inline double table_at(const double* base, unsigned bytes) {
  return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(base) + bytes);
}

// --------------------------------------------------------------------------
// The reduced system of the flux families as a generator: the flux unknowns
// eliminated through the reference decomposition (build_flux_ref),
//   R = R0 - s_r sum_(e,e') W(e, e') H_ee',   s_r = -1 on the potential rows,
// +1 (Darcy) or -1 (elasticity) on the trace rows, R0 = [A_uu A_ub b_u; A_bu
// A_bb 0].  Nothing of R is kept in memory: the elimination asks for every
// entry once, 12 products at most on the potential columns, 4 with a trace
// column and 2 between traces, from tables that all cells share (L2) and the
// cell's weights (LDS).  A singular C leaves a zero system.
// --------------------------------------------------------------------------
template <int PHYS, int D, int MAXNR, int MAXZ>
struct RefGen {
  static constexpr int ND = PHYS == kDarcy ? 1 : D;              // potential components
  static constexpr int NP = PHYS == kDarcy ? D * (D + 1) / 2 : D * D;
  static constexpr int NW = ND * ND * D * D;
  static constexpr int TA = PHYS == kDarcy ? 28 : 63;            // alpha: tau terms
  static constexpr bool kHeavy = true;     // an entry's own loads fill the registers
  static constexpr bool kStoresY = true;   // out.Y is always there
  Tables T;
  MeshDev M;
  struct Shared {
    double alpha[kMaxAlpha];
    double W[NW];                                // [d][d'][e][e']
    double rhs[MAXNR];
    double z[PHYS == kDarcy ? MAXZ : 1];
    // potential row: scalar index | component << 16; trace column: scalar index |
    // its place in W's [d'][.][e'] << 10 | component << 16 | facet << 20
    int idx[MAXNR];
  };

  __device__ void start(Shared& sh, int tid, int nthreads) const {
    const int nq = T.nq, nm = T.nm, nu = ND * nq;
    for (int r = tid; r < nu + T.nb; r += nthreads) {
      if (r < nu) {
        const int d = r / nq;
        sh.idx[r] = (r - d * nq) | d << 16;
      } else {
        const int b = r - nu, f = b / T.ntf, c = b - f * T.ntf, d = c / nm;
        sh.idx[r] = (f * nm + c - d * nm) | (d * D * D + D - 1 - f / 2) << 10 | d << 16 | f << 20;
      }
    }
  }
  __device__ double cof(const Shared& sh, int e, int a) const {
    return PHYS == kDarcy ? -sh.alpha[1 + e * D + a] : sh.alpha[36 + e * D + a];
  }
  __device__ void begin(int64_t cell, Shared& sh) const {
    // (opaque: what begin() addresses, kept for the next cell, spills)
    const int tid = opaque_v(threadIdx.x), nthreads = blockDim.x;
    const int na = T.na, nu = ND * T.nq, nr = nu + T.nb;
    const double* al = M.alpha + cell * kMaxAlpha;
    const double* b = M.srcq + cell * srcq_stride(T);
    for (int t = tid; t < kMaxAlpha; t += nthreads) sh.alpha[t] = al[t];
    const double* bu = b + (T.fo_P ? T.ni : na);  // in the basis of the tables
    for (int t = tid; t < nr; t += nthreads) sh.rhs[t] = t < nu ? bu[t] : 0.0;
    int load = 0;  // the flux equation's load (none: its terms are skipped)
    if (PHYS == kDarcy)
      for (int t = tid; t < na; t += nthreads) load |= b[t] != 0.0;
    load = __syncthreads_or(load);
    bool bad;
    double inva = 0.0, cd = 0.0, co = 0.0, cs = 0.0;
    if (PHYS == kDarcy) {
      bad = !(sh.alpha[0] != 0.0);
      inva = bad ? 0.0 : 1.0 / sh.alpha[0];
    } else {
      // C: k0 on the normal components, k1 between them, ks on the shear ones
      const double k0 = sh.alpha[0], k1 = sh.alpha[D == 3 ? 3 : 2], ks = sh.alpha[7];
      const double dm = k0 - k1, dn = k0 + (D - 1) * k1;
      bad = dm == 0.0 || dn == 0.0 || ks == 0.0;
      cd = bad ? 0.0 : (k0 + (D - 2) * k1) / (dm * dn);
      co = bad ? 0.0 : -k1 / (dm * dn);
      cs = bad ? 0.0 : 1.0 / ks;
    }
    for (int t = tid; t < NW; t += nthreads) {
      const int e2 = t % D, e = t / D % D;
      double v = 0.0;
      if (PHYS == kDarcy) {
#pragma unroll
        for (int a = 0; a < D; ++a) v = fma(cof(sh, e, a), cof(sh, e2, a), v);
        v *= inva;
      } else {
        // W(e, e') = sum over the stress components s of d and s' of d' of
        // C^-1[s][s'] c_e,partner c_e',partner
        const int d2 = t / (D * D) % D, d = t / (D * D * D);
        double x = 0.0;
        if (d == d2) {
#pragma unroll
          for (int a = 0; a < D; ++a)
            if (a != d) x = fma(cof(sh, e, a), cof(sh, e2, a), x);
        } else {
          x = cof(sh, e, d2) * cof(sh, e2, d);
        }
        v = fma(cs, x, (d == d2 ? cd : co) * (cof(sh, e, d) * cof(sh, e2, d2)));
      }
      sh.W[t] = v;
    }
    if (PHYS == kDarcy && load) {  // rhs += s_r sum_e H_e^T z_e, z_e = C^-1 sum_a c_ea b_q,a
      const int np = T.np, nk = D * np, nrs = T.nq + T.nF * T.nm;
      for (int t = tid; t < nk; t += nthreads) {
        const int e = t / np, j = t - e * np;
        double v = 0.0;
#pragma unroll
        for (int a = 0; a < D; ++a) v = fma(cof(sh, e, a), b[a * np + j], v);
        sh.z[t] = v * inva;
      }
      __syncthreads();
      for (int r = tid; r < nr; r += nthreads) {
        // (a trace column has its facet's direction only)
        const int f = r < nu ? -1 : D - 1 - (sh.idx[r] >> 20) / 2;
        const int k0 = f < 0 ? 0 : f * np, k1 = f < 0 ? nk : k0 + np;
        double x = 0.0;
#pragma unroll 4
        for (int k = k0; k < k1; ++k) x = fma(T.fr_hm[k * nrs + r], sh.z[k], x);
        sh.rhs[r] = r < nu ? sh.rhs[r] + x : -x;
      }
    }
    if (bad) {
      __syncthreads();
      for (int t = tid; t < 2 * D; t += nthreads) sh.alpha[TA + t] = 0.0;
      for (int t = tid; t < nr; t += nthreads) sh.rhs[t] = 0.0;
    }
  }
  // entry (r, c) of R_uu; keep: R0's term of it, of the first component.  (H_ee'
  // read as the transpose of H_e'e: consecutive lanes, rows, read consecutive
  // values.  A lane per cache line, the elimination of Darcy 24^3 k=3 took 5.0
  // instead of 2.9 ms.)
  __device__ double uu(const Shared& sh, int r, int c, double* keep) const {
    const int nq = T.nq, nqq = nq * nq;
    double x = 0.0, t = 0.0;
    bool own = true;
    unsigned at;
    if (PHYS == kDarcy) {
      at = 8 * (c * nq + r);
      int p = 0;
#pragma unroll
      for (int e = 0; e < D; ++e)
#pragma unroll
        for (int e2 = e; e2 < D; ++e2, ++p)
          x = fma(sh.W[e * D + e2], table_at(T.fr_uu + p * nqq, at), x);
    } else {
      const int ir = sh.idx[r], ic = sh.idx[c], d = ir >> 16, d2 = ic >> 16;
      at = 8 * ((ic & 0xffff) * nq + (ir & 0xffff));
      own = d == d2;
      const double* w = sh.W + (d * D + d2) * D * D;
#pragma unroll
      for (int p = 0; p < NP; ++p)
        x = fma(w[p], table_at(T.fr_uu + (p % D * D + p / D) * nqq, at), x);
    }
#pragma unroll
    for (int f = 0; f < 2 * D; ++f) t = fma(sh.alpha[TA + f], table_at(T.Fqq + f * nqq, at), t);
    if (PHYS != kDarcy) t = keep_if(own, t);
    if (keep && r < nq && c < nq) keep[c * nq + r] = t;
    return t + x;
  }
  // A trace column and what its entries share.
  struct Col {
    unsigned at;  // byte offset of its scalar index
    int id;
    double tau, w[PHYS == kDarcy ? D : 1];
  };
  __device__ Col col(const Shared& sh, int b) const {  // b: the trace unknown
    Col k;
    k.id = sh.idx[ND * T.nq + b];
    k.at = 8 * (k.id & 1023);
    const int f = k.id >> 20;
    k.tau = sh.alpha[TA + f];
    if (PHYS == kDarcy)
#pragma unroll
      for (int e = 0; e < D; ++e) k.w[e] = sh.W[e * D + D - 1 - f / 2];
    return k;
  }
  // the potential row u of it
  __device__ double ub(const Shared& sh, const Col& k, int u) const {
    const int nq = T.nq, nbs = T.nF * T.nm;
    double x = 0.0, tau = k.tau;
    unsigned at;
    if (PHYS == kDarcy) {
      at = k.at + 8u * nbs * u;
#pragma unroll
      for (int e = 0; e < D; ++e) x = fma(k.w[e], table_at(T.fr_ub + e * nq * nbs, at), x);
    } else {
      const int iu = sh.idx[u], d = iu >> 16;
      at = k.at + 8u * nbs * (iu & 0xffff);
      const double* w = sh.W + d * D * D * D + (k.id >> 10 & 31);
#pragma unroll
      for (int e = 0; e < D; ++e) x = fma(w[e * D], table_at(T.fr_ub + e * nq * nbs, at), x);
      tau = keep_if(d == (k.id >> 16 & 15), tau);
    }
    return fma(-tau, table_at(T.fr_qm, at), x);
  }
  // the trace row k, column b of A_bb
  __device__ double bb(const Shared& sh, const Col& k, int b) const {
    const int nbs = T.nF * T.nm;
    const int id = sh.idx[ND * T.nq + b], d = k.id >> 16 & 15, fix = D - 1 - (k.id >> 20) / 2;
    const unsigned at = k.at + 8u * nbs * (id & 1023);  // (symmetric: consecutive lanes, rows)
    const double w = sh.W[d * D * D * D + fix * D + (id >> 10 & 31)];
    double tau = k.tau;
    if (PHYS != kDarcy) tau = keep_if(d == (id >> 16 & 15), tau);
    const double x = fma(tau, table_at(T.fr_mm, at), w * table_at(T.fr_bb, at));
    return PHYS == kDarcy ? -x : x;
  }
};
template <int PHYS, int D, int MAXNR, int MAXZ>
struct TileSrc<RefGen<PHYS, D, MAXNR, MAXZ>> {
  using G = RefGen<PHYS, D, MAXNR, MAXZ>;
  using Sh = typename G::Shared;
  static constexpr bool kSym = true;
  using Col = typename G::Col;
  __device__ static Col col(const G& g, const Sh& sh, int c, int nb) {
    return g.col(sh, min(c, nb - 1));
  }
  __device__ static double ii(const G& g, const Sh& sh, int r, int c, int64_t, double* keep) {
    return g.uu(sh, r, c, keep);
  }
  __device__ static double ib(const G& g, const Sh& sh, const Col& b, int r, int, int, int64_t) {
    return g.ub(sh, b, r);
  }
  __device__ static double bi(const G& g, const Sh& sh, const Col& b, int k, int, int, int64_t) {
    const double x = g.ub(sh, b, k);
    return PHYS == kDarcy ? -x : x;
  }
  __device__ static double bb(const G& g, const Sh& sh, const Col& r, int c, int, int nb, int64_t) {
    return g.bb(sh, r, min(c, nb - 1));
  }
};
template <int PHYS, int D, int MAXNR, int MAXZ>
struct GenCall<RefGen<PHYS, D, MAXNR, MAXZ>> {  // (the backward map only)
  using G = RefGen<PHYS, D, MAXNR, MAXZ>;
  __device__ static double entry(const G&, const typename G::Shared&, int, int, int64_t) {
    return 0.0;
  }
};
template <int PHYS, int D, int MAXNR, int MAXZ>
__device__ inline void tile_start(const RefGen<PHYS, D, MAXNR, MAXZ>& g,
                                  typename RefGen<PHYS, D, MAXNR, MAXZ>::Shared& sh, int tid,
                                  int nthreads) {
  g.start(sh, tid, nthreads);
  __syncthreads();
}

// The factored interior block F of one cell in LDS and the products with it.
// One lane's share of a 16 x 16 tile: row or k index 4 v + q4, column i16.
template <int NT>
struct Tile {
  static constexpr int N = 16 * NT;
  // (with at most two tiles the last few hundred bytes buy another cell on the CU)
  static constexpr int LD = N + (NT <= 2 ? 4 : 8);
  static constexpr int T = N > 64 ? 2 : 1;  // rows per lane of a panel
  static constexpr int kF = N * LD;         // doubles of F
  static constexpr int YLD = N + 4;         // a staged strip's column: lanes 4 banks apart
  static constexpr int kStrip = YLD * 16;   // doubles of a staged strip
  double* F;
  int lane, i16, q4;

  __device__ Tile(double* f, int lane_) : F(f), lane(lane_), i16(lane_ & 15), q4(lane_ >> 4) {}

  // A operands [i16][4 v + q4] of the triangular tiles.  L(I, J), I > J, and
  // U(I, J), I < J, share one form.  The diagonal tile holds L_II^-1 strictly
  // below (unit diagonal) and on and above it U_II with the 4 x 4 blocks on its
  // diagonal replaced by their inverses, for a substitution by groups of 4 rows.  (L_II^-1 is harmless, its multipliers being at most 1;
  // an explicit U_II^-1 was measured 10 to 20 times less exact in S for 2D
  // elasticity with k = 3, a group's error stays in the group's residual.)
  __device__ double lu(int I, int J, int v) const {
    return F[(16 * J + 4 * v + q4) * LD + 16 * I + i16];
  }
  __device__ double lut(int I, int J, int v) const {  // of the transposes: tile (J, I)
    return F[(16 * I + i16) * LD + 16 * J + 4 * v + q4];
  }
  __device__ double loinv(int I, int v) const {
    const int k = 4 * v + q4;
    return pick(k < i16, lu(I, I, v), k == i16 ? 1.0 : 0.0);
  }
  __device__ double loinvt(int I, int v) const {  // L_II^-T
    const int k = 4 * v + q4;
    return pick(k > i16, lut(I, I, v), k == i16 ? 1.0 : 0.0);
  }
  __device__ double utinv(int I, int v) const {  // the inverse of group v of U_II^T
    return keep_if(i16 >> 2 == v && 4 * v + q4 <= i16, lut(I, I, v));
  }
  __device__ double utoff(int I, int v) const {  // -U_II^T, columns of group v below it
    return keep_if(i16 >> 2 > v, -lut(I, I, v));
  }
  __device__ double upinv(int I, int v) const {  // the same of U_II
    return keep_if(i16 >> 2 == v && i16 <= 4 * v + q4, lu(I, I, v));
  }
  __device__ double upoff(int I, int v) const {
    return keep_if(i16 >> 2 < v, -lu(I, I, v));
  }
  // a strip x of 16 columns: x <- L^-1 x
  __device__ void forward(dbl4 (&x)[NT]) const {
#pragma unroll
    for (int I = 0; I < NT; ++I) {
      if (NT > 1) __builtin_amdgcn_sched_barrier(0);  // operands of one row of tiles at a time
      dbl4 acc = x[I];
#pragma unroll
      for (int J = 0; J < I; ++J) {
        if (NT > 4) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int v = 0; v < 4; ++v)
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-lu(I, J, v), x[J][v], acc, 0, 0, 0);
      }
      dbl4 r = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int v = 0; v < 4; ++v)
        r = __builtin_amdgcn_mfma_f64_16x16x4f64(loinv(I, v), acc[v], r, 0, 0, 0);
      x[I] = r;
    }
  }
  // x <- U^-T x
  __device__ void forward_ut(dbl4 (&x)[NT]) const {
    const dbl4 zero = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int I = 0; I < NT; ++I) {
      if (NT > 1) __builtin_amdgcn_sched_barrier(0);  // operands of one row of tiles at a time
      dbl4 acc = x[I];
#pragma unroll
      for (int J = 0; J < I; ++J) {
        if (NT > 4) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int v = 0; v < 4; ++v)
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-lut(I, J, v), x[J][v], acc, 0, 0, 0);
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        // (the product has the group's rows only: element v of every lane)
        const dbl4 r = __builtin_amdgcn_mfma_f64_16x16x4f64(utinv(I, v), acc[v], zero, 0, 0, 0);
        acc[v] = r[v];
        if (v < 3)
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(utoff(I, v), acc[v], acc, 0, 0, 0);
      }
      x[I] = acc;
    }
  }
  // x <- L^-T x
  __device__ void backward_lt(dbl4 (&x)[NT]) const {
#pragma unroll
    for (int I = NT - 1; I >= 0; --I) {
      if (NT > 1) __builtin_amdgcn_sched_barrier(0);  // operands of one row of tiles at a time
      dbl4 acc = x[I];
#pragma unroll
      for (int J = I + 1; J < NT; ++J) {
        if (NT > 4) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int v = 0; v < 4; ++v)
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-lut(I, J, v), x[J][v], acc, 0, 0, 0);
      }
      dbl4 r = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int v = 0; v < 4; ++v)
        r = __builtin_amdgcn_mfma_f64_16x16x4f64(loinvt(I, v), acc[v], r, 0, 0, 0);
      x[I] = r;
    }
  }
  // x <- U^-1 x
  __device__ void backward(dbl4 (&x)[NT]) const {
    const dbl4 zero = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int I = NT - 1; I >= 0; --I) {
      if (NT > 1) __builtin_amdgcn_sched_barrier(0);  // operands of one row of tiles at a time
      dbl4 acc = x[I];
#pragma unroll
      for (int J = I + 1; J < NT; ++J) {
        if (NT > 4) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int v = 0; v < 4; ++v)
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-lu(I, J, v), x[J][v], acc, 0, 0, 0);
      }
#pragma unroll
      for (int v = 3; v >= 0; --v) {
        const dbl4 r = __builtin_amdgcn_mfma_f64_16x16x4f64(upinv(I, v), acc[v], zero, 0, 0, 0);
        acc[v] = r[v];
        if (v > 0)
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(upoff(I, v), acc[v], acc, 0, 0, 0);
      }
      x[I] = acc;
    }
  }

  // Factors the 16 columns from c0 on, one wavefront, one row per lane (T
  // rows).  Each step eliminates the column in slot 0 and stores the others
  // one slot lower, so the loop stays rolled (unrolled, the
  // kernel was 83 KB of code and slower); after 16 steps the columns are back in order.  A
  // pivoted row keeps its place in the later steps' columns already
  // eliminated, which leaves L^-1 of the block below its diagonal.  The
  // identity padding (rows and columns from ni on) takes no part: its columns
  // only pass through the slots.  s_pos receives the
  // position of every row, dinv 1 / U[c][c] (0 for a zero pivot).
  __device__ void panel(int c0, int ni, int* s_pos, double* dinv, int& info) const {
    double a[T][16];
    int pos[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int r = lane + 64 * t;
      pos[t] = r;
#pragma unroll
      for (int c = 0; c < 16; ++c) a[t][c] = r < N ? F[(c0 + c) * LD + r] : 0.0;
    }
    const int jn = min(16, ni - c0);
#pragma unroll 1
    for (int j = 0; j < jn; ++j) {
      const int col = c0 + j;
      // every lane's own reciprocal, off the pivot's critical path
      double ri[T];
#pragma unroll
      for (int t = 0; t < T; ++t) ri[t] = a[t][0] != 0.0 ? 1.0 / a[t][0] : 0.0;
      // largest magnitude, smallest position on ties
      int64_t key = -1;
      int kpos = INT_MAX;
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const bool cand = lane + 64 * t < ni && pos[t] >= col;
        const int64_t kt = cand ? dbits(fabs(a[t][0])) : (int64_t)-1;
        const bool take = kt > key || (kt == key && pos[t] < kpos);
        key = take ? kt : key;
        kpos = take ? pos[t] : kpos;
      }
      const int hi = (int)(key >> 32);
      const int mhi = wave_max_i32(hi);
      uint64_t who = __ballot(hi == mhi);
      if (who & (who - 1)) {  // several lanes share the high word
        const int64_t m = wave_max_i64(hi == mhi ? key : (int64_t)-1);
        const int mp = wave_min_i32(key == m ? kpos : INT_MAX);
        who = __ballot(key == m && kpos == mp);
      }
      const int p = __builtin_ffsll((long long)who) - 1;
      const int ppos = __builtin_amdgcn_readlane(kpos, p);
      const int tp = T > 1 && __builtin_amdgcn_readlane(pos[0], p) != ppos ? 1 : 0;
      double prow[16], rinv;
      if (T == 1 || tp == 0) {  // wave-uniform
        rinv = wave_readlane_f64(ri[0], p);
#pragma unroll
        for (int c = 0; c < 16; ++c) prow[c] = wave_readlane_f64(a[0][c], p);
      } else {
        rinv = wave_readlane_f64(ri[T - 1], p);
#pragma unroll
        for (int c = 0; c < 16; ++c) prow[c] = wave_readlane_f64(a[T - 1][c], p);
      }
      const double pv = prow[0];
      if (pv == 0.0 && info == 0) info = col + 1;
      if (lane == 0) dinv[col] = rinv;
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const bool isp = lane == p && t == tp;
        if (pos[t] == col) pos[t] = ppos;  // LAPACK interchange of col and ppos
        if (isp) pos[t] = col;
        const bool act = pos[t] > col;
        const double a0 = a[t][0];
        const double l = act ? a0 * rinv : 0.0;
        if ((N >= 64 * (t + 1) || lane + 64 * t < N) && (act || isp))
          F[col * LD + lane + 64 * t] = isp ? pv : l;
#pragma unroll
        for (int c = 1; c < 16; ++c) a[t][c - 1] = fma(-l, prow[c], a[t][c]);
        a[t][15] = act ? -l : (isp ? 1.0 : a0);
      }
    }
#pragma unroll 1
    for (int j = jn; j < 16; ++j)
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const double a0 = a[t][0];
#pragma unroll
        for (int c = 1; c < 16; ++c) a[t][c - 1] = a[t][c];
        a[t][15] = a0;
      }
    // the panel's pivot rows: U above the diagonal, L^-1 below it
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int r = lane + 64 * t, jj = pos[t] - c0;
      if (r < N) {
        s_pos[r] = pos[t];
        if (jj >= 0 && jj < 16)
#pragma unroll
          for (int c = 0; c < 16; ++c)
            if (c != jj) F[(c0 + c) * LD + r] = a[t][c];
      }
    }
  }
  // Moves the rows of strip s to their positions.
  __device__ void permute(int s, const int* s_pos) const {
    double b[T][16];
    int ps[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int r = lane + 64 * t;
      ps[t] = r < N ? s_pos[r] : r;
#pragma unroll
      for (int c = 0; c < 16; ++c) b[t][c] = r < N ? F[(16 * s + c) * LD + r] : 0.0;
    }
    wave_sync_lds();
#pragma unroll
    for (int t = 0; t < T; ++t)
      if (lane + 64 * t < N && ps[t] != lane + 64 * t)
#pragma unroll
        for (int c = 0; c < 16; ++c) F[(16 * s + c) * LD + ps[t]] = b[t][c];
    wave_sync_lds();
  }
  // U_Js and the rank-16 update of strip s behind panel J.
  __device__ void update(int J, int s) const {
    dbl4 u = {0.0, 0.0, 0.0, 0.0};
    double* const col = F + (16 * s + i16) * LD;
#pragma unroll
    for (int v = 0; v < 4; ++v)
      u = __builtin_amdgcn_mfma_f64_16x16x4f64(loinv(J, v), col[16 * J + 4 * v + q4], u, 0, 0, 0);
#pragma unroll
    for (int v = 0; v < 4; ++v) col[16 * J + 4 * v + q4] = u[v];
#pragma unroll 1
    for (int I = J + 1; I < NT; I += 2) {  // two tiles in flight
      const int I2 = min(I + 1, NT - 1);
      dbl4 acc, acc2;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        acc[v] = col[16 * I + 4 * v + q4];
        acc2[v] = col[16 * I2 + 4 * v + q4];
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-lu(I, J, v), u[v], acc, 0, 0, 0);
        acc2 = __builtin_amdgcn_mfma_f64_16x16x4f64(-lu(I2, J, v), u[v], acc2, 0, 0, 0);
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        col[16 * I + 4 * v + q4] = acc[v];
        if (I + 1 < NT) col[16 * I2 + 4 * v + q4] = acc2[v];
      }
    }
  }
  // The inverses of the diagonal 4 x 4 blocks of U_JJ in their place, a lane per
  // column.
  __device__ void factor_diag(int J, const double* dinv) const {
    const int v = 4 * (i16 >> 2);
    double* const D = F + (16 * J + v) * LD + 16 * J + v;  // the column's block
    const double* di = dinv + 16 * J + v;
    double r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = v + i == i16 ? 1.0 : 0.0;
#pragma unroll
    for (int i = 3; i >= 0; --i) {
      r[i] *= di[i];
#pragma unroll
      for (int h = 0; h < i; ++h) r[h] = fma(-D[i * LD + h], r[i], r[h]);
    }
    wave_sync_lds();
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (v + i <= i16 && q4 == 0) D[(i16 - v) * LD + i] = r[i];
  }
};

// A_ii into F, padded to whole tiles with the identity, by nthreads threads.
// (Every entry by itself also where A_ii is symmetric: the mirrored triangle
// was measured 8 times less exact in S, 5.3e-11 against 6.3e-12 of the largest
// entry, for elasticity with k = 3 in the displacement's nodal basis.)
template <int NT, class Gen>
__device__ inline void tile_load(const Gen& gen, const typename Gen::Shared& sh, double* F,
                                 int64_t cell, int ni, int tid, int nthreads, double* keep) {
  constexpr int N = Tile<NT>::N, LD = Tile<NT>::LD;
  constexpr int AT = Gen::kHeavy ? 1 : 4;  // entries in flight
  for (int t0 = tid; t0 < N * N; t0 += AT * nthreads) {
    double v[AT];
#pragma unroll
    for (int u = 0; u < AT; ++u) {
      const int t = t0 + u * nthreads, c = t / N, r = t - c * N;
      const bool in = r < ni && c < ni;
      const double x = TileSrc<Gen>::ii(gen, sh, min(r, ni - 1), min(c, ni - 1), cell,
                                        in ? keep : nullptr);
      v[u] = pick(in, x, r == c ? 1.0 : 0.0);
    }
#pragma unroll
    for (int u = 0; u < AT; ++u) {
      const int t = t0 + u * nthreads, c = t / N, r = t - c * N;
      if (t < N * N) F[c * LD + r] = v[u];
    }
  }
}

// One strip of P [A_ib b_i] (column c of this lane) and of A_bi^T (row c).
template <int NT, class Gen>
__device__ inline void tile_strip_y(const Gen& gen, const typename Gen::Shared& sh,
                                    const int* perm, const typename TileSrc<Gen>::Col& b,
                                    dbl4 (&y)[NT], int c, int q, int ni, int nb, int64_t cell) {
#pragma unroll
  for (int I = 0; I < NT; ++I) {
    __builtin_amdgcn_sched_barrier(0);  // a tile's loads in flight, not the strip's
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int k = 16 * I + 4 * v + q;
      const double x = TileSrc<Gen>::ib(gen, sh, b, perm[min(k, ni - 1)], ni, nb, cell);
      y[I][v] = keep_if(k < ni, x);  // (columns past nb repeat the last: not stored)
    }
  }
  if constexpr (TileSrc<Gen>::kSym)
    if (__ballot(c == nb)) {  // wave-uniform: the strip with b_i
#pragma unroll
      for (int I = 0; I < NT; ++I)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int k = 16 * I + 4 * v + q;
          const double x = sh.rhs[perm[min(k, ni - 1)]];
          y[I][v] = pick(c == nb, keep_if(k < ni, x), y[I][v]);
        }
    }
}
template <int NT, class Gen>
__device__ inline void tile_strip_z(const Gen& gen, const typename Gen::Shared& sh,
                                    const typename TileSrc<Gen>::Col& b, dbl4 (&z)[NT], int q,
                                    int ni, int nb, int64_t cell) {
#pragma unroll
  for (int I = 0; I < NT; ++I) {
    __builtin_amdgcn_sched_barrier(0);  // a tile's loads in flight, not the strip's
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int k = 16 * I + 4 * v + q;
      const double x = TileSrc<Gen>::bi(gen, sh, b, min(k, ni - 1), ni, nb, cell);
      z[I][v] = keep_if(k < ni, x);
    }
  }
}
// S^T tile: columns 16 s + 4 v + q of [A_bb b_b], row r of this lane (b its Col).
template <class Gen>
__device__ inline dbl4 tile_bb(const Gen& gen, const typename Gen::Shared& sh,
                               const typename TileSrc<Gen>::Col& b, int r, int s, int q, int ni,
                               int nb, int64_t cell) {
  dbl4 a;
#pragma unroll
  for (int v = 0; v < 4; ++v)
    a[v] = TileSrc<Gen>::bb(gen, sh, b, 16 * s + 4 * v + q, ni, nb, cell);
  if constexpr (TileSrc<Gen>::kSym)
    if (16 * s + 16 > nb) {  // wave-uniform: the strip with b_b
      const double x = sh.rhs[ni + min(r, nb - 1)];
#pragma unroll
      for (int v = 0; v < 4; ++v) a[v] = pick(16 * s + 4 * v + q == nb, x, a[v]);
    }
  return a;
}
// (mirror: and its transpose, of a symmetric S)
__device__ inline void tile_store_s(const CondenseOut& out, const dbl4& acc, int r, int s, int q,
                                    int nb, int64_t cell, bool mirror) {
  if (r >= nb) return;
  if (mirror && out.S) {
    double* dst = out.S + (cell * nb + r) * nb + 16 * s + q;
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (16 * s + 4 * v + q < nb) dst[4 * v] = acc[v];
  }
  if (16 * s + 16 <= nb) {  // (wave-uniform: a whole tile needs no guards)
    if (out.S) {
      double* dst = out.S + (cell * nb + 16 * s + q) * nb + r;
#pragma unroll
      for (int v = 0; v < 4; ++v) dst[4 * v * nb] = acc[v];
    }
    return;
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int c = 16 * s + 4 * v + q;
    if (c < nb) {
      if (out.S) out.S[(cell * nb + c) * nb + r] = acc[v];
    } else if (c == nb && out.g) {
      out.g[cell * nb + r] = acc[v];
    }
  }
}
// The first column strip from s on whose tile row strip t forms: every one, or
// of a symmetric S one of each pair (t, s), (s, t), as many to each t: the last
// strip (with g) and the half of the others that follow t cyclically.
template <bool SYM>
__device__ inline int tile_next(int t, int s, int s1, int nstrip) {
  if (SYM)
    for (; s < s1; ++s) {
      const int m = nstrip - 1, d = s < t ? s - t + m : s - t;
      if (s == m || (t < m && (2 * d < m || (2 * d == m && t < s)))) break;
    }
  return s;
}
// Column c of an [col][row] output of ni rows from a strip.
template <int NT>
__device__ inline void tile_store_strip(double* dst, const dbl4 (&y)[NT], int c, int q, int ni) {
  dst += (int64_t)c * ni + q;
#pragma unroll
  for (int I = 0; I < NT; ++I) {
    if (16 * I + 16 <= ni) {
#pragma unroll
      for (int v = 0; v < 4; ++v) dst[16 * I + 4 * v] = y[I][v];
    } else if (16 * I < ni) {
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (16 * I + 4 * v + q < ni) dst[16 * I + 4 * v] = y[I][v];
    }
  }
}

// Rows 16 s + i16 of A_ii^-1, stored [col][row].
template <int NT>
__device__ inline void tile_inverse(const Tile<NT>& tl, const int* perm, dbl4 (&x)[NT], int s,
                                    int ni, double* dst) {
  const int c = 16 * s + opaque_v(tl.i16), q = opaque_v(tl.q4);
#pragma unroll
  for (int I = 0; I < NT; ++I)
#pragma unroll
    for (int v = 0; v < 4; ++v) x[I][v] = 16 * I + 4 * v + q == c ? 1.0 : 0.0;
  tl.forward_ut(x);
  tl.backward_lt(x);
  if (c >= ni) return;
  dst += c;
#pragma unroll
  for (int I = 0; I < NT; ++I) {
    if (16 * I + 16 <= ni) {
#pragma unroll
      for (int v = 0; v < 4; ++v) dst[perm[16 * I + 4 * v + q] * ni] = x[I][v];
    } else if (16 * I < ni) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int k = 16 * I + 4 * v + q;
        if (k < ni) dst[perm[k] * ni] = x[I][v];
      }
    }
  }
}

// --------------------------------------------------------------------------
// A workgroup per cell: interiors of 33 to 128 rows, and any with more than 63
// boundary columns.
// --------------------------------------------------------------------------
template <int NT, class Gen>
struct TileGroup {
  static constexpr int kWaves = NT <= 5 ? 4 : 8;
  // strips per wavefront.  (A generator whose Y is stored anyway rereads it; one
  // that keeps its strips of Y in registers beside Z's has room for two of four
  // tiles each, two of five with one of Z's at a time, or one of seven.)
  static constexpr int kStrips = NT <= 5 || Gen::kStoresY ? 2 : 1;
  static constexpr int kHold = NT <= 4 || (NT > 5 && !Gen::kStoresY) ? kStrips : 1;  // strips of Z at a time
  static constexpr int kMinBlocks = NT <= 5 ? 2 : 1;  // workgroups per CU: two wavefronts a SIMD
};

template <int NT, class Gen, bool BACKSUB>
__global__ void __launch_bounds__((64 * TileGroup<NT, Gen>::kWaves), 2)
    condense_tile_kernel(Gen gen, CondenseOut out, int64_t ncells, int ni_, int nb_, int chunk) {
  using TL = Tile<NT>;
  using SRC = TileSrc<Gen>;
  constexpr int N = TL::N, LD = TL::LD;
  extern __shared__ double s_tile[];
  double* const F = s_tile;            // A_ii, then its factors, [col][row]
  double* const sY = s_tile + TL::kF;  // [chunk][16][YLD]
  __shared__ typename Gen::Shared sh;
  __shared__ int s_pos[N];      // the panel's row moves: row -> position
  __shared__ int s_perm[2][N];  // row of A_ii at each position
  __shared__ double s_dinv[N];  // 1 / U[c][c], 0 for a zero pivot
  __shared__ double s_rhs[BACKSUB ? N : 1];
  const int nthreads = blockDim.x, nw = blockDim.x >> 6;
  const int64_t us = ustride(out, ni_), ys = ystride(out, ni_, nb_);
  tile_start(gen, sh, threadIdx.x, nthreads);
  for (int64_t cell = blockIdx.x; cell < ncells; cell += gridDim.x) {
    const int tid = opaque_v(threadIdx.x), ni = opaque_s(ni_), nb = opaque_s(nb_);
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    // (every phase looks at its lane anew: nothing of one lives through another)
    auto here = [&] { return TL(F, opaque_v(threadIdx.x) & 63); };
    const int lane = opaque_v(threadIdx.x) & 63;
    const int ncol = nb + 1, nstrip = (ncol + 15) >> 4;
    gen.begin(cell, sh);
    __syncthreads();
    // ---- A_ii -------------------------------------------------------------------
    tile_load<NT>(gen, sh, F, cell, ni, tid, nthreads, out.Auu ? out.Auu + cell * us : nullptr);
    for (int t = tid; t < N; t += nthreads) {
      s_perm[0][t] = t;
      if (t >= ni) s_dinv[t] = 1.0;
      if (BACKSUB) s_rhs[t] = t < ni ? GenCall<Gen>::entry(gen, sh, t, ni, cell) : 0.0;
    }
    __syncthreads();
    // ---- P A_ii = L U, 16 columns at a time -------------------------------------
    // (the panel's wavefront rotates with the cell, for the SIMDs' sake)
    int info = 0, pb = 0;
    const int npanel = (ni + 15) >> 4;
    const int pw = (int)((blockIdx.x / 256 + cell / gridDim.x) % nw);
#pragma unroll 1
    for (int J = 0; J < npanel; ++J) {
      if (w == pw) here().panel(16 * J, ni, s_pos, s_dinv, info);  // wave-uniform
      __syncthreads();
      for (int t = tid; t < N; t += nthreads) s_perm[pb ^ 1][s_pos[t]] = s_perm[pb][t];
      pb ^= 1;
      for (int s = w; s < NT; s += nw) here().permute(s, s_pos);
      __syncthreads();  // the panel's strip is in position order
      for (int s = J + 1 + w; s < NT; s += nw) here().update(J, s);
      __syncthreads();
    }
    // ---- U out, then its diagonal tiles in the form of their substitution -------
    const int* perm = s_perm[pb];
    if (out.U)
      for (int c = w; c < ni; c += nw)
        for (int k = lane; k <= c; k += 64) out.U[cell * us + c * (c + 1) / 2 + k] = F[c * LD + k];
    if (out.info && w == pw && lane == 0) out.info[cell] = info;
    __syncthreads();
    for (int J = w; J < NT; J += nw) here().factor_diag(J, s_dinv);
    __syncthreads();
    // ---- backward map: x = U^-1 L^-1 P b_i, one column -----------------------------
    if (BACKSUB) {
      if (w == 0 && out.X) {
        const TL tl = here();
        const int i16 = tl.i16, q4 = tl.q4;
        dbl4 x[NT];
#pragma unroll
        for (int I = 0; I < NT; ++I)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int k = 16 * I + 4 * v + q4;
            x[I][v] = i16 == 0 ? s_rhs[perm[k]] : 0.0;
          }
        tl.forward(x);
        tl.backward(x);
        if (i16 == 0) tile_store_strip(out.X + cell * ni, x, 0, q4, ni);
      }
      __syncthreads();
      continue;
    }
    // ---- Y = L^-1 P [A_ib b_i]: strips w, w + nw, ... ------------------------------
    // (all but a stored one stay in registers)
    constexpr int SPW = TileGroup<NT, Gen>::kStrips, HOLD = TileGroup<NT, Gen>::kHold;
    constexpr int KEEP = Gen::kStoresY ? 1 : SPW;
    dbl4 y[KEEP][NT];
#pragma unroll KEEP
    for (int h = 0; h < SPW; ++h) {
      const int s = w + h * nw;
      if (s >= nstrip) continue;
      dbl4(&yh)[NT] = y[h % KEEP];
      const TL tl = here();
      const int c = 16 * s + tl.i16;
      tile_strip_y<NT>(gen, sh, perm, SRC::col(gen, sh, c, nb), yh, c, tl.q4, ni, nb, cell);
      tl.forward(yh);
      if (out.Y && c < ncol) tile_store_strip(out.Y + cell * ys, yh, c, tl.q4, ni);
    }
    if (Gen::kStoresY) {
      __threadfence_block();
      __syncthreads();
    }
    // ---- Z = U^-T A_bi^T, S = A_bb - Z^T Y, g = b_b - Z^T y: 16 rows per strip of Z --
    // (HOLD strips of Z at a time; Y's strips by way of LDS, `chunk` at a time: from
    // out.Y, or from their wavefronts' registers)
#pragma unroll 1
    for (int h0 = 0; h0 < SPW && 16 * h0 * nw < nb; h0 += HOLD) {
      dbl4 z[HOLD][NT];
#pragma unroll
      for (int h = 0; h < HOLD; ++h) {
        const int s = w + (h0 + h) * nw;
        if (16 * s >= nb) continue;
        const TL tl = here();
        tile_strip_z<NT>(gen, sh, SRC::col(gen, sh, 16 * s + tl.i16, nb), z[h], tl.q4, ni, nb,
                         cell);
        tl.forward_ut(z[h]);
      }
#pragma unroll 1
      for (int s0 = 0; s0 < nstrip; s0 += chunk) {
        const int s1 = min(s0 + chunk, nstrip);
        const int i16 = opaque_v(lane) & 15, q4 = opaque_v(lane) >> 4;
        if (Gen::kStoresY) {
          const double* src = out.Y + cell * ys;
          for (int c = 16 * s0 + w; c < 16 * s1; c += nw)
#pragma unroll
            for (int k0 = 0; k0 < N; k0 += 64) {
              const int k = k0 + lane;
              const double x = src[(int64_t)min(c, nb) * ni + min(k, ni - 1)];
              if (k < N) sY[(c - 16 * s0) * TL::YLD + k] = keep_if(k < ni, x);
            }
        } else {
#pragma unroll
          for (int h = 0; h < SPW; ++h) {
            const int s = w + h * nw;
            if (s < s0 || s >= s1) continue;
            double* const dst = sY + (s - s0) * TL::kStrip + i16 * TL::YLD + q4;
#pragma unroll
            for (int I = 0; I < NT; ++I)
#pragma unroll
              for (int v = 0; v < 4; ++v) dst[16 * I + 4 * v] = y[h % KEEP][I][v];
          }
        }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < HOLD; ++h) {
          const int t = w + (h0 + h) * nw, r = 16 * t + i16;
          if (16 * t >= nb) continue;
          const typename SRC::Col rc = SRC::col(gen, sh, r, nb);
          int s = tile_next<SRC::kSym>(t, s0, s1, nstrip);
          dbl4 nxt = {0.0, 0.0, 0.0, 0.0};
          if (s < s1) nxt = tile_bb(gen, sh, rc, r, s, q4, ni, nb, cell);
          while (s < s1) {
            const double* const ysrc = sY + (s - s0) * TL::kStrip + i16 * TL::YLD + q4;
            dbl4 acc = nxt;  // (the next tile's entries come in behind this one's products)
            const int sn = tile_next<SRC::kSym>(t, s + 1, s1, nstrip);
            if (sn < s1) nxt = tile_bb(gen, sh, rc, r, sn, q4, ni, nb, cell);
#pragma unroll
            for (int I = 0; I < NT; ++I)
#pragma unroll
              for (int v = 0; v < 4; ++v)
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-ysrc[16 * I + 4 * v], z[h][I][v], acc,
                                                           0, 0, 0);
            tile_store_s(out, acc, r, s, q4, nb, cell, SRC::kSym && s != t);
            s = sn;
          }
        }
        __syncthreads();
      }
    }
    // ---- A_ii^-1 for the recovery, by rows: P^T L^-T U^-T ---------------------------
    if (out.Rinv)
      for (int s = w; 16 * s < ni; s += nw)
        tile_inverse<NT>(here(), perm, y[0], s, ni, out.Rinv + cell * us);
    __syncthreads();  // LDS reuse by the next cell
  }
}

// --------------------------------------------------------------------------
// A wavefront per cell: interiors of at most 32 rows and 63 boundary columns
// (SPW strips).  Every strip of Y stays in the wavefront's registers and is
// the operand of the S tiles as it is, so nothing is exchanged and nothing
// waits for another wavefront: up to 16 cells share a CU.
// --------------------------------------------------------------------------
template <int NT, int SPW, class Gen, bool BACKSUB>
__global__ void __launch_bounds__(64, 3)
    condense_wtile_kernel(Gen gen, CondenseOut out, int64_t ncells, int ni_, int nb_) {
  using TL = Tile<NT>;
  using SRC = TileSrc<Gen>;
  constexpr int N = TL::N, LD = TL::LD;
  __shared__ double F[TL::kF];
  __shared__ typename Gen::Shared sh;
  __shared__ int s_pos[N], s_perm[N];
  __shared__ double s_dinv[N];
  const int64_t us = ustride(out, ni_), ys = ystride(out, ni_, nb_);
  tile_start(gen, sh, threadIdx.x, 64);
  for (int64_t cell = blockIdx.x; cell < ncells; cell += gridDim.x) {
    const int ni = opaque_s(ni_), nb = opaque_s(nb_), ncol = nb + 1;
    // (every phase looks at its lane anew: nothing of one lives through another)
    auto here = [&] { return TL(F, opaque_v(threadIdx.x)); };
    const int lane = opaque_v(threadIdx.x);
    gen.begin(cell, sh);
    wave_sync_lds();
    tile_load<NT>(gen, sh, F, cell, ni, lane, 64, out.Auu ? out.Auu + cell * us : nullptr);
    if (lane < N) {
      s_perm[lane] = lane;
      s_dinv[lane] = 1.0;
    }
    wave_sync_lds();
    int info = 0;
    const int npanel = (ni + 15) >> 4;
#pragma unroll 1
    for (int J = 0; J < npanel; ++J) {
      here().panel(16 * J, ni, s_pos, s_dinv, info);
      wave_sync_lds();
      const int row = lane < N ? s_perm[lane] : 0;
      wave_sync_lds();
      if (lane < N) s_perm[s_pos[lane]] = row;
#pragma unroll 1
      for (int s = 0; s < NT; ++s) here().permute(s, s_pos);
#pragma unroll 1
      for (int s = J + 1; s < NT; ++s) here().update(J, s);
      wave_sync_lds();
    }
    if (out.U)
#pragma unroll 4
      for (int c = 0; c < ni; ++c)
        if (lane <= c) out.U[cell * us + c * (c + 1) / 2 + lane] = F[c * LD + lane];
    if (out.info && lane == 0) out.info[cell] = info;
    wave_sync_lds();
#pragma unroll 1
    for (int J = 0; J < NT; ++J) here().factor_diag(J, s_dinv);
    wave_sync_lds();
    if (BACKSUB) {
      if (out.X) {
        const double b = lane < ni ? GenCall<Gen>::entry(gen, sh, lane, ni, cell) : 0.0;
        const TL tl = here();
        dbl4 x[NT];
#pragma unroll
        for (int I = 0; I < NT; ++I)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const double t = __shfl(b, s_perm[16 * I + 4 * v + tl.q4]);
            x[I][v] = tl.i16 == 0 ? t : 0.0;
          }
        tl.forward(x);
        tl.backward(x);
        if (tl.i16 == 0) tile_store_strip(out.X + cell * ni, x, 0, tl.q4, ni);
      }
      wave_sync_lds();
      continue;
    }
    if constexpr (SRC::kSym) {
      // Z's strips stay, a strip of Y meets those up to its own
      dbl4 z[SPW][NT];
#pragma unroll
      for (int s = 0; s < SPW; ++s)
        if (16 * s < ncol) {
          const TL tl = here();
          const int c = 16 * s + tl.i16;
          const typename SRC::Col b = SRC::col(gen, sh, c, nb);
          if (16 * s < nb) {
            tile_strip_z<NT>(gen, sh, b, z[s], tl.q4, ni, nb, cell);
            tl.forward_ut(z[s]);
          }
          dbl4 y[NT];
          tile_strip_y<NT>(gen, sh, s_perm, b, y, c, tl.q4, ni, nb, cell);
          tl.forward(y);
          if (out.Y && c < ncol) tile_store_strip(out.Y + cell * ys, y, c, tl.q4, ni);
#pragma unroll
          for (int t = 0; t <= s; ++t)
            if (16 * t < nb) {
              __builtin_amdgcn_sched_barrier(0);
              const int q = opaque_v(tl.q4), r = 16 * t + opaque_v(tl.i16);
              dbl4 acc = tile_bb(gen, sh, SRC::col(gen, sh, r, nb), r, s, q, ni, nb, cell);
#pragma unroll
              for (int I = 0; I < NT; ++I)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                  acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-y[I][v], z[t][I][v], acc, 0, 0, 0);
              tile_store_s(out, acc, r, s, q, nb, cell, t != s);
            }
        }
    } else {
      dbl4 y[SPW][NT];
#pragma unroll
      for (int s = 0; s < SPW; ++s)
        if (16 * s < ncol) {
          const TL tl = here();
          const int c = 16 * s + tl.i16;
          tile_strip_y<NT>(gen, sh, s_perm, SRC::col(gen, sh, c, nb), y[s], c, tl.q4, ni, nb, cell);
          tl.forward(y[s]);
          if (out.Y && c < ncol) tile_store_strip(out.Y + cell * ys, y[s], c, tl.q4, ni);
        }
#pragma unroll 1
      for (int t = 0; 16 * t < nb; ++t) {
        const TL tl = here();
        const int r = 16 * t + tl.i16;
        const typename SRC::Col b = SRC::col(gen, sh, r, nb);
        dbl4 z[NT];
        tile_strip_z<NT>(gen, sh, b, z, tl.q4, ni, nb, cell);
        tl.forward_ut(z);
#pragma unroll
        for (int s = 0; s < SPW; ++s)
          if (16 * s < ncol) {
            __builtin_amdgcn_sched_barrier(0);
            const int q = opaque_v(tl.q4);
            dbl4 acc = tile_bb(gen, sh, b, r, s, q, ni, nb, cell);
#pragma unroll
            for (int I = 0; I < NT; ++I)
#pragma unroll
              for (int v = 0; v < 4; ++v)
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-y[s][I][v], z[I][v], acc, 0, 0, 0);
            tile_store_s(out, acc, r, s, q, nb, cell, false);
          }
      }
    }
    if (out.Rinv)
#pragma unroll 1
      for (int s = 0; 16 * s < ni; ++s) {
        dbl4 x[NT];
        tile_inverse<NT>(here(), s_perm, x, s, ni, out.Rinv + cell * us);
      }
    wave_sync_lds();  // LDS reuse by the next cell
  }
}

// Rows and columns the kernels take: the interior tiles in LDS, one strip of
// boundary columns per wavefront (a wavefront per cell: four strips).
static bool tile_one_wave(int ni, int nb) { return ni <= 32 && nb < 64; }

// Row tiles of a workgroup's kernel.  With seven, 65 to 80 rows took a workgroup a
// CU and up to 1.16 times the time of the panel kernel they had before on few
// boundary columns and many cells; with five, two workgroups share a CU
// (forward map with the caller's transposes, panel kernel, seven and five tiles:
// 3,000 cells of 72 + 16 1,325, 1,474 and 817 us, 6,000 of 80 + 40 3,868, 3,501
// and 2,055 us).
static int tile_nt(int ni) { return ni <= 64 ? 4 : ni <= 80 ? 5 : ni <= 112 ? 7 : 8; }

// (stored: the generators that store Y, with two strips a wavefront throughout)
static bool tile_ok(int ni, int nb, bool stored = false) {
  if (ni < 1 || ni > 128) return false;
  return (nb + 16) / 16 <= (stored && tile_nt(ni) > 4 ? 16 : 8);
}

template <int NT, class Gen, bool BACKSUB>
static hipError_t launch_tile_nt(const Gen& gen, const CondenseOut& out, int64_t ncells, int ni,
                                 int nb, hipStream_t st, int gridmul) {
  using TL = Tile<NT>;
  using TG = TileGroup<NT, Gen>;
  const int nstrip = (nb + 16) / 16;
  const int waves = TG::kWaves;
  // the Y strips that keep kMinBlocks workgroups on a CU, all of them if they fit
  const int budget =
      (160 * 1024 / TG::kMinBlocks - 3072 - (int)sizeof(typename Gen::Shared)) / 8 - TL::kF;
  const int chunk = BACKSUB ? 0 : std::max(1, std::min(nstrip, budget / TL::kStrip));
  const size_t lds = (size_t)(TL::kF + chunk * TL::kStrip) * sizeof(double);
  if (nstrip > waves * TG::kStrips || lds + sizeof(typename Gen::Shared) > 160 * 1024 - 3072)
    return hipErrorInvalidValue;
  const auto kernel = condense_tile_kernel<NT, Gen, BACKSUB>;
  if (lds > 48 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void*)kernel,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  const int64_t per = gridmul > 0 ? gridmul : 4 * TG::kMinBlocks;
  const int grid = (int)std::min<int64_t>(ncells, 256 * per);
  ClockScope clk_(st, "condense_tile");
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * waves), lds, st, gen, out, ncells, ni, nb, chunk);
  return hipGetLastError();
}

template <int NT, class Gen, bool BACKSUB>
static hipError_t launch_wtile_nt(const Gen& gen, const CondenseOut& out, int64_t ncells, int ni,
                                  int nb, hipStream_t st, int gridmul) {
  const int64_t per = gridmul > 0 ? gridmul : 48;
  const int grid = (int)std::min<int64_t>(ncells, 256 * per);
  ClockScope clk_(st, "condense_tile");
  hipLaunchKernelGGL((condense_wtile_kernel<NT, 4, Gen, BACKSUB>), dim3(grid), dim3(64), 0, st,
                     gen, out, ncells, ni, nb);
  return hipGetLastError();
}

template <class Gen, bool BACKSUB>
static hipError_t launch_tile_small(const Gen& gen, const CondenseOut& out, int64_t ncells, int ni,
                                    int nb, hipStream_t st, int gridmul) {
  return ni <= 16 ? launch_wtile_nt<1, Gen, BACKSUB>(gen, out, ncells, ni, nb, st, gridmul)
                  : launch_wtile_nt<2, Gen, BACKSUB>(gen, out, ncells, ni, nb, st, gridmul);
}

template <class Gen, bool BACKSUB>
static hipError_t launch_tile(const Gen& gen, const CondenseOut& out, int64_t ncells, int ni,
                              int nb, hipStream_t st, int gridmul) {
  if (!tile_ok(ni, nb)) return hipErrorInvalidValue;
  if (tile_one_wave(ni, nb))
    return launch_tile_small<Gen, BACKSUB>(gen, out, ncells, ni, nb, st, gridmul);
  switch (tile_nt(ni)) {
    case 4: return launch_tile_nt<4, Gen, BACKSUB>(gen, out, ncells, ni, nb, st, gridmul);
    case 5: return launch_tile_nt<5, Gen, BACKSUB>(gen, out, ncells, ni, nb, st, gridmul);
    case 7: return launch_tile_nt<7, Gen, BACKSUB>(gen, out, ncells, ni, nb, st, gridmul);
    default: return launch_tile_nt<8, Gen, BACKSUB>(gen, out, ncells, ni, nb, st, gridmul);
  }
}

// The reduced systems of every cell from the reference decomposition.
constexpr int kRefSmallNr = 96, kRefMaxNr = 304, kRefMaxNp = 64;

static bool ref_tile_ok(int nu, int nb, int np) {
  return np <= kRefMaxNp && nu <= 112 && nu + nb <= kRefMaxNr && tile_ok(nu, nb, true);
}

template <int PHYS, int D>
static hipError_t launch_tile_ref(const Tables& T, const MeshDev& M, const CondenseOut& out,
                                  hipStream_t st, int gridmul) {
  const int nu = T.ni - T.na, nb = T.nb;
  if (!ref_tile_ok(nu, nb, T.np)) return hipErrorInvalidValue;
  if (tile_one_wave(nu, nb) && T.np <= 32)
    return launch_tile_small<RefGen<PHYS, D, kRefSmallNr, 32 * D>, false>(
        RefGen<PHYS, D, kRefSmallNr, 32 * D>{T, M}, out, M.ncells, nu, nb, st, gridmul);
  using Gen = RefGen<PHYS, D, kRefMaxNr, kRefMaxNp * D>;
  return nu <= 64 ? launch_tile_nt<4, Gen, false>(Gen{T, M}, out, M.ncells, nu, nb, st, gridmul)
                  : launch_tile_nt<7, Gen, false>(Gen{T, M}, out, M.ncells, nu, nb, st, gridmul);
}
