#pragma once
// Darcy's flux recovery through the reference decomposition (build_flux_ref), a
// workgroup per 16 cells (included by hdg_kernels.hip).
//
// On affine cells every block of the interior system but R_uu^-1 is a
// combination, with a few coefficients per cell, of matrices that all cells
// share:
//   A_qq = alpha_0 (I (x) M),  A_q,(u|b) = sum_e c_ea G_e,  A_uq = -A_qu^T,
//   A_uu = sum_F tau_F Fqq_F,  A_ub = -tau_F Fqm_F.
// So 16 cells are the 16 columns of FP64 MFMA products with those tables as the
// other operand: a lane's column is its cell, and mixing the directions of an
// accumulator by its coefficients is a lane's own work.  Wavefront w owns the
// rows 16 w .. 16 w + 15 of the scalar bases (np flux functions, nq potential
// functions); vectors that are the B operand of the next product pass through
// LDS as [row][cell].  R_uu^-1, the one block of a cell's own, is applied with a
// thread per (cell, row), the only large read of a step.
//
// What bounds it: the latency of R_uu^-1's columns (8 in flight a thread; 3.0
// TB/s at 64^3 k=2, read once a step) and of the chained products; MFMA issue is
// a fifth.  Measured against a wavefront per cell (recover_flux_kernel):
//   64^3 k=2 7.61 -> 1.74 ms, 24^3 k=3 3.08 -> 0.62 ms, 2D k=3, 16,247 cells,
//   136 -> 56 us, 3D k=1, 13,547 cells, 92 -> 46 us.
// Elasticity's six components and 12 to 21 coefficients a cell fill the
// registers of a wavefront a SIMD here: 5,814 cells of k=2 241 -> 206 us, but
// 125 cells 60 -> 168 us, so it stays with the wavefront per cell.
//
// With c = b_i - A_ib lambda, the structured solve of a right-hand side r is
//   z = A_qq^-1 r_q (A_qq^-1 = C^-1 (x) M^-1),  d_u = R_uu^-1 (r_u - A_uq z),
//   d_q = z - A_qq^-1 A_qu d_u,
// applied to c and then, up to kFluxRefineSteps times, to the residual of the
// full interior system, r = c - A_ii x.  All of it is in the principal basis of
// the potential (build_flux_ref), where R_uu^-1 is exact enough however small the
// flux block is (large kappa); x_u returns to the nodal one at the end.  c_q -
// A_qu x_u is carried from step to step, and r_u - A_uq z is formed as
// c_u - A_uu x_u - A_uq (x_q + z), whose rounding is that of the residual
// itself.  A cell's columns rest once its correction is below 2^-44 of its
// solution: the next would be smaller by the ratio of this one to the error it
// removed.  (With 2^-48, or without resting, the errors of 60 to 500 cells each
// of 2D k=3 and 4 and of 3D k=1 and 2, kappa up to lognormal(0, 3), have the same
// quantiles to a few percent.)  The workgroup ends when all 16 do.

constexpr int kRecLd = 17;    // doubles between rows of a vector in LDS
constexpr int kRecCoef = 17;  // coefficients of a cell, at most

// E tables' 16 rows against N vectors: acc[e N + n] += A_e x_n over K columns.
// a(e, k): the entry of table e in this lane's row and column k; x(n, k): row k
// of vector n in this lane's cell, 0 from K on.  The table entries of the next
// U steps load behind this one's products.
template <int E, int N, class A, class X>
__device__ inline void rec_mm(dbl4 (&acc)[E * N], int K, int q4_, A a, X x) {
  constexpr int U = E > 1 ? 2 : N > 1 ? 4 : 8;
  __builtin_amdgcn_sched_barrier(0);
  const int q4 = opaque_v(q4_);  // (addresses hoisted out of the step loop spill)
  double av[U][E];
  auto load = [&](int k0) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < E; ++e) av[u][e] = a(e, min(k0 + 4 * u + q4, K - 1));
  };
  load(0);
#pragma unroll 1
  for (int k0 = 0; k0 < K; k0 += 4 * U) {
    double cur[U][E];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < E; ++e) cur[u][e] = av[u][e];
    load(k0 + 4 * U);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (k0 + 4 * u < K)
#pragma unroll
        for (int n = 0; n < N; ++n) {
          const double xv = x(n, k0 + 4 * u + q4);
#pragma unroll
          for (int e = 0; e < E; ++e)
            acc[e * N + n] =
                __builtin_amdgcn_mfma_f64_16x16x4f64(cur[u][e], xv, acc[e * N + n], 0, 0, 0);
        }
  }
}

// doubles of LDS: the vectors of the flux rows and of the directions, three of
// the potential rows, the convergence maxima, and the cells' coefficients
__host__ __device__ inline int rec_ref_lds(int D, int np, int nq, int nb) {
  const int np4 = (np + 3) & ~3, nq4 = (nq + 3) & ~3, rows = D * np4 + ((D * np + 3) & ~3);
  return ((rows > nb ? rows : nb) + 3 * nq4) * kRecLd + 2 * 8 * 16 + kRecCoef * 16;
}

template <int D>
__global__ void __launch_bounds__(512, 2)
    recover_ref_kernel(Tables T, MeshDev M, const double* __restrict__ slots, int64_t usz,
                       const int32_t* __restrict__ cell_dofs, const double* __restrict__ lam_free,
                       const double* __restrict__ lam_dir, double* __restrict__ out) {
  constexpr int KT = D * D, KC = KT + 2 * D;  // coef: c_ea, tau_F, alpha_0 and its inverse
  extern __shared__ double s_rec[];
  const int np = T.np, nq = T.nq, nm = T.nm, nb = T.nb, na = D * np;
  const int np4 = (np + 3) & ~3, nq4 = (nq + 3) & ~3, nr = nq + nb;
  const int dp4 = (D * np + 3) & ~3, vrows = max(D * np4 + dp4, nb);
  // k / nq = k invq >> 20 up to 2^20 / nq
  const int invq = (1 << 20) / nq + 1, invm = (1 << 20) / nm + 1;
  double* const V = s_rec;                   // [D][np4] flux rows
  double* const TV = V + D * np4 * kRecLd;   // [D np] directions, padded
  double* const LAM = V;                     // [nb], before the first step
  double* const XU = s_rec + vrows * kRecLd; // x_u
  double* const UV = XU + nq4 * kRecLd;      // reduced right-hand side
  double* const DU = UV + nq4 * kRecLd;      // reduced correction
  double* const smax = DU + nq4 * kRecLd;    // [2][wavefront][cell]
  double* const coef = smax + 2 * 8 * 16;    // [coefficient][cell]
  const int tid = threadIdx.x, nthreads = blockDim.x, nw = nthreads >> 6;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int i16 = lane & 15, q4 = lane >> 4;
  const int64_t ncells = M.ncells;
  const bool prow = 16 * w < np, qrow = 16 * w < nq;  // wave-uniform
  const int pr = min(16 * w + i16, np - 1);           // table rows of this lane
  const int qr = min(16 * w + i16, nq - 1);
  const dbl4 zero = {0.0, 0.0, 0.0, 0.0};
  // row k of vector n of the flux rows, of the directions, of the potential rows
  auto vrow = [&](int n, int k) { return V[(n * np4 + k) * kRecLd + i16]; };
  auto trow = [&](int, int k) { return TV[k * kRecLd + i16]; };
  auto drow = [&](int, int k) { return DU[k * kRecLd + i16]; };
  auto mass = [&](int, int k) { return table_at(T.Mpp, 8u * (pr + k * np)); };
  auto minv = [&](int, int k) { return table_at(T.fb_minv, 8u * (pr + k * np)); };
  // rows 16 w + 4 v + q4 of this lane's accumulators, in LDS and for reading
  auto put = [&](double* vec, const dbl4& x, int n) {
    const int r0 = 16 * w + opaque_v(q4), at = r0 * kRecLd + i16;
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (r0 + 4 * v < n) vec[at + 4 * v * kRecLd] = x[v];
  };

  for (int64_t c0 = (int64_t)blockIdx.x * 16; c0 < ncells; c0 += (int64_t)gridDim.x * 16) {
    const int64_t cell = min(c0 + i16, ncells - 1);
    // ---- the cells' coefficients (in LDS: in registers all through the steps they
    // spill; 0 for the inverse of a singular flux block)
    if (tid < 16) {
      const double* const al = M.alpha + cell * kMaxAlpha;
      for (int k = 0; k < KT; ++k) coef[k * 16 + i16] = -al[1 + k];
      for (int f = 0; f < 2 * D; ++f) coef[(KT + f) * 16 + i16] = al[28 + f];
      coef[KC * 16 + i16] = al[0];
      coef[(KC + 1) * 16 + i16] = al[0] != 0.0 ? 1.0 / al[0] : 0.0;
    }
    auto at = [&](int k) { return coef[k * 16 + opaque_v(i16)]; };
    auto scale = [&](dbl4(&y)[D], double c) {
#pragma unroll
      for (int a = 0; a < D; ++a) y[a] *= c;
    };
    // flux rows of sum_e c_ea t_e
    auto mix = [&](dbl4(&q)[D], const dbl4(&t)[D]) {
#pragma unroll
      for (int a = 0; a < D; ++a) {
        q[a] = zero;
#pragma unroll
        for (int e = 0; e < D; ++e) q[a] += at(e * D + a) * t[e];
      }
    };
    // ---- lambda of the 16 cells -----------------------------------------------------
    for (int t = tid; t < 16 * nb; t += nthreads) {
      const int ci = t / nb, j = t - ci * nb;
      const int32_t d = cell_dofs[min(c0 + ci, ncells - 1) * nb + j];
      LAM[j * kRecLd + ci] = d >= 0 ? lam_free[d] : lam_dir[-(int64_t)d - 1];
    }
    __syncthreads();
    // ---- c = b_i - A_ib lambda ------------------------------------------------------
    const double* const bi = M.srcq + cell * srcq_stride(T);
    dbl4 ca[D], xq[D], cu[1];  // c_q - A_qu x_u, x_q, c_u
#pragma unroll
    for (int a = 0; a < D; ++a) {
      xq[a] = zero;
#pragma unroll
      for (int v = 0; v < 4; ++v) ca[a][v] = bi[a * np + min(16 * w + 4 * v + q4, np - 1)];
    }
    const double* const bu = bi + (T.fo_P ? T.ni : na);  // in the basis of the tables
#pragma unroll
    for (int v = 0; v < 4; ++v) cu[0][v] = bu[min(16 * w + 4 * v + q4, nq - 1)];
    {
      dbl4 t[D], q[D];
#pragma unroll
      for (int e = 0; e < D; ++e) t[e] = zero;
      if (prow)
#pragma unroll
        for (int e = 0; e < D; ++e) {  // facets 2 (D - 1 - e) and the next: direction e
          dbl4 y[1] = {zero};
          const int b0 = 2 * (D - 1 - e) * nm;
          rec_mm<1, 1>(
              y, 2 * nm, q4,
              [&](int, int k) { return table_at(T.fr_Gt, 8u * (pr + (e * nr + nq + b0 + k) * np)); },
              [&](int, int k) {
                return keep_if(k < 2 * nm, -LAM[(b0 + min(k, 2 * nm - 1)) * kRecLd + i16]);
              });
          t[e] = y[0];
        }
      if (qrow)
        rec_mm<1, 1>(
            cu, nb, q4, [&](int, int k) { return table_at(T.fr_qm, 8u * (qr * nb + k)); },
            [&](int, int k_) {
              const int k = min(k_, nb - 1);
              return keep_if(k_ < nb, coef[(KT + (k * invm >> 20)) * 16 + i16] *
                                          LAM[k * kRecLd + i16]);
            });
      mix(q, t);
#pragma unroll
      for (int a = 0; a < D; ++a) ca[a] += q[a];
    }
    __syncthreads();  // lambda read: V and TV from here on
    for (int t = tid; t < (vrows + 3 * nq4) * kRecLd; t += nthreads) s_rec[t] = 0.0;
    __syncthreads();
    // ---- the structured solve of c, then of the residuals of the full interior system
    bool act = true;  // this lane's cell
#pragma unroll 1
    for (int it = 0; it <= kFluxRefineSteps; ++it) {
      // r_q = c_q - A_qu x_u - (C (x) M) x_q  (x_q in V), then z = A_qq^-1 r_q
      dbl4 z[D];
#pragma unroll
      for (int a = 0; a < D; ++a) z[a] = zero;
      if (it > 0) {
        if (prow) rec_mm<1, D>(z, np, q4, mass, vrow);
        scale(z, at(KC));
        __syncthreads();
      }
#pragma unroll
      for (int a = 0; a < D; ++a) put(V + a * np4 * kRecLd, ca[a] - z[a], np);
      __syncthreads();
#pragma unroll
      for (int a = 0; a < D; ++a) z[a] = zero;
      if (prow) rec_mm<1, D>(z, np, q4, minv, vrow);
      scale(z, at(KC + 1));
      // r_u - A_uq z = c_u - A_uu x_u - A_uq (x_q + z), A_uq = -A_qu^T
#pragma unroll
      for (int e = 0; e < D; ++e) {
        dbl4 s = zero;
#pragma unroll
        for (int a = 0; a < D; ++a) s += at(e * D + a) * (xq[a] + z[a]);
        put(TV + e * np * kRecLd, s, np);
      }
      __syncthreads();
      if (qrow) {
        dbl4 ru[1] = {cu[0]};
        if (it > 0)  // the facets one after the other: rows tau_F x_u
          rec_mm<1, 1>(
              ru, 2 * D * nq, q4,
              [&](int, int k) { return table_at(T.Fqq, 8u * (qr + k * nq)); },  // (symmetric)
              [&](int, int k) {
                const int f = min(k * invq >> 20, 2 * D - 1), j = min(k - f * nq, nq - 1);
                const double x = coef[(KT + f) * 16 + i16] * XU[j * kRecLd + i16];
                return keep_if(k < 2 * D * nq, -x);
              });
        rec_mm<1, 1>(
            ru, D * np, q4, [&](int, int k) { return table_at(T.fr_G, 8u * (qr + k * nr)); }, trow);
        put(UV, ru[0], nq);
      }
      __syncthreads();
      // d_u = R_uu^-1 (.): a thread per (cell, row), the next CH columns in flight
      {
        constexpr int CH = 8;
        const int nch = (nq + CH - 1) / CH, total = ((16 * nq + nthreads - 1) / nthreads) * nch;
        double nxt[CH], x = 0.0;
        auto at_pair = [&](int t, int& ci, int& r) {
          t = min(t, 16 * nq - 1);
          ci = t / nq;
          r = t - ci * nq;
        };
        int t = tid, ci, r, j0 = 0;
        at_pair(t, ci, r);
        const double* ri = slots + min(c0 + ci, ncells - 1) * usz + r;
#pragma unroll
        for (int u = 0; u < CH; ++u) nxt[u] = ri[(int64_t)min(u, nq - 1) * nq];
#pragma unroll 1
        for (int k = 0; k < total; ++k) {
          double cur[CH];
#pragma unroll
          for (int u = 0; u < CH; ++u) cur[u] = nxt[u];
          const bool last = j0 + CH >= nq;  // wave-uniform
          const int cj = ci, row = r, mine = t;
          const double* const uv = UV + j0 * kRecLd + cj;
          if (last) {
            t += nthreads;
            at_pair(t, ci, r);
            ri = slots + min(c0 + ci, ncells - 1) * usz + r;
          }
          const int jn = last ? 0 : j0 + CH;
#pragma unroll
          for (int u = 0; u < CH; ++u) nxt[u] = ri[(int64_t)min(jn + u, nq - 1) * nq];
#pragma unroll
          for (int u = 0; u < CH; ++u)
            if (j0 + u < nq) x = fma(cur[u], uv[u * kRecLd], x);
          if (last) {
            if (mine < 16 * nq) DU[row * kRecLd + cj] = x;
            x = 0.0;
          }
          j0 = jn;
        }
      }
      __syncthreads();
      // A_qu d_u; d_q = z - A_qq^-1 A_qu d_u
      {
        dbl4 t[D], q[D];
#pragma unroll
        for (int e = 0; e < D; ++e) t[e] = zero;
        if (prow)
          rec_mm<D, 1>(
              t, nq, q4,
              [&](int e, int k) { return table_at(T.fr_Gt, 8u * (pr + (e * nr + k) * np)); }, drow);
        mix(q, t);
#pragma unroll
        for (int a = 0; a < D; ++a) {
          ca[a] -= q[a];
          put(V + a * np4 * kRecLd, q[a], np);
        }
      }
      __syncthreads();
      double dmax = 0.0, xmax = 0.0;
      {
        dbl4 y[D];
#pragma unroll
        for (int a = 0; a < D; ++a) y[a] = zero;
        if (prow) rec_mm<1, D>(y, np, q4, minv, vrow);
        scale(y, at(KC + 1));
#pragma unroll
        for (int a = 0; a < D; ++a)
#pragma unroll
          for (int v = 0; v < 4; ++v)
            if (16 * w + 4 * v + opaque_v(q4) < np) {
              const double d = z[a][v] - y[a][v];
              if (act) xq[a][v] += d;
              dmax = fmax(dmax, fabs(d));
              xmax = fmax(xmax, fabs(xq[a][v]));
            }
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = 16 * w + 4 * v + opaque_v(q4);
        if (r < nq) {
          const double dx = DU[r * kRecLd + i16], x = XU[r * kRecLd + i16] + (act ? dx : 0.0);
          XU[r * kRecLd + i16] = x;
          dmax = fmax(dmax, fabs(dx));
          xmax = fmax(xmax, fabs(x));
        }
      }
#pragma unroll
      for (int o = 16; o < 64; o *= 2) {
        dmax = fmax(dmax, __shfl_xor(dmax, o));
        xmax = fmax(xmax, __shfl_xor(xmax, o));
      }
      if (q4 == 0) {
        smax[w * 16 + i16] = dmax;
        smax[128 + w * 16 + i16] = xmax;
      }
      __syncthreads();  // (V read as well)
      for (int k = 0; k < nw; ++k) {
        dmax = fmax(dmax, smax[k * 16 + i16]);
        xmax = fmax(xmax, smax[128 + k * 16 + i16]);
      }
      if (it > 0 && dmax <= 0x1p-44 * xmax) act = false;
      if (!__ballot(act)) break;  // (the same cells in every wavefront)
#pragma unroll
      for (int a = 0; a < D; ++a) put(V + a * np4 * kRecLd, xq[a], np);
      __syncthreads();
    }
    dbl4 ux[1] = {zero};
    if (T.fo_P && qrow)  // x_u = P x_u'
      rec_mm<1, 1>(
          ux, nq, q4, [&](int, int k) { return table_at(T.fo_Pt, 8u * (qr + k * nq)); },
          [&](int, int k) { return XU[k * kRecLd + i16]; });
    if (c0 + i16 < ncells) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = 16 * w + 4 * v + q4;
        if (r < np)
#pragma unroll
          for (int a = 0; a < D; ++a) out[cell * na + a * np + r] = xq[a][v];
        if (r < nq) out[ncells * na + cell * nq + r] = T.fo_P ? ux[0][v] : XU[r * kRecLd + i16];
      }
    }
    __syncthreads();  // LDS reuse by the next cells
  }
}

// Which cells come here: with one row tile (np, nq <= 16) a wavefront per cell
// is faster below about 2,000 cells (77 cells of 2D k=3 23 against 33 us, 2,400
// cells 36 against 33, 125 cells of 3D k=1 18 against 31); in 2D with more
// below about 1,000 (a recovery with its launch and copies, k=4: 256 cells 52
// against 65 us, 1,024 53 against 65, 2,116 72 against 65; k=5: 73 against 82, 76
// against 82, 144 against 84; k=6: 93 against 109, 111 against 110, 215 against
// 117); in 3D with more never (8 cells of k=2 59 and 59 us, of k=3 168 and 127).
// Asked by whoever condenses, once, with the cells of one recovery: it decides
// whether A_uu is kept (a batch's class has more cells than each of its meshes).
bool recover_by_group(const Tables& T, int64_t ncells) {
  const int rows = std::max(T.np, T.nq);
  return T.phys == kDarcy && rows <= 128 &&
         rec_ref_lds(T.D, T.np, T.nq, T.nb) * sizeof(double) <= 160 * 1024 &&
         ncells >= (rows <= 16 ? 2048 : T.D == 2 ? 1024 : 0);
}

template <int D>
static hipError_t launch_recover_ref(const Tables& T, const MeshDev& M, const double* rinv,
                                     int64_t usz, const int32_t* cell_dofs, const double* lam_free,
                                     const double* lam_dir, double* out, hipStream_t st) {
  const size_t lds = rec_ref_lds(D, T.np, T.nq, T.nb) * sizeof(double);
  const int64_t groups = (M.ncells + 15) / 16;
  int waves = (std::max(T.np, T.nq) + 15) / 16;
  // a CU to itself: two more wavefronts share R_uu^-1 (75 -> 63 us for 10^3
  // cells of k=2; 1.74 -> 2.46 ms where they take the place of other groups)
  if (groups <= 256) waves = std::max(waves, 4);
  const auto kernel = recover_ref_kernel<D>;
  if (lds > 48 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void*)kernel,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  const int grid = (int)std::min<int64_t>(groups, 1 << 16);
  ClockScope clk_(st, "recover_flux");
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * waves), lds, st, T, M, rinv, usz, cell_dofs,
                     lam_free, lam_dir, out);
  return hipGetLastError();
}
