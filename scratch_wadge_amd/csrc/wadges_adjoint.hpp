// wadges_adjoint.hpp -- discrete adjoint (vector-Jacobian products) of the
// WADGES stage, included by wadges.hip.
//
// Forward stage (okl/Euler3D.okl:2123-2884, euler.c:3656-3666):
//   R   = vol(u~q, u~f) + lift(surf(u~f, u~f[nbr]) + rhsQf)      (RHS)
//   r   = VqPq diag(1/J) VqPq (-2 R)
//   res'= fa res + dt r ;  Q' = Q + fb res'
//   v~  = VqPq diag(1/J) VqPq (J v(Q')) ; u~q' = u(VqPq v~), u~f' = u(VfPq v~)
// The VJPs below run that sequence backwards:
//   sbar_kernel      s_bar = VqLq^T R_bar per element (the lift transposed); the
//                    RHS VJP needs it at neighbour face points, hence a pass of
//                    its own
//   rhs_vjp_kernel   (u~q_bar, u~f_bar) from R_bar: the flux-differencing pairs on
//                    the same diagonal schedules as the forward volume kernel (each
//                    symmetric pair differentiated once, partner cotangents
//                    accumulated in LDS), then the surface flux and LF penalty of
//                    this element's face points and of the neighbour's matching
//                    points (recomputed locally, so no scatter between elements)
//   update_vjp_kernel (Q_bar, res_bar, R_bar) from the stage outputs' cotangents,
//                    recomputing the projection from Q'
//   proj_vjp_kernel  the initial-state projection u~q = u(VqPq v(Q0)),
//                    u~f = u(VfPq v(Q0)) (euler.c:4028-4133)
// Included inside namespace wadges, after the forward kernels it reuses.
#pragma once

template <class S, int TS, int TPW>
__global__ void __launch_bounds__(WAVE * 4)
sbar_kernel(int K, const double *__restrict__ VqLq, const double *__restrict__ Rb,
            double *__restrict__ sbar) {
  constexpr int NQ = S::NQ, NFN = S::NFN, NFLD = S::NFLD;
  constexpr int EPB = 4 * TPW;
  __shared__ double sR[EPB][NFLD][NQ];
  const int wave = threadIdx.x / WAVE;
  const int wl = threadIdx.x % WAVE;
  const int tw = wl / TS;
  const int lane = wl - tw * TS;
  const bool active = tw < TPW;
  const int e = wave * TPW + (active ? tw : 0);
  const int k = blockIdx.x * EPB + e;
  const bool valid = active && k < K;
  if (valid && lane < NQ)
    for (int f = 0; f < NFLD; ++f) sR[e][f][lane] = Rb[(size_t)k * NQ * NFLD + f * NQ + lane];
  __syncthreads();
  if (valid && lane < NFN) {
    double v[NFLD];
    for (int f = 0; f < NFLD; ++f) v[f] = 0.0;
#pragma unroll 4
    for (int i = 0; i < NQ; ++i) {
      const double L = ld_off(VqLq, (unsigned)(i + lane * NQ));
      for (int f = 0; f < NFLD; ++f) v[f] += L * sR[e][f][i];
    }
    for (int f = 0; f < NFLD; ++f) sbar[(size_t)k * NFN * NFLD + f * NFN + lane] = v[f];
  }
}

template <class S> struct VjpSmem {
  static constexpr int NPB = S::DIM + 2;  // primitive cotangent components
  static constexpr int acc_v = NPB * S::NQ;
  static constexpr int phase1 = S::VREC * S::NQ + S::NFLD * S::NQ;
  static constexpr int phase2 = (S::FREC + S::NFLD + NPB) * S::NFN;
  static constexpr int per_elem = acc_v + (phase1 > phase2 ? phase1 : phase2);
};

template <int DIM>
__device__ __forceinline__ void lds_add_primbar(double *acc, int stride, int j,
                                                const PrimBar<DIM> &g) {
  lds_add(&acc[0 * stride + j], g.rho);
  for (int d = 0; d < DIM; ++d) lds_add(&acc[(1 + d) * stride + j], g.u[d]);
  lds_add(&acc[(DIM + 1) * stride + j], g.beta);
}

template <int DIM>
__device__ __forceinline__ void add_lds_primbar(PrimBar<DIM> &g, const double *acc, int stride,
                                                int j) {
  g.rho += acc[0 * stride + j];
  for (int d = 0; d < DIM; ++d) g.u[d] += acc[(1 + d) * stride + j];
  g.beta += acc[(DIM + 1) * stride + j];
}

template <class S, int TPW>
__global__ void __launch_bounds__(WAVE)
rhs_vjp_kernel(int K, const double *__restrict__ vgeo, const double *__restrict__ vfgeo,
               const double *__restrict__ fgeo, const uint32_t *__restrict__ mapPq,
               const double *__restrict__ nrJ, const double *__restrict__ nsJ,
               const double *__restrict__ ntJ, const double *__restrict__ ws,
               const double *__restrict__ Uq, const double *__restrict__ Uf,
               const double *__restrict__ Rb, const double *__restrict__ sbar,
               double *__restrict__ uqb, double *__restrict__ ufb, double gamma, double gm1,
               double inv2gm1, double ltau) {
  constexpr int DIM = S::DIM, NQ = S::NQ, NFQ = S::NFQ, NFN = S::NFN, NFLD = S::NFLD;
  constexpr int NG = S::NG, TVT = S::TVT, VS = S::VS, VREC = S::VREC, FREC = S::FREC;
  constexpr int NPB = VjpSmem<S>::NPB, PER = VjpSmem<S>::per_elem, NFG = DIM + 1;
  constexpr int T = vf_steps<S>();
  extern __shared__ double smem[];
  __shared__ double s_nref[S::NFACES][DIM];

  const int lane = threadIdx.x;
  const int team = lane / NQ;
  const int i = lane - team * NQ;
  const bool active = team < TPW;
  const int k = blockIdx.x * TPW + team;
  const bool valid = active && k < K;
  const size_t kk = valid ? (size_t)k : 0;

  load_nref<S>(lane, nrJ, nsJ, ntJ, s_nref);
  double *gV = smem + (active ? team : 0) * PER;   // [NPB][NQ] partner cotangents
  double *vrec = gV + NPB * NQ;                    // phase 1
  double *RbV = vrec + VREC * NQ;                  // phase 1: R_bar rows [NFLD][NQ]
  double *frec = vrec;                             // phase 2
  double *sbF = frec + FREC * NFN;                 // phase 2: s_bar own [NFLD][NFN]
  double *gF = sbF + NFLD * NFN;                   // phase 2: [NPB][NFN]

  // ---------------- phase 1: records, volume-volume pairs
  Node<DIM> me;
  double hG[NG], Rbi[NFLD];
  PrimBar<DIM> gI;
  primbar_zero<DIM>(gI);
  if (valid) {
    double U[NFLD];
    for (int f = 0; f < NFLD; ++f) U[f] = Uq[kk * NQ * NFLD + f * NQ + i];
    me = make_node<DIM, false>(U, gm1);
    for (int c = 0; c < NG; ++c) hG[c] = 0.5 * vgeo[kk * NQ * NG + c * NQ + i];
    store_node<DIM>(vrec, NQ, i, me);
    for (int c = 0; c < NG; ++c) vrec[(VS + c) * NQ + i] = hG[c];
    for (int f = 0; f < NFLD; ++f) {
      Rbi[f] = Rb[kk * NQ * NFLD + f * NQ + i];
      RbV[f * NQ + i] = Rbi[f];
    }
    for (int c = 0; c < NPB; ++c) gV[c * NQ + i] = 0.0;
  }
  __syncthreads();
  // logarithms of the records only where the wave is not smooth (as in the forward
  // volume term: a smooth wave's pairs all take the series branch)
  const double rho_ref = smem[NPB * NQ], beta_ref = smem[NPB * NQ + (DIM + 1) * NQ];
  const bool smooth_v = uniform_flag(
      wave_all(!valid || in_smooth_band<DIM>(me.rho, me.beta, rho_ref, beta_ref)));
  auto own_logs = [&]() {
    if (!valid) return;
    me.lrho = ln(me.rho);
    me.lbeta = ln(me.beta);
  };
  if (!smooth_v) {
    own_logs();
    if (valid) {
      vrec[(DIM + 2) * NQ + i] = me.lrho;
      vrec[(DIM + 3) * NQ + i] = me.lbeta;
    }
    __syncthreads();
  }
  // Loops kept rolled where unrolled completely they spill or leave one wave per SIMD
  // (3D N = 1, 2; 2D from N = 2 on): 3D N = 2, K = 16,464, 101 -> 81 us; 2D N = 4, K =
  // 8,192, 36 -> 30 us; 2D N = 2, K = 12,288 and 32,768, 39 -> 29 and 65 -> 50 us (8,192
  // and less the same).  The other shapes lose 5 % by it.
  constexpr bool ROLLED = DIM == 3 ? NQ <= 11 : NQ >= 6;
  auto bound = [](int v) { return ROLLED ? opaque_bound(v) : v; };
  if (valid) {
    const double *Dfw = ws;
    const double *Dbw = ws + DIM * TVT * NQ;
    const int steps = bound(TVT);
    for (int t = 0; t < steps; ++t) {
      if (2 * t > NQ) break;
      if (2 * t == NQ && i >= NQ / 2) continue;
      int j = i + t;
      if (j >= NQ) j -= NQ;
      const Node<DIM> pj = load_node<DIM>(vrec, NQ, j);
      double Ga[NG];
      for (int c = 0; c < NG; ++c) Ga[c] = hG[c] + vrec[(VS + c) * NQ + j];
      double Dxf[DIM], Dxb[DIM];
      for (int d = 0; d < DIM; ++d) Dxf[d] = Dxb[d] = 0.0;
      for (int r = 0; r < DIM; ++r) {
        const double a = ld_off(Dfw, (unsigned)((r * TVT + t) * NQ + i));
        const double b = ld_off(Dbw, (unsigned)((r * TVT + t) * NQ + i));
        for (int d = 0; d < DIM; ++d) {
          Dxf[d] = Dxf[d] + a * Ga[r * DIM + d];
          Dxb[d] = Dxb[d] + b * Ga[r * DIM + d];
        }
      }
      // cotangent Rb_i (x) Dxf + Rb_j (x) Dxb (the partner row only off the diagonal)
      PrimBar<DIM> gj;
      primbar_zero<DIM>(gj);
      if (t > 0) {
        double nk[2][DIM], ck[2][NFLD];
        for (int d = 0; d < DIM; ++d) {
          nk[0][d] = Dxf[d];
          nk[1][d] = Dxb[d];
        }
        for (int f = 0; f < NFLD; ++f) {
          ck[0][f] = Rbi[f];
          ck[1][f] = RbV[f * NQ + j];
        }
        flux_dot_vjp_k<DIM, 2>(me, pj, nk, ck, inv2gm1, gI, gj);
      } else {
        flux_dot_vjp<DIM>(me, pj, Dxf, Rbi, inv2gm1, gI, gj);
      }
      if (t == 0) {
        gI.rho += gj.rho;
        for (int d = 0; d < DIM; ++d) gI.u[d] += gj.u[d];
        gI.beta += gj.beta;
      } else {
        lds_add_primbar<DIM>(gV, NQ, j, gj);
      }
    }
  }
  __syncthreads();

  // ---------------- phase 2: face records, s_bar, volume-face pairs.  Face
  // point work of all teams is spread over the whole wave.
  auto team_base = [&](int t) { return smem + t * PER; };
  bool ok_f = true;
  constexpr int OFF_FREC = NPB * NQ, OFF_SBF = OFF_FREC + FREC * NFN, OFF_GF = OFF_SBF + NFLD * NFN;
  for (int p = lane; p < TPW * NFN; p += WAVE) {
    const int t = p / NFN;
    const int fn = p - t * NFN;
    const size_t kt = (size_t)blockIdx.x * TPW + t;
    if (kt >= (size_t)K) continue;
    double *frt = team_base(t) + OFF_FREC;
    double *sbt = team_base(t) + OFF_SBF;
    double *gft = team_base(t) + OFF_GF;
    double U[NFLD];
    for (int f = 0; f < NFLD; ++f) U[f] = Uf[kt * NFN * NFLD + f * NFN + fn];
    const Node<DIM> nf = make_node<DIM, false>(U, gm1);
    ok_f = ok_f && in_smooth_band<DIM>(nf.rho, nf.beta, rho_ref, beta_ref);
    store_node<DIM>(frt, NFN, fn, nf);
    const int face = fn / NFQ;
    for (int d = 0; d < DIM; ++d) {
      double b = 0.0;
      for (int r = 0; r < DIM; ++r)
        b = b + 0.5 * vfgeo[kt * NFN * NG + (r * DIM + d) * NFN + fn] * s_nref[face][r];
      frt[(VS + d) * NFN + fn] = b;
    }
    for (int f = 0; f < NFLD; ++f) sbt[f * NFN + fn] = sbar[kt * NFN * NFLD + f * NFN + fn];
    for (int c = 0; c < NPB; ++c) gft[c * NFN + fn] = 0.0;
  }
  __syncthreads();
  if (!uniform_flag(smooth_v && wave_all(ok_f))) {
    if (smooth_v) own_logs();
    for (int p = lane; p < TPW * NFN; p += WAVE) {
      const int t = p / NFN;
      const int fn = p - t * NFN;
      if ((size_t)blockIdx.x * TPW + t >= (size_t)K) continue;
      double *frt = team_base(t) + OFF_FREC;
      frt[(DIM + 2) * NFN + fn] = ln(frt[fn]);
      frt[(DIM + 3) * NFN + fn] = ln(frt[(DIM + 1) * NFN + fn]);
    }
    __syncthreads();
  }
  if (valid) {
    const double *W1 = ws + S::WS_D;
    const double *W2 = W1 + T * NQ;
    auto vf_pair = [&](int t, int fn, const double (&a)[DIM]) {
      const Node<DIM> pf = load_node<DIM>(frec, NFN, fn);
      double n[DIM];
      for (int d = 0; d < DIM; ++d) n[d] = a[d] + frec[(VS + d) * NFN + fn];
      const double w1 = ld_off(W1, (unsigned)(t * NQ + i));
      const double w2 = ld_off(W2, (unsigned)(t * NQ + i));
      double c[NFLD];
      for (int f = 0; f < NFLD; ++f) c[f] = w1 * Rbi[f] + w2 * sbF[f * NFN + fn];
      PrimBar<DIM> gf;
      primbar_zero<DIM>(gf);
      flux_dot_vjp<DIM>(me, pf, n, c, inv2gm1, gI, gf);
      lds_add_primbar<DIM>(gF, NFN, fn, gf);
    };
    auto own_normal = [&](int face, double (&a)[DIM]) {
      for (int d = 0; d < DIM; ++d) {
        double v = 0.0;
        for (int r = 0; r < DIM; ++r) v = v + hG[r * DIM + d] * s_nref[face][r];
        a[d] = v;
      }
    };
    if constexpr (face_chunked<S>()) {
      const int g = i / NFQ, o = i - (i / NFQ) * NFQ;
      const int faces = bound(S::NFACES), points = bound(NFQ);
      for (int c = 0; c < faces; ++c) {
        int face = c + g;
        if (face >= S::NFACES) face -= S::NFACES;
        double a[DIM];
        own_normal(face, a);
        for (int m = 0; m < points; ++m) {
          int node = o + m;
          if (node >= NFQ) node -= NFQ;
          vf_pair(c * NFQ + m, face * NFQ + node, a);
        }
      }
    } else {
      const int steps = bound(T);
      for (int t = 0; t < steps; ++t) {
        const int fn = vf_partner<S>(t, i);
        if (fn >= NFN) continue;
        double a[DIM];
        own_normal(fn / NFQ, a);
        vf_pair(t, fn, a);
      }
    }
  }
  __syncthreads();

  // ---------------- phase 3: surface terms at the face points, spread over the
  // whole wave.  A point's conservative-space part overwrites its s_bar slot
  // (only this lane reads that slot from here on).
  for (int p = lane; p < TPW * NFN; p += WAVE) {
    const int t = p / NFN;
    const int fn = p - t * NFN;
    const size_t kt = (size_t)blockIdx.x * TPW + t;
    if (kt >= (size_t)K) continue;
    double *sbt = team_base(t) + OFF_SBF;
    double *gft = team_base(t) + OFF_GF;
    const double *g = fgeo + kt * NFN * NFG;
    const size_t idM = (size_t)fn + kt * NFN * NFLD;
    const size_t idP = mapPq[kt * NFN + fn];
    double UM[NFLD], UP[NFLD], sbM[NFLD], cons[NFLD];
    for (int f = 0; f < NFLD; ++f) {
      UM[f] = Uf[idM + (size_t)f * NFN];
      UP[f] = Uf[idP + (size_t)f * NFN];
      sbM[f] = sbt[f * NFN + fn];
      cons[f] = 0.0;
    }
    Node<DIM> a = make_node<DIM, false>(UM, gm1);
    Node<DIM> b = make_node<DIM, false>(UP, gm1);
    double hnM[DIM];
    for (int d = 0; d < DIM; ++d) hnM[d] = 0.5 * g[fn + d * NFN];
    const double sJM = g[fn + DIM * NFN];
    PrimBar<DIM> ga, gb;
    primbar_zero<DIM>(ga);
    primbar_zero<DIM>(gb);
    flux_dot_vjp<DIM, true>(a, b, hnM, sbM, inv2gm1, ga, gb);
    double dlM[NFLD], dlP[NFLD];
    const double lamM = wavespeed<DIM>(UM, gamma, gm1, dlM);
    const double lamP = wavespeed<DIM>(UP, gamma, gm1, dlP);
    if (idP == idM) {
      // no neighbour: u~P = u~M, zero jump; both flux arguments are this point
      ga.rho += gb.rho;
      for (int d = 0; d < DIM; ++d) ga.u[d] += gb.u[d];
      ga.beta += gb.beta;
    } else {
      // own LF term  -ltau max(lamM, lamP) sJM (UP - UM) . sbM
      const double LfM = ltau * fmax(lamM, lamP) * sJM;
      double S1 = 0.0;
      for (int f = 0; f < NFLD; ++f) S1 = S1 + sbM[f] * (UP[f] - UM[f]);
      const double dM = (lamM >= lamP) ? -S1 * ltau * sJM : 0.0;
      for (int f = 0; f < NFLD; ++f) cons[f] += LfM * sbM[f] + dM * dlM[f];
      // the neighbour's terms at its matching point, where this point is the
      // second flux argument and the P side of its penalty
      const size_t eN = idP / ((size_t)NFN * NFLD);
      const int pN = (int)(idP - eN * (size_t)NFN * NFLD);
      const double *gN = fgeo + eN * NFN * NFG;
      double hnP[DIM], sbP[NFLD];
      for (int d = 0; d < DIM; ++d) hnP[d] = 0.5 * gN[pN + d * NFN];
      const double sJP = gN[pN + DIM * NFN];
      for (int f = 0; f < NFLD; ++f) sbP[f] = sbar[idP + (size_t)f * NFN];
      PrimBar<DIM> gx;
      primbar_zero<DIM>(gx);
      flux_dot_vjp<DIM>(b, a, hnP, sbP, inv2gm1, gx, ga);   // logarithms: taken above if needed
      const double LfP = ltau * fmax(lamP, lamM) * sJP;
      double S2 = 0.0;
      for (int f = 0; f < NFLD; ++f) S2 = S2 + sbP[f] * (UM[f] - UP[f]);
      const double dP = (lamM > lamP) ? -S2 * ltau * sJP : 0.0;
      for (int f = 0; f < NFLD; ++f) cons[f] += -LfP * sbP[f] + dP * dlM[f];
    }
    // plain adds: this lane owns face point (t, fn) after the barrier
    gft[0 * NFN + fn] += ga.rho;
    for (int d = 0; d < DIM; ++d) gft[(1 + d) * NFN + fn] += ga.u[d];
    gft[(DIM + 1) * NFN + fn] += ga.beta;
    for (int f = 0; f < NFLD; ++f) sbt[f * NFN + fn] = cons[f];
  }
  __syncthreads();

  // ---------------- phase 4: primitive -> conservative cotangents
  if (valid) {
    add_lds_primbar<DIM>(gI, gV, NQ, i);
    double Ub[NFLD];
    primbar_to_cons<DIM>(me, gI, gm1, Ub);
    for (int f = 0; f < NFLD; ++f) uqb[kk * NQ * NFLD + f * NQ + i] = Ub[f];
  }
  for (int p = lane; p < TPW * NFN; p += WAVE) {
    const int t = p / NFN;
    const int fn = p - t * NFN;
    const size_t kt = (size_t)blockIdx.x * TPW + t;
    if (kt >= (size_t)K) continue;
    const double *frt = team_base(t) + OFF_FREC;
    const double *sbt = team_base(t) + OFF_SBF;
    double *gft = team_base(t) + OFF_GF;
    const Node<DIM> nf = load_node<DIM>(frt, NFN, fn);
    PrimBar<DIM> gf;
    primbar_zero<DIM>(gf);
    add_lds_primbar<DIM>(gf, gft, NFN, fn);
    double Ub[NFLD];
    primbar_to_cons<DIM>(nf, gf, gm1, Ub);
    for (int f = 0; f < NFLD; ++f) ufb[kt * NFN * NFLD + f * NFN + fn] = Ub[f] + sbt[f * NFN + fn];
  }
}

// (Q_bar, res_bar) <- stage VJP; R_bar written.  Q is the stage's output state.
// Workgroup shape of the update VJPs.  2D: one wave (its barriers cost nothing).  3D:
// four waves; at N = 1 they share the operators staged in LDS (the transposed products
// read them along rows, which through L1 touches a cache line per lane).
template <class S> constexpr int uvjp_wg_waves() { return S::DIM == 2 ? 1 : 4; }
// Whether the products next to the nonlinear maps, in these kernels and in
// proj_vjp_kernel, are unrolled completely.  In parts elsewhere: completely, the larger
// shapes spill and 2D N = 3 to 5 lose waves (4 to 10 % at K >= 12,288).  2D N = 2, K =
// 2,048, four at a time / completely: update VJP 9.3 / 8.6 us, projection VJP 8.9 / 7.9;
// 3D N = 1: projection VJP 8.5 / 8.2; 2D N = 5, four / eight at a time: 12.0 / 10.8.
template <class S> constexpr bool vjp_unrolled() { return S::NQ <= 6; }

template <class S, int TPW>
__global__ void __launch_bounds__(WAVE * uvjp_wg_waves<S>())
update_vjp_kernel(int K, const double *__restrict__ Jq, const double *__restrict__ VqPq,
                  const double *__restrict__ VfPq, double fa, double fb, double fdt,
                  const double *__restrict__ Q, double *__restrict__ Qb,
                  double *__restrict__ resb, const double *__restrict__ uqb,
                  const double *__restrict__ ufb, double *__restrict__ Rb, double gamma,
                  double lgm1, const double *__restrict__ VqLq, double *__restrict__ sbar) {
  constexpr int DIM = S::DIM, NQ = S::NQ, NFN = S::NFN, NFLD = S::NFLD;
  constexpr int WPB = uvjp_wg_waves<S>();
  constexpr bool OPS_LDS = WPB > 1;
  constexpr int EPB = WPB * TPW;
  constexpr int UNROLL = vjp_unrolled<S>() ? NQ : 4, UNROLLF = vjp_unrolled<S>() ? NFN : 8;
  __shared__ double sP[OPS_LDS ? NQ * NQ : 1];
  __shared__ double sPf[OPS_LDS ? NFN * NQ : 1];
  __shared__ double bufA[EPB][NFLD][NQ];
  __shared__ double bufB[EPB][NFLD][NQ];
  __shared__ double bufF[EPB][NFLD][NFN];
  if constexpr (OPS_LDS) {
    for (int idx = threadIdx.x; idx < NQ * NQ; idx += blockDim.x) sP[idx] = VqPq[idx];
    for (int idx = threadIdx.x; idx < NFN * NQ; idx += blockDim.x) sPf[idx] = VfPq[idx];
  }
  auto Pv = [&](int idx) {      // VqPq, column-major
    if constexpr (OPS_LDS) return sP[idx]; else return ld_off(VqPq, (unsigned)idx);
  };
  auto Pf = [&](int idx) {      // VfPq, column-major
    if constexpr (OPS_LDS) return sPf[idx]; else return ld_off(VfPq, (unsigned)idx);
  };
  const int wave = threadIdx.x / WAVE;
  const int wl = threadIdx.x % WAVE;
  const int tw = wl / NQ;
  const int i = wl - tw * NQ;
  const bool active = tw < TPW;
  const int e = wave * TPW + (active ? tw : 0);
  const int k = blockIdx.x * EPB + e;
  const bool valid = active && k < K;
  const size_t base = (valid ? (size_t)k : 0) * NQ * NFLD;

  // A x (row i) and A^T x (column i) with A = VqPq
  auto mv = [&](double (*in)[NQ], double (&r)[NFLD]) {
    for (int f = 0; f < NFLD; ++f) r[f] = 0.0;
#pragma unroll 8
    for (int j = 0; j < NQ; ++j) {
      const double P = Pv(i + j * NQ);
      for (int f = 0; f < NFLD; ++f) r[f] += P * in[f][j];
    }
  };
  auto mvT = [&](double (*in)[NQ], double (&r)[NFLD]) {
    for (int f = 0; f < NFLD; ++f) r[f] = 0.0;
#pragma unroll 8
    for (int j = 0; j < NQ; ++j) {
      const double P = Pv(j + i * NQ);
      for (int f = 0; f < NFLD; ++f) r[f] += P * in[f][j];
    }
  };

  double U[NFLD], J = 1.0, invJ = 1.0;
  if (valid) {
    J = Jq[(size_t)k * NQ + i];
    invJ = rcp(J);
    for (int f = 0; f < NFLD; ++f) U[f] = Q[base + i + f * NQ];
    double V[NFLD];
    entropy_vars<DIM>(U, gamma, V);
    for (int f = 0; f < NFLD; ++f) bufA[e][f][i] = V[f] * J;
  }
  __syncthreads();
  if (valid) {
    double r[NFLD];
    mv(bufA[e], r);
    for (int f = 0; f < NFLD; ++f) bufB[e][f][i] = r[f] * invJ;
  }
  __syncthreads();
  if (valid) {
    double r[NFLD];
    mv(bufB[e], r);
    for (int f = 0; f < NFLD; ++f) bufA[e][f][i] = r[f];  // v~
  }
  __syncthreads();
  // cotangents of v~ through u(v~) and u(VfPq v~): the stage writes rhsQ = u(v~)
  // (v~ already lies in the range of the projection VqPq).  This phase reads
  // only bufA; bufB was last read before the barrier above and bufF is read
  // after the next one, so the results go straight to LDS.
  if (valid) {
    double V[NFLD], Ub[NFLD], g[NFLD];
    for (int f = 0; f < NFLD; ++f) V[f] = bufA[e][f][i];
    for (int f = 0; f < NFLD; ++f) Ub[f] = uqb[base + i + f * NQ];
    conservative_vars_vjp<DIM>(V, gamma, lgm1, Ub, g);
    for (int f = 0; f < NFLD; ++f) bufB[e][f][i] = g[f];
  }
  // face points of the wave's TPW elements, spread over all its lanes
  for (int p = wl; p < TPW * NFN; p += WAVE) {
    const int t = p / NFN;
    const int fn = p - t * NFN;
    const int et = wave * TPW + t;
    const int kt = blockIdx.x * EPB + et;
    if (kt >= K) continue;
    double V[NFLD], Ub[NFLD], g[NFLD];
    for (int f = 0; f < NFLD; ++f) V[f] = 0.0;
#pragma unroll UNROLL
    for (int j = 0; j < NQ; ++j) {
      const double P = Pf(fn + j * NFN);
      for (int f = 0; f < NFLD; ++f) V[f] += P * bufA[et][f][j];
    }
    for (int f = 0; f < NFLD; ++f) Ub[f] = ufb[(size_t)kt * NFN * NFLD + fn + f * NFN];
    conservative_vars_vjp<DIM>(V, gamma, lgm1, Ub, g);
    for (int f = 0; f < NFLD; ++f) bufF[et][f][fn] = g[f];
  }
  __syncthreads();
  // v~_bar = g_q + VfPq^T g_f ; then through VqPq diag(1/J) VqPq
  if (valid) {
    double r[NFLD];
    for (int f = 0; f < NFLD; ++f) r[f] = bufB[e][f][i];
#pragma unroll UNROLLF
    for (int fn = 0; fn < NFN; ++fn) {
      const double P = Pf(fn + i * NFN);
      for (int f = 0; f < NFLD; ++f) r[f] += P * bufF[e][f][fn];
    }
    for (int f = 0; f < NFLD; ++f) bufA[e][f][i] = r[f];
  }
  __syncthreads();
  if (valid) {
    double r[NFLD];
    mvT(bufA[e], r);
    for (int f = 0; f < NFLD; ++f) bufB[e][f][i] = r[f] * invJ;
  }
  __syncthreads();
  double rb[NFLD];
  if (valid) {
    double wb[NFLD], Vb[NFLD], Ub[NFLD];
    mvT(bufB[e], wb);
    for (int f = 0; f < NFLD; ++f) Vb[f] = J * wb[f];
    entropy_vars_vjp<DIM>(U, gamma, Vb, Ub);
    for (int f = 0; f < NFLD; ++f) {
      const size_t id = base + i + f * NQ;
      const double qb = Qb[id] + Ub[f];        // cotangent of Q'
      const double resb_tot = resb[id] + fb * qb;  // Q' = Q + fb res'
      Qb[id] = qb;
      resb[id] = fa * resb_tot;
      rb[f] = fdt * resb_tot;
    }
  }
  __syncthreads();
  // R_bar = -2 VqPq^T diag(1/J) VqPq^T r_bar
  if (valid)
    for (int f = 0; f < NFLD; ++f) bufA[e][f][i] = rb[f];
  __syncthreads();
  if (valid) {
    double r[NFLD];
    mvT(bufA[e], r);
    for (int f = 0; f < NFLD; ++f) bufB[e][f][i] = r[f] * invJ;
  }
  __syncthreads();
  double rbar[NFLD];
  if (valid) {
    double r[NFLD];
    mvT(bufB[e], r);
    for (int f = 0; f < NFLD; ++f) {
      rbar[f] = -2.0 * r[f];
      Rb[base + i + f * NQ] = rbar[f];
    }
  }
  if (!sbar) return;  // uniform: a kernel argument
  // s_bar = VqLq^T R_bar at this element's face points (what sbar_kernel computes)
  __syncthreads();
  if (valid)
    for (int f = 0; f < NFLD; ++f) bufA[e][f][i] = rbar[f];
  __syncthreads();
  for (int p = wl; p < TPW * NFN; p += WAVE) {
    const int t = p / NFN;
    const int fn = p - t * NFN;
    const int et = wave * TPW + t;
    const int kt = blockIdx.x * EPB + et;
    if (kt >= K) continue;
    double v[NFLD];
    for (int f = 0; f < NFLD; ++f) v[f] = 0.0;
#pragma unroll 4
    for (int j = 0; j < NQ; ++j) {
      const double L = ld_off(VqLq, (unsigned)(j + fn * NQ));
      for (int f = 0; f < NFLD; ++f) v[f] += L * bufA[et][f][j];
    }
    for (int f = 0; f < NFLD; ++f) sbar[(size_t)kt * NFN * NFLD + f * NFN + fn] = v[f];
  }
}

// The update VJP with its eight products on MFMA.  A lane per row reads an operator
// entry and NFLD inputs from LDS for NFLD multiply-adds, and the LDS ports bound the
// kernel; a 16 x 16 tile reads two values for 16.  The operators come through L1: staged
// in LDS they cost workgroups per CU and gained nothing.  Bound by the memory it moves
// and the chain of barriers between the products.  Used where the rows fill enough of a
// tile: 3D from N = 2, 2D from N = 4.  A pass of two steps and their reverse (four in
// 2D), a lane per row -> this kernel: 3D N = 2, K = 16,464: 2.32 -> 2.28 ms; N = 3,
// K = 10,368: 4.15 -> 3.88 ms (update VJP 87 -> 56 us); N = 4, K = 3,072: 3.24 -> 3.10 ms;
// 2D K = 8,192, N = 4: 1.83 -> 1.74 ms; N = 5: 4.05 -> 3.89 ms.  Below, it loses: 2D
// N = 1: 0.90 -> 1.03 ms, N = 2: 1.235 -> 1.28 ms, N = 3 (K = 2,048): 1.77 -> 1.80 ms;
// 3D N = 1: 1.17 -> 1.23 ms.
template <class S> constexpr bool uvjp_mfma() { return S::DIM == 3 ? S::NQ >= 11 : S::NQ >= 16; }

// OUT[c][i] = sum_j M(i, j) IN[c][j] for the NCOL columns of a workgroup on MFMA, the
// 16 x 16 tiles spread over its W waves; sums in ascending j, one fused multiply-add
// per term.  M(i, j) is read through `m` (LDS or L1), IN and OUT are LDS with leading
// dimensions LDI and LDO.  Columns are independent: those of absent elements hold
// whatever the LDS held.
template <int W, int NCOL, int ROWS, int KD, int LDI, int LDO, class M>
__device__ __forceinline__ void uvjp_product(M m, const double *in, double *out, int lane,
                                             int wave) {
  constexpr int MT = (ROWS + 15) / 16, NT = (NCOL + 15) / 16, KS = (KD + 3) / 4;
  const int lr = lane & 15, lk = lane >> 4;
  double a[KS];
  auto load_a = [&](int mt) {
    const int row = 16 * mt + lr;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int j = 4 * ks + lk;
      a[ks] = (j < KD && row < ROWS) ? m(row, j) : 0.0;
    }
  };
  constexpr bool FIXED = W % MT == 0;    // a wave's tiles are of one row block
  if constexpr (FIXED) load_a(wave % MT);
  for (int t = wave; t < MT * NT; t += W) {
    const int mt = t % MT;
    const int c = 16 * (t / MT) + lr;
    const double *x = in + (c < NCOL ? c : 0) * LDI;
    double b[KS];
    if constexpr (!FIXED) load_a(mt);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int j = 4 * ks + lk;
      b[ks] = j < KD ? x[j] : 0.0;
    }
    dbl4 acc = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) acc = mfma_f64_16x16x4(a[ks], b[ks], acc);
    if (c < NCOL)
      for (int r = 0; r < 4; ++r) {
        const int i = 16 * mt + lk + 4 * r;
        if (i < ROWS) out[c * LDO + i] = acc[r];
      }
  }
}

template <class S, int TPW>
__global__ void __launch_bounds__(WAVE * uvjp_wg_waves<S>())
update_vjp_mfma_kernel(int K, const double *__restrict__ Jq, const double *__restrict__ VqPq,
                  const double *__restrict__ VfPq, double fa, double fb, double fdt,
                  const double *__restrict__ Q, double *__restrict__ Qb,
                  double *__restrict__ resb, const double *__restrict__ uqb,
                  const double *__restrict__ ufb, double *__restrict__ Rb, double gamma,
                  double lgm1, const double *__restrict__ VqLq, double *__restrict__ sbar) {
  constexpr int DIM = S::DIM, NQ = S::NQ, NFN = S::NFN, NFLD = S::NFLD;
  constexpr int W = uvjp_wg_waves<S>();
  constexpr int EPB = W * TPW, NCOL = EPB * NFLD;
  constexpr int LQ = NQ | 1, LF = NFN | 1;     // odd: no bank conflicts across columns
  __shared__ double bufA[NCOL * LQ];
  __shared__ double bufB[NCOL * LQ];
  __shared__ double bufF[NCOL * LF];
  auto P = [&](int i, int j) { return ld_off(VqPq, (unsigned)(i + j * NQ)); };
  auto Pt = [&](int i, int j) { return ld_off(VqPq, (unsigned)(j + i * NQ)); };
  auto Pf = [&](int i, int j) { return ld_off(VfPq, (unsigned)(i + j * NFN)); };
  auto Pft = [&](int i, int j) { return ld_off(VfPq, (unsigned)(j + i * NFN)); };
  auto Lt = [&](int i, int j) { return ld_off(VqLq, (unsigned)(j + i * NQ)); };
  const int wave = threadIdx.x / WAVE;
  const int wl = threadIdx.x % WAVE;
  const int tw = wl / NQ;
  const int i = wl - tw * NQ;
  const bool active = tw < TPW;
  const int e = wave * TPW + (active ? tw : 0);
  const int k = blockIdx.x * EPB + e;
  const bool valid = active && k < K;
  const size_t base = (valid ? (size_t)k : 0) * NQ * NFLD;
  double *A = bufA + e * NFLD * LQ + (active ? i : 0), *B = bufB + e * NFLD * LQ + (active ? i : 0);
  auto mv = [&](double *in, double *out) {
    uvjp_product<W, NCOL, NQ, NQ, LQ, LQ>(P, in, out, wl, wave);
  };
  auto mvT = [&](double *in, double *out) {
    uvjp_product<W, NCOL, NQ, NQ, LQ, LQ>(Pt, in, out, wl, wave);
  };

  double U[NFLD], J = 1.0, invJ = 1.0;
  if (valid) {
    J = Jq[(size_t)k * NQ + i];
    invJ = rcp(J);
    for (int f = 0; f < NFLD; ++f) U[f] = Q[base + i + f * NQ];
    double V[NFLD];
    entropy_vars<DIM>(U, gamma, V);
    for (int f = 0; f < NFLD; ++f) A[f * LQ] = V[f] * J;
  }
  __syncthreads();
  mv(bufA, bufB);
  __syncthreads();
  if (valid)
    for (int f = 0; f < NFLD; ++f) B[f * LQ] *= invJ;
  __syncthreads();
  mv(bufB, bufA);                                    // v~
  __syncthreads();
  // cotangents of v~ through u(v~) and u(VfPq v~): the stage writes rhsQ = u(v~)
  // (v~ already lies in the range of the projection VqPq)
  uvjp_product<W, NCOL, NFN, NQ, LQ, LF>(Pf, bufA, bufF, wl, wave);
  double gq[NFLD];
  if (valid) {
    double V[NFLD], Ub[NFLD];
    for (int f = 0; f < NFLD; ++f) V[f] = A[f * LQ];
    for (int f = 0; f < NFLD; ++f) Ub[f] = uqb[base + i + f * NQ];
    conservative_vars_vjp<DIM>(V, gamma, lgm1, Ub, gq);
  }
  __syncthreads();
  // face points of the wave's TPW elements, spread over all its lanes
  for (int p = wl; p < TPW * NFN; p += WAVE) {
    const int t = p / NFN;
    const int fn = p - t * NFN;
    const int et = wave * TPW + t;
    const int kt = blockIdx.x * EPB + et;
    if (kt >= K) continue;
    double *F = bufF + et * NFLD * LF + fn;
    double V[NFLD], Ub[NFLD], g[NFLD];
    for (int f = 0; f < NFLD; ++f) V[f] = F[f * LF];
    for (int f = 0; f < NFLD; ++f) Ub[f] = ufb[(size_t)kt * NFN * NFLD + fn + f * NFN];
    conservative_vars_vjp<DIM>(V, gamma, lgm1, Ub, g);
    for (int f = 0; f < NFLD; ++f) F[f * LF] = g[f];
  }
  __syncthreads();
  // v~_bar = g_q + VfPq^T g_f ; then through VqPq diag(1/J) VqPq
  uvjp_product<W, NCOL, NQ, NFN, LF, LQ>(Pft, bufF, bufB, wl, wave);
  __syncthreads();
  if (valid)
    for (int f = 0; f < NFLD; ++f) B[f * LQ] += gq[f];
  __syncthreads();
  mvT(bufB, bufA);
  __syncthreads();
  if (valid)
    for (int f = 0; f < NFLD; ++f) A[f * LQ] *= invJ;
  __syncthreads();
  mvT(bufA, bufB);
  __syncthreads();
  if (valid) {
    double Vb[NFLD], Ub[NFLD];
    for (int f = 0; f < NFLD; ++f) Vb[f] = J * B[f * LQ];
    entropy_vars_vjp<DIM>(U, gamma, Vb, Ub);
    for (int f = 0; f < NFLD; ++f) {
      const size_t id = base + i + f * NQ;
      const double qb = Qb[id] + Ub[f];        // cotangent of Q'
      const double resb_tot = resb[id] + fb * qb;  // Q' = Q + fb res'
      Qb[id] = qb;
      resb[id] = fa * resb_tot;
      A[f * LQ] = fdt * resb_tot;              // r_bar
    }
  }
  // R_bar = -2 VqPq^T diag(1/J) VqPq^T r_bar
  __syncthreads();
  mvT(bufA, bufB);
  __syncthreads();
  if (valid)
    for (int f = 0; f < NFLD; ++f) B[f * LQ] *= invJ;
  __syncthreads();
  mvT(bufB, bufA);
  __syncthreads();
  if (valid)
    for (int f = 0; f < NFLD; ++f) {
      const double rbar = -2.0 * A[f * LQ];
      Rb[base + i + f * NQ] = rbar;
      A[f * LQ] = rbar;
    }
  if (!sbar) return;  // uniform: a kernel argument
  // s_bar = VqLq^T R_bar at this element's face points (what sbar_kernel computes)
  __syncthreads();
  uvjp_product<W, NCOL, NFN, NQ, LQ, LF>(Lt, bufA, bufF, wl, wave);
  __syncthreads();
  for (int p = threadIdx.x; p < NCOL * NFN; p += WAVE * W) {
    const int c = p / NFN;
    const size_t at = (size_t)blockIdx.x * NCOL * NFN + p;
    if ((int)blockIdx.x * EPB + c / NFLD < K) sbar[at] = bufF[c * LF + p - c * NFN];
  }
}

template <class S>
inline void launch_update_vjp(int K, const double *Jq, const double *VqPq, const double *VfPq,
                              double fa, double fb, double fdt, const double *Q, double *Qb,
                              double *resb, const double *uqb, const double *ufb, double *Rb,
                              double gamma, const double *VqLq, double *sbar, hipStream_t st) {
  constexpr int TPW = WAVE / S::NQ, T = WAVE * uvjp_wg_waves<S>();
  constexpr int EPB = uvjp_wg_waves<S>() * TPW;
  const int blocks = (K + EPB - 1) / EPB;
  const double lgm1 = std::log(gamma - 1.0);
  if constexpr (uvjp_mfma<S>())
    update_vjp_mfma_kernel<S, TPW><<<blocks, T, 0, st>>>(K, Jq, VqPq, VfPq, fa, fb, fdt, Q, Qb, resb, uqb,
                                                         ufb, Rb, gamma, lgm1, VqLq, sbar);
  else
    update_vjp_kernel<S, TPW><<<blocks, T, 0, st>>>(K, Jq, VqPq, VfPq, fa, fb, fdt, Q, Qb, resb, uqb,
                                                    ufb, Rb, gamma, lgm1, VqLq, sbar);
}

// Q_bar += VJP of (u~q, u~f) = (u(VqPq v(Q)), u(VfPq v(Q))) at Q.
template <class S, int TPW>
__global__ void __launch_bounds__(WAVE * 4)
proj_vjp_kernel(int K, const double *__restrict__ VqPq, const double *__restrict__ VfPq,
                const double *__restrict__ Q, const double *__restrict__ uqb,
                const double *__restrict__ ufb, double *__restrict__ Qb, double gamma,
                double lgm1) {
  constexpr int DIM = S::DIM, NQ = S::NQ, NFN = S::NFN, NFLD = S::NFLD;
  constexpr int EPB = 4 * TPW;
  constexpr int PART = DIM == 2 && NQ >= 16 ? 8 : 4;
  constexpr int UNROLL = vjp_unrolled<S>() ? NQ : PART, UNROLLF = vjp_unrolled<S>() ? NFN : PART;
  __shared__ double bufA[EPB][NFLD][NQ];
  __shared__ double bufB[EPB][NFLD][NQ];
  __shared__ double bufF[EPB][NFLD][NFN];
  const int wave = threadIdx.x / WAVE;
  const int wl = threadIdx.x % WAVE;
  const int tw = wl / NQ;
  const int i = wl - tw * NQ;
  const bool active = tw < TPW;
  const int e = wave * TPW + (active ? tw : 0);
  const int k = blockIdx.x * EPB + e;
  const bool valid = active && k < K;
  const size_t base = (valid ? (size_t)k : 0) * NQ * NFLD;
  double U[NFLD];
  if (valid) {
    double V[NFLD];
    for (int f = 0; f < NFLD; ++f) U[f] = Q[base + i + f * NQ];
    entropy_vars<DIM>(U, gamma, V);
    for (int f = 0; f < NFLD; ++f) bufA[e][f][i] = V[f];
  }
  __syncthreads();
  // cotangents through u(VqPq v) and u(VfPq v), straight to LDS; the face points of the
  // wave's elements spread over all its lanes
  if (valid) {
    double V[NFLD], Ub[NFLD], g[NFLD];
    for (int f = 0; f < NFLD; ++f) V[f] = 0.0;
#pragma unroll UNROLL
    for (int j = 0; j < NQ; ++j) {
      const double P = ld_off(VqPq, (unsigned)(i + j * NQ));
      for (int f = 0; f < NFLD; ++f) V[f] += P * bufA[e][f][j];
    }
    for (int f = 0; f < NFLD; ++f) Ub[f] = uqb[base + i + f * NQ];
    conservative_vars_vjp<DIM>(V, gamma, lgm1, Ub, g);
    for (int f = 0; f < NFLD; ++f) bufB[e][f][i] = g[f];
  }
  for (int p = wl; p < TPW * NFN; p += WAVE) {
    const int t = p / NFN;
    const int fn = p - t * NFN;
    const int et = wave * TPW + t;
    const int kt = blockIdx.x * EPB + et;
    if (kt >= K) continue;
    double V[NFLD], Ub[NFLD], g[NFLD];
    for (int f = 0; f < NFLD; ++f) V[f] = 0.0;
#pragma unroll UNROLL
    for (int j = 0; j < NQ; ++j) {
      const double P = ld_off(VfPq, (unsigned)(fn + j * NFN));
      for (int f = 0; f < NFLD; ++f) V[f] += P * bufA[et][f][j];
    }
    for (int f = 0; f < NFLD; ++f) Ub[f] = ufb[(size_t)kt * NFN * NFLD + fn + f * NFN];
    conservative_vars_vjp<DIM>(V, gamma, lgm1, Ub, g);
    for (int f = 0; f < NFLD; ++f) bufF[et][f][fn] = g[f];
  }
  __syncthreads();
  if (valid) {
    double vb[NFLD], Ub[NFLD];
    for (int f = 0; f < NFLD; ++f) vb[f] = 0.0;
#pragma unroll UNROLL
    for (int j = 0; j < NQ; ++j) {
      const double P = ld_off(VqPq, (unsigned)(j + i * NQ));
      for (int f = 0; f < NFLD; ++f) vb[f] += P * bufB[e][f][j];
    }
#pragma unroll UNROLLF
    for (int fn = 0; fn < NFN; ++fn) {
      const double P = ld_off(VfPq, (unsigned)(fn + i * NFN));
      for (int f = 0; f < NFLD; ++f) vb[f] += P * bufF[e][f][fn];
    }
    entropy_vars_vjp<DIM>(U, gamma, vb, Ub);
    for (int f = 0; f < NFLD; ++f) Qb[base + i + f * NQ] += Ub[f];
  }
}

// Initial projection of a conservative state: u~q = u(VqPq v(Q)), u~f = u(VfPq v(Q))
// (euler.c:4028-4133).  Bound by its launch on the meshes of one card's adjoint: as
// tensor operations the same maps were some sixty launches, two operator uploads and
// 0.65 ms of a 2.44 ms pass (2D N = 3, K = 2,048, two steps and their reverse; now
// 1.79 ms), 0.6 ms of 4.76 ms at 3D N = 3, K = 10,368 (now 4.17 ms).  Each row has its
// own lane, the face points of a wave's elements are spread over all of its lanes;
// the operators (<= 30 KB) come through L1.
template <class S, int TPW>
__global__ void __launch_bounds__(WAVE * 4)
project_kernel(int K, const double *__restrict__ VqPq, const double *__restrict__ VfPq,
               const double *__restrict__ Q, double *__restrict__ rhsQ, double *__restrict__ Qf,
               double gamma, double lgm1) {
  constexpr int DIM = S::DIM, NQ = S::NQ, NFN = S::NFN, NFLD = S::NFLD;
  constexpr int EPB = 4 * TPW;
  __shared__ double buf[EPB][NFLD][NQ];
  const int wave = threadIdx.x / WAVE;
  const int wl = threadIdx.x % WAVE;
  const int tw = wl / NQ;
  const int i = wl - tw * NQ;
  const bool active = tw < TPW;
  const int e = wave * TPW + (active ? tw : 0);
  const int k = blockIdx.x * EPB + e;
  const bool valid = active && k < K;
  const size_t base = (valid ? (size_t)k : 0) * NQ * NFLD;
  if (valid) {
    double U[NFLD], V[NFLD];
    for (int f = 0; f < NFLD; ++f) U[f] = Q[base + i + f * NQ];
    entropy_vars<DIM>(U, gamma, V);
    for (int f = 0; f < NFLD; ++f) buf[e][f][i] = V[f];
  }
  __syncthreads();
  if (valid) {
    double U[NFLD], V[NFLD];
    for (int f = 0; f < NFLD; ++f) V[f] = 0.0;
#pragma unroll 4
    for (int j = 0; j < NQ; ++j) {
      const double P = ld_off(VqPq, (unsigned)(i + j * NQ));
      for (int f = 0; f < NFLD; ++f) V[f] += P * buf[e][f][j];
    }
    conservative_vars<DIM>(V, gamma, lgm1, U);
    for (int f = 0; f < NFLD; ++f) rhsQ[base + i + f * NQ] = U[f];
  }
  for (int p = wl; p < TPW * NFN; p += WAVE) {
    const int t = p / NFN;
    const int fn = p - t * NFN;
    const int et = wave * TPW + t;
    const int kt = blockIdx.x * EPB + et;
    if (kt >= K) continue;
    double U[NFLD], V[NFLD];
    for (int f = 0; f < NFLD; ++f) V[f] = 0.0;
#pragma unroll 4
    for (int j = 0; j < NQ; ++j) {
      const double P = ld_off(VfPq, (unsigned)(fn + j * NFN));
      for (int f = 0; f < NFLD; ++f) V[f] += P * buf[et][f][j];
    }
    conservative_vars<DIM>(V, gamma, lgm1, U);
    for (int f = 0; f < NFLD; ++f) Qf[(size_t)kt * NFN * NFLD + fn + f * NFN] = U[f];
  }
}
