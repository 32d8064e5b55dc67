// wadges_team.hpp -- volume term and fused stage of the shapes with two rows per lane
// (3D N = 3), one wave per face.  Included by wadges.hip after the packed
// stage, whose sums these kernels form in the same parts (the same bits).
//
// A workgroup of NFACES waves holds the E = TPW elements that one wave of the
// packed stage holds.  Wave w takes group w of the volume-volume steps, face w of
// the volume-face block and the face points of face w; its lanes own rows l and
// l + LPE of element `team` as in the packed stage, and face point l of face w.
// The instructions per element are the packed stage's, but
//   * the four waves share one LDS tile (49 KB for 5 elements instead of 20 KB per
//     wave), so registers, not LDS, set the occupancy: three waves per SIMD;
//   * a wave's walk is a quarter as long (3 + 12 steps instead of 12 + 48), so a
//     small mesh finishes in a third of the time.
// Used for every mesh: faster than the packed kernels that give the same bits at every
// size.  Fused stage, packed / this, microseconds on one card, launches back to back: K =
// 750 56.5 / 21.2; 2,058 61.9 / 30.1; 6,000 91.2 / 61.4; 10,368 146 / 101; 24,576 248 /
// 229; 82,944 793 / 754; 196,608 1,808 / 1,774.  Volume kernel: 24,576 190 / 179; 82,944
// 533 / 493; 196,608 1,230 / 1,188.  (A packed kernel that sums straight through, without
// the parts and so in other bits, takes 759 and 496 at 82,944, 1,742 and 1,158 at
// 196,608, where its fewer LDS reads weigh more.)  The LDS is busy
// 70 % of the time: a row's own record is read once per wave, the stride of an
// element is LPE mod 32 doubles (3 % against a stride that makes the elements of a
// wave meet in the banks), and neither records held in more registers (two waves per
// SIMD: 14 % slower) nor operator entries fetched ahead (2 %) pay.

template <class S> struct Team {
  static constexpr int NW = S::NFACES, T = WAVE * NW, E = S::TPW;
  static constexpr int TG = S::TVT / NW;                 // volume-volume steps per wave
  // per-element LDS (doubles): volume accumulators of the waves, volume records
  // (then face records, in the face's block the wave's row sums), face accumulators
  static constexpr int RQ = S::NFLD * S::NQ;
  static constexpr int VOFF = NW * RQ;
  static constexpr int FB = S::FREC * S::NFQ;            // one face's records
  static constexpr int AFOFF = VOFF + Max<S::VREC * S::NQ, NW * FB>::value;
  // LPE mod 32, so that the LPE-lane windows of a wave's elements lie next to each
  // other in the LDS banks
  static constexpr int END = AFOFF + S::NFLD * S::NFN;
  static constexpr int per_elem = END + (32 + S::LPE - END % 32) % 32;
  // the update's buffers, over the accumulators and the face records
  static constexpr int AOFF = 0, BOFF = RQ, TOFF = 2 * RQ;
  static constexpr int bytes = 8 * E * per_elem;
  static_assert(S::R == 2 && S::LPE == S::NFQ && S::TVT % NW == 0 && S::NQ % 2 == 1 && TG > 1,
                "two rows per lane, a face's points on an element's lanes, equal groups of steps");
  static_assert(RQ <= FB && TOFF + S::NFLD * S::NFN <= AFOFF, "regions");
};

// The lane's place in the workgroup.
template <class S> struct TeamLane {
  int tid, wave, lane, team, l;
  bool valid;                       // element `team` exists
  bool rv[S::R];                    // row l + r LPE exists
  __device__ __forceinline__ TeamLane(int t, int nvalid) {
    tid = t;
    wave = __builtin_amdgcn_readfirstlane(t / WAVE);
    lane = t - wave * WAVE;
    team = lane / S::LPE;
    l = lane - team * S::LPE;
    valid = team < nvalid;          // nvalid <= E
    if (!valid) team = 0;
    for (int r = 0; r < S::R; ++r) rv[r] = valid && l + r * S::LPE < S::NQ;
  }
};

// Volume term of the workgroup's elements.  On return LDS holds, per element, the
// volume accumulators T_w of the waves from 0 on, the row sums P_w of face w at the
// start of that face's record block, and the face rows (rhsQf) at AFOFF (this wave's
// face complete, the others' after a barrier).
template <class S>
__device__ __forceinline__ void team_volume(const TeamLane<S> &L, int kfirst, int nvalid,
                                            const double *Uq, const double *Uf, const double *vgeo,
                                            const double *vfgeo, const double *nrJ,
                                            const double *nsJ, const double *ntJ, const double *ws,
                                            double gm1, double inv2gm1, double *smem) {
  using X = Team<S>;
  constexpr int DIM = S::DIM, NQ = S::NQ, NFQ = S::NFQ, NFN = S::NFN, NFLD = S::NFLD, NG = S::NG;
  constexpr int R = S::R, LPE = S::LPE, VS = S::VS, TVT = S::TVT, PER = X::per_elem, TG = X::TG;
  double *el = smem + L.team * PER;
  double *vrec = el + X::VOFF;
  const int w = L.wave;

  // records: the lane's face point (kept in registers), then the volume nodes
  const size_t kt = kfirst + L.team;
  const int fn = w * NFQ + L.l;
  Node<DIM> nf;
  double nref[DIM];
  nref[0] = nrJ[w * NFQ];
  nref[1] = nsJ[w * NFQ];
  if constexpr (DIM == 3) nref[2] = ntJ[w * NFQ];
  {
    double U[NFLD];
    for (int f = 0; f < NFLD; ++f) U[f] = Uf[kt * NFN * NFLD + fn + f * NFN];
    nf = make_node<DIM, false>(U, gm1);
  }
  // the face node waits in its accumulators' place (registers for the block below)
  double *park = el + X::AFOFF + fn;
  if (L.valid) {
    park[0] = nf.rho;
    for (int d = 0; d < DIM; ++d) park[(1 + d) * NFN] = nf.hv[d];
    park[(1 + DIM) * NFN] = nf.beta;
  }
  for (int p = L.tid; p < nvalid * NQ; p += X::T) {
    const int e = p / NQ;
    const int i = p - e * NQ;
    const size_t k = kfirst + e;
    double U[NFLD];
    for (int f = 0; f < NFLD; ++f) U[f] = Uq[k * NQ * NFLD + i + f * NQ];
    double *rec = smem + e * PER + X::VOFF;
    for (int c = 0; c < NG; ++c) rec[(VS + c) * NQ + i] = 0.5 * vgeo[k * NQ * NG + i + c * NQ];
    store_node<DIM>(rec, NQ, i, make_node<DIM>(U, gm1));
  }
  __syncthreads();

  const double rho_ref = smem[X::VOFF], beta_ref = smem[X::VOFF + (DIM + 1) * NQ];
  bool in_band = true;
  for (int r = 0; r < R; ++r)
    if (L.rv[r])
      in_band = in_band && in_smooth_band<DIM>(vrec[L.l + r * LPE], vrec[(DIM + 1) * NQ + L.l + r * LPE],
                                               rho_ref, beta_ref);
  const bool smooth_v = uniform_flag(wave_all(in_band));

  // ---------------- volume-volume block: this wave's steps, one row of the lane after
  // the other (a row's record is read once); after its steps a row adds its own part
  double *accV = el + w * X::RQ;
  if (L.valid) {
    for (int r = 0; r < R; ++r)
      if (L.rv[r])
        for (int f = 0; f < NFLD; ++f) accV[f * NQ + L.l + r * LPE] = 0.0;
    wave_fence();
    const double *Dbw = ws + DIM * TVT * NQ;
    for (int r = 0; r < R; ++r) {
      if (!L.rv[r]) continue;
      const int i = L.l + r * LPE;
      const Node<DIM> pi = load_node<DIM>(vrec, NQ, i);
      double hG[NG], own[NFLD];
      for (int c = 0; c < NG; ++c) hG[c] = vrec[(VS + c) * NQ + i];
      for (int f = 0; f < NFLD; ++f) own[f] = 0.0;
#pragma unroll 1
      for (int t = w * TG; t < (w + 1) * TG; ++t) {
        int j = i + t;
        if (j >= NQ) j -= NQ;
        double Df[DIM], Db[DIM];
        for (int q = 0; q < DIM; ++q) {
          Df[q] = ld_off(ws, (unsigned)((q * TVT + t) * NQ + i));
          Db[q] = ld_off(Dbw, (unsigned)((q * TVT + t) * NQ + i));
        }
        const Node<DIM> pj = load_node<DIM>(vrec, NQ, j);
        double Ga[NG];
        for (int c = 0; c < NG; ++c) Ga[c] = hG[c] + vrec[(VS + c) * NQ + j];
        const PairFlux<DIM> P = pair_flux<DIM>(pi, pj, inv2gm1, smooth_v);
        double Dx[DIM];
        for (int d = 0; d < DIM; ++d) Dx[d] = 0.0;
        for (int q = 0; q < DIM; ++q)
          for (int d = 0; d < DIM; ++d) Dx[d] = Dx[d] + Df[q] * Ga[q * DIM + d];
        double c[NFLD];
        flux_dot<DIM>(P, Dx, c);
        for (int f = 0; f < NFLD; ++f) own[f] += c[f];
        if (t > 0) {
          for (int d = 0; d < DIM; ++d) Dx[d] = 0.0;
          for (int q = 0; q < DIM; ++q)
            for (int d = 0; d < DIM; ++d) Dx[d] = Dx[d] + Db[q] * Ga[q * DIM + d];
          flux_dot<DIM>(P, Dx, c);
          for (int f = 0; f < NFLD; ++f) lds_add(&accV[f * NQ + j], c[f]);
        }
      }
      for (int f = 0; f < NFLD; ++f) lds_add(&accV[f * NQ + i], own[f]);
    }
  }
  // the rows' records, and the own-side part of their averaged normals on this face
  Node<DIM> me[R];
  double a[R][DIM];
  for (int r = 0; r < R; ++r) {
    const int i = L.rv[r] ? L.l + r * LPE : 0;
    me[r] = load_node<DIM>(vrec, NQ, i);
    for (int d = 0; d < DIM; ++d) {
      double v = 0.0;
      for (int q = 0; q < DIM; ++q) v = v + vrec[(VS + q * DIM + d) * NQ + i] * nref[q];
      a[r][d] = v;
    }
  }
  __syncthreads();                  // the face records overwrite the volume records

  // ---------------- volume-face block: this wave's face
  double acc[R][NFLD];
  for (int r = 0; r < R; ++r)
    for (int f = 0; f < NFLD; ++f) acc[r][f] = 0.0;
  double *frec = vrec + w * X::FB;
  double *accF = el + X::AFOFF + w * NFQ;
  if (L.valid) {
    nf.rho = park[0];
    double hh = 0.0;
    for (int d = 0; d < DIM; ++d) {
      nf.hv[d] = park[(1 + d) * NFN];
      hh = d == 0 ? nf.hv[0] * nf.hv[0] : hh + nf.hv[d] * nf.hv[d];
    }
    nf.beta = park[(1 + DIM) * NFN];
    nf.hq = 2.0 * hh;               // |u|^2 / 2 of the halved velocity: exact scaling
  }
  const bool smooth_f = uniform_flag(
      smooth_v && wave_all(!L.valid || in_smooth_band<DIM>(nf.rho, nf.beta, rho_ref, beta_ref)));
  if (L.valid) {
    if (!smooth_f) {
      nf.lrho = ln(nf.rho);
      nf.lbeta = ln(nf.beta);
    }
    store_node<DIM>(frec, NFQ, L.l, nf);
    for (int d = 0; d < DIM; ++d) {
      double b = 0.0;
      for (int q = 0; q < DIM; ++q)
        b = b + 0.5 * vfgeo[kt * NFN * NG + fn + (q * DIM + d) * NFN] * nref[q];
      frec[(VS + d) * NFQ + L.l] = b;
    }
    wave_fence();
    int iw[R];
    for (int r = 0; r < R; ++r) iw[r] = L.rv[r] ? L.l + r * LPE : 0;
    const double *W1 = ws + S::WS_D + S::WS_W;
    const double *W2 = W1 + NFN * NQ;
    // the weights of a step are loaded during the one before
    double w1n[R], w2n[R];
    auto fetch = [&](int m) {
      for (int r = 0; r < R; ++r) {
        w1n[r] = ld_off(W1, (unsigned)((w * NFQ + m) * NQ + iw[r]));
        w2n[r] = ld_off(W2, (unsigned)((w * NFQ + m) * NQ + iw[r]));
      }
    };
    fetch(0);
    auto vf_step = [&](int m, bool first) {
      int q = L.l + m;
      if (q >= NFQ) q -= NFQ;
      double w1[R], w2[R];
      for (int r = 0; r < R; ++r) {
        w1[r] = w1n[r];
        w2[r] = w2n[r];
      }
      if (m + 1 < NFQ) fetch(m + 1);
      const Node<DIM> pf = load_node<DIM>(frec, NFQ, q);
      double pb[DIM];
      for (int d = 0; d < DIM; ++d) pb[d] = frec[(VS + d) * NFQ + q];
      double sF[NFLD];
      for (int f = 0; f < NFLD; ++f) sF[f] = 0.0;
      for (int r = 0; r < R; ++r) {
        if (!L.rv[r]) continue;
        double n[DIM];
        for (int d = 0; d < DIM; ++d) n[d] = a[r][d] + pb[d];
        const PairFlux<DIM> P = pair_flux<DIM>(me[r], pf, inv2gm1, smooth_f);
        double Fn[NFLD];
        flux_dot<DIM>(P, n, Fn);
        for (int f = 0; f < NFLD; ++f) {
          acc[r][f] += w1[r] * Fn[f];
          sF[f] += w2[r] * Fn[f];
        }
      }
      for (int f = 0; f < NFLD; ++f) {
        if (first) accF[f * NFN + q] = sF[f];
        else lds_add(&accF[f * NFN + q], sF[f]);
      }
    };
    vf_step(0, true);               // every point once: stores
    wave_fence();
#pragma unroll 1
    for (int m = 1; m < NFQ; ++m) vf_step(m, false);
    wave_fence();
    // the row sums, over this face's records
    for (int r = 0; r < R; ++r)
      if (L.rv[r])
        for (int f = 0; f < NFLD; ++f) frec[f * NQ + L.l + r * LPE] = acc[r][f];
    wave_fence();
  }
}

// Row i, field f of an element: the parts of the volume term in the packed stage's order.
template <class S> __device__ __forceinline__ double team_row(const double *el, int f, int i) {
  using X = Team<S>;
  double v = el[f * S::NQ + i];
  for (int w = 1; w < X::NW; ++w) v += el[w * X::RQ + f * S::NQ + i];
  for (int w = 0; w < X::NW; ++w) v += el[X::VOFF + w * X::FB + f * S::NQ + i];
  return v;
}

constexpr int kTeamWaves = 3;   // per SIMD: the LDS tile of 3D N = 3 allows three workgroups per CU

template <class S>
__global__ void __launch_bounds__(Team<S>::T) __attribute__((amdgpu_waves_per_eu(kTeamWaves)))
team_vol_kernel(int K, const double *__restrict__ vgeo, const double *__restrict__ vfgeo,
         const double *__restrict__ nrJ, const double *__restrict__ nsJ,
         const double *__restrict__ ntJ, const double *__restrict__ ws,
         const double *__restrict__ Qf, double *rhsQ, double *__restrict__ rhsQf, double gm1,
         double inv2gm1) {
  using X = Team<S>;
  constexpr int NQ = S::NQ, NFN = S::NFN, NFLD = S::NFLD;
  extern __shared__ double smem[];
  const int kfirst = blockIdx.x * X::E;
  const int nvalid = K - kfirst < X::E ? K - kfirst : X::E;
  const TeamLane<S> L(threadIdx.x, nvalid);
  team_volume<S>(L, kfirst, nvalid, rhsQ, Qf, vgeo, vfgeo, nrJ, nsJ, ntJ, ws, gm1, inv2gm1, smem);
  __syncthreads();
  for (int p = L.tid; p < nvalid * X::RQ; p += X::T) {
    const int e = p / X::RQ;
    const int c = p - e * X::RQ;
    const int f = c / NQ;
    rhsQ[(size_t)kfirst * X::RQ + p] = team_row<S>(smem + e * X::per_elem, f, c - f * NQ);
  }
  for (int p = L.tid; p < nvalid * NFLD * NFN; p += X::T) {
    const int e = p / (NFLD * NFN);
    rhsQf[(size_t)kfirst * NFLD * NFN + p] =
        smem[e * X::per_elem + X::AFOFF + (p - e * NFLD * NFN)];
  }
}

// A wave's tiles (idx = wave + NW x; row tile idx % MT, column tile idx / MT) of a
// product of all the workgroup's elements on the matrix cores: the A operands, and
// the product (sums in ascending index order, one fused multiply-add per term, as
// wave_product_mfma).
template <class S, int ROWS, int KD> struct TeamTiles {
  using X = Team<S>;
  static constexpr int MT = (ROWS + 15) / 16, NT = (X::E * S::NFLD + 15) / 16, KS = (KD + 3) / 4;
  static constexpr int TX = (MT * NT + X::NW - 1) / X::NW;
  double a[TX][KS];
  __device__ __forceinline__ void load(const double *M, const TeamLane<S> &L) {
    const int lr = L.lane & 15, lk = L.lane >> 4;
    for (int x = 0; x < TX; ++x) {
      const int row = 16 * ((L.wave + X::NW * x) % MT) + lr;
      for (int ks = 0; ks < KS; ++ks) {
        const int j = 4 * ks + lk;
        a[x][ks] = (j < KD && row < ROWS) ? ld_off(M, (unsigned)(row + j * ROWS)) : 0.0;
      }
    }
  }
  __device__ __forceinline__ void product(int in_off, int out_off, double *smem,
                                          const TeamLane<S> &L, int nvalid) const {
    const int lr = L.lane & 15, lk = L.lane >> 4;
    for (int x = 0; x < TX; ++x) {
      const int idx = L.wave + X::NW * x;
      if (MT * NT % X::NW != 0 && idx >= MT * NT) break;     // uniform over the wave
      const int mt = idx % MT, c = 16 * (idx / MT) + lr;
      const int e = c / S::NFLD;
      const int f = c - e * S::NFLD;
      const bool ok = c < X::E * S::NFLD && e < nvalid;
      const double *in = smem + (ok ? e * X::per_elem + in_off + f * KD : 0);
      double *out = smem + (ok ? e * X::per_elem + out_off + f * ROWS : 0);
      dbl4 acc = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int j = 4 * ks + lk;
        acc = mfma_f64_16x16x4(a[x][ks], (ok && j < KD) ? in[j] : 0.0, acc);
      }
      if (ok)
        for (int r = 0; r < 4; ++r) {
          const int i = 16 * mt + lk + 4 * r;
          if (i < ROWS) out[i] = acc[r];
        }
    }
  }
};

template <class S>
__global__ void __launch_bounds__(Team<S>::T) __attribute__((amdgpu_waves_per_eu(kTeamWaves)))
team_stage_kernel(StageArgs args) {
  using X = Team<S>;
  constexpr int DIM = S::DIM, NQ = S::NQ, NFQ = S::NFQ, NFN = S::NFN, NFLD = S::NFLD;
  constexpr int NFG = DIM + 1, PER = X::per_elem;
  extern __shared__ double smem[];
  const ConstArgs *A = (const ConstArgs *)&args;
  const double gamma = A->gamma, gm1 = A->gm1, lgm1 = A->lgm1;
  const int kfirst = blockIdx.x * X::E;
  const int nvalid = A->K - kfirst < X::E ? A->K - kfirst : X::E;
  const TeamLane<S> L(threadIdx.x, nvalid);
  team_volume<S>(L, kfirst, nvalid, A->rhsQ_in, A->Qf_in, A->vgeo, A->vfgeo, A->nrJ, A->nsJ, A->ntJ,
                 A->ws, gm1, A->inv2gm1, smem);

  // ---------------- surface flux + LF penalty at the lane's face point, in place
  if (L.valid) {
    const size_t k = kfirst + L.team;
    const int fn = L.wave * NFQ + L.l;
    const double *Qf = A->Qf_in;
    const size_t idM = k * NFN * NFLD + fn;
    const size_t idP = A->mapPq[k * NFN + fn];
    const double *g = A->fgeo + k * NFN * NFG;
    double UM[NFLD], UP[NFLD], nJ[DIM];
    for (int f = 0; f < NFLD; ++f) {
      UM[f] = Qf[idM + (size_t)f * NFN];
      UP[f] = Qf[idP + (size_t)f * NFN];
    }
    for (int d = 0; d < DIM; ++d) nJ[d] = g[fn + d * NFN];
    const double sJ = g[fn + DIM * NFN];
    const Node<DIM> na = make_node<DIM, false>(UM, gm1);
    const Node<DIM> nb = make_node<DIM, false>(UP, gm1);
    const double Lfc = A->ltau * fmax(node_speed<DIM>(na, gamma), node_speed<DIM>(nb, gamma)) * sJ;
    const PairFlux<DIM> P = pair_flux<DIM, true>(na, nb, A->inv2gm1);
    double Fn[NFLD];
    flux_dot<DIM>(P, nJ, Fn);
    double *s = smem + L.team * PER + X::AFOFF + fn;
    for (int f = 0; f < NFLD; ++f)
      s[f * NFN] = 0.5 * Fn[f] + s[f * NFN] - Lfc * (UP[f] - UM[f]);
  }
  // rows of the update, one per lane on the last waves (the first two hold more of
  // the products' tiles), and their inputs
  constexpr int RPAD = X::T - ((X::E * NQ + WAVE - 1) / WAVE) * WAVE;
  static_assert(RPAD >= 0, "one row per lane");
  const int row = L.tid - RPAD;
  const bool rv = row >= 0 && row < nvalid * NQ;
  const int re = rv ? row / NQ : 0, ri = rv ? row - re * NQ : 0;
  const size_t rbase = (size_t)(kfirst + re) * X::RQ + ri;
  double *el = smem + re * PER;
  double J = 1.0, Qin[NFLD], resin[NFLD];
  if (rv) {
    J = A->Jq[(size_t)(kfirst + re) * NQ + ri];
    for (int f = 0; f < NFLD; ++f) {
      Qin[f] = A->Q_in[rbase + f * NQ];
      resin[f] = A->resQ_in[rbase + f * NQ];
    }
  }
  // RHS rows = volume part + lift of the face terms
  double *a = el + X::AOFF + ri, *b = el + X::BOFF + ri;
  double rhs[NFLD];
  TeamTiles<S, NQ, NQ> aP;
  {
    TeamTiles<S, NQ, NFN> aL;
    aL.load(A->VqLq, L);
    __syncthreads();
    if (rv)
      for (int f = 0; f < NFLD; ++f) rhs[f] = team_row<S>(el, f, ri);
    __syncthreads();
    aL.product(X::AFOFF, X::BOFF, smem, L, nvalid);
  }
  aP.load(A->VqPq, L);
  __syncthreads();
  if (rv)
    for (int f = 0; f < NFLD; ++f) a[f * NQ] = rhs[f] + b[f * NQ];
  __syncthreads();
  const double invJ = rcp(J);
  auto product = [&](int in_off, int out_off) {
    aP.product(in_off, out_off, smem, L, nvalid);
    __syncthreads();
  };
  auto over_J = [&](double *x, double scale) {
    if (rv)
      for (int f = 0; f < NFLD; ++f) {
        const double r = scale * x[f * NQ];
        x[f * NQ] = (DIM == 3) ? r * invJ : quot(r, J, invJ);
      }
    __syncthreads();
  };
  product(X::AOFF, X::BOFF);
  over_J(b, -2.0);
  product(X::BOFF, X::AOFF);
  if (rv) {
    double U[NFLD], V[NFLD];
    for (int f = 0; f < NFLD; ++f) {
      const double rq = A->fa * resin[f] + A->fdt * a[f * NQ];
      A->resQ[rbase + f * NQ] = rq;
      U[f] = Qin[f] + A->fb * rq;
      A->Q[rbase + f * NQ] = U[f];
    }
    entropy_vars<DIM>(U, gamma, V);
    for (int f = 0; f < NFLD; ++f) a[f * NQ] = V[f] * J;
  }
  __syncthreads();
  product(X::AOFF, X::BOFF);
  over_J(b, 1.0);
  product(X::BOFF, X::AOFF);
  {
    TeamTiles<S, NFN, NQ> aF;
    aF.load(A->VfPq, L);
    aF.product(X::AOFF, X::TOFF, smem, L, nvalid);
  }
  __syncthreads();
  if (L.valid) {
    const int fn = L.wave * NFQ + L.l;
    const double *v = smem + L.team * PER + X::TOFF + fn;
    double V[NFLD], U[NFLD];
    for (int f = 0; f < NFLD; ++f) V[f] = v[f * NFN];
    conservative_vars<DIM>(V, gamma, lgm1, U);
    double *qf = A->Qf_out + (size_t)(kfirst + L.team) * NFN * NFLD + fn;
    for (int f = 0; f < NFLD; ++f) qf[f * NFN] = U[f];
  }
  if (rv) {
    double V[NFLD], U[NFLD];
    for (int f = 0; f < NFLD; ++f) V[f] = a[f * NQ];
    conservative_vars<DIM>(V, gamma, lgm1, U);
    for (int f = 0; f < NFLD; ++f) A->rhsQ[rbase + f * NQ] = U[f];
  }
}
