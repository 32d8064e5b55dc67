// wadges_wide.hpp -- the fused stage for launches too small to fill the chip:
// an element's pairs spread over all lanes of a workgroup.  Included by
// wadges.hip after the packed fused stage whose results it reproduces.
//
// stage_body packs several elements into a wave and gives each lane a row, which
// then walks its partners one after the other: few instructions per element,
// but a wave takes its whole walk (3D N = 4: 67 pair fluxes in a row) however few
// waves there are.  Here a workgroup of W waves holds E elements and every
// lane evaluates one pair at a time, so the walk is E * pairs / (64 W) long.  The
// contributions go to LDS and are then added, one lane per (row, field) and per
// (face point, field), in the order in which stage_body adds them: the results
// are the same bits, and an ensemble's packed stage and a problem's own wide one
// agree.

// E elements per workgroup of W waves; the contributions of CV steps of the
// volume-volume block, or of CF steps of the volume-face block, lie in LDS at a
// time.
template <class S_, int E_, int W_, int CV_, int CF_> struct Wide {
  using S = S_;
  static constexpr int E = E_, W = W_, CV = CV_, CF = CF_;
  static constexpr int T = WAVE * W;
  static_assert(S::R == 1, "one row per lane in the packed stage");
  using Vf = VfWalk<S>;
  static constexpr int CVP = CV * S::NQ, CFP = CF * Vf::P;
  // per-element LDS (doubles): volume records, normal parts of the rows on each
  // face, face records, contributions
  static constexpr int VOFF = 0;
  static constexpr int NOFF = VOFF + S::VREC * S::NQ;
  static constexpr int FOFF = NOFF + S::NFACES * S::DIM * S::NQ;
  static constexpr int COFF = FOFF + S::FREC * S::NFN;
  static constexpr int CSZ = Max<2 * S::NFLD * CVP, (S::NFLD + 2) * CFP>::value;
  // after the pairs, from the front: face terms, two row buffers, traces
  static constexpr int SOFF = 0;
  static constexpr int AOFF = SOFF + S::NFLD * S::NFN;
  static constexpr int BOFF = AOFF + S::NFLD * S::NQ;
  static constexpr int TOFF = BOFF + S::NFLD * S::NQ;
  static constexpr int END = TOFF + S::NFLD * S::NFN;
  static constexpr int per_elem = Max<COFF + CSZ, END>::value;
  static constexpr int bytes = 8 * E * per_elem;
};

// Shapes of the wide launch.  Small: up to two elements per CU; Large: as long as all
// its workgroups are resident at once.  Beyond that the packed stage is faster: its
// waves take as long whatever their number (until they fill the chip) and issue a
// half to a third of the instructions.  One stage, packed / wide, microseconds
// (chosen from sweeps of E, W and the chunks at K = 128 .. 16,000):
//   2D N = 1   K = 1,058  16.9 / 8.9    8,192  17.6 / 13.5   16,200  18.8 / 25.0
//   2D N = 2   K = 128    18.5 / 8.3    4,050  18.8 / 13.3    8,192  20.7 / 23.5
//   2D N = 3   K = 128    15.6 / 9.4    2,048  16.1 / 13.2    3,200  16.7 / 24.0
//   2D N = 4   K = 128    18.2 / 11.6   2,048  18.6 / 16.1    3,200  19.7 / 28.8
//   2D N = 5   K = 512    26.5 / 16.9   1,058  27.1 / 30.3
//   3D N = 1   K = 384    21.5 / 9.8    6,000  24.6 / 16.8   10,368  26.8 / 26.4
//   3D N = 2   K = 162    25.0 / 10.5     750  25.5 / 12.7    1,296  26.2 / 24.0
//   3D N = 4   K = 384    47.3 / 36.0     750  49.1 / 45.1    1,296  67.8 / 83.9
template <class S> struct WideChoice;
template <> struct WideChoice<Shape<2, 3, 2>> {
  using Small = Wide<Shape<2, 3, 2>, 4, 2, 2, 6>;
  using Large = Small;
};
template <> struct WideChoice<Shape<2, 6, 3>> {
  using Small = Wide<Shape<2, 6, 3>, 1, 1, 4, 9>;
  using Large = Wide<Shape<2, 6, 3>, 2, 1, 4, 9>;
};
template <> struct WideChoice<Shape<2, 12, 4>> {
  using Small = Wide<Shape<2, 12, 4>, 1, 2, 7, 12>;
  using Large = Wide<Shape<2, 12, 4>, 2, 2, 7, 12>;
};
template <> struct WideChoice<Shape<2, 16, 5>> {
  using Small = Wide<Shape<2, 16, 5>, 1, 2, 9, 16>;
  using Large = Wide<Shape<2, 16, 5>, 2, 2, 9, 16>;
};
template <> struct WideChoice<Shape<2, 25, 6>> {
  using Small = Wide<Shape<2, 25, 6>, 1, 4, 13, 25>;
  using Large = Wide<Shape<2, 25, 6>, 1, 2, 13, 25>;
};
template <> struct WideChoice<Shape<3, 4, 3>> {
  using Small = Wide<Shape<3, 4, 3>, 3, 1, 3, 12>;
  using Large = Small;
};
template <> struct WideChoice<Shape<3, 11, 6>> {
  using Small = Wide<Shape<3, 11, 6>, 1, 2, 6, 24>;
  using Large = Small;
};
template <> struct WideChoice<Shape<3, 44, 16>> {
  using Small = Wide<Shape<3, 44, 16>, 1, 4, 6, 4>;
  using Large = Small;
};

// The A operand (16-row tiles mt = wave + W x of M, ROWS x KD, column major) of
// wide_product, loaded ahead of it.
template <int W, int ROWS, int KD> struct TileA {
  static constexpr int MT = (ROWS + 15) / 16, KS = (KD + 3) / 4, TX = (MT + W - 1) / W;
  double a[TX][KS];
  __device__ __forceinline__ void load(const double *M, int lane, int wave) {
    const int lr = lane & 15, lk = lane >> 4;
    for (int x = 0; x < TX; ++x) {
      const int row = 16 * (wave + W * x) + lr;
      for (int ks = 0; ks < KS; ++ks) {
        const int j = 4 * ks + lk;
        a[x][ks] = (j < KD && row < ROWS) ? ld_off(M, (unsigned)(row + j * ROWS)) : 0.0;
      }
    }
  }
};

// OUT[c][i] = sum_j M[i][j] IN[c][j] for the E NFLD columns of the workgroup, the
// row tiles spread over its waves; sums in ascending j, one fused multiply-add
// per term, as wave_product_mfma.
template <int E, int W, int NFLD, int PER, int ROWS, int KD>
__device__ __forceinline__ void wide_product(const TileA<W, ROWS, KD> &A, int in_off, int out_off,
                                             double *smem, int lane, int wave, int nvalid) {
  using TA = TileA<W, ROWS, KD>;
  constexpr int NCOL = E * NFLD, NT = (NCOL + 15) / 16;
  const int lr = lane & 15, lk = lane >> 4;
  for (int nt = 0; nt < NT; ++nt) {
    const int c = 16 * nt + lr;
    const int e = c / NFLD;
    const int f = c - e * NFLD;
    const bool ok = c < NCOL && e < nvalid;
    const double *in = smem + (ok ? e * PER + in_off + f * KD : 0);
    double *out = smem + (ok ? e * PER + out_off + f * ROWS : 0);
    double b[TA::KS];
    for (int ks = 0; ks < TA::KS; ++ks) {
      const int j = 4 * ks + lk;
      b[ks] = (ok && j < KD) ? in[j] : 0.0;
    }
    for (int x = 0; x < TA::TX; ++x) {
      const int mt = wave + W * x;
      if (TA::MT % W != 0 && mt >= TA::MT) continue;   // uniform over the wave
      dbl4 acc = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int ks = 0; ks < TA::KS; ++ks) acc = mfma_f64_16x16x4(A.a[x][ks], b[ks], acc);
      if (ok)
        for (int r = 0; r < 4; ++r) {
          const int i = 16 * mt + lk + 4 * r;
          if (i < ROWS) out[i] = acc[r];
        }
    }
  }
}

// Two waves per SIMD declared: 128 or 168 registers spill in several shapes (the batched
// LDS reads of the sums), and a launch that fills more goes to the packed stage.
template <class X>
__global__ void __launch_bounds__(X::T) __attribute__((amdgpu_waves_per_eu(2)))
stage_wide(StageArgs args) {
  using S = typename X::S;
  constexpr int E = X::E, W = X::W, CV = X::CV, CF = X::CF;
  using Vf = typename X::Vf;
  constexpr int DIM = S::DIM, NQ = S::NQ, NFQ = S::NFQ, NFN = S::NFN, NFLD = S::NFLD, NG = S::NG;
  constexpr int NFACES = S::NFACES, NFG = DIM + 1, VS = S::VS, TVT = S::TVT;
  constexpr int T = X::T, PER = X::per_elem, CVP = X::CVP, CFP = X::CFP;
  extern __shared__ double smem[];
  __shared__ double s_nref[NFACES][DIM];
  const ConstArgs *A = (const ConstArgs *)&args;
  const double gamma = A->gamma, gm1 = A->gm1, inv2gm1 = A->inv2gm1, ltau = A->ltau, lgm1 = A->lgm1;
  const double fa = A->fa, fb = A->fb, fdt = A->fdt;
  const int tid = threadIdx.x;
  const int wave = W > 1 ? __builtin_amdgcn_readfirstlane(tid / WAVE) : 0;
  const int lane = tid - wave * WAVE;
  const int kfirst = blockIdx.x * E;
  const int nvalid = A->K - kfirst < E ? A->K - kfirst : E;   // elements of this workgroup, >= 1

  // ---------------- records of all nodes; the other inputs are loaded on the way
  load_nref<S>(tid, A->nrJ, A->nsJ, A->ntJ, s_nref);
  constexpr int NN = NQ + NFN;
  for (int q = tid; q < nvalid * NN; q += T) {
    const int e = q / NN;
    const int c = q - e * NN;
    const bool vol = c < NQ;
    const int i = vol ? c : c - NQ;
    const int n = vol ? NQ : NFN;
    const size_t k = kfirst + e;
    const double *src = vol ? A->rhsQ_in + k * NQ * NFLD : A->Qf_in + k * NFN * NFLD;
    const double *geo = vol ? A->vgeo + k * NQ * NG : A->vfgeo + k * NFN * NG;
    double U[NFLD], g[NG];
    for (int f = 0; f < NFLD; ++f) U[f] = src[i + f * n];
    for (int x = 0; x < NG; ++x) g[x] = geo[i + x * n];
    double *rec = smem + e * PER + (vol ? X::VOFF : X::FOFF);
    store_node<DIM>(rec, n, i, make_node<DIM>(U, gm1));
    if (vol) {
      for (int x = 0; x < NG; ++x) rec[(VS + x) * NQ + i] = 0.5 * g[x];
    } else {
      const int p = (i / NFQ) * NFQ;
      double nr[DIM];
      nr[0] = A->nrJ[p];
      nr[1] = A->nsJ[p];
      if constexpr (DIM == 3) nr[2] = A->ntJ[p];
      for (int d = 0; d < DIM; ++d) {
        double b = 0.0;
        for (int r = 0; r < DIM; ++r) b = b + 0.5 * g[r * DIM + d] * nr[r];
        rec[(VS + d) * NFN + i] = b;
      }
    }
  }
  // Rows of the update, on the last lanes of the workgroup (the face points are
  // on the first ones), and their inputs
  constexpr int RN = E * NQ, RX = (RN + T - 1) / T;
  constexpr int RPAD = RX > 1 ? 0 : T - ((RN + WAVE - 1) / WAVE) * WAVE;
  double Qin[RX][NFLD], resin[RX][NFLD], J[RX];
  int re[RX], ri[RX];
  bool rv[RX];
  for (int x = 0; x < RX; ++x) {
    const int r = tid - RPAD + x * T;
    rv[x] = r >= 0 && r < nvalid * NQ;
    re[x] = rv[x] ? r / NQ : 0;
    ri[x] = rv[x] ? r - re[x] * NQ : 0;
    J[x] = 1.0;
    if (rv[x]) {
      const size_t k = kfirst + re[x];
      J[x] = A->Jq[k * NQ + ri[x]];
      for (int f = 0; f < NFLD; ++f) {
        const size_t id = k * NQ * NFLD + ri[x] + f * NQ;
        Qin[x][f] = A->Q_in[id];
        resin[x][f] = A->resQ_in[id];
      }
    }
  }
  // Face points and their matching points
  constexpr int FN = E * NFN, FX = (FN + T - 1) / T;
  size_t idP[FX];
  for (int x = 0; x < FX; ++x) {
    const int p = tid + x * T;
    idP[x] = p < nvalid * NFN ? A->mapPq[(size_t)kfirst * NFN + p] : 0;
  }
  __syncthreads();
  // own-side part of the averaged normals: sum_q (G_qd / 2) nref_q of each row and face
  for (int q = tid; q < nvalid * NFACES * NQ; q += T) {
    const int e = q / (NFACES * NQ);
    const int c = q - e * NFACES * NQ;
    const int face = c / NQ;
    const int i = c - face * NQ;
    const double *rec = smem + e * PER + X::VOFF;
    for (int d = 0; d < DIM; ++d) {
      double v = 0.0;
      for (int r = 0; r < DIM; ++r) v = v + rec[(VS + r * DIM + d) * NQ + i] * s_nref[face][r];
      smem[e * PER + X::NOFF + (face * DIM + d) * NQ + i] = v;
    }
  }

  // ---------------- volume-volume pairs.  Row sums: one lane per (row, field);
  // acc holds the row's own part, accv what its partners add.
  constexpr int RS = E * NFLD * NQ, SX = (RS + T - 1) / T;
  double acc[SX], accv[SX];
  int se[SX], sf[SX], si[SX];
  bool sv[SX];
  for (int x = 0; x < SX; ++x) {
    const int r = tid + x * T;
    const bool v = r < nvalid * NFLD * NQ;
    sv[x] = v;
    se[x] = v ? r / (NFLD * NQ) : 0;
    const int c = v ? r - se[x] * NFLD * NQ : 0;
    sf[x] = c / NQ;
    si[x] = c - sf[x] * NQ;
    acc[x] = accv[x] = 0.0;
  }
  for (int t0 = 0; t0 < TVT; t0 += CV) {
    const int nst = TVT - t0 < CV ? TVT - t0 : CV;
    const int np = E == 1 ? nst * NQ : nvalid * CVP;
    // the operator entries of a lane's next pair are loaded during the one before
    double Df_n[DIM], Db_n[DIM];
    auto fetch = [&](int p) {
      const int c = E == 1 ? p : p % CVP;
      const int t = t0 + c / NQ;
      if (p >= np || t >= TVT) return;
      const int i = c - (c / NQ) * NQ;
      for (int q = 0; q < DIM; ++q) {
        Df_n[q] = ld_off(A->ws, (unsigned)((q * TVT + t) * NQ + i));
        Db_n[q] = ld_off(A->ws, (unsigned)(((DIM + q) * TVT + t) * NQ + i));
      }
    };
    fetch(tid);
    for (int p = tid; p < np; p += T) {
      const int e = E == 1 ? 0 : p / CVP;
      const int c = p - e * CVP;
      const int tl = c / NQ;
      const int i = c - tl * NQ;
      const int t = t0 + tl;
      double Df[DIM], Db[DIM];
      for (int q = 0; q < DIM; ++q) {
        Df[q] = Df_n[q];
        Db[q] = Db_n[q];
      }
      fetch(p + T);
      if (t >= TVT || (2 * t == NQ && i >= NQ / 2)) continue;
      int j = i + t;
      if (j >= NQ) j -= NQ;
      const double *vrec = smem + e * PER + X::VOFF;
      double *out = smem + e * PER + X::COFF + c;
      const Node<DIM> pi = load_node<DIM>(vrec, NQ, i);
      const Node<DIM> pj = load_node<DIM>(vrec, NQ, j);
      double Ga[NG];
      for (int x = 0; x < NG; ++x) Ga[x] = vrec[(VS + x) * NQ + i] + vrec[(VS + x) * NQ + j];
      const PairFlux<DIM> F = pair_flux<DIM>(pi, pj, inv2gm1);
      double Dx[DIM], c1[NFLD];
      for (int d = 0; d < DIM; ++d) Dx[d] = 0.0;
      for (int q = 0; q < DIM; ++q)
        for (int d = 0; d < DIM; ++d) Dx[d] = Dx[d] + Df[q] * Ga[q * DIM + d];
      flux_dot<DIM>(F, Dx, c1);
      for (int f = 0; f < NFLD; ++f) out[f * CVP] = c1[f];
      if (t > 0) {
        for (int d = 0; d < DIM; ++d) Dx[d] = 0.0;
        for (int q = 0; q < DIM; ++q)
          for (int d = 0; d < DIM; ++d) Dx[d] = Dx[d] + Db[q] * Ga[q * DIM + d];
        flux_dot<DIM>(F, Dx, c1);
        for (int f = 0; f < NFLD; ++f) out[(NFLD + f) * CVP] = c1[f];
      }
    }
    __syncthreads();
    for (int x = 0; x < SX; ++x) {
      const int i = si[x];
      const double *own = smem + se[x] * PER + X::COFF + sf[x] * CVP;
      const double *part = own + NFLD * CVP;
#pragma unroll
      for (int tl = 0; tl < CV; ++tl) {
        const int t = t0 + tl;
        if (TVT % CV != 0 && t >= TVT) break;
        int ip = i - t;                       // the row whose partner is i
        if (ip < 0) ip += NQ;
        const double o = own[tl * NQ + i], q = part[tl * NQ + ip];
        acc[x] += 2 * t != NQ || i < NQ / 2 ? o : 0.0;
        accv[x] += t > 0 && (2 * t != NQ || ip < NQ / 2) ? q : 0.0;
      }
    }
    __syncthreads();
  }
  if constexpr (Vf::COL)
    for (int x = 0; x < SX; ++x) {
      accv[x] = acc[x] + accv[x];
      acc[x] = 0.0;
    }

  // ---------------- volume-face pairs.  Face sums: one lane per (face point,
  // field), the points of a face and their fields next to each other.
  constexpr int GS = E * NFN * NFLD, GX = (GS + T - 1) / T;
  double accf[GX];
  int ge[GX], gf[GX], gn[GX];
  bool gv[GX];
  for (int x = 0; x < GX; ++x) {
    const int r = tid + x * T;
    const bool v = r < nvalid * NFN * NFLD;
    gv[x] = v;
    ge[x] = v ? r / (NFN * NFLD) : 0;
    const int c = v ? r - ge[x] * NFN * NFLD : 0;
    const int face = c / (NFQ * NFLD);
    const int d = c - face * NFQ * NFLD;
    gf[x] = d / NFQ;
    gn[x] = face * NFQ + (d - gf[x] * NFQ);
    accf[x] = 0.0;
  }
  const uint32_t *codes = (const uint32_t *)(A->ws + Vf::CODES);
  static_assert(Vf::STEPS % CF == 0, "equal chunks of the walk");
  for (int s0 = 0; s0 < Vf::STEPS; s0 += CF) {
    const int np = nvalid * CFP;
    // the code and weights of a lane's next pair are loaded during the one before
    uint32_t code_n = Vf::NONE;
    double w1_n = 0.0, w2_n = 0.0;
    auto fetch = [&](int p) {
      const unsigned at = s0 * Vf::P + (E == 1 ? p : p % CFP);
      if (p < np) {
        code_n = codes[at];
        w1_n = ld_off(A->ws, Vf::W1 + at);
        w2_n = ld_off(A->ws, Vf::W2 + at);
      }
    };
    fetch(tid);
    for (int p = tid; p < np; p += T) {
      const int e = E == 1 ? 0 : p / CFP;
      const int c = p - e * CFP;
      const uint32_t code = code_n;
      const double w1 = w1_n, w2 = w2_n;
      fetch(p + T);
      if (code == Vf::NONE) continue;
      const int i = code & 255, fn = (code >> 8) & 255, face = code >> 16;
      const double *base = smem + e * PER;
      const double *frec = base + X::FOFF;
      const Node<DIM> pv = load_node<DIM>(base + X::VOFF, NQ, i);
      const Node<DIM> pf = load_node<DIM>(frec, NFN, fn);
      double n[DIM];
      for (int d = 0; d < DIM; ++d)
        n[d] = base[X::NOFF + (face * DIM + d) * NQ + i] + frec[(VS + d) * NFN + fn];
      const PairFlux<DIM> F = pair_flux<DIM>(pv, pf, inv2gm1);
      double Fn[NFLD];
      flux_dot<DIM>(F, n, Fn);
      double *out = smem + e * PER + X::COFF + c;
      for (int f = 0; f < NFLD; ++f) out[f * CFP] = Fn[f];
      out[NFLD * CFP] = w1;
      out[(NFLD + 1) * CFP] = w2;
    }
    __syncthreads();
    for (int x = 0; x < SX; ++x) {
      const double *F = smem + se[x] * PER + X::COFF + sf[x] * CFP;
      const double *w1 = smem + se[x] * PER + X::COFF + NFLD * CFP;
      if constexpr (Vf::COL) {
        int l = si[x] - s0;                   // face points l and l + NQ visit this row
        if (l < 0) l += NQ;
#pragma unroll
        for (int sl = 0; sl < CF; ++sl) {
          const int at = sl * Vf::P + l;
          const double c = w1[at] * F[at];
          accv[x] += c;
          const bool second = l + NQ < NFN;
          const int at2 = second ? at + NQ : at;
          const double c2 = w1[at2] * F[at2];
          accv[x] += second ? c2 : 0.0;
          l = l == 0 ? NQ - 1 : l - 1;
        }
      } else {
#pragma unroll
        for (int sl = 0; sl < CF; ++sl) {
          const int at = sl * Vf::P + si[x];
          if constexpr (Vf::CHUNKED) {
            acc[x] += w1[at] * F[at];
          } else {
            int fn = si[x] + s0 + sl;         // no pair beyond the face points
            if (fn >= S::L) fn -= S::L;
            const double v = acc[x] + w1[at] * F[at];
            acc[x] = fn < NFN ? v : acc[x];
          }
        }
      }
    }
    for (int x = 0; x < GX; ++x) {
      const double *F = smem + ge[x] * PER + X::COFF + gf[x] * CFP;
      const double *w2 = smem + ge[x] * PER + X::COFF + (NFLD + 1) * CFP;
      const int face = gn[x] / NFQ;
      const int q = gn[x] - face * NFQ;
      if constexpr (Vf::COL) {
#pragma unroll
        for (int sl = 0; sl < CF; ++sl) {
          const int at = sl * Vf::P + gn[x];
          accf[x] += w2[at] * F[at];
        }
      } else if constexpr (Vf::CHUNKED) {
        constexpr int GR = face_groups<S>(), FH = Vf::FH;
        static_assert(CF == Vf::STEPS, "whole walk at a time");
        const int h = face / FH, fh = face - h * FH;
        // 3D N = 2: with the sums of both faces of a part in flight the kernel spilled
        // (28 bytes a lane; a stage at K = 162, 750 and 1,000 13.7, 16.0 and 17.1 us,
        // one face at a time 13.2, 15.3 and 16.5)
#pragma unroll (DIM == 3 && NQ == 11 ? 1 : FH)
        for (int u = 0; u < FH; ++u) {
          int g0 = fh - u;
          if (g0 < 0) g0 += FH;
#pragma unroll
          for (int m = 0; m < NFQ; ++m) {
            int o = q - m;
            if (o < 0) o += NFQ;
#pragma unroll
            for (int gg = 0; gg < GR; gg += FH) {
              const int i = (g0 + gg) * NFQ + o;
              const bool ok = i < NQ && g0 + gg < GR;
              const int at = ((h * FH + u) * NFQ + m) * Vf::P + (ok ? i : 0);
              const double c = w2[at] * F[at];
              accf[x] += ok ? c : 0.0;
            }
          }
        }
      } else {
        int i = gn[x] - s0;
        if (i < 0) i += S::L;
#pragma unroll
        for (int sl = 0; sl < CF; ++sl) {
          const int at = sl * Vf::P + i;
          const double c = w2[at] * F[at];
          accf[x] += c;
          i = i == 0 ? S::L - 1 : i - 1;
        }
      }
    }
    __syncthreads();
  }

  // ---------------- surface flux + LF penalty at the face points
  TileA<W, NQ, NFN> aL;
  aL.load(A->VqLq, lane, wave);
  // states and normals of the surface flux
  double UM[FX][NFLD], UP[FX][NFLD], nJ[FX][DIM], sJ[FX];
  for (int x = 0; x < FX; ++x) {
    const int p = tid + x * T;
    if (p >= nvalid * NFN) continue;
    const int e = p / NFN;
    const int fn = p - e * NFN;
    const size_t k = kfirst + e;
    const size_t idM = (size_t)fn + k * NFN * NFLD;
    const double *g = A->fgeo + k * NFN * NFG;
    for (int f = 0; f < NFLD; ++f) {
      UM[x][f] = A->Qf_in[idM + (size_t)f * NFN];
      UP[x][f] = A->Qf_in[idP[x] + (size_t)f * NFN];
    }
    for (int d = 0; d < DIM; ++d) nJ[x][d] = g[fn + d * NFN];
    sJ[x] = g[fn + DIM * NFN];
  }

  Node<DIM> own[FX];
  for (int x = 0; x < FX; ++x) {
    const int p = tid + x * T;
    const int e = p < nvalid * NFN ? p / NFN : 0;
    own[x] = load_node<DIM>(smem + e * PER + X::FOFF, NFN, p < nvalid * NFN ? p - e * NFN : 0);
  }
  if constexpr (X::END > X::FOFF) __syncthreads();   // the face terms may overlap the records
  for (int x = 0; x < SX; ++x)
    if (sv[x]) smem[se[x] * PER + X::AOFF + sf[x] * NQ + si[x]] = acc[x] + accv[x];
  for (int x = 0; x < GX; ++x)
    if (gv[x]) smem[ge[x] * PER + X::SOFF + gf[x] * NFN + gn[x]] = accf[x];
  __syncthreads();
  for (int x = 0; x < FX; ++x) {
    const int p = tid + x * T;
    if (p >= nvalid * NFN) continue;
    const int e = p / NFN;
    const int fn = p - e * NFN;
    double *s = smem + e * PER + X::SOFF;
    const Node<DIM> &a = own[x];
    const Node<DIM> b = make_node<DIM, false>(UP[x], gm1);
    const double Lfc = ltau * fmax(node_speed<DIM>(a, gamma), node_speed<DIM>(b, gamma)) * sJ[x];
    const PairFlux<DIM> P = pair_flux<DIM, true>(a, b, inv2gm1);
    double Fn[NFLD];
    flux_dot<DIM>(P, nJ[x], Fn);
    for (int f = 0; f < NFLD; ++f)
      s[f * NFN + fn] = 0.5 * Fn[f] + s[f * NFN + fn] - Lfc * (UP[x][f] - UM[x][f]);
  }
  __syncthreads();

  // ---------------- lift, weight-adjusted inverse mass, RK update, projection
  TileA<W, NQ, NQ> aP;
  aP.load(A->VqPq, lane, wave);
  wide_product<E, W, NFLD, PER, NQ, NFN>(aL, X::SOFF, X::BOFF, smem, lane, wave, nvalid);
  __syncthreads();
  double invJ[RX];
  for (int x = 0; x < RX; ++x) {
    invJ[x] = rcp(J[x]);
    if (!rv[x]) continue;
    double *a = smem + re[x] * PER + X::AOFF + ri[x];
    const double *b = smem + re[x] * PER + X::BOFF + ri[x];
    for (int f = 0; f < NFLD; ++f) a[f * NQ] = a[f * NQ] + b[f * NQ];
  }
  __syncthreads();
  auto product = [&](int in_off, int out_off) {
    wide_product<E, W, NFLD, PER, NQ, NQ>(aP, in_off, out_off, smem, lane, wave, nvalid);
    __syncthreads();
  };
  // the row's values at off, scaled, over J
  auto over_J = [&](int off, double scale) {
    for (int x = 0; x < RX; ++x) {
      if (!rv[x]) continue;
      double *b = smem + re[x] * PER + off + ri[x];
      for (int f = 0; f < NFLD; ++f) {
        const double r = scale * b[f * NQ];
        b[f * NQ] = (DIM == 3) ? r * invJ[x] : quot(r, J[x], invJ[x]);
      }
    }
    __syncthreads();
  };
  product(X::AOFF, X::BOFF);
  over_J(X::BOFF, -2.0);
  product(X::BOFF, X::AOFF);
  for (int x = 0; x < RX; ++x) {
    if (!rv[x]) continue;
    double *a = smem + re[x] * PER + X::AOFF + ri[x];
    double U[NFLD], V[NFLD];
    for (int f = 0; f < NFLD; ++f) {
      const size_t id = (size_t)(kfirst + re[x]) * NQ * NFLD + ri[x] + f * NQ;
      const double rq = fa * resin[x][f] + fdt * a[f * NQ];
      A->resQ[id] = rq;
      U[f] = Qin[x][f] + fb * rq;
      A->Q[id] = U[f];
    }
    entropy_vars<DIM>(U, gamma, V);
    for (int f = 0; f < NFLD; ++f) a[f * NQ] = V[f] * J[x];
  }
  __syncthreads();
  TileA<W, NFN, NQ> aF;
  aF.load(A->VfPq, lane, wave);
  product(X::AOFF, X::BOFF);
  over_J(X::BOFF, 1.0);
  product(X::BOFF, X::AOFF);
  wide_product<E, W, NFLD, PER, NFN, NQ>(aF, X::AOFF, X::TOFF, smem, lane, wave, nvalid);
  __syncthreads();
  for (int x = 0; x < FX; ++x) {
    const int p = tid + x * T;
    if (p >= nvalid * NFN) continue;
    const int e = p / NFN;
    const int fn = p - e * NFN;
    const double *v = smem + e * PER + X::TOFF + fn;
    double V[NFLD], U[NFLD];
    for (int f = 0; f < NFLD; ++f) V[f] = v[f * NFN];
    conservative_vars<DIM>(V, gamma, lgm1, U);
    double *qf = A->Qf_out + (size_t)(kfirst + e) * NFN * NFLD;
    for (int f = 0; f < NFLD; ++f) qf[fn + f * NFN] = U[f];
  }
  for (int x = 0; x < RX; ++x) {
    if (!rv[x]) continue;
    const double *a = smem + re[x] * PER + X::AOFF + ri[x];
    double V[NFLD], U[NFLD];
    for (int f = 0; f < NFLD; ++f) V[f] = a[f * NQ];
    conservative_vars<DIM>(V, gamma, lgm1, U);
    const size_t base = (size_t)(kfirst + re[x]) * NQ * NFLD;
    for (int f = 0; f < NFLD; ++f) A->rhsQ[base + ri[x] + f * NQ] = U[f];
  }
}
