// What a workgroup of the segment kernels does with the chunks c0 .. c0 + nc - 1 of segment `seg` (see gdr_chunk_kernels.h): the
// body of gdr_segment_kernel, with its template and function parameters and hv, flags and map (where the composite goes) in
// scope. A text of its own and not a function: as one that is inlined, the compiler schedules the output pass worse (64 x 128
// value columns: 39.2 -> 41.5 us of a call on 25 080 tokens x 5 heads).
  // OT: the 16-bit type of every MFMA operand (tiles in LDS, T, R, v_new, P, the state as operand, M' of the
  // composites): the input type, so that fp16 inputs run on the fp16 MFMA without losing mantissa bits
  using X8 = typename OpVec<OT>::x8;
  using X4 = typename OpVec<OT>::x4;
  constexpr bool SCALED = !PASS_B && SCALED_K;
  constexpr bool SWZ = GdrSegShape<KT, VT, PASS_B, CW>::SWIZZLED;
  // narrow chain waves: the k, q and T tiles keep every 32 columns in the order of op_perm32 (gdr_ops.h)
  constexpr bool P16 = CW == 16;
  // The narrow form keeps the k, q and T tiles in op_perm32 order (one 16-byte read per operand fragment). With the
  // tiles in plain order and two 8-byte reads per fragment the output pass is slower: 71.0 against 68.2 us at
  // K = V = 64, 1 463 against 1 290 us at K = V = 128 (config 4).
  constexpr bool PERM = P16;
  // 32-column output pass: the o tile of a chunk is written to HBM by the STAGER waves (after the next chunk's barrier
  // B, whole rows), so the read-back and the stores are off the recurrence waves' chain.
  constexpr bool STAGER_FLUSH = PASS_B && CW == 32 && KT + VT <= 128;  // (the wider heads have no registers for it)
  static_assert(STAGER_FLUSH || !PASS_B || !KEEP, "o_width is applied where the stagers write o");
  // Output pass at K <= 64: a stager builds the P tiles of the q rows it staged itself (stager 0 the tile (0,0),
  // stager 1 the tiles (1,0) and (1,1)), so no barrier separates staging q from building P. At K = 128 a P tile is
  // twice the work, the two stagers share the middle tile, and the barrier Qb(c) (q(c) is staged) comes back.
  constexpr bool OWN_Q = KT <= 64 || CW == 16;  // (the narrow form's q / P stagers have registers of their own to spare)
  // Narrow form of the heads wider than 64 x 64 (one workgroup per CU, LDS to spare): q, P and the q factor rows exist
  // twice, so the q / P stagers stage q(c + 1) while the chain waves still read q(c) and P(c).
  constexpr bool DBQ = GdrSegShape<KT, VT, PASS_B, CW>::DOUBLE_Q;
  using SM = GdrSegSmem<KT, VT, PASS_B, SCALED, DBQ ? 2 : 1>;
  constexpr int NSLAB = GdrSegShape<KT, VT, PASS_B, CW>::SLABS;
  constexpr int SK = SM::SK, SV = SM::SV, ST = SM::ST;
  extern __shared__ __align__(16) unsigned char smem[];
  auto tiles = [&](int par) {
    unsigned char* base = smem + par * SM::TILE_BYTES;
    GdrTilesT<OT> t;
    t.k = reinterpret_cast<OT*>(base + SM::T_OFF_K);
    t.kd = reinterpret_cast<OT*>(base + (SCALED ? SM::T_OFF_KD : SM::T_OFF_K));
    t.v = reinterpret_cast<OT*>(base + SM::T_OFF_V);
    t.t = reinterpret_cast<OT*>(base + SM::T_OFF_T);
    t.beta = reinterpret_cast<float*>(base + SM::T_OFF_F);
    t.ek = t.beta + 64;
    t.dk = t.beta + 128;
    t.gamma = t.beta + 192;
    t.rk = t.beta + 256;
    t.misc = t.beta + 320;
    return t;
  };
  OT* const s_q0 = reinterpret_cast<OT*>(smem + SM::OFF_Q);
  unsigned char* const s_P0 = smem + SM::OFF_P;
  T* s_o = reinterpret_cast<T*>(smem + SM::OFF_O);
  float* const s_qs0 = reinterpret_cast<float*>(smem + SM::OFF_QF);  // scale e^{gamma_i} rq_i, then rq_i
  // the copy of the q tile / the P fragments / the factor rows that belongs to a chunk of parity par
#define GDR_Q_BUFFERS(par)                                                          \
  OT* const s_q = s_q0 + (DBQ ? (par) : 0) * (SM::Q_BYTES / 2);                     \
  unsigned char* const s_P = s_P0 + (DBQ ? (par) : 0) * SM::P_BYTES;                \
  float* const s_qs = s_qs0 + (DBQ ? (par) : 0) * (SM::QF_BYTES / 4);               \
  float* const s_rq = s_qs + 64;                                                    \
  (void)s_q; (void)s_P; (void)s_qs; (void)s_rq

  const int h = hv / (HV / H);
  const int c1 = c0 + nc;
  // (the per-chunk tables are separate restrict parameters: read through the view they could alias the kernel's
  // stores, would be fetched with vector loads and would sit in the same queue as the stagers' prefetches)
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, hh = lane >> 5, ln = lane & 31;
  // Segments that cut off what lies before them are found (see the end of the kernel), in the composite pass of the plain rule.
  constexpr bool CUTS = !PASS_B && SCALED_K;
  constexpr bool SKIP_M = CUTS && KT + VT > 128;

  if (wave >= NSLAB) {
    // ================================================ stager ================================================
    // Narrow output pass: with eight or more chain waves beside them the four stagers are the longer pole, so they get
    // the SIMDs' issue slots first (config 4: output pass 1 168 -> 993 - 1 012 us). In the other forms the chain is
    // the longer pole and a raised priority on either side changes nothing or costs a little.
    if constexpr (PASS_B && CW == 16) __builtin_amdgcn_s_setprio(3);
    constexpr int KU = KT / 16, VU = VT / 16;  // 16-byte pieces per thread: half a row of k / q, of v
    // (narrow form: pair 0 = waves NSLAB, NSLAB + 1 stages k, v, T and the factors, pair 1 = the next two q and P; a
    // pair is the 128 threads the staging code is written for)
    const int spair = P16 ? (wave - NSLAB) >> 1 : 0;
    const int stid = tid - 64 * (NSLAB + 2 * spair), sw = (wave - NSLAB) & 1;
    const int srow = stid >> 1, spart = stid & 1;
    // PASS_A keeps the raw k rows of two chunks (sets by chunk parity): the scaled tiles are written from the
    // registers after the row norms are known, and the next k loads must already be on their way by then
    typename Raw8<T>::type rk0_[KU], rk1_[SCALED ? KU : 1], rv_[VU];
    typename Raw8<T>::type rq0_[PASS_B ? KU : 1], rq1_[PASS_B ? KU : 1];  // q of even / odd chunks of the segment
    X8 rt_[3];
    float rg = 0.0f, rb = 0.0f;
    float grow = 0.0f;  // gamma of row srow of the chunk whose tiles were staged last
    float ghalf = 0.0f;  // half the total log-decay of that chunk
    bool pfast = false;  // that chunk's P takes the factored gating (stage_factors)
    // where this thread's pieces of the packed diagonal blocks of T go in the LDS tile; the pieces above the diagonal
    // are never staged and are zeroed once, in both tile sets
    int ta_off, tb_off;  // element offsets into the T area of a tile set of this thread's two packed pieces
    {
      int row, part;
      const int da = stid, db = 128 + (stid & 31);  // indices among the 160 packed pieces (T11: 0 .. 79, T22: 80 .. 159)
      tri_piece(da < T_DIAG_PIECES ? da : da - T_DIAG_PIECES, row, part);
      ta_off = ((da < T_DIAG_PIECES ? 0 : 2) * 32 + row) * ST + (PERM ? op_perm32_piece(part) : 8 * part);
      tri_piece(db - T_DIAG_PIECES, row, part);
      tb_off = (2 * 32 + row) * ST + (PERM ? op_perm32_piece(part) : 8 * part);
    }
    const int t21_off = (1 * 32 + (stid >> 2)) * ST + (PERM ? op_perm32_piece(stid & 3) : 8 * (stid & 3));
    // a 16-byte piece of T into a tile: as it is, or (P16) its two halves 8 elements apart
    auto put_t = [&](OT* at, X8 v) __attribute__((always_inline)) {
      if constexpr (PERM) {
        X4 lo, hi;
#pragma unroll
        for (int e = 0; e < 4; ++e) { lo[e] = v[e]; hi[e] = v[4 + e]; }
        *reinterpret_cast<X4*>(at) = lo;
        *reinterpret_cast<X4*>(at + 8) = hi;
      } else {
        *reinterpret_cast<X8*>(at) = v;
      }
    };
    if (stid < 128 - T_DIAG_PIECES) {
      int ur, up;
      tri_upper_piece(stid, ur, up);
      X8 z8;
#pragma unroll
      for (int e = 0; e < 8; ++e) z8[e] = (OT)0.0f;
#pragma unroll
      for (int par = 0; par < 2; ++par) {
        OT* tt = tiles(par).t;
        put_t(&tt[(0 * 32 + ur) * ST + (PERM ? op_perm32_piece(up) : 8 * up)], z8);
        put_t(&tt[(2 * 32 + ur) * ST + (PERM ? op_perm32_piece(up) : 8 * up)], z8);
      }
    }
    // Loads are unconditional (rows past the end of a partial chunk read its last row and are zeroed when staged):
    // a select on a freshly loaded value would make the wave wait for the load at once.
    // (tok0, len: the chunk's entries of the tables, which the caller holds in scalar registers: fetched here they
    // would put a dependent scalar-memory round trip in front of every use)
    auto issue_tiles = [&](int c, int tok0, int len, typename Raw8<T>::type* rk_) {  // k, v, T
      c = uniform(c);
      const T* kb = k + ((size_t)tok0 * H + h) * KT;
      const T* vb = v + ((size_t)tok0 * HV + hv) * VT;
      const int r = min(srow, len - 1);
      const int koff = r * H * KT + spart * (KT / 2), voff = r * HV * VT + spart * (VT / 2);
#pragma unroll
      for (int u = 0; u < KU; ++u) rk_[u] = *reinterpret_cast<const typename Raw8<T>::type*>(kb + koff + 8 * u);
#pragma unroll
      for (int u = 0; u < VU; ++u) rv_[u] = *reinterpret_cast<const typename Raw8<T>::type*>(vb + voff + 8 * u);
      // three pieces per thread, unconditional loads (the last 32 pieces are loaded by four threads each, which then
      // store the same values to the same place)
      const X8* tp = reinterpret_cast<const X8*>(tmat + ((size_t)c * HV + hv) * REC_BYTES);
      rt_[0] = tp[stid];                    // T21
      rt_[1] = tp[128 + stid];              // packed diagonal pieces 0 .. 127 (T11, then the first 48 of T22)
      rt_[2] = tp[256 + (stid & 31)];       // packed diagonal pieces 128 .. 159 (the rest of T22), four times over
    };
    auto issue_gb = [&](int c) {  // cumulative log-decay and beta of the chunk's tokens (lane = token)
      c = uniform(c);
      const float* fact = reinterpret_cast<const float*>(tmat + ((size_t)c * HV + hv) * REC_BYTES + T_BYTES);
      rg = fact[lane];
      rb = fact[64 + lane];
    };
    auto issue_q = [&](int tok0, int len, typename Raw8<T>::type* rq_) {
      const T* qb = q + ((size_t)tok0 * H + h) * KT;
      const int koff = min(srow, len - 1) * H * KT + spart * (KT / 2);
#pragma unroll
      for (int u = 0; u < KU; ++u) rq_[u] = *reinterpret_cast<const typename Raw8<T>::type*>(qb + koff + 8 * u);
    };
    typename Raw8<T>::type zero;
#pragma unroll
    for (int e = 0; e < 8; ++e) zero[e] = (T)0.0f;
    const bool want_ss = l2norm != GDR_L2_NONE;

    float kss = 0.0f;  // sum of squares of this thread's half of k row srow (stage_data -> stage_factors)
    // k, v and T of chunk c from the registers to tile set par
    // rows past the end of a partial chunk become zero (a uniform branch: whole chunks pay nothing for it)
    auto zero_dead_rows = [&](int len, typename Raw8<T>::type* regs, int n) __attribute__((always_inline)) {
      if (len < 64) {
        const bool live = srow < len;
#pragma unroll
        for (int u = 0; u < n; ++u) regs[u] = live ? regs[u] : zero;
      }
    };
    auto stage_data = [&](int len, int par, typename Raw8<T>::type* rk_) {
      const GdrTilesT<OT> tl = tiles(par);
      zero_dead_rows(len, rk_, KU);
      zero_dead_rows(len, rv_, VU);
      put_t(&tl.t[t21_off], rt_[0]);
      put_t(&tl.t[ta_off], rt_[1]);
      put_t(&tl.t[tb_off], rt_[2]);
      kss = 0.0f;
      if constexpr (PERM) {
#pragma unroll
        for (int u = 0; u < KU; u += 4) {  // (a thread's half row is one or two groups of 32 columns)
          X8 p0 = raw_to_op<T, OT>(rk_[u], kss, want_ss), p1 = raw_to_op<T, OT>(rk_[u + 1], kss, want_ss);
          X8 p2 = raw_to_op<T, OT>(rk_[u + 2], kss, want_ss), p3 = raw_to_op<T, OT>(rk_[u + 3], kss, want_ss);
          op_perm32<OT>(p0, p1, p2, p3);
          OT* at = &tl.k[srow * SK + spart * (KT / 2) + 8 * u];
          *reinterpret_cast<X8*>(at) = p0;
          *reinterpret_cast<X8*>(at + 8) = p1;
          *reinterpret_cast<X8*>(at + 16) = p2;
          *reinterpret_cast<X8*>(at + 24) = p3;
        }
      }
#pragma unroll
      for (int u = 0; u < (PERM ? 0 : KU); u += 2) {
        X8 pa = raw_to_op<T, OT>(rk_[u], kss, want_ss), pb = raw_to_op<T, OT>(rk_[u + 1], kss, want_ss);
        if constexpr (!SCALED) {
          if constexpr (SWZ) op_swizzle16<OT>(pa, pb);
          *reinterpret_cast<X8*>(&tl.k[srow * SK + spart * (KT / 2) + 8 * u]) = pa;
          *reinterpret_cast<X8*>(&tl.k[srow * SK + spart * (KT / 2) + 8 * u + 8]) = pb;
        }
      }
#pragma unroll
      for (int u = 0; u < VU; ++u) {
        float unused = 0.0f;
        *reinterpret_cast<X8*>(&tl.v[srow * SV + spart * (VT / 2) + 8 * u]) =
            raw_to_op<T, OT>(rv_[u], unused, false);
      }
    };
    // per-token factors of chunk c (gate, beta, norms) into tile set par
    auto stage_factors = [&](int c, int par, const typename Raw8<T>::type* rk_) {
      const GdrTilesT<OT> tl = tiles(par);
      // in-chunk cumulative log-decay in units of log 2 (exp2 is a single instruction) and beta, lane = token; both
      // come ready from the chunk's record (zero decay increment and zero beta past the end of a partial chunk)
      const float bv = rb, gv = rg;
      const float g_last = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(gv), 63));
      const float kss2 = kss + dpp_f32<GDR_DPP_QUAD_XOR1, 0xF>(0.0f, kss);
      // the thread that owns row srow derives that token's factors (gamma / beta of the row sit in lane srow)
      grow = __shfl(gv, srow);
      const float brow = __shfl(bv, srow);
      const float rk = l2_factor(kss2, l2norm);
      const float ekr = __builtin_amdgcn_exp2f(grow) * rk, dkr = safe_exp2(g_last - grow) * rk;
      if constexpr (PASS_B && OWN_Q) {  // (the 128-wide heads have no registers to spare for a second form)
        // Gating of P in factored form, e^{gamma_i - gamma_j} = E_i / E_j with E = 2^(gamma - gamma_last / 2): one exp2
        // per token instead of one per element. Allowed while no exponent can leave the fp32 range (the chunk's total
        // decay above 2^-120) and no log-decay of the chunk is positive (the cumulative sums never rise); otherwise
        // every ratio goes through safe_exp2 one by one. Lanes past the end of a partial chunk repeat the last sum.
        const float gprev = __shfl_up(gv, 1);
        pfast = !__ballot(lane > 0 && gv > gprev) && !__ballot(gv > 0.0f) && g_last > -120.0f;
        ghalf = 0.5f * g_last;
      }
      if (spart == 0) {
        tl.beta[srow] = brow;
        tl.ek[srow] = ekr;
        tl.dk[srow] = dkr;
        tl.gamma[srow] = grow;
        tl.rk[srow] = (PASS_B && pfast) ? rk * __builtin_amdgcn_exp2f(ghalf - grow) : rk;  // column factor of P
        if (srow == 0) {
          tl.misc[0] = __builtin_amdgcn_exp2f(g_last);
          tl.misc[1] = (PASS_B && pfast) ? 1.0f : 0.0f;
          tl.misc[2] = ghalf;
        }
      }
      if constexpr (SCALED) {  // the two scaled k tiles, from the raw row that is still in registers
#pragma unroll
        for (int u = 0; u < KU; u += 2) {
          X8 pe[2], pd[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const typename Raw8<T>::type piece = rk_[u + h];  // (dead rows were zeroed by stage_data)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const float f = (float)piece[e];
              pe[h][e] = (OT)(f * ekr);
              pd[h][e] = (OT)(f * dkr);
            }
          }
          if constexpr (SWZ) { op_swizzle16<OT>(pe[0], pe[1]); op_swizzle16<OT>(pd[0], pd[1]); }
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            *reinterpret_cast<X8*>(&tl.k[srow * SK + spart * (KT / 2) + 8 * (u + h)]) = pe[h];
            *reinterpret_cast<X8*>(&tl.kd[srow * SK + spart * (KT / 2) + 8 * (u + h)]) = pd[h];
          }
        }
      }
    };
    auto stage_q = [&](int len, typename Raw8<T>::type* rq_, int par = 0) {
      GDR_Q_BUFFERS(par);
      if constexpr (P16) {  // the factors of this chunk were derived by the other pair of stagers
        const GdrTilesT<OT> tl = tiles(par);
        grow = tl.gamma[srow];
        pfast = tl.misc[1] != 0.0f;
        ghalf = tl.misc[2];
      }
      zero_dead_rows(len, rq_, KU);
      float qss = 0.0f;
      if constexpr (PERM) {
#pragma unroll
        for (int u = 0; u < KU; u += 4) {
          X8 p0 = raw_to_op<T, OT>(rq_[u], qss, want_ss), p1 = raw_to_op<T, OT>(rq_[u + 1], qss, want_ss);
          X8 p2 = raw_to_op<T, OT>(rq_[u + 2], qss, want_ss), p3 = raw_to_op<T, OT>(rq_[u + 3], qss, want_ss);
          op_perm32<OT>(p0, p1, p2, p3);
          OT* at = &s_q[srow * SK + spart * (KT / 2) + 8 * u];
          *reinterpret_cast<X8*>(at) = p0;
          *reinterpret_cast<X8*>(at + 8) = p1;
          *reinterpret_cast<X8*>(at + 16) = p2;
          *reinterpret_cast<X8*>(at + 24) = p3;
        }
      }
#pragma unroll
      for (int u = 0; u < (PERM ? 0 : KU); u += 2) {
        X8 pa = raw_to_op<T, OT>(rq_[u], qss, want_ss), pb = raw_to_op<T, OT>(rq_[u + 1], qss, want_ss);
        if constexpr (SWZ) op_swizzle16<OT>(pa, pb);
        *reinterpret_cast<X8*>(&s_q[srow * SK + spart * (KT / 2) + 8 * u]) = pa;
        *reinterpret_cast<X8*>(&s_q[srow * SK + spart * (KT / 2) + 8 * u + 8]) = pb;
      }
      qss += dpp_f32<GDR_DPP_QUAD_XOR1, 0xF>(0.0f, qss);
      if (spart == 0) {
        const float rq = l2_factor(qss, l2norm);
        s_qs[srow] = scale * __builtin_amdgcn_exp2f(grow) * rq;
        s_rq[srow] = pfast ? rq * __builtin_amdgcn_exp2f(grow - ghalf) : rq;  // row factor of P (without scale)
      }
    };

    auto build_p = [&](int par) {
      if constexpr (PASS_B) {
        GDR_Q_BUFFERS(par);
        const GdrTilesT<OT> tl = tiles(par);
        // P^T tiles (0,0), (0,1), (1,1) -> P fragments; tile (1,0) is zero. Stager 0 takes tile 0, stager 1 tile 2,
        // and they share tile 1: both run its four MFMAs, each finishes and stores one of its two fragments.
        const bool fast = OWN_Q && uniform(__float_as_int(tl.misc[1])) != 0;
        auto p_tile = [&](int t, int half) {  // half: -1 = whole tile, 0 / 1 = accumulator registers 0-7 / 8-15
          const int jm = t == 2 ? 1 : 0, tn = t == 0 ? 0 : 1;
          X8 fa[KT / 16], fb[KT / 16];
#pragma unroll
          for (int ks = 0; ks < KT / 16; ++ks) {
            fa[ks] = *reinterpret_cast<const X8*>(&tl.k[(32 * jm + ln) * SK + 16 * ks + 8 * hh]);
            fb[ks] = *reinterpret_cast<const X8*>(&s_q[(32 * tn + ln) * SK + 16 * ks + 8 * hh]);
          }
          f32x4 gj[4], rj[4];  // gamma_j (slow path only) and the column factor of this lane's 16 accumulator rows
#pragma unroll
          for (int b4 = 0; b4 < 4; ++b4) {
            if (!fast) gj[b4] = *reinterpret_cast<const f32x4*>(&tl.gamma[32 * jm + 8 * b4 + 4 * hh]);
            rj[b4] = *reinterpret_cast<const f32x4*>(&tl.rk[32 * jm + 8 * b4 + 4 * hh]);
          }
          const int i = 32 * tn + ln;
          const float gi = fast ? 0.0f : tl.gamma[i], fi = scale * s_rq[i];
          lds_fence();
          f32x16 acc = zero16();
#pragma unroll
          for (int ks = 0; ks < KT / 16; ++ks) acc = mfma32(fa[ks], fb[ks], acc);
          if constexpr (P16) {
            // Narrow chain waves read P as the B operand of the 16x16x32 shape: lane 16 g + i' of fragment (tt, ts)
            // holds P[token 16 tt + i'][32 ts + 4 g .. + 3 and 32 ts + 16 + 4 g .. + 3]. Of this tile (columns = tokens
            // 32 tn + ln, rows j = 32 jm + 8 b + 4 hh + e in register 4 b + e) a lane therefore holds two pieces:
            // registers {0-3, 8-11} for g = hh and {4-7, 12-15} for g = hh + 2, both of fragment (2 tn + ln / 16, jm).
            const int tt = 2 * tn + (ln >> 4), f16 = tt < 2 ? tt : 2 + 2 * (tt - 2) + jm;
#pragma unroll
            for (int pc = 0; pc < 2; ++pc) {
              if (half >= 0 && half != pc) continue;
              X8 piece;
              if (fast) {  // (one branch per piece, not per element)
#pragma unroll
                for (int x = 0; x < 8; ++x) {
                  const int r = (x < 4 ? 0 : 8) + 4 * pc + (x & 3);
                  const float t = acc[r] * (fi * rj[r / 4][r % 4]);
                  piece[x] = (OT)((jm != tn || ln >= acc_row(r, hh)) ? t : 0.0f);
                }
              } else {
#pragma unroll
                for (int x = 0; x < 8; ++x) {
                  const int r = (x < 4 ? 0 : 8) + 4 * pc + (x & 3);
                  const int j = 32 * jm + acc_row(r, hh);
                  piece[x] = (OT)(acc[r] * (fi * rj[r / 4][r % 4] * safe_exp2(i >= j ? gi - gj[r / 4][r % 4] : 1.0f)));
                }
              }
              op_frag_store<OT>(s_P, f16, 16 * (hh + 2 * pc) + (ln & 15), piece);
            }
            return;
          }
          const int f0 = tn == 0 ? 0 : 2 + 2 * jm;  // fragments: tm=0 -> 0,1 ; tm=1 -> 2..5
#pragma unroll
          for (int part = 0; part < 2; ++part) {
            if (half >= 0 && half != part) continue;
            if (fast) {
#pragma unroll
              for (int r = 8 * part; r < 8 * part + 8; ++r) {
                const float val = acc[r] * (fi * rj[r / 4][r % 4]);
                acc[r] = (jm != tn || ln >= acc_row(r, hh)) ? val : 0.0f;  // (the tile below the diagonal is full)
              }
            } else {
#pragma unroll
              for (int r = 8 * part; r < 8 * part + 8; ++r) {  // the mask goes on the exponent: branch-free
                const int j = 32 * jm + acc_row(r, hh);
                acc[r] *= fi * rj[r / 4][r % 4] * safe_exp2(i >= j ? gi - gj[r / 4][r % 4] : 1.0f);
              }
            }
            op_frag_store<OT>(s_P, f0 + part, lane, acc_to_op<OT>(acc, 8 * part));
          }
        };
        if constexpr (P16 && KT <= 64) {
          // Narrow form (the P builders are on the critical path there): one batch of operand reads for all tiles of the
          // wave -- stager 1's two tiles share their q rows --, the tiles' MFMA chains interleaved, the column factors
          // requested behind the MFMAs. Fragment layout as in p_tile.
          const int tn = sw;
          const int i = 32 * tn + ln;
          X8 fb[KT / 16], fa0[KT / 16], fa1[KT / 16];
#pragma unroll
          for (int ks = 0; ks < KT / 16; ++ks) {
            fb[ks] = *reinterpret_cast<const X8*>(&s_q[(32 * tn + ln) * SK + 16 * ks + 8 * hh]);
            fa0[ks] = *reinterpret_cast<const X8*>(&tl.k[ln * SK + 16 * ks + 8 * hh]);
            if (sw == 1) fa1[ks] = *reinterpret_cast<const X8*>(&tl.k[(32 + ln) * SK + 16 * ks + 8 * hh]);
          }
          const float gi = fast ? 0.0f : tl.gamma[i], fi = scale * s_rq[i];
          lds_fence();
          f32x16 acc0 = zero16(), acc1 = zero16();
#pragma unroll
          for (int ks = 0; ks < KT / 16; ++ks) {
            acc0 = mfma32(fa0[ks], fb[ks], acc0);
            if (sw == 1) acc1 = mfma32(fa1[ks], fb[ks], acc1);
          }
          asm volatile("" ::: "memory");
          auto finish = [&](const f32x16& acc, int jm) __attribute__((always_inline)) {
            f32x4 gj[4], rj[4];
#pragma unroll
            for (int b4 = 0; b4 < 4; ++b4) {
              if (!fast) gj[b4] = *reinterpret_cast<const f32x4*>(&tl.gamma[32 * jm + 8 * b4 + 4 * hh]);
              rj[b4] = *reinterpret_cast<const f32x4*>(&tl.rk[32 * jm + 8 * b4 + 4 * hh]);
            }
            const int tt = 2 * tn + (ln >> 4), f16 = tt < 2 ? tt : 2 + 2 * (tt - 2) + jm;
            f32x16 val;
            if (fast) {  // (one branch for the tile: inside the element loop it becomes a branch per element)
#pragma unroll
              for (int r = 0; r < 16; ++r) {
                const float t = acc[r] * (fi * rj[r / 4][r % 4]);
                val[r] = (jm != tn || ln >= acc_row(r, hh)) ? t : 0.0f;
              }
            } else {
#pragma unroll
              for (int r = 0; r < 16; ++r) {
                const int j = 32 * jm + acc_row(r, hh);
                val[r] = acc[r] * (fi * rj[r / 4][r % 4] * safe_exp2(i >= j ? gi - gj[r / 4][r % 4] : 1.0f));
              }
            }
#pragma unroll
            for (int pc = 0; pc < 2; ++pc) {
              X8 piece;
#pragma unroll
              for (int x = 0; x < 8; ++x) piece[x] = (OT)val[(x < 4 ? 0 : 8) + 4 * pc + (x & 3)];
              op_frag_store<OT>(s_P, f16, 16 * (hh + 2 * pc) + (ln & 15), piece);
            }
          };
          finish(acc0, 0);
          if (sw == 1) finish(acc1, 1);
          return;
        }
        // P^T tiles (0,0), (0,1), (1,1) -> P fragments; tile (1,0) is zero.
        if constexpr (OWN_Q) {  // a stager builds the tiles whose q rows it staged itself
          if (sw == 0) p_tile(0, -1);
          else { p_tile(1, -1); p_tile(2, -1); }
        } else {                // stager 0 takes tile 0, stager 1 tile 2, and they share tile 1: both run its MFMAs,
          p_tile(sw == 0 ? 0 : 2, -1);  // each finishes and stores one of its two fragments
          p_tile(1, sw);
        }
      }
    };
    // Chunk indices past the end of the segment are clamped (the last chunk is fetched again for nothing), so that
    // every iteration issues the same loads: with conditional issues the compiler could not count the loads in
    // flight any more and would drain the queue at every wait. q(c) / q(c+2) share a register set.
    const int cl = c1 - 1;
    if constexpr (P16) {
      if (nc > 0) {
        const int ca = uniform(c0), cb = uniform(min(c0 + 1, cl)), cc = uniform(min(c0 + 2, cl));
        const int tk0 = chunk_tok0[ca], ln0 = chunk_len[ca], tk1 = chunk_tok0[cb], ln1 = chunk_len[cb];
        int ln_c = ln0, ln_c1 = ln1, tk_c1 = tk1, tk_c2 = chunk_tok0[cc], ln_c2 = chunk_len[cc];
        if (spair == 0) {
          // ---- k, v, T and the factors: tiles and factors (c + 1) are staged and the loads (c + 2) issued before B(c)
          issue_tiles(c0, tk0, ln0, rk0_);
          issue_gb(c0);
          stage_data(ln0, 0, rk0_);
          stage_factors(c0, 0, rk0_);
          issue_tiles(min(c0 + 1, cl), tk1, ln1, rk0_);
          issue_gb(min(c0 + 1, cl));
          lds_barrier();  // tiles (c0) are ready
          for (int c = c0; c < c1; ++c) {
            const int par = (c - c0) & 1;
            const int cn = uniform(min(c + 3, cl));
            const int tk_n = chunk_tok0[cn], ln_n = chunk_len[cn];
            if constexpr (!OWN_Q) lds_barrier();  // Qb(c) (this pair only takes part)
            if (c + 1 < c1) {
              stage_data(ln_c1, par ^ 1, rk0_);
              stage_factors(c + 1, par ^ 1, rk0_);  // (that set's factor rows are free since B(c - 1))
            }
            issue_tiles(min(c + 2, cl), tk_c2, ln_c2, rk0_);
            issue_gb(min(c + 2, cl));
            lds_barrier();  // B(c)
            lds_barrier();  // C(c)
            ln_c = ln_c1; ln_c1 = ln_c2; tk_c2 = tk_n; ln_c2 = ln_n;
          }
        } else {
          // ---- q and P: q(c) staged and P(c) built before B(c) (from the k tile and the factors of chunk c, complete
          //      since C(c - 1)); the loads of q(c + 1) follow the staging of q(c) into the same registers
          issue_q(tk0, ln0, rq0_);
          lds_barrier();  // tiles (c0) are ready
          if constexpr (DBQ) {
            // q and P exist twice: q(c + 1) is staged between B(c) and C(c) (its factors are complete at B(c), its buffer
            // free since C(c - 1)), P(c + 1) is built after C(c) -- so only the P products sit between C(c) and B(c + 1)
            stage_q(ln_c, rq0_, 0);
            issue_q(tk_c1, ln_c1, rq0_);
            lds_fence();
            build_p(0);
            for (int c = c0; c < c1; ++c) {
              const int par = (c - c0) & 1;
              const int cn = uniform(min(c + 3, cl));
              const int tk_n = chunk_tok0[cn], ln_n = chunk_len[cn];
              lds_barrier();  // B(c)
              if (c + 1 < c1) {
                stage_q(ln_c1, rq0_, par ^ 1);
                issue_q(tk_c2, ln_c2, rq0_);
              }
              lds_barrier();  // C(c)
              if (c + 1 < c1) build_p(par ^ 1);
              ln_c = ln_c1; tk_c1 = tk_c2; ln_c1 = ln_c2; tk_c2 = tk_n; ln_c2 = ln_n;
            }
          } else
          for (int c = c0; c < c1; ++c) {
            const int par = (c - c0) & 1;
            const int cn = uniform(min(c + 3, cl));
            const int tk_n = chunk_tok0[cn], ln_n = chunk_len[cn];
            stage_q(ln_c, rq0_, par);
            issue_q(tk_c1, ln_c1, rq0_);
            if constexpr (OWN_Q) lds_fence();  // this wave's own q rows are in LDS (it builds P from no others)
            else lds_barrier();                // Qb(c)
            build_p(par);
            lds_barrier();  // B(c)
            lds_barrier();  // C(c)
            ln_c = ln_c1; tk_c1 = tk_c2; ln_c1 = ln_c2; tk_c2 = tk_n; ln_c2 = ln_n;
          }
        }
        lds_barrier();  // the o tile of the last chunk is complete (the chain waves' last flush)
      }
      return;
    }
    if (nc > 0) {
      typename Raw8<T>::type* const rkA = rk0_;
      typename Raw8<T>::type* const rkB = SCALED ? rk1_ : rk0_;
      // the chunks' table entries live in scalar registers and are fetched a chunk period before their first use
      const int ca = uniform(c0), cb = uniform(min(c0 + 1, cl)), cc = uniform(min(c0 + 2, cl));
      const int tk0 = chunk_tok0[ca], ln0 = chunk_len[ca], tk1 = chunk_tok0[cb], ln1 = chunk_len[cb];
      int ln_c = ln0, ln_c1 = ln1, tk_c2 = chunk_tok0[cc], ln_c2 = chunk_len[cc];  // of chunks c, c + 1, c + 2 (clamped)
      int tk_c = tk0, tk_c1 = tk1, tk_p = 0, ln_p = 0;                              // (tk_p, ln_p: of chunk c - 1)
      // the o tile (rows of chunk `tok0`) -> HBM, 16-byte pieces, whole rows (non-temporal: o is not read again here)
      auto stager_flush = [&](int tok0, int len) __attribute__((always_inline)) {
        constexpr int PPR = VT / 8, NP = 64 * PPR / 128;
        const int ow = KEEP ? o_width : VT;
        T* ob = o + ((size_t)tok0 * HV + hv) * ow;
        uint4 val[NP];
#pragma unroll
        for (int j = 0; j < NP; ++j) {
          const int x = stid + 128 * j;
          val[j] = *reinterpret_cast<const uint4*>(&s_o[(x / PPR) * SV + 8 * (x % PPR)]);
        }
#pragma unroll
        for (int j = 0; j < NP; ++j) {
          const int x = stid + 128 * j, row = x / PPR, part = x % PPR;
          typedef unsigned int nt_u32x4 __attribute__((ext_vector_type(4)));
          nt_u32x4 nv;
          nv[0] = val[j].x; nv[1] = val[j].y; nv[2] = val[j].z; nv[3] = val[j].w;
          if (row < len && (!KEEP || 8 * part < ow))
            __builtin_nontemporal_store(nv, reinterpret_cast<nt_u32x4*>(ob + (unsigned)(row * (HV * ow) + 8 * part)));
        }
      };
      issue_tiles(c0, tk0, ln0, rkA);
      issue_gb(c0);
      if constexpr (PASS_B) { issue_q(tk0, ln0, rq0_); issue_q(tk1, ln1, rq1_); }
      stage_data(ln0, 0, rkA);
      stage_factors(c0, 0, rkA);
      issue_tiles(min(c0 + 1, cl), tk1, ln1, rkB);
      issue_gb(min(c0 + 1, cl));
      lds_barrier();  // tiles (c0) are ready
      // rk_next holds the raw k rows of chunk c + 1, rk_free is loaded with those of chunk c + 2
      auto one_chunk = [&](int c, int par, typename Raw8<T>::type* rq_, typename Raw8<T>::type* rk_next,
                           typename Raw8<T>::type* rk_free) {
        const int cn = uniform(min(c + 3, cl));
        const int tk_n = chunk_tok0[cn], ln_n = chunk_len[cn];  // used from the next chunk on
        if (c + 1 < c1) stage_data(ln_c1, par ^ 1, rk_next);
        issue_tiles(min(c + 2, cl), tk_c2, ln_c2, rk_free);
        if constexpr (PASS_B) {
          stage_q(ln_c, rq_);
          issue_q(tk_c2, ln_c2, rq_);
          if constexpr (OWN_Q) lds_fence();  // this wave's own q rows are in LDS (it builds P from no others)
          else lds_barrier();                // Qb(c)
          build_p(par);
          lds_barrier();  // B(c)
          if constexpr (STAGER_FLUSH) {
            if (c > c0) stager_flush(tk_p, ln_p);  // o(c - 1): written after C(c - 1), next written after C(c)
          }
          if (c + 1 < c1) stage_factors(c + 1, par ^ 1, rk_next);
          issue_gb(min(c + 2, cl));
          lds_barrier();  // C(c)
        } else {
          if (c + 1 < c1) stage_factors(c + 1, par ^ 1, rk_next);
          issue_gb(min(c + 2, cl));
          lds_barrier();  // B(c)
        }
        tk_p = tk_c; ln_p = ln_c; tk_c = tk_c1; tk_c1 = tk_c2;
        ln_c = ln_c1; ln_c1 = ln_c2; tk_c2 = tk_n; ln_c2 = ln_n;
      };
      for (int c = c0; c < c1; c += 2) {
        one_chunk(c, 0, rq0_, rkB, rkA);
        if (c + 1 < c1) one_chunk(c + 1, 1, rq1_, rkA, rkB);
      }
      if constexpr (STAGER_FLUSH) {
        lds_barrier();  // the o tile of the last chunk is complete
        stager_flush(tk_p, ln_p);
      }
    }
    return;
  }

  if constexpr (CW == 16) {
    // ============================================ narrow chain wave ============================================
    // Wave w owns the 16 value columns 16 w .. + 15 and all K rows of them: S as K / 16 accumulator tiles of the
    // 16x16x32 shape (lane 16 g + i: rows 16 km + 4 g + r, column i). Same stages and barriers as the 32-column chain
    // wave below; every operand fragment from memory is one 16-byte LDS read (tiles in op_perm32 order).
    constexpr int NKM = KT / 16, NKS = KT / 32, NF = 4 * NKS;  // state tiles, contraction steps over K, k / q fragments
    const int g4 = lane >> 4, li = lane & 15;
    const int col = 16 * wave + li;
    f32x4 S[NKM];
    // where this lane's part of a state tile sits in the 32-column accumulator order the scan kernels use: tile
    // (column slab wave / 2, row block km / 2), plane 2 (km % 2) + g / 2, lane 32 (g % 2) + 16 (wave % 2) + i
    const int lane32 = 32 * (g4 & 1) + 16 * (wave & 1) + li;
    auto slab_piece = [&](int km) { return ((km >> 1) * 4 + 2 * (km & 1) + (g4 >> 1)) * 64 + lane32; };
    bool walked = false;
    if constexpr (KT == 64) if (gmax > 0) {
      walked = true;
      // second level of the two-level scan (see the 32-column chain wave): the composites of the groups before this
      // segment's group, then of the segments before it inside its group
      constexpr int M_BYTES = KT * KT * 2, N_BYTES = KT * 32 * 4;
      const int seq = pv.seg_seq[seg], local = seg - pv.seq_seg0[seq];
      const int lead = local / GDR_SCAN_GROUP, nst = lead + local % GDR_SCAN_GROUP;
      const int item0 = seg - local % GDR_SCAN_GROUP;
#pragma unroll
      for (int km = 0; km < NKM; ++km)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          S[km][r] = h0 ? h0[(((size_t)seq * HV + hv) * KT + 16 * km + 4 * g4 + r) * VT + col] : 0.0f;
      X8 rm[2][NKM * NKS];
      f32x4 rn[2][NKM];
      float rd[2];
      // M' is stored as A-operand fragments of the 32x32x16 shape: element (row, c) in fragment (row / 32, c / 16), lane
      // 32 ((c % 16 / 4) & 1) + row % 32, slot 4 (c % 16 / 8) + c % 4. This lane's share of the step ks (columns
      // 32 ks + 4 g .. and 32 ks + 16 + 4 g ..) of rows 16 km + i: the 8-byte half g / 2 of lane 32 (g % 2) + (16 km + i) % 32
      // in the fragments (km / 2, 2 ks) and (km / 2, 2 ks + 1).
      auto issue = [&](int p, X8* m, f32x4* n, float& d) __attribute__((always_inline)) {
        p = uniform(max(0, min(p, nst - 1)));
        const bool top = p < lead;
        const size_t sh = (size_t)(top ? seq * gmax + p : item0 + (p - lead)) * HV + hv;
        const unsigned char* M = (top ? Mgrp : Mcomp) + sh * M_BYTES;
        const f32x4* N = reinterpret_cast<const f32x4*>((top ? Ngrp : Ncomp) + (sh * (VT / 32) + (wave >> 1)) * N_BYTES);
#pragma unroll
        for (int km = 0; km < NKM; ++km)
#pragma unroll
          for (int ks = 0; ks < NKS; ++ks) {
            const int l32 = 32 * (g4 & 1) + 16 * (km & 1) + li;
            const unsigned char* f = M + ((size_t)((km >> 1) * (KT / 16) + 2 * ks) * 64 + l32) * 16 + 8 * (g4 >> 1);
            const X4 lo = *reinterpret_cast<const X4*>(f), hi = *reinterpret_cast<const X4*>(f + 1024);
            X8 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) { v[e] = lo[e]; v[4 + e] = hi[e]; }
            m[km * NKS + ks] = v;
          }
#pragma unroll
        for (int km = 0; km < NKM; ++km) n[km] = N[slab_piece(km)];
        d = (top ? Dgrp : Dcomp)[sh];
      };
      auto step = [&](const X8* m, const f32x4* n, float d) __attribute__((always_inline)) {
        X8 Sb[NKS];
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) Sb[ks] = acc2_to_op<OT>(S[2 * ks], S[2 * ks + 1]);
#pragma unroll
        for (int km = 0; km < NKM; ++km) {
          f32x4 acc;
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf(d, S[km][e], n[km][e]);
#pragma unroll
          for (int ks = 0; ks < NKS; ++ks) acc = mfma16(m[km * NKS + ks], Sb[ks], acc);
          S[km] = acc;
        }
      };
      if (nst > 0) {
        issue(0, rm[0], rn[0], rd[0]);
        issue(1, rm[1], rn[1], rd[1]);
        for (int p = 0; p < nst; p += 2) {
          step(rm[0], rn[0], rd[0]);
          issue(p + 2, rm[0], rn[0], rd[0]);
          if (p + 1 < nst) step(rm[1], rn[1], rd[1]);
          issue(p + 3, rm[1], rn[1], rd[1]);
        }
      }
    }
    if (!walked) {  // the scan leaves every segment's initial state as 32-column slabs in accumulator order
      const f32x4* si = reinterpret_cast<const f32x4*>(Sinit + (((size_t)seg * HV + hv) * (VT / 32) + (wave >> 1)) * (KT * 32));
#pragma unroll
      for (int km = 0; km < NKM; ++km) S[km] = si[slab_piece(km)];
    }

    // this wave's rows of the o tile -> HBM: 64 / NSLAB whole rows of V values, two 16-byte pieces per lane (piece
    // lane + 64 j of the wave's rows: the same part of a row 64 / PPR rows further down)
    constexpr int RW = 64 / NSLAB, PPR = VT / 8;
    const int fo_row = wave * RW + lane / PPR;
    const T* fo_lds = s_o + fo_row * SV + 8 * (lane % PPR);
    const unsigned fo_off = (unsigned)(fo_row * (HV * VT) + 8 * (lane % PPR));  // elements, from the chunk's first o row
    auto flush_o = [&](int tok0, int len) __attribute__((always_inline)) {
      T* ob = o + ((size_t)tok0 * HV + hv) * VT;  // uniform base; per-lane 32-bit offsets
      const uint4 v0 = *reinterpret_cast<const uint4*>(fo_lds);
      const uint4 v1 = *reinterpret_cast<const uint4*>(fo_lds + (64 / PPR) * SV);
      // (o is written once and not read again by this pipeline: non-temporal, see the 32-column chain wave)
      typedef unsigned int nt_u32x4 __attribute__((ext_vector_type(4)));
      nt_u32x4 n0, n1;
      n0[0] = v0.x; n0[1] = v0.y; n0[2] = v0.z; n0[3] = v0.w;
      n1[0] = v1.x; n1[1] = v1.y; n1[2] = v1.z; n1[3] = v1.w;
      if (fo_row < len) __builtin_nontemporal_store(n0, reinterpret_cast<nt_u32x4*>(ob + fo_off));
      if (fo_row + 64 / PPR < len)
        __builtin_nontemporal_store(n1, reinterpret_cast<nt_u32x4*>(ob + fo_off + (unsigned)((64 / PPR) * (HV * VT))));
    };
    // A-operand fragment of a row-major tile: row `row`, the 32-wide contraction step that starts at column c32, in
    // the slot order of the narrow shape (columns 4 g .. + 3 and 16 + 4 g .. + 3): one 16-byte piece of a tile in
    // op_perm32 order, two 8-byte pieces otherwise
    auto row_frag = [&](const OT* arr, int stride, int row, int c32) __attribute__((always_inline)) {
      if constexpr (PERM) {
        return *reinterpret_cast<const X8*>(&arr[row * stride + c32 + 8 * g4]);
      } else {
        const X4 lo = *reinterpret_cast<const X4*>(&arr[row * stride + c32 + 4 * g4]);
        const X4 hi = *reinterpret_cast<const X4*>(&arr[row * stride + c32 + 16 + 4 * g4]);
        X8 out;
#pragma unroll
        for (int e = 0; e < 4; ++e) { out[e] = lo[e]; out[4 + e] = hi[e]; }
        return out;
      }
    };
    // T fragment (tm, ts): rows 16 tm + i of the block T11 (tm < 2) or of T21 / T22 (tm >= 2, ts = 0 / 1)
    auto t_frag = [&](const OT* tt, int tm, int ts) {
      const int blk = tm < 2 ? 0 : 1 + ts;
      return row_frag(tt, ST, blk * 32 + 16 * (tm & 1) + li, 0);
    };

    int o_tok0 = 0, o_len = 0, p_tok0 = 0, p_len = 0;  // table entries of this chunk and of the one before it
    if (nc > 0) { o_tok0 = chunk_tok0[uniform(c0)]; o_len = chunk_len[uniform(c0)]; }
    if (nc > 0) lds_barrier();  // tiles (c0) are ready
    for (int c = c0; c < c1; ++c) {
      const GdrTilesT<OT> tl = tiles((c - c0) & 1);
      GDR_Q_BUFFERS((c - c0) & 1);
      if constexpr (!OWN_Q) lds_barrier();  // Qb(c) (the chain waves only take part)
      const int c_nx = uniform(min(c + 1, c1 - 1));
      const int n_tok0 = chunk_tok0[c_nx], n_len = chunk_len[c_nx];
      // Registers: four waves share a SIMD at K = V = 64 (128 registers each), so every batch of LDS reads is requested
      // behind the MFMAs whose operands it replaces (an MFMA has read its operands once it is issued), not a stage ahead;
      // the MFMAs in flight and the epilogue arithmetic cover the reads. (The empty asm statements keep the compiler from
      // hoisting the reads back up.)
      X8 fk[NF];  // K rows (stage 1), K^T rows (stage 3), Q rows (output)
      X8 ft[6];   // T (stage 2), P (output)
#pragma unroll
      for (int tm = 0; tm < 4; ++tm)
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
          fk[tm * NKS + ks] = row_frag(tl.k, SK, 16 * tm + li, 32 * ks);
      X8 Sb[NKS];
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) Sb[ks] = acc2_to_op<OT>(S[2 * ks], S[2 * ks + 1]);
      lds_fence();
      f32x4 R[4];
#pragma unroll
      for (int tm = 0; tm < 4; ++tm) {  // K S
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) acc = mfma16(fk[tm * NKS + ks], Sb[ks], acc);
        R[tm] = acc;
      }
      asm volatile("" ::: "memory");
      // the per-token factors and the v tile (in accumulator layout) of stage 1's epilogue, then the T fragments
      f32x4 be[4], ek[4];
      X4 vv[4];
#pragma unroll
      for (int tm = 0; tm < 4; ++tm) {
        be[tm] = *reinterpret_cast<const f32x4*>(&tl.beta[16 * tm + 4 * g4]);
        ek[tm] = *reinterpret_cast<const f32x4*>(&tl.ek[16 * tm + 4 * g4]);
        vv[tm] = op_lds_read_tr4<OT>(tl.v + (16 * tm + 4 * g4 + (li >> 2)) * SV + 16 * wave + 4 * (li & 3));
      }
      ft[0] = t_frag(tl.t, 0, 0); ft[1] = t_frag(tl.t, 1, 0); ft[2] = t_frag(tl.t, 2, 0);
      ft[3] = t_frag(tl.t, 2, 1); ft[4] = t_frag(tl.t, 3, 0); ft[5] = t_frag(tl.t, 3, 1);
#pragma unroll
      for (int tm = 0; tm < 4; ++tm)  // R = beta (v - ek (K S))
#pragma unroll
        for (int e = 0; e < 4; ++e) R[tm][e] = be[tm][e] * ((float)vv[tm][e] - ek[tm][e] * R[tm][e]);
      X8 Rb[2];
      Rb[0] = acc2_to_op<OT>(R[0], R[1]);
      Rb[1] = acc2_to_op<OT>(R[2], R[3]);
      f32x4 Vn[4];
#pragma unroll
      for (int tm = 0; tm < 4; ++tm) {  // v_new = T R (T is lower triangular: rows 32 .. 63 need both steps)
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        acc = mfma16(ft[tm < 2 ? tm : 2 * tm - 2], Rb[0], acc);
        if (tm >= 2) acc = mfma16(ft[2 * tm - 1], Rb[1], acc);
        Vn[tm] = acc;
      }
      asm volatile("" ::: "memory");
      // K^T fragments (transposing reads of the row-major k tile) and the decay factors of the state update
#pragma unroll
      for (int km = 0; km < NKM; ++km)
#pragma unroll
        for (int ts = 0; ts < 2; ++ts) fk[km * 2 + ts] = op_ld_tr16<OT, PERM>(tl.k, SK, 16 * km, 32 * ts, lane);
      f32x4 dk[4];
#pragma unroll
      for (int tm = 0; tm < 4; ++tm) dk[tm] = *reinterpret_cast<const f32x4*>(&tl.dk[16 * tm + 4 * g4]);
      const float dec = tl.misc[0];
      X8 Vb[2], Vsb[2];
#pragma unroll
      for (int ts = 0; ts < 2; ++ts) {
        Vb[ts] = acc2_to_op<OT>(Vn[2 * ts], Vn[2 * ts + 1]);
        f32x4 a = Vn[2 * ts], b = Vn[2 * ts + 1];
#pragma unroll
        for (int e = 0; e < 4; ++e) { a[e] *= dk[2 * ts][e]; b[e] *= dk[2 * ts + 1][e]; }
        Vsb[ts] = acc2_to_op<OT>(a, b);
      }
      lds_fence();
      lds_barrier();  // B(c): every operand that comes from the k, v and T tiles of chunk c is in registers; the o
                      // tile of chunk c - 1 is complete
#pragma unroll
      for (int km = 0; km < NKM; ++km) {  // S <- dec S + K^T (dk v_new)
#pragma unroll
        for (int e = 0; e < 4; ++e) S[km][e] *= dec;
#pragma unroll
        for (int ts = 0; ts < 2; ++ts) S[km] = mfma16(fk[km * 2 + ts], Vsb[ts], S[km]);
      }
      asm volatile("" ::: "memory");
      if (c > c0) flush_o(p_tok0, p_len);  // (behind the MFMAs of the state update, where few registers are live)
      asm volatile("" ::: "memory");
      // Q rows, P fragments, output factors
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
          fk[tt * NKS + ks] = row_frag(s_q, SK, 16 * tt + li, 32 * ks);
#pragma unroll
      for (int f = 0; f < 6; ++f) ft[f] = op_frag_load<OT>(s_P, f, lane);
      float qsv[4];
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) qsv[tt] = s_qs[16 * tt + li];  // scale e^{gamma} rq of this lane's token per row tile
      lds_fence();
      lds_barrier();  // C(c): the q and P operands of chunk c are in registers, the o tile of chunk c - 1 has been read
      // o^T = S_old^T (qs Q)^T + v_new^T P^T (computed transposed: the lane holds a token and four value columns, see
      // the 32-column chain wave): tile tt = tokens 16 tt .. + 15, rows of the result = this wave's 16 value columns
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        f32x4 a1 = {0.0f, 0.0f, 0.0f, 0.0f}, a2 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) a1 = mfma16(Sb[ks], fk[tt * NKS + ks], a1);
        a2 = mfma16(Vb[0], ft[tt < 2 ? tt : 2 * tt - 2], a2);
        if (tt >= 2) a2 = mfma16(Vb[1], ft[2 * tt - 1], a2);
        typedef T T4 __attribute__((ext_vector_type(4)));
        T4 pk;
#pragma unroll
        for (int e = 0; e < 4; ++e) pk[e] = GdrElem<T>::from_float(__builtin_fmaf(qsv[tt], a1[e], a2[e]));
        *reinterpret_cast<T4*>(&s_o[(16 * tt + li) * SV + 16 * wave + 4 * g4]) = pk;
      }
      p_tok0 = o_tok0; p_len = o_len;
      o_tok0 = n_tok0; o_len = n_len;
    }
    if (nc > 0) {
      lds_barrier();  // the o tile of the last chunk is complete
      flush_o(p_tok0, p_len);
    }
    int late = 0;  // (keeps the compiler from computing these addresses before the loop)
    asm volatile("" : "+v"(late));
    if (ht && (flags & SEG_LAST)) {
      const int seq = pv.seg_seq[seg];
      float* out = ht + ((size_t)seq * HV + hv) * KT * VT + late;
#pragma unroll
      for (int km = 0; km < NKM; ++km)
#pragma unroll
        for (int r = 0; r < 4; ++r) out[(16 * km + 4 * g4 + r) * VT + col] = S[km][r];
    }
    return;
  } else {

  // ================================================== chain ==================================================
  // this wave's 32 columns: PASS_B value columns; PASS_A columns of [M | N]
  const bool is_m = !PASS_B && wave < KT / 32;
  const int vslab = PASS_B ? wave : (is_m ? 0 : wave - KT / 32);
  const int col = 32 * vslab + ln;  // value column (unused for M slabs)
  const float vmask = is_m ? 0.0f : 1.0f;
  const unsigned vkeep = uniform(is_m ? 0 : -1);

  f32x16 S[KT / 32];
  bool walked = false;
  if constexpr (PASS_B && KT == 64) if (gmax > 0) {
    walked = true;
    // Two-level scan, second level done here: the state this segment starts from = the sequence's initial state
    // pushed through the composites of the groups before this segment's group (Mgrp / Ngrp / Dgrp, written by the
    // group pass) and then through the composites of the segments before it inside its group (at most
    // 2 (GDR_SCAN_GROUP - 1) steps S <- d S + N + M' S). This wave owns all rows of its 32 columns, so the state
    // feeds the next step's B operand straight from the accumulators.
    constexpr int NKS = KT / 16, NKM = KT / 32;
    constexpr int M_BYTES = KT * KT * 2, N_BYTES = KT * 32 * 4;
    const int seq = pv.seg_seq[seg], local = seg - pv.seq_seg0[seq];
    const int lead = local / GDR_SCAN_GROUP, nst = lead + local % GDR_SCAN_GROUP;
    const int item0 = seg - local % GDR_SCAN_GROUP;
#pragma unroll
    for (int km = 0; km < NKM; ++km)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        S[km][r] = h0 ? h0[(((size_t)seq * HV + hv) * KT + 32 * km + acc_row(r, hh)) * VT + col] : 0.0f;
    X8 rm[2][NKM * NKS];
    f32x4 rn[2][NKM * 4];
    float rd[2];
    auto issue = [&](int p, X8* m, f32x4* n, float& d) __attribute__((always_inline)) {
      p = uniform(max(0, min(p, nst - 1)));
      const bool top = p < lead;
      const size_t sh = (size_t)(top ? seq * gmax + p : item0 + (p - lead)) * HV + hv;
      const X8* M = reinterpret_cast<const X8*>((top ? Mgrp : Mcomp) + sh * M_BYTES);
      const f32x4* N = reinterpret_cast<const f32x4*>((top ? Ngrp : Ncomp) + (sh * (VT / 32) + vslab) * N_BYTES);
#pragma unroll
      for (int f = 0; f < NKM * NKS; ++f) m[f] = M[f * 64 + lane];
#pragma unroll
      for (int f = 0; f < NKM * 4; ++f) n[f] = N[f * 64 + lane];
      d = (top ? Dgrp : Dcomp)[sh];
    };
    auto step = [&](const X8* m, const f32x4* n, float d) __attribute__((always_inline)) {
      X8 Sb[NKS];
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) Sb[ks] = acc_to_op<OT>(S[ks / 2], 8 * (ks % 2));
#pragma unroll
      for (int km = 0; km < NKM; ++km) {
        f32x16 acc;
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[4 * q4 + e] = __builtin_fmaf(d, S[km][4 * q4 + e], n[km * 4 + q4][e]);
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) acc = mfma32(m[km * NKS + ks], Sb[ks], acc);
        S[km] = acc;
      }
    };
    if (nst > 0) {
      // (strong decays: the walk starts at the last map of a run of maps that cut off what lies before them; 60 000 tokens x
      // 8 heads at e^-0.8 a token: pass 60.1 -> 57.2 us, call 131 -> 124.5; 6 007 tokens where none does 39.6 -> 38.7)
      const int pl = min(lane, nst - 1);
      const float dl = (pl < lead ? Dgrp : Dcomp)[(size_t)(pl < lead ? seq * gmax + pl : item0 + (pl - lead)) * HV + hv];
      issue(0, rm[0], rn[0], rd[0]);
      issue(1, rm[1], rn[1], rd[1]);
      int from = max(0, uniform(gdr_leading_cuts(dl, nst, lane)) - 1);
      // (the decays' scalar loads stay in front of the branch: the compiler moves them behind it, a memory latency more in
      // front of the first step; 15 000 tokens x 6 heads where nothing cuts off: pass 24.7 -> 25.0 us)
      asm volatile("" : "+s"(rd[0]), "+s"(rd[1]));
      if (from > 0 && h0) {
        float probe = 0.0f;
#pragma unroll
        for (int km = 0; km < NKM; ++km)
#pragma unroll
          for (int r = 0; r < 16; ++r) probe = __builtin_fmaf(S[km][r], 0.0f, probe);
        if (__ballot(!(probe == 0.0f))) from = 0;
      }
      if (from > 0) {
        issue(from, rm[0], rn[0], rd[0]);
        issue(from + 1, rm[1], rn[1], rd[1]);
      }
      for (int p = from; p < nst; p += 2) {
        step(rm[0], rn[0], rd[0]);
        issue(p + 2, rm[0], rn[0], rd[0]);
        if (p + 1 < nst) step(rm[1], rn[1], rd[1]);
        issue(p + 3, rm[1], rn[1], rd[1]);
      }
    }
  }
  if (walked) {
  } else if (PASS_B) {  // the scan leaves every segment's initial state as 32-column slabs in accumulator order
    const f32x4* si = reinterpret_cast<const f32x4*>(Sinit + (((size_t)seg * HV + hv) * (VT / 32) + vslab) * (KT * 32));
#pragma unroll
    for (int km = 0; km < KT / 32; ++km)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const f32x4 t = si[(km * 4 + q4) * 64 + lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) S[km][4 * q4 + e] = t[e];
      }
  } else {
#pragma unroll
    for (int km = 0; km < KT / 32; ++km)
#pragma unroll
      for (int r = 0; r < 16; ++r) S[km][r] = (is_m && 32 * km + acc_row(r, hh) == 32 * wave + ln) ? 1.0f : 0.0f;
  }

  GDR_Q_BUFFERS(0);
  float dtot = 1.0f;  // product of the chunks' decays over the segment (PASS_A)
  // The LDS operand reads of a stage are issued as one batch one stage ahead of the MFMAs that use them
  // (lds_fence() pins that order); left alone the compiler fetches each fragment right before its MFMA and
  // pays the LDS latency once per MFMA.
  // The q rows and the P fragments of the output are requested right after B(c), before the state update's MFMAs,
  // where the registers allow a second set of fragments (K = 64 and below).
  constexpr bool EARLY_Q = PASS_B && KT <= 64;
  int o_tok0 = 0, o_len = 0;  // table entries of the chunk whose o rows are stored, fetched a chunk ahead
  if (PASS_B && nc > 0) { o_tok0 = chunk_tok0[uniform(c0)]; o_len = chunk_len[uniform(c0)]; }
  // Output pass at K <= 64: the K rows of chunk c + 1 are requested behind the barrier C(c), in front of the output's
  // MFMAs (the fragment registers are free from the state update on, and the tiles of chunk c + 1 are complete since
  // B(c)), so the next chunk does not start with an LDS round trip.
  constexpr bool EARLY_K = EARLY_Q && KT == 64;  // (the 32 x 32 form has no registers for it)
  X8 fk[2 * (KT / 16)];  // K rows (stage 1), K^T rows (stage 3), Q rows (output)
  auto load_k_rows = [&](const GdrTilesT<OT>& tx) __attribute__((always_inline)) {
#pragma unroll
    for (int tm = 0; tm < 2; ++tm)
#pragma unroll
      for (int ks = 0; ks < KT / 16; ++ks) fk[tm * (KT / 16) + ks] = SWZ ? op_ld_kappa_swz<OT>(tx.k, SK, 32 * tm + ln, 16 * ks, hh)
                                        : op_ld_kappa<OT>(tx.k, SK, 32 * tm + ln, 16 * ks, hh);
  };
  bool faded = false;  // the decays' product is zero (of a wide head: has been)
  bool gone = false;   // (M) this wave's columns are zero
  auto m_is_zero = [&]() __attribute__((always_inline)) {
    unsigned any = 0;
#pragma unroll
    for (int km = 0; km < KT / 32; ++km)
#pragma unroll
      for (int r = 0; r < 16; ++r) any |= __float_as_uint(S[km][r]) << 1;
    return __ballot(any != 0) == 0;
  };
  if (nc > 0) lds_barrier();  // tiles (c0) are ready
  if constexpr (EARLY_K) load_k_rows(tiles(0));
  int c = c0;
  for (; c < c1 && !(SKIP_M && gone); ++c) {
    const GdrTilesT<OT> tl = tiles((c - c0) & 1);
    if constexpr (PASS_B && !OWN_Q) lds_barrier();  // Qb(c) (the chain waves only take part)
    const int c_nx = uniform(min(c + 1, c1 - 1));
    const int n_tok0 = PASS_B ? chunk_tok0[c_nx] : 0, n_len = PASS_B ? chunk_len[c_nx] : 0;
    X8 fq[EARLY_Q ? 2 * (KT / 16) : 1];
    X8 ft[6];              // T (stage 2), P (output)
    if constexpr (!EARLY_K) load_k_rows(tl);
    X8 Sb[KT / 16];
#pragma unroll
    for (int ks = 0; ks < KT / 16; ++ks) Sb[ks] = acc_to_op<OT>(S[ks / 2], 8 * (ks % 2));
    if constexpr (KEEP && PASS_B) {
      unsigned char* st = keep + (((size_t)uniform(c) * HV + hv) * (VT / 32) + vslab) * (KT * 32 * 2);
#pragma unroll
      for (int ks = 0; ks < KT / 16; ++ks) op_frag_store<OT>(st, ks, lane, Sb[ks]);
    }
    lds_fence();
    // batch for stage 2: T fragments and the per-token factors / v tile of stage 1's epilogue
#pragma unroll
    for (int tm = 0; tm < 2; ++tm)
#pragma unroll
      for (int ks = 0; ks < 2 * (tm + 1); ++ks)  // blocks T11 | T21, T22
        ft[2 * tm + ks] = op_ld_kappa<OT>(tl.t + (tm == 0 ? 0 : (ks < 2 ? 1 : 2)) * 32 * ST, ST, ln, 16 * (ks & 1), hh);
    f32x4 be[8], ek[8];
    X4 vv[8];
#pragma unroll
    for (int t8 = 0; t8 < 8; ++t8) {
      const int i0 = 8 * t8 + 4 * hh;
      be[t8] = *reinterpret_cast<const f32x4*>(&tl.beta[i0]);
      if constexpr (!SCALED) ek[t8] = *reinterpret_cast<const f32x4*>(&tl.ek[i0]);
      // v[8 t8 + 4 hh + e][col]. The M slabs (v = 0) issue the same transposing loads and drop the result with
      // vmask: the load must run with every lane enabled, so it is kept out of any per-wave branch.
      vv[t8] = op_ld_col4<OT>(tl.v, SV, 32 * vslab, 8 * t8, lane);
    }
    X8 Rb[4];
#pragma unroll
    for (int tm = 0; tm < 2; ++tm) {  // R = beta (v - ek (K S))
      f32x16 acc = zero16();
#pragma unroll
      for (int ks = 0; ks < KT / 16; ++ks) acc = mfma32(fk[tm * (KT / 16) + ks], Sb[ks], acc);
#pragma unroll
      for (int b4 = 0; b4 < 4; ++b4)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float ks_ = SCALED ? acc[4 * b4 + e] : ek[4 * tm + b4][e] * acc[4 * b4 + e];
          // (training form: selected, not multiplied away, so that a v that is not finite stays out of M' and with it out
          // of the gradients of the tokens before it; so with SKIP_M, where it would reach M, and through M the other value
          // columns behind the segment, only as long as M lives on)
          const float v_ = SKIP_M ? (__is_same(OT, __bf16) ? 1.0f : vmask) * op_elem_keep<OT>(vv[4 * tm + b4], e, vkeep)
                           : KEEP ? (is_m ? 0.0f : (float)vv[4 * tm + b4][e])
                                  : vmask * (float)vv[4 * tm + b4][e];
          acc[4 * b4 + e] = be[4 * tm + b4][e] * (v_ - ks_);
        }
      Rb[2 * tm + 0] = acc_to_op<OT>(acc, 0);
      Rb[2 * tm + 1] = acc_to_op<OT>(acc, 8);
    }
    lds_fence();
    // batch for stage 3: K^T fragments (transposing reads of the row-major k tile) and the decay factors
#pragma unroll
    for (int km = 0; km < KT / 32; ++km)
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) fk[km * 4 + ks] = op_ld_kappa_tr<OT, SWZ>(tl.kd, SK, 32 * km, 16 * ks, lane);
    f32x4 dk[8];
    if constexpr (!SCALED) {
#pragma unroll
      for (int t8 = 0; t8 < 8; ++t8) dk[t8] = *reinterpret_cast<const f32x4*>(&tl.dk[8 * t8 + 4 * hh]);
    }
    const float dec = tl.misc[0];
    X8 Vb[4], Vsb[4];
#pragma unroll
    for (int tm = 0; tm < 2; ++tm) {  // v_new = T R (T is lower triangular: tile tm needs 2 (tm + 1) steps)
      f32x16 acc = zero16();
#pragma unroll
      for (int ks = 0; ks < 2 * (tm + 1); ++ks) acc = mfma32(ft[2 * tm + ks], Rb[ks], acc);
      Vb[2 * tm + 0] = acc_to_op<OT>(acc, 0);
      Vb[2 * tm + 1] = acc_to_op<OT>(acc, 8);
      if constexpr (!SCALED) {
#pragma unroll
        for (int b4 = 0; b4 < 4; ++b4)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[4 * b4 + e] *= dk[4 * tm + b4][e];
        Vsb[2 * tm + 0] = acc_to_op<OT>(acc, 0);
        Vsb[2 * tm + 1] = acc_to_op<OT>(acc, 8);
      } else {  // (the decay factors are in the kd tile)
        Vsb[2 * tm + 0] = Vb[2 * tm + 0];
        Vsb[2 * tm + 1] = Vb[2 * tm + 1];
      }
    }
    lds_fence();
    lds_barrier();  // B(c): every operand that comes from the k, v and T tiles of chunk c is in registers
    dtot *= dec;
    float qs0 = 0.0f, qs1 = 0.0f;
    if constexpr (EARLY_Q) {  // batch: Q rows, P fragments, output factors (in flight during the state update)
#pragma unroll
      for (int tm = 0; tm < 2; ++tm)
#pragma unroll
        for (int ks = 0; ks < KT / 16; ++ks) fq[tm * (KT / 16) + ks] = SWZ ? op_ld_kappa_swz<OT>(s_q, SK, 32 * tm + ln, 16 * ks, hh)
                                        : op_ld_kappa<OT>(s_q, SK, 32 * tm + ln, 16 * ks, hh);
#pragma unroll
      for (int f = 0; f < 6; ++f) ft[f] = op_frag_load<OT>(s_P, f, lane);
      qs0 = s_qs[ln];
      qs1 = s_qs[32 + ln];
    }
#pragma unroll
    for (int km = 0; km < KT / 32; ++km) {  // S <- dec S + K^T (dk v_new)
#pragma unroll
      for (int r = 0; r < 16; ++r) S[km][r] *= dec;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) S[km] = mfma32(fk[km * 4 + ks], Vsb[ks], S[km]);
    }
    if constexpr (SKIP_M) {
      // Columns of M that have become zero stay zero, whatever chunks follow: a wave whose columns all have only takes part
      // in the barriers from there on and leaves the LDS and the matrix cores, which bound this pass at the wide heads, to
      // the columns of N. The result is the same to the bit (a k, g or beta of a later chunk that is not finite reaches
      // every column of N, and through N what comes after the segment; a v, its own column of N alone). With decays of e^-0.8
      // a token a segment's M has left the fp32 range after three chunks, with e^-0.24 after eight, with e^-0.04 after 47;
      // looked at only once the decays' own product has. 16 packed events of 520 000 tokens, 8 x 128 x 128, e^-0.8: pass
      // 890 -> 691 us, call 2 166 -> 2 000. Where M lives on, calls of 25 080 tokens x 5 heads take 0.6 us less (64 x 128) to
      // 1 us more (128 x 64, of 98: other registers; as a branch of which the compiler does not know that the whole wave takes
      // it, 2 us). Heads up to 64 x 64 are bound by the chain of a chunk and gain nothing.
      faded |= uniform(__float_as_int(dtot)) == 0;
      if (uniform(is_m) && faded) gone = m_is_zero();
    }
    if constexpr (PASS_B) {
      if constexpr (!EARLY_Q) {  // batch: Q rows, P fragments, output factors
#pragma unroll
        for (int tm = 0; tm < 2; ++tm)
#pragma unroll
          for (int ks = 0; ks < KT / 16; ++ks) fk[tm * (KT / 16) + ks] = SWZ ? op_ld_kappa_swz<OT>(s_q, SK, 32 * tm + ln, 16 * ks, hh)
                                          : op_ld_kappa<OT>(s_q, SK, 32 * tm + ln, 16 * ks, hh);
#pragma unroll
        for (int f = 0; f < 6; ++f) ft[f] = op_frag_load<OT>(s_P, f, lane);
        qs0 = s_qs[ln];  // scale e^{gamma_i} rq_i of this lane's token in either row tile
        qs1 = s_qs[32 + ln];
      }
      lds_fence();
      lds_barrier();  // C(c): the q and P operands of chunk c are in registers
      if constexpr (EARLY_K) load_k_rows(tiles((c + 1 - c0) & 1));  // (after the last chunk: read and dropped)
      // o^T = S_old^T (qs Q)^T + v_new^T P^T: the state and v_new, which this wave holds in accumulator layout (lane =
      // value column), are read as the A operands (operand row = value column), the Q and P fragments as the B
      // operands (operand column = token). The result tile has the TOKEN in the lane and 16 value columns (four runs
      // of four) in the registers, so the token's factor is one scalar per lane and a run packs into one 8-byte piece
      // of the token's row without any exchange between lanes. The slab goes to this wave's own part of the o tile
      // and from there to HBM in 16-byte pieces.
#pragma unroll
      for (int tm = 0; tm < 2; ++tm) {
        f32x16 a1 = zero16(), a2 = zero16();
#pragma unroll
        for (int ks = 0; ks < KT / 16; ++ks) a1 = mfma32(Sb[ks], (EARLY_Q ? fq : fk)[tm * (KT / 16) + ks], a1);
#pragma unroll
        for (int ks = 0; ks < 2 * (tm + 1); ++ks) a2 = mfma32(Vb[ks], ft[2 * tm + ks], a2);
        const float qsv = tm ? qs1 : qs0;
        typedef T T4 __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int b4 = 0; b4 < 4; ++b4) {
          T4 pk;
#pragma unroll
          for (int e = 0; e < 4; ++e) pk[e] = GdrElem<T>::from_float(__builtin_fmaf(qsv, a1[4 * b4 + e], a2[4 * b4 + e]));
          *reinterpret_cast<T4*>(&s_o[(32 * tm + ln) * SV + 32 * vslab + 8 * b4 + 4 * hh]) = pk;
        }
      }
      if constexpr (!STAGER_FLUSH) {
        lds_fence();
        const int tok0 = o_tok0, len = o_len;
        T* ob = o + ((size_t)tok0 * HV + hv) * VT;  // uniform base; per-lane 32-bit offsets below
        const int rs = HV * VT;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int piece = lane + 64 * j, row = piece >> 2, part = piece & 3;
          const uint4 val = *reinterpret_cast<const uint4*>(&s_o[row * SV + 32 * vslab + 8 * part]);
          // o is written once and not read again by this pipeline: a non-temporal store keeps it from pushing the
          // tiles and composites out of the L2 (layer 136.6 -> 132.9 us; the same hint on the loads of q, k, v costs
          // 10 - 30 us, on the records' stores it changes nothing)
          typedef unsigned int nt_u32x4 __attribute__((ext_vector_type(4)));
          nt_u32x4 nv;
          nv[0] = val.x; nv[1] = val.y; nv[2] = val.z; nv[3] = val.w;
          if (row < len) __builtin_nontemporal_store(nv, reinterpret_cast<nt_u32x4*>(ob + row * rs + 32 * vslab + 8 * part));
        }
      }
      o_tok0 = n_tok0;
      o_len = n_len;
    }
  }

  if constexpr (STAGER_FLUSH) {
    if (nc > 0) lds_barrier();  // the o tile of the last chunk is complete (the stagers write it out)
  }
  if constexpr (SKIP_M) {
    for (; c < c1; ++c) lds_barrier();  // B(c)
  } else if constexpr (CUTS) {
    faded = uniform(__float_as_int(dtot)) == 0;
  }
  // epilogue; the opaque zero keeps the compiler from computing all these addresses before the loop
  int late = 0;
  asm volatile("" : "+v"(late));
  if constexpr (CUTS) {
    // A segment whose M is zero and whose N is finite hands N on whatever finite state it starts from: its decay is
    // stored as -0 (gdr_d_cut), which those who walk the composites look for. Every wave notes what it knows of its own
    // columns, wave 0 stores the decay. Looked at only where the decays' product has left the fp32 range, which all chain
    // waves see at the same chunk; the stagers may have ended, a barrier does not wait for waves that have. (With a note and
    // a barrier in every segment, 9 000 tokens x 6 x 128 x 128 where none does: pass 25.0 us; so 23.9, without any look 23.7.)
    if (faded) {
      float probe = 0.0f;  // 0 x every entry: NaN unless all are finite
#pragma unroll
      for (int km = 0; km < KT / 32; ++km)
#pragma unroll
        for (int r = 0; r < 16; ++r) probe = __builtin_fmaf(S[km][r], 0.0f, probe);
      const bool fine = is_m ? gone || m_is_zero() : __ballot(!(probe == 0.0f)) == 0;
      float* note = tiles(0).misc + 8;
      if (lane == 0) note[wave] = fine ? 0.0f : 1.0f;
      lds_barrier();
      if (wave == 0) {
        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < NSLAB; ++w) sum += note[w];
        if (sum == 0.0f) dtot = -0.0f;
      }
    }
  }
  if constexpr (PASS_B) {
    if (ht && (flags & SEG_LAST)) {
      const int seq = pv.seg_seq[seg];
      float* out = ht + ((size_t)seq * HV + hv) * KT * VT + late;
#pragma unroll
      for (int km = 0; km < KT / 32; ++km)
#pragma unroll
        for (int r = 0; r < 16; ++r) out[(32 * km + acc_row(r, hh)) * VT + col] = S[km][r];
    }
  } else if (is_m) {
    // M = dtot I + M': M' as bf16 A-operand fragments (rows = state rows, contraction over the columns in
    // accumulator slot order), element (row, col) -> fragment (row/32, col/16), lane 32*hh' + row%32, slot s
    // (a piece's M' is kept as pairs of value and remainder: gdr_scan2_kernel<PIECES>)
    unsigned char* out = Mcomp + ((size_t)map * HV + hv) * (KT * KT * 2) + late;
    if constexpr (PIECES) out += gmax > 0 ? ((size_t)map * HV + hv) * (KT * KT * 2) : 0;
    const int mcol = 32 * wave + ln, ks = mcol >> 4, c16 = mcol & 15;
    const int hs = (c16 >> 2) & 1, slot = 4 * (c16 >> 3) + (c16 & 3);
#pragma unroll
    for (int km = 0; km < KT / 32; ++km)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = 32 * km + acc_row(r, hh);
        const float val = S[km][r] - (row == mcol ? dtot : 0.0f);
        if constexpr (PIECES) {
          const size_t at = (size_t)((km * (KT / 16) + ks) * 64 + 32 * hs + (row & 31)) * 8 + slot;
          if (gmax > 0) {
            typename OpVec<OT>::x2 pair;
            pair[0] = (OT)val;
            pair[1] = (OT)(val - (float)pair[0]);
            reinterpret_cast<typename OpVec<OT>::x2*>(out)[at] = pair;
          } else {
            reinterpret_cast<OT*>(out)[at] = (OT)val;
          }
        } else {
          *reinterpret_cast<OT*>(out + ((size_t)((km * (KT / 16) + ks) * 64 + 32 * hs + (row & 31))) * 16 + 2 * slot) =
              (OT)val;
        }
      }
    if (wave == 0 && lane == 0) Dcomp[(size_t)map * HV + hv] = dtot;
    if constexpr (KEEP) {  // accumulator tiles read as A operand are the transpose
      unsigned char* mt = keep + ((size_t)seg * HV + hv) * (KT * KT * 2);
#pragma unroll
      for (int km = 0; km < KT / 32; ++km) {
        f32x16 m = S[km];
#pragma unroll
        for (int r = 0; r < 16; ++r) m[r] -= (32 * km + acc_row(r, hh) == mcol) ? dtot : 0.0f;
        op_frag_store<OT>(mt, wave * (KT / 16) + 2 * km + 0, lane, acc_to_op<OT>(m, 0));
        op_frag_store<OT>(mt, wave * (KT / 16) + 2 * km + 1, lane, acc_to_op<OT>(m, 8));
      }
    }
  } else {
    // N slab in accumulator order: tile (vslab, km), plane q (registers 4q..4q+3), lane -> 16 bytes
    unsigned char* out = Ncomp + (((size_t)map * HV + hv) * (VT / 32) + vslab) * (KT * 32 * 4) + late;
#pragma unroll
    for (int km = 0; km < KT / 32; ++km)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        f32x4 t;
#pragma unroll
        for (int e = 0; e < 4; ++e) t[e] = S[km][4 * q4 + e];
        reinterpret_cast<f32x4*>(out)[(km * 4 + q4) * 64 + lane] = t;
      }
  }
  }  // (the 32-column chain wave)
#undef GDR_Q_BUFFERS
