// Body of dQ, taken in by its kernel, by the one that runs it beside dK/dV and by the function of that name in attn.hip.  (Text, because as an inlined function
// it takes four registers and 7 % more time, 2 x 4096, 32 heads 965 -> 1016 us a backward pass: the mask of each score becomes a compare and a select that every tile pays, here a branch around it.  With the soft-cap at head_dim 128 the function takes 18 registers
// less, which the launch of both needs; by itself it would be 1 % faster on some lengths and 1 % slower on others, 2 x 4096, 32/16 heads 1144 -> 1128, 2 x 1777, 32/8 heads 267 -> 269.)
// Expects the kernel's arguments, smem, and the workgroup's id among nwg; DELTA may be null.
  constexpr int TILE = 64 * D * 2;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform for the compiler too
  const int l32 = lane & 31, lhi = lane >> 5;
  const int qw = wave % QW, ks = wave / QW;
  constexpr int QR = QW * 32;         // queries of the workgroup
  constexpr int TEAMS = QW * KS / 4;  // tiles are fetched by teams of 4 waves
  const int nqt = (S + QR - 1) / QR;
  const WgCoord wg = decode_wg(id, (int)(nwg / (nqt * (H / KH))), H / KH);
  const int qt = nqt - 1 - wg.rank;  // longest rows first
  const int b = wg.group / KH, kh = wg.group % KH;
  const int h = kh * (H / KH) + wg.r;
  const int i0 = qt * QR;
  const int iw0 = i0 + qw * 32;
  const int qi = iw0 + l32;
  const int qic = min(qi, S - 1);

  bf16x8 qf[D / 16], dof[D / 16];
  // delta[b,h,i] = sum_d dO[i,h,d] * O[i,h,d]: the two lanes of a query each hold half of its dO
  // row already, so the row sum costs one pass over O here; it is also written out (DELTA) for a
  // dK/dV kernel that runs after this one.  In one launch dK/dV forms its own and DELTA is null.
  float dlt = 0.f;
  {
    const bf16* qp = Q + ((int64_t)b * S + qic) * ldq + h * D + lhi * 8;
    const bf16* dp = dO + ((int64_t)b * S + qic) * lddo + h * D + lhi * 8;
    const bf16* op = O + ((int64_t)b * S + qic) * ldo + h * D + lhi * 8;
#pragma unroll
    for (int s = 0; s < D / 16; s++) {
      qf[s] = *reinterpret_cast<const bf16x8*>(qp + s * 16);
      dof[s] = *reinterpret_cast<const bf16x8*>(dp + s * 16);
      const bf16x8 of = *reinterpret_cast<const bf16x8*>(op + s * 16);
#pragma unroll
      for (int e = 0; e < 8; e++) dlt += bf2f(of[e]) * bf2f(dof[s][e]);
    }
  }
  dlt = half_swap_sum(dlt);
  // stored NEGATED: the dK/dV kernel starts its dP accumulators from it, so that dP - delta
  // comes out of the MFMAs and costs that kernel no subtraction
  if (DELTA && lhi == 0 && ks == 0 && qi < S) DELTA[((int64_t)b * H + h) * S + qi] = -dlt;
  const float lse2 = LSE[((int64_t)b * H + h) * S + qic] * LOG2E;
  const int j_lo = window >= 0 ? max(0, i0 - window) : 0;
  const int t_lo = j_lo >> 6;
  const int t_hi = min(i0 + QR - 1, S - 1) >> 6;

  f32x16 dq[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
    for (int r = 0; r < 16; r++) dq[dt][r] = 0.f;

  const bf16* kbase = K + (int64_t)b * S * ldk + kh * D;
  const bf16* vbase = V + (int64_t)b * S * ldv + kh * D;
  const unsigned lds0 = lds_addr_of(smem);
  const int wv = wave & 3, team = wave >> 2;
  TileDma<64, D> dk, dv;
  dk.init(ldk, wv, lane);
  dv.init(ldv, wv, lane);
  // K/V tiles of round r: tile t_lo + r KS + g for key group g
  auto load_kv = [&](int round, int stage) {
#pragma unroll
    for (int g0 = 0; g0 < KS / TEAMS; g0++) {
      const int g = g0 * TEAMS + team, t = t_lo + round * KS + g;
      if (KS > 1 && t > t_hi) break;
      const unsigned dst = lds0 + (g * 2 + stage) * (2 * TILE);
      if (t * 64 + 64 <= S) {
        dk.issue(kbase + (int64_t)t * 64 * ldk, dst, wv);
        dv.issue(vbase + (int64_t)t * 64 * ldv, dst + TILE, wv);
      } else {
        dma_tile<64, D>(kbase, ldk, t * 64, S, dst, wv, lane);
        dma_tile<64, D>(vbase, ldv, t * 64, S, dst + TILE, wv, lane);
      }
    }
  };
  const float sc2 = scale * LOG2E;
  const float cap_c1 = CAP ? 2.f * sc2 / cap : 0.f, cap_l2 = cap * LOG2E;  // soft-cap: see cap_tanh

  FragAddr<D, CAP && D == 128> fa;  // the soft-cap variant is the one short of registers
  fa.init(lane);

  load_kv(0, 0);
  dma_wait_all();
  __syncthreads();
  const int rounds = (t_hi - t_lo + KS) / KS;
  for (int r0 = 0; r0 < rounds; r0++) {
    const int cur = r0 & 1;
    if (r0 + 1 < rounds) load_kv(r0 + 1, cur ^ 1);
    const int t = t_lo + r0 * KS + ks, j0 = t * 64;
    const bool visible = (KS == 1 || t <= t_hi) && (j0 <= iw0 + 31) && (window < 0 || j0 + 63 >= iw0 - window);
    if (visible) {
      const unsigned char* sk = smem + (ks * 2 + cur) * (2 * TILE);
      const unsigned char* sv = sk + TILE;
      const bool need_mask = (j0 + 63 > iw0) || (window >= 0 && j0 < iw0 + 31 - window);
      // dS of one 32-key half from its scores and dP, packed as the B operand of the dQ product
      bf16x8 dsb[4];
      auto finish_half = [&](int jt, f32x16& sj, const f32x16& dpj) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
          float s = sj[r], chain = 1.f, p;
          if (CAP) {
            const float th = cap_tanh_of<D>(s, cap_c1, scale, cap);
            p = fexp2(__builtin_fmaf(th, cap_l2, -lse2));
            chain = 1.f - th * th;
          } else {
            p = fexp2(__builtin_fmaf(s, sc2, -lse2));
          }
          if (need_mask) {
            const int j = j0 + jt * 32 + (r >> 2) * 8 + lhi * 4 + (r & 3);
            const bool ok = (j <= qi) && (window < 0 || j >= qi - window);
            p = ok ? p : 0.f;
          }
          sj[r] = p * (dpj[r] - dlt) * chain;
        }
        dsb[2 * jt] = pack_bf16x8(sj, 0);
        dsb[2 * jt + 1] = pack_bf16x8(sj, 8);
      };
      f32x16 st[2], dpt[2];
#pragma unroll
      for (int jt = 0; jt < 2; jt++) {
#pragma unroll
        for (int r = 0; r < 16; r++) { st[jt][r] = 0.f; dpt[jt][r] = 0.f; }
#pragma unroll
        for (int s = 0; s < D / 16; s++) {
          st[jt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa.load_kc(sk, jt * 32, s), qf[s], st[jt], 0, 0, 0);
          dpt[jt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa.load_kc(sv, jt * 32, s), dof[s], dpt[jt], 0, 0, 0);
        }
        // with the soft-cap's extra temporaries both halves do not fit the register file at once:
        // finish each half before the next one's products start
        if (CAP) finish_half(jt, st[jt], dpt[jt]);
      }
      if (!CAP) {
#pragma unroll
        for (int jt = 0; jt < 2; jt++) finish_half(jt, st[jt], dpt[jt]);
      }
#pragma unroll
      for (int u = 0; u < 4; u++)
#pragma unroll
        for (int dt = 0; dt < D / 32; dt++)
          dq[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa.load_tr(sk, u * 16, dt), dsb[u], dq[dt], 0, 0, 0);
    }
    dma_wait_all();
    __syncthreads();
  }
  float zeros = 0.f;  // see redo_rows
  auto store4 = [&](int dt, int g, const f32x4& v) {
    bf16* op = dQ + ((int64_t)b * S + qic) * lddq + h * D;
    Pack4 pk;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const float x = v[e] * scale;
      if (D == 64) zeros = __builtin_fmaf(x, 0.f, zeros);
      pk.e[e] = f2bf(x);
    }
    *reinterpret_cast<u32x2*>(op + dt * 32 + g * 8 + lhi * 4) = pk.u;
  };
  if constexpr (KS == 1) {
    if (qi < S) {
#pragma unroll
      for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
        for (int g = 0; g < 4; g++) store4(dt, g, f32x4{dq[dt][g * 4], dq[dt][g * 4 + 1], dq[dt][g * 4 + 2], dq[dt][g * 4 + 3]});
    }
  } else {
    add_partials<D, KS>(smem, dq, qw, ks, lane, [&](int u, const f32x4& v) {
      if (qi < S) store4(u >> 2, u & 3, v);
    });
  }
  if constexpr (D == 64)
    redo_rows(zeros, [&](int r) {
      const int64_t at = (int64_t)b * S + iw0 + r;
      redo_dq<CAP>(Q + at * ldq + h * D, kbase, ldk, vbase, ldv, O + at * ldo + h * D, dO + at * lddo + h * D, LSE[((int64_t)b * H + h) * S + iw0 + r],
                   dQ + at * lddq + h * D, iw0 + r, window, scale, cap, lane, ks * (D / KS), (ks + 1) * (D / KS));
    });
