// What a workgroup of decode.hip does once its record is there: part of decode_kernel's body, which includes it with XI, the number of
// token rows per lane group, as a constant (it has no guard and stands alone nowhere).
  // ---- round trip 2: issue every load ---------------------------------------------------------
  const int nks = K / 32;  // k-steps of the contraction
  const int ks0 = KSPW > 0 ? wave * KSPW : wave * nks / kNW;
  const int ks1 = KSPW > 0 ? ks0 + KSPW : (wave + 1) * nks / kNW;
  Pack8 xa[CH], aw[RB][CH];
  i32x4 xst[TR ? 4 * ROUNDS : 1], ast[TR ? RB : 1][TR ? 4 * ROUNDS : 1];
  if constexpr (TR) {
    // row-contiguous: lane = (row group lane/16, 16-byte chunk lane%16 of a 256-byte K range);
    // one such range (four k-steps) per round
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
      const int64_t koff = static_cast<int64_t>(ks0 + 4 * r) * 32 + (lane & 15) * 8;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (i < XI) xst[4 * r + i] = load128(static_cast<const T*>(xv) + static_cast<int64_t>(rows4[i]) * xs + koff);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
          const int rr = rb * 16 + 4 * lg + i;
          if (!MASKED || RB == 1 || rb < rb_n) ast[rb][4 * r + i] = load128(A + static_cast<int64_t>(rr < rbuf ? rr : rbuf - 1) * K + koff);
          else ast[rb][4 * r + i] = i32x4{0, 0, 0, 0};
        }
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int ks = ks0 + i;
      if (KSPW > 0 || ks < ks1) {
        xa[i].raw = load128(xrow + ks * 32);  // absent tokens read row 0; their results are never stored
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) aw[rb][i].raw = load128(arow[rb] + ks * 32);
      }
    }
  }
  if constexpr (URGENT) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
  }
  constexpr int kSpansAhead = SA;
  Pack8 bop[kSpansAhead][4][KSTEPS], yreg[kSpansAhead][2];
  uint2 yq[TR ? kSpansAhead : 1][TR ? 4 : 1];  // TR: four columns of four tokens per lane and span
  T* const ycols = static_cast<T*>(yv_) + sp.y_col;
  // TR span: MFMA j takes column c0 + 4 * (lane % 16) + j, so a lane ends up with four consecutive
  // columns of tokens 4 * (lane / 16) .. + 3
  constexpr bool K16 = TR && R == 16;  // expand on the 16x16x16 MFMA: 64-bit operand pieces
  auto load_span_tr = [&](int c0, Pack8(&bo)[4][KSTEPS], uint2(&yy)[4]) {
    if constexpr (K16) {
      // A span's 64 B rows of 32 bytes are 2 KB of contiguous memory: fetched as such (lane l takes
      // 16 bytes of row c0 + l / 2 and of row c0 + 32 + l / 2, eight cache lines per instruction
      // instead of sixteen quarter-used ones); finish_span_tr turns them into operand pieces.
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        int n = c0 + 32 * h + (lane >> 1);
        n = n < sp.n1 ? n : sp.n1 - 1;
        bo[h][0].raw = load128(B + static_cast<int64_t>(n) * R + (lane & 1) * 8);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        int n = c0 + 4 * lr + j;
        n = n < sp.n1 ? n : sp.n1 - 1;
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) {
          int kc = (lg + 4 * ks) & (R / 8 - 1);
          if (GR && kc * 8 >= rbuf) kc = rbuf / 8 - 1;  // (masked where it is used)
          bo[j][ks].raw = load128(B + static_cast<int64_t>(n) * rbuf + kc * 8);
        }
      }
    }
    const int c = c0 + 4 * lr < sp.n1 ? c0 + 4 * lr : sp.n1 - 4;
#pragma unroll
    for (int i = 0; i < XI; ++i) yy[i] = *reinterpret_cast<const uint2*>(ycols + static_cast<int64_t>(rows4[i]) * ys + c);
  };
#pragma unroll
  for (int s = 0; s < kSpansAhead; ++s) {
    const int c0 = sp.n0 + (wave + s * kNW) * 64;
    if constexpr (TR) {
      // requested whether the span exists or not (the addresses of one that does not are clamped
      // into the range: a cache line or two, never stored): values that are requested in a branch
      // and used in a later one are unpacked by the compiler where they are requested, and the
      // wavefront then waits for them before it has requested anything else
      load_span_tr(c0, bop[s], yq[s]);
    } else if (c0 < sp.n1) {
      {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          int n = c0 + 16 * (lr >> 2) + 4 * j + (lr & 3);
          n = n < sp.n1 ? n : sp.n1 - 1;
#pragma unroll
          for (int ks = 0; ks < KSTEPS; ++ks) {
            // lanes whose chunk lies beyond the rank fetch a valid chunk anyway: their H operand is
            // zero, and an unconditional load keeps the whole batch of loads in flight together
            int kc = (lg + 4 * ks) & (R / 8 - 1);
            if (GR && kc * 8 >= rbuf) kc = rbuf / 8 - 1;  // (masked where it is used)
            bop[s][j][ks].raw = load128(B + static_cast<int64_t>(n) * rbuf + kc * 8);
          }
        }
#pragma unroll
        for (int half = 0; half < 2; ++half)
          if (live && c0 + 16 * lg + 8 * half < sp.n1) yreg[s][half].raw = load128(yrow + c0 + 8 * half);
      }
    }
  }

  MLORA_STAMP(2);  // every load is issued
  // ---- shrink: H[token, rank] partial over this wavefront's K range ----------------------------
  f32x4 acc[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) acc[rb] = f32x4{0.f, 0.f, 0.f, 0.f};
  if constexpr (TR) {
    // through the wavefront's LDS block: written row-contiguously, read in operand layout
    // (k-step i of lane group g is chunk 4 * i + g, the same elements the direct loads take)
    i32x4* stage = s_stage + wave * (1 + SB) * 16 * kStageRow;
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
#pragma unroll
      for (int i = 0; i < XI; ++i) stage[(4 * lg + i) * kStageRow + (lane & 15)] = xst[4 * r + i];
#pragma unroll
      for (int p = 0; p < RB / SB; ++p) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
          for (int sb = 0; sb < SB; ++sb) stage[((1 + sb) * 16 + 4 * lg + i) * kStageRow + (lane & 15)] = ast[p * SB + sb][4 * r + i];
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (p == 0) xa[i].raw = stage[lr * kStageRow + 4 * i + lg];
#pragma unroll
          for (int sb = 0; sb < SB; ++sb) aw[p * SB + sb][i].raw = stage[((1 + sb) * 16 + lr) * kStageRow + 4 * i + lg];
        }
        __builtin_amdgcn_wave_barrier();  // the block is rewritten by the next pass or round (and later by the expand)
      }
      // this round's k-steps, in ascending order as the direct form takes them
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) acc[rb] = Mma<T>::run(xa[i], aw[rb][i], acc[rb]);
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      if (KSPW > 0 || ks0 + i < ks1) {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) acc[rb] = Mma<T>::run(xa[i], aw[rb][i], acc[rb]);
      }
    }
  }
  if (KSPW == 0) {
    for (int ksb = ks0 + CH; ksb < ks1; ksb += CH) {  // K not known at compile time: further batches
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        const int ks = ksb + i;
        if (ks < ks1) {
          xa[i].raw = load128(xrow + ks * 32);
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) aw[rb][i].raw = load128(arow[rb] + ks * 32);
        }
      }
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        if (ksb + i < ks1) {
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) acc[rb] = Mma<T>::run(xa[i], aw[rb][i], acc[rb]);
        }
      }
    }
  }

  // Sum the K-partials of the wavefronts.  D layout: lane holds H[token 4*(lane/16)+i][rank lane%16].
  if constexpr (KSPW == 0) mfma_settle(acc);  // k-steps past the end of K were skipped by branches
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) *reinterpret_cast<f32x4*>(&s_red[((wave * RB + rb) * 64 + lane) * 4]) = acc[rb];
  MLORA_STAMP(3);  // wavefront 0: x and A arrived, staged and multiplied
  __syncthreads();
  MLORA_STAMP(4);  // every wavefront's partial is in LDS
  for (int e = tid; e < RB * 256; e += NT) {
    const int rb = e >> 8, ln = (e & 255) >> 2, i = e & 3;
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < kNW; ++w) sum += s_red[((w * RB + rb) * 64 + ln) * 4 + i];
    const int tok = 4 * (ln >> 4) + i, r = rb * 16 + (ln & 15);
    if (r < R) {
      const float v = (!MASKED || r < eff) ? sum * scaling : 0.f;  // ranks the adapter does not have contribute nothing
      const T hi = from_f32<T>(v);
      s_hi[tok * HSTRIDE + r] = hi;
      s_lo[tok * HSTRIDE + r] = from_f32<T>(v - to_f32(hi));
    }
  }
  __syncthreads();
  MLORA_STAMP(5);  // the intermediate is in LDS

  // ---- expand ---------------------------------------------------------------------------------
  Pack8 hop[KSTEPS], hlo[KSTEPS];
#pragma unroll
  for (int ks = 0; ks < KSTEPS; ++ks) {
    const int kc = lg + 4 * ks;
    if (kc * 8 < R) {
      hop[ks].raw = load128(&s_hi[lr * HSTRIDE + kc * 8]);
      hlo[ks].raw = load128(&s_lo[lr * HSTRIDE + kc * 8]);
    } else {
      hop[ks].raw = i32x4{0, 0, 0, 0};
      hlo[ks].raw = i32x4{0, 0, 0, 0};
    }
  }

  // Ranks at or above the adapter's are cleared in the B operands where they are used, not where
  // they were requested: cleared at the request, every load is waited for on the spot.
  auto mask_b = [&](Pack8(&bo)[4][KSTEPS]) {
    if (MASKED && eff < R) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) mask_ranks(bo[j][ks], ((lg + 4 * ks) & (R / 8 - 1)) * 8, eff);
    }
  };
  auto finish_span = [&](int c0, Pack8(&bo)[4][KSTEPS], Pack8(&yy)[2]) {
    f32x4 out[4];
    mask_b(bo);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      out[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) {
        out[j] = Mma<T>::run(bo[j][ks], hlo[ks], out[j]);
        out[j] = Mma<T>::run(bo[j][ks], hop[ks], out[j]);
      }
    }
    if (live) {
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        if (c0 + 16 * lg + 8 * half < sp.n1) {
          float yf[8];
          unpack8<T>(yy[half], yf);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            yf[i] += out[2 * half][i];
            yf[4 + i] += out[2 * half + 1][i];
          }
          Pack8 r;
          pack8<T>(yf, r);
          store128(yrow + c0 + 8 * half, r.raw);
        }
      }
    }
  };
  // tokens as MFMA rows: lane holds out[row 4 * lg + i][column c0 + 4 * lr + j]
  uint2 hop16 = {0, 0}, hlo16 = {0, 0};
  if constexpr (K16) {
    hop16 = *reinterpret_cast<const uint2*>(&s_hi[lr * HSTRIDE + 4 * lg]);
    hlo16 = *reinterpret_cast<const uint2*>(&s_lo[lr * HSTRIDE + 4 * lg]);
  }
  auto finish_span_tr = [&](int c0, Pack8(&bo)[4][KSTEPS], uint2(&yy)[4]) {
    f32x4 out[4];
    uint2 pieces[4];
    if constexpr (K16) {
      if (MASKED && eff < R) {
        mask_ranks(bo[0][0], (lane & 1) * 8, eff);
        mask_ranks(bo[1][0], (lane & 1) * 8, eff);
      }
      // B rows -> operand pieces through the wavefront's LDS block: four rows (128 bytes) per
      // group, groups 144 bytes apart so that the sixteen lanes of a piece read hit every bank
      // once.  MFMA j of lane (lr, lg) takes ranks 4*lg .. 4*lg+3 of column c0 + 4*lr + j.
      char* blk = reinterpret_cast<char*>(s_stage + wave * (1 + SB) * 16 * kStageRow);
      *reinterpret_cast<i32x4*>(blk + (lane >> 3) * 144 + (lane & 7) * 16) = bo[0][0].raw;
      *reinterpret_cast<i32x4*>(blk + ((lane >> 3) + 8) * 144 + (lane & 7) * 16) = bo[1][0].raw;
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int j = 0; j < 4; ++j) pieces[j] = *reinterpret_cast<const uint2*>(blk + lr * 144 + j * 32 + lg * 8);
      __builtin_amdgcn_wave_barrier();
    } else {
      mask_b(bo);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      out[j] = f32x4{0.f, 0.f, 0.f, 0.f};
      if constexpr (K16) {
        const uint2 piece = pieces[j];
        out[j] = Mma16<T>::run(hlo16, piece, out[j]);
        out[j] = Mma16<T>::run(hop16, piece, out[j]);
      } else {
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) {
          out[j] = Mma<T>::run(hlo[ks], bo[j][ks], out[j]);
          out[j] = Mma<T>::run(hop[ks], bo[j][ks], out[j]);
        }
      }
    }
    const int c = c0 + 4 * lr;
    // (the y values are taken as they are only here: left to itself the compiler unpacks them
    // where they were requested, and the wavefront then waits for their arrival before it has
    // requested its other spans and before the shrink)
#pragma unroll
    for (int i = 0; i < XI; ++i) asm volatile("" : "+v"(yy[i].x), "+v"(yy[i].y));
    if (c < sp.n1) {
#pragma unroll
      for (int i = 0; i < XI; ++i) {
        if ((SHORT ? lg + 4 * i : 4 * lg + i) < m) {
          union { uint2 raw; T e[4]; } v;
          v.raw = yy[i];
#pragma unroll
          for (int j = 0; j < 4; ++j) v.e[j] = from_f32<T>(to_f32(v.e[j]) + out[j][i]);
          T* const to = ycols + static_cast<int64_t>(rows4[i]) * ys + c;
          if constexpr (THROUGH) store_through(to, __builtin_bit_cast(u32x2, v.raw));
          else *reinterpret_cast<uint2*>(to) = v.raw;
        }
      }
    }
  };

#pragma unroll
  for (int s = 0; s < kSpansAhead; ++s) {
    const int c0 = sp.n0 + (wave + s * kNW) * 64;
    if (c0 < sp.n1) {
      if constexpr (TR) finish_span_tr(c0, bop[s], yq[s]);
      else finish_span(c0, bop[s], yreg[s]);
    }
  }
  MLORA_STAMP(6);  // wavefront 0: its first spans are multiplied and their stores issued
  for (int c0 = sp.n0 + (wave + kSpansAhead * kNW) * 64; c0 < sp.n1; c0 += kNW * 64) {  // wide ranges
    Pack8 bo[4][KSTEPS], yy[2];
    if constexpr (TR) {
      uint2 yt[4];
      load_span_tr(c0, bo, yt);
      finish_span_tr(c0, bo, yt);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        int n = c0 + 16 * (lr >> 2) + 4 * j + (lr & 3);
        n = n < sp.n1 ? n : sp.n1 - 1;
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) {
          int kc = (lg + 4 * ks) & (R / 8 - 1);
          if (GR && kc * 8 >= rbuf) kc = rbuf / 8 - 1;  // (masked where it is used)
          bo[j][ks].raw = load128(B + static_cast<int64_t>(n) * rbuf + kc * 8);
        }
      }
#pragma unroll
      for (int half = 0; half < 2; ++half)
        if (live && c0 + 16 * lg + 8 * half < sp.n1) yy[half].raw = load128(yrow + c0 + 8 * half);
      finish_span(c0, bo, yy);
    }
  }
#ifdef MLORA_TRACE
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  MLORA_STAMP(7);  // wavefront 0: its stores are acknowledged
  __syncthreads();
  MLORA_STAMP(8);  // every wavefront is done
#endif
