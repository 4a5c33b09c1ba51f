// What a workgroup of slot.hip does once its record is there: part of slot_tile's body, which includes it with XI, the number of token
// rows per lane group, as a constant (it has no guard and stands alone nowhere).
  // ---- the rows the record names --------------------------------------------------------------
  i32x4 xst[4 * ROUNDS];
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const int64_t koff = static_cast<int64_t>(ks0 + 4 * r) * 32 + (lane & 15) * 8;
#pragma unroll
    for (int i = 0; i < XI; ++i) xst[4 * r + i] = load128(static_cast<const T*>(xv) + static_cast<int64_t>(rows4[i]) * xs + koff);
  }
  if constexpr (URGENT) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
  }
  // (the B rows behind the x rows: they are not needed before the expand, and in front of the
  // record's wait they would hold the x rows up for as long as it takes to hand them over)
  request_b(slot);
  uint2 yq[SA][4];  // four columns of four tokens per lane and span
  T* const ycols = static_cast<T*>(yv_) + y_col;
  auto request_y = [&](int c0, uint2(&yy)[4]) {
    const int c = c0 + 4 * lr < sp.n1 ? c0 + 4 * lr : sp.n1 - 4;
#pragma unroll
    for (int i = 0; i < XI; ++i) yy[i] = *reinterpret_cast<const uint2*>(ycols + static_cast<int64_t>(rows4[i]) * ys + c);
  };
#pragma unroll
  for (int s = 0; s < SA; ++s) request_y(sp.n0 + (wave + s * NW) * 64, yq[s]);
  MLORA_STAMP(2);  // every load is issued

  // ---- shrink: H[token, rank] partial over this wavefront's K range ----------------------------
  i32x4* stage = s_stage + wave * (1 + SB) * 16 * kStageRow;
  // x rows and A rows, fetched row-contiguously, through the wavefront's LDS block into operand
  // layout, and multiplied: k-steps in ascending order
  auto stage_and_multiply = [&](const i32x4(&xs_)[4 * ROUNDS], const i32x4(&as_)[RB][4 * ROUNDS], f32x4(&acc)[RB], const bool clear_blocks) {
    Pack8 xa[4], aw[RB][4];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) acc[rb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
#pragma unroll
      for (int i = 0; i < XI; ++i) stage[(4 * lg + i) * kStageRow + (lane & 15)] = xs_[4 * r + i];
#pragma unroll
      for (int p = 0; p < RB / SB; ++p) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
          for (int sb = 0; sb < SB; ++sb) {
            i32x4 v = as_[p * SB + sb][4 * r + i];
            // rank blocks the adapter does not have were requested before its rank was known: they
            // never reach a multiplier
            if (MASKED && RB > 1 && clear_blocks && p * SB + sb >= rb_n) v = i32x4{0, 0, 0, 0};
            stage[((1 + sb) * 16 + 4 * lg + i) * kStageRow + (lane & 15)] = v;
          }
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
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) acc[rb] = Mma<T>::run(xa[i], aw[rb][i], acc[rb]);
      }
    }
  };
  // Sum of the wavefronts' partial tiles, wavefront 0 first: out[j] is word tid + j * NT.
  // D layout: lane holds H[token 4*(lane/16)+i][rank lane%16].
  auto sum_wavefronts = [&](const f32x4(&acc)[RB], float(&out)[EPT]) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) *reinterpret_cast<f32x4*>(&s_red[((wave * RB + rb) * 64 + lane) * 4]) = acc[rb];
    MLORA_STAMP(3);
    __syncthreads();
    MLORA_STAMP(4);
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
      const int e = tid + j * NT;
      float sum = 0.f;
      if (WORDS % NT == 0 || e < WORDS) {
        const int rb = e >> 8, ln = (e & 255) >> 2, i = e & 3;
#pragma unroll
        for (int w = 0; w < NW; ++w) sum += s_red[((w * RB + rb) * 64 + ln) * 4 + i];
      }
      out[j] = sum;
    }
  };
  f32x4 acc[RB];
  float total[EPT];
  if (KP > 1 && tid == 0) *s_ok = 1;  // (seen by everyone behind the barrier of the sum below)
  stage_and_multiply(xst, ast, acc, EARLY);
  sum_wavefronts(acc, total);

  if constexpr (KP > 1) {
    // ---- the other K parts: from the tile's other workgroups, or multiplied here -----------------
    u64* const xchg = reinterpret_cast<u64*>(reinterpret_cast<char*>(xc.ws) + kWsXchgOff) +
                      xc.tile * (KP * WORDS);  // the KP parts of this (tile, slice)
    float part[KP][EPT];
#pragma unroll
    for (int q = 0; q < KP; ++q)
#pragma unroll
      for (int j = 0; j < EPT; ++j) part[q][j] = 0.f;
    if (xok) {
#pragma unroll
      for (int j = 0; j < EPT; ++j) {
        const int e = tid + j * NT;
        if (WORDS % NT == 0 || e < WORDS)
          __hip_atomic_store(xchg + kp * WORDS + e, (static_cast<u64>(tag) << 32) | __float_as_uint(total[j]), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
    MLORA_STAMP(9);  // this workgroup's partial sums are on their way to the L2
    int ok = xok && xc.spin_ticks >= 0;
    if (ok) {
      const long long t0 = wall_clock64();
      for (;;) {
        // every part's words are requested together, this workgroup's own among them (a request
        // behind a test on the part number is a round trip of its own); its own are not looked at
        u64 w[KP][EPT];
#pragma unroll
        for (int q = 0; q < KP; ++q) {
#pragma unroll
          for (int j = 0; j < EPT; ++j) {
            const int e = (WORDS % NT == 0 || tid + j * NT < WORDS) ? tid + j * NT : 0;
            w[q][j] = __hip_atomic_load(xchg + q * WORDS + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
        }
        bool all = true;
#pragma unroll
        for (int q = 0; q < KP; ++q) {
#pragma unroll
          for (int j = 0; j < EPT; ++j) {
            const bool mine = !(WORDS % NT == 0 || tid + j * NT < WORDS) || q == kp;
            all &= mine | (static_cast<uint32_t>(w[q][j] >> 32) == tag);
            part[q][j] = __uint_as_float(static_cast<uint32_t>(w[q][j]));
          }
        }
        if (__builtin_amdgcn_ballot_w64(all) == __builtin_amdgcn_ballot_w64(true)) break;
        if (wall_clock64() - t0 >= xc.spin_ticks) { ok = 0; break; }
        __builtin_amdgcn_s_sleep(1);
      }
      if (!ok && xc.spin_ticks > 0 && lane == 0) atomicAdd(xc.ws + kWsTimeoutsWord, 1u);  // diagnostic: a wait ran out
    }
    MLORA_STAMP(10);  // the wait for the partners is over
    // one verdict for the workgroup (through a flag in LDS: the library's block-wide AND reads the
    // launch's shape from memory first, two trips); the barrier also ends the reading of s_red
    if (!ok) *s_ok = 0;
    __syncthreads();
    ok = *s_ok;
    if (!ok) {
      // every other part multiplied here as its own workgroup multiplies it
      for (int q = 0; q < KP; ++q) {
        if (q == kp) continue;
        i32x4 xo[4 * ROUNDS], ao[RB][4 * ROUNDS];
        const T* A = static_cast<const T*>(sp.a) + static_cast<int64_t>(slot) * rbuf * K;
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
          const int64_t koff = static_cast<int64_t>(q * (KPART / 32) + wave * KSPW + 4 * r) * 32 + (lane & 15) * 8;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if (i < XI) xo[4 * r + i] = load128(static_cast<const T*>(xv) + static_cast<int64_t>(rows4[i]) * xs + koff);
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
              const int rr = rb * 16 + 4 * lg + i;
              if (!MASKED || RB == 1 || rb < rb_n) ao[rb][4 * r + i] = load128(A + static_cast<int64_t>(rr < rbuf ? rr : rbuf - 1) * K + koff);
              else ao[rb][4 * r + i] = i32x4{0, 0, 0, 0};
            }
          }
        }
        f32x4 acc2[RB];
        float got[EPT];
        stage_and_multiply(xo, ao, acc2, false);
        sum_wavefronts(acc2, got);
        __syncthreads();  // s_red is rewritten by the next part
#pragma unroll
        for (int qq = 0; qq < KP; ++qq) {
          if (qq == q) {
#pragma unroll
            for (int j = 0; j < EPT; ++j) part[qq][j] = got[j];
          }
        }
      }
    }
    // all parts added up in part order, this workgroup's own at its place
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
      const float own = total[j];
      float sum = 0.f;
#pragma unroll
      for (int q = 0; q < KP; ++q) sum += q == kp ? own : part[q][j];
      total[j] = sum;
    }
  }
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int e = tid + j * NT;
    if (WORDS % NT == 0 || e < WORDS) {
      const int rb = e >> 8, ln = (e & 255) >> 2, i = e & 3;
      const int tok = 4 * (ln >> 4) + i, r = rb * 16 + (ln & 15);
      if (r < R) {
        const float v = (!MASKED || r < eff) ? total[j] * scaling : 0.f;  // ranks the adapter does not have contribute nothing
        const T hi = from_f32<T>(v);
        s_hi[tok * HSTRIDE + r] = hi;
        s_lo[tok * HSTRIDE + r] = from_f32<T>(v - to_f32(hi));
      }
    }
  }
  __syncthreads();
  MLORA_STAMP(5);  // the intermediate is in LDS
  report();  // this workgroup reads the exchange area no more

  // ---- expand: tokens as MFMA rows, lane holds out[row 4 * lg + i][column c0 + 4 * lr + j] ----
  Pack8 hop[KSTEPS], hlo[KSTEPS];
  uint2 hop16 = {0, 0}, hlo16 = {0, 0};
  if constexpr (K16) {
    hop16 = *reinterpret_cast<const uint2*>(&s_hi[lr * HSTRIDE + 4 * lg]);
    hlo16 = *reinterpret_cast<const uint2*>(&s_lo[lr * HSTRIDE + 4 * lg]);
  } else {
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
  }
  auto finish_span = [&](int c0, Pack8(&bo)[4][KSTEPS], uint2(&yy)[4]) {
    f32x4 out[4];
    uint2 pieces[4];
    if constexpr (K16) {
      if (MASKED && eff < R) {
        mask_ranks(bo[0][0], (lane & 1) * 8, eff);
        mask_ranks(bo[1][0], (lane & 1) * 8, eff);
      }
      // B rows -> operand pieces through the wavefront's LDS block: four rows (128 bytes) per
      // group, groups 144 bytes apart.  MFMA j of lane (lr, lg) takes ranks 4*lg .. 4*lg+3 of
      // column c0 + 4*lr + j.
      char* blk = reinterpret_cast<char*>(stage);
      *reinterpret_cast<i32x4*>(blk + (lane >> 3) * 144 + (lane & 7) * 16) = bo[0][0].raw;
      *reinterpret_cast<i32x4*>(blk + ((lane >> 3) + 8) * 144 + (lane & 7) * 16) = bo[1][0].raw;
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int j = 0; j < 4; ++j) pieces[j] = *reinterpret_cast<const uint2*>(blk + lr * 144 + j * 32 + lg * 8);
      __builtin_amdgcn_wave_barrier();
    } else if (MASKED && eff < R) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) mask_ranks(bo[j][ks], ((lg + 4 * ks) & (R / 8 - 1)) * 8, eff);
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
    // (the y values are taken as they are only here: unpacked where they were requested, the
    // wavefront would wait for their arrival before the shrink)
#pragma unroll
    for (int i = 0; i < XI; ++i) asm volatile("" : "+v"(yy[i].x), "+v"(yy[i].y));
    if (c < sp.n1) {
#pragma unroll
      for (int i = 0; i < XI; ++i) {
        if ((SPREAD ? lg + 4 * i : 4 * lg + i) < m) {
          union { uint2 raw; T e[4]; } v;
          v.raw = yy[i];
#pragma unroll
          for (int j = 0; j < 4; ++j) v.e[j] = from_f32<T>(to_f32(v.e[j]) + out[j][i]);
          *reinterpret_cast<uint2*>(ycols + static_cast<int64_t>(rows4[i]) * ys + c) = v.raw;
        }
      }
    }
  };
#pragma unroll
  for (int s = 0; s < SA; ++s) {
    const int c0 = sp.n0 + (wave + s * NW) * 64;
    if (c0 < sp.n1) finish_span(c0, bop[s], yq[s]);
  }
  MLORA_STAMP(6);
#ifdef MLORA_TRACE
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  MLORA_STAMP(7);
  __syncthreads();
  MLORA_STAMP(8);
#endif
