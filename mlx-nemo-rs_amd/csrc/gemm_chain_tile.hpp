// The bf16 GEMM of few output tiles, for the GEMM dispatcher. Included inside
// namespace mhsa { namespace { ... } } after common.hpp, kernels.hpp,
// quant.hpp and gemm_tile.hpp.
#pragma once

// Waits until at most `n` of this wave's loads are in flight.
template <int N>
__device__ __forceinline__ void wait_loads() {
  static_assert(N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (15 << 8) | (7 << 4));
  asm volatile("" ::: "memory");
}

// The epilogue of 4 columns [col, col + 4) of a row in the reference's order,
// each step stored in bf16: the sums `s`, bias, SiLU, scaled residual.
__device__ __forceinline__ void bf16_store4(const GemmParams& p, int row, int col, floatx4 s, const floatx4& bias,
                                            const bf16x4& res) {
#pragma unroll
  for (int e = 0; e < 4; ++e) s[e] = round_to<bf16>(s[e]);
  if (p.bias) {
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] = round_to<bf16>(s[e] + bias[e]);
  }
  if (p.act == kActSilu) {
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] = silu_value<bf16>(s[e]);
  }
  if (p.R) {
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] = round_to<bf16>((float)res[e] + p.res_scale * s[e]);
  }
  bf16x4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = (bf16)s[e];
  *reinterpret_cast<bf16x4*>(reinterpret_cast<bf16*>(p.C) + row_offset(p, row) + col) = v;
}

// bf16 projections with too few output tiles to fill the GPU (one utterance,
// a short position table). Every sum is the tile kernels' one chain of MFMAs
// along K, bit for bit, so a row gives the same result alone and in a batch;
// what the waves of a workgroup share is the rest. TM x TN consumer waves own
// a 32 x 32 tile each and issue nothing but fragment reads and MFMAs; four
// loader waves bring the operands straight to LDS in phases of 4 / TN stages
// of 64 k-columns, R - 2 phases ahead; eight dequantiser waves turn codes into
// fragments in LDS a phase ahead of their products. One barrier per phase.
//
// The 64 x 64 tile kernel's four waves do all of it in turn, 0.35 us a stage
// of u8 weights and 0.2 dense: every weight dequantised by two waves, a barrier
// and its latencies per 64 columns. Here a phase of 256 columns takes 0.24 us
// dense, of which the chain itself is 0.21 (16 MFMAs of 32 cycles), and 0.38
// u8, where the dequantisers that share the consumer's SIMD end last. Loads
// and dequantisation in the same waves measured 0.46 (a wave is held up about
// 80 cycles by each load to LDS), stage addresses by division and branches
// between a consumer's MFMAs 0.42 dense. Measured, us a launch, 64 x 64 tiles
// / this: u8 125 x 1024 x 1024 8.7 / 6.2, 203 x 1024 x 4096 23.9 / 12.0, 203 x
// 4096 x 1024 11.4 / 10.3; bf16 125 x 1024 x 4096 14.7 / 8.7, 125 x 512 x 512
// 5.5 / 4.8. (The waves sharing the contraction, eight chains to a sum, take
// 4.4 and 9.1 on the first two, but round bf16 results the other way here and
// there: a row's result would depend on how many come with it.)
template <int TM, int TN, int R_, bool QUANT>
struct ChainTile {
  // waves: consumers, loaders, dequantisers
  static constexpr int NC = TM * TN, NLD = 4, NDQ = QUANT ? 8 : 0, NT = 64 * (NC + NLD + NDQ);
  static constexpr int BM = 32 * TM, BN = 32 * TN, G = NLD / TN, R = R_;  // G stages a phase, R phases in LDS
  // A ring of phases of A's rows (and dense W's), one of codes with {scale,
  // bias}, and the dequantised fragments of two phases
  static constexpr int ABYTES = BM * 128, STAGE = ABYTES + (QUANT ? 0 : BN * 128), PHASE = G * STAGE;
  static constexpr int CSTAGE = QUANT ? BN * 72 : 0, CPHASE = G * CSTAGE;
  static constexpr int FRAGS = QUANT ? G * TN * 4096 : 0;
  static constexpr int C_OFF = R * PHASE, F_OFF = C_OFF + R * CPHASE, LDS = F_OFF + 2 * FRAGS;
  static constexpr int NA = 4 * TM / TN, NW = QUANT ? 3 : 4, NL = NA + NW;  // loads per loader and phase
  static constexpr int PITCH = BN * 4 + 16;  // epilogue row (bytes)
  static constexpr int RUNS = BM * BN / 4, RIT = (RUNS + NT - 1) / NT;
  static_assert(LDS <= 160 * 1024 && BM * PITCH <= LDS && R >= 3 && R <= 5 && R * NL < 64, "limits");
};

template <int TM, int TN, int R, bool QUANT>
__device__ __forceinline__ void chain_tile_body(const GemmParams& p, int block, char* smem) {
  using C = ChainTile<TM, TN, R, QUANT>;
  const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5, c32 = lane & 31;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);

  // contiguous tile ranges per XCD, walked down the rows 8 tiles at a time
  const int tilesM = (int)m_tiles<C::BM>(p), tilesN = p.N / C::BN, nt = tilesM * tilesN;
  const int per = (nt + 7) / 8;
  const int W = (int)((unsigned)block % 8u) * per + (int)((unsigned)block / 8u);
  if ((int)((unsigned)block / 8u) >= per || W >= nt) return;  // (whole workgroup)
  constexpr int GM = 8;
  const int gsz = GM * tilesN, first = W / gsz * GM, gm = min(tilesM - first, GM);
  const int n0 = (W % gsz) / gm * C::BN;
  int m0, m_end, seg;
  tile_rows<C::BM>(p, first + (W % gsz) % gm, m0, m_end, seg);
  const bool vt_tile = p.vt && n0 >= p.vt_col0;

  // the epilogue's bias and residual runs, ahead of the operand stream
  floatx4 bpre[C::RIT];
  bf16x4 rpre[C::RIT];
  if (!vt_tile) {
#pragma unroll
    for (int it = 0; it < C::RIT; ++it) {
      const int id = it * C::NT + tid, r = id / (C::BN / 4), col = n0 + id % (C::BN / 4) * 4;
      const bool ok = (C::RUNS % C::NT == 0 || id < C::RUNS) && m0 + r < m_end;
      if (p.bias && ok) bpre[it] = *reinterpret_cast<const floatx4*>(p.bias + col);
      if (p.R && ok)
        rpre[it] = *reinterpret_cast<const bf16x4*>(reinterpret_cast<const bf16*>(p.R) + (int64_t)(m0 + r) * p.ldr + col);
    }
  }

  const int nk = p.K / 64, nph = (nk + C::G - 1) / C::G;
  // (dequantised fragments: [phase parity][stage][column block][sub-step][lane])
  floatx16 acc{};
  const int ci = w % TM, cj = w / TM;  // a consumer's block
  if (w < C::NC) {
    // Fragments of a sub-step: row l % 32, columns as in the tile kernel. A
    // stage's MFMAs have the next stage's reads between them; phases are
    // straight-line code but for the last.
    bf16x8 fa[2][4], fb[2][4];
    int sat = 0, fat = C::F_OFF;  // this phase's stages and fragments
    int ao[4], bo[4];
    auto base = [&]() {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int so = 16 * ((QUANT ? 4 * hh + s : 2 * s + hh) ^ ((lane >> 1) & 7));
        ao[s] = sat + (32 * ci + c32) * 128 + so;
        bo[s] = QUANT ? fat + cj * 4096 + s * 1024 + lane * 16 : sat + C::ABYTES + (32 * cj + c32) * 128 + so;
      }
    };
    auto next_phase = [&]() {
      sat = sat + C::PHASE == C::R * C::PHASE ? 0 : sat + C::PHASE;
      fat = 2 * C::F_OFF + C::FRAGS - fat;
      base();
    };
    auto rd = [&](int g, int s, int b) {
      fa[b][s] = *reinterpret_cast<const bf16x8*>(smem + ao[s] + g * C::STAGE);
      fb[b][s] = *reinterpret_cast<const bf16x8*>(smem + bo[s] + g * (QUANT ? TN * 4096 : C::STAGE));
    };
    auto mma = [&](int b, int s) {
      acc = mma32(fb[b][s], fa[b][s], acc);
      __builtin_amdgcn_sched_barrier(0);
    };
    base();
    __builtin_amdgcn_s_setprio(2);
    if constexpr (QUANT) asm volatile("s_barrier" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int s = 0; s < 4; ++s) rd(0, s, 0);
    int ph = 0;
    for (; ph + 1 < nph; ++ph) {
#pragma unroll
      for (int g = 0; g < C::G; ++g) {
        const int b = g & 1;
        if (g + 1 < C::G) {
#pragma unroll
          for (int s = 0; s < 4; ++s) mma(b, s), rd(g + 1, s, b ^ 1);
        } else {
          mma(b, 0);
          mma(b, 1);
          __builtin_amdgcn_s_waitcnt((15) | (3 << 14) | (7 << 4));  // lgkmcnt(0): the phase is read
          asm volatile("s_barrier" ::: "memory");
          next_phase();
          rd(0, 0, 0);
          rd(0, 1, 0);
          mma(b, 2);
          rd(0, 2, 0);
          rd(0, 3, 0);
          mma(b, 3);
        }
      }
    }
    const int left = nk - ph * C::G;
#pragma unroll
    for (int g = 0; g < C::G; ++g) {
      if (g < left) {
        if (g + 1 < left) {
#pragma unroll
          for (int s = 0; s < 4; ++s) rd(g + 1, s, (g & 1) ^ 1);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 4; ++s) mma(g & 1, s);
      }
    }
    __builtin_amdgcn_s_setprio(0);
  } else if (w < C::NC + C::NLD) {
    // Loader of stage g of each phase and 32 columns j: its share of A's loads
    // of 8 rows, rows 32 j + [0, 32) of W. Stage rows as in the tile kernel:
    // 128-byte rows of A and dense W with chunk c at c ^ (row / 2 % 8), 64-byte
    // rows of codes with chunk c at c ^ (row / 4 % 4); rows of A past the
    // matrix read as zero.
    const int g = (w - C::NC) / TN, j = (w - C::NC) % TN;
    const char* Ab = reinterpret_cast<const char*>(p.A) + (int64_t)m0 * p.lda * 2;
    const __amdgpu_buffer_rsrc_t ra =
        __builtin_amdgcn_make_buffer_rsrc((void*)Ab, (short)0, (int)((int64_t)(p.M - m0) * p.lda * 2), kRawBuffer);
    const char* Bb = reinterpret_cast<const char*>(p.W) + (int64_t)n0 * p.K * (QUANT ? 1 : 2);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        (void*)Bb, (short)0, (int)((int64_t)C::BN * p.K * (QUANT ? 1 : 2)), kRawBuffer);
    const int groups = p.K / 64;
    __amdgpu_buffer_rsrc_t rs;
    if constexpr (QUANT)
      rs = __builtin_amdgcn_make_buffer_rsrc((void*)(p.sb + 2 * (int64_t)n0 * groups), (short)0,
                                             (int)((int64_t)C::BN * groups * 8), kRawBuffer);
    int aoff[C::NA], woff[QUANT ? 2 : 4];
#pragma unroll
    for (int i = 0; i < C::NA; ++i) {
      const int row = (j * C::NA + i) * 8 + (lane >> 3);
      aoff[i] = (int)(row * p.lda * 2) + 16 * ((lane & 7) ^ ((row >> 1) & 7));
    }
#pragma unroll
    for (int i = 0; i < (QUANT ? 2 : 4); ++i) {
      const int row = 32 * j + (QUANT ? 16 * i + (lane >> 2) : 8 * i + (lane >> 3));
      woff[i] = QUANT ? row * p.K + 16 * ((lane & 3) ^ ((row >> 2) & 3))
                      : row * p.K * 2 + 16 * ((lane & 7) ^ ((row >> 1) & 7));
    }
    const int soff = (32 * j + (lane >> 1)) * groups * 8 + 4 * (lane & 1);
    const int n = nk > g ? (nk - g + C::G - 1) / C::G : 0;  // phases in which stage g exists
    auto issue_w = [&](int ph) {
      const int kt = ph * C::G + g;
      char* S = smem + (QUANT ? C::C_OFF + ph % R * C::CPHASE + g * C::CSTAGE + j * 2048
                              : ph % R * C::PHASE + g * C::STAGE + C::ABYTES + j * 4096);
#pragma unroll
      for (int i = 0; i < (QUANT ? 2 : 4); ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_void*)(S + i * 1024), 16, woff[i], kt * (QUANT ? 64 : 128), 0, 0);
      if constexpr (QUANT)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rs, (lds_void*)(smem + C::C_OFF + ph % R * C::CPHASE + g * C::CSTAGE + C::BN * 64 + j * 256), 4, soff, kt * 8,
            0, 0);
    };
    // Batch b: A of phase b, and W of phase b, or, as codes are read a phase
    // before they are dequantised and that is a phase before their products,
    // of phase b + 2. Slot i, between barriers i - 1 and i, issues batch
    // i - 2 + R (the consumers are past phase i - 2, the dequantisers have
    // read phase i) and ends when batch i has landed.
    constexpr int AHEAD = QUANT ? 2 : 0;
    auto batch = [&](int b) {
      if (b + AHEAD < n) issue_w(b + AHEAD);
      char* S = smem + b % R * C::PHASE + g * C::STAGE;
#pragma unroll
      for (int i = 0; i < C::NA; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void*)(S + (j * C::NA + i) * 1024), 16, aoff[i],
                                                 (b * C::G + g) * 128, 0, 0);
    };
    // the wait for batch n - 1 - rem behind the batches issued after it, of
    // which the last AHEAD bring no W
    auto wait = [&](int rem) {
      constexpr int NL = C::NL, NX = QUANT ? C::NW : 0;
      if (rem >= R) wait_loads<(R - 2) * NL>();
      else if (rem == R - 1) wait_loads<(R - 2) * NL - NX>();
      else if (rem == 3) wait_loads<(R > 4 ? 3 * NL - 2 * NX : 0)>();
      else if (rem == 2) wait_loads<(R > 3 ? 2 * NL - 2 * NX : 0)>();
      else if (rem == 1) wait_loads<NL - NX>();
      else wait_loads<0>();
    };
    constexpr int PRO = R - AHEAD;  // batches that find their buffers free
    if constexpr (QUANT) {
      if (n > 0) issue_w(0);
      if (n > 1) issue_w(1);
      for (int b = 0; b < min(PRO, n); ++b) batch(b);
      // W of phases 0 and 1, then batch 0, the only one without R - 2 behind it
      if (n >= R) wait_loads<PRO * C::NL>();
      else wait_loads<C::NA>();
      asm volatile("s_barrier" ::: "memory");
      if (n >= R) wait_loads<(PRO - 1) * C::NL>();
      else if (PRO > 1 && n > 1) wait_loads<C::NA>();
      else wait_loads<0>();
      asm volatile("s_barrier" ::: "memory");
      if (PRO < n) batch(PRO);
    } else {
      for (int b = 0; b < min(PRO, n); ++b) batch(b);
    }
    int i = QUANT ? 1 : 0;
    auto edge = [&](int end) {
      for (; i < end; ++i) {
        if ((QUANT || i >= 2) && i - 2 + R < n) batch(i - 2 + R);
        if (i < n) wait(n - 1 - i);
        asm volatile("s_barrier" ::: "memory");
      }
    };
    edge(min(2, nph));
    for (; i + R < n; ++i) {
      batch(i - 2 + R);
      wait_loads<(R - 2) * C::NL>();
      asm volatile("s_barrier" ::: "memory");
    }
    edge(nph);
  } else {
    // Dequantiser of rows 16 q + [0, 16) of W in stage g of each phase. Lane l
    // holds codes 16 (l / 16) + [0, 16) of row 16 q + l % 16, which are
    // sub-steps 2 (l / 16 % 2) + {0, 1} of half l / 32.
    const int d = w - C::NC - C::NLD, g = d / (2 * TN), q = d % (2 * TN), r = lane & 15, c = lane >> 4;
    const int co = C::C_OFF + g * C::CSTAGE + q * 1024 + r * 64 + 16 * (c ^ ((r >> 2) & 3));
    const int qo = C::C_OFF + g * C::CSTAGE + C::BN * 64 + (16 * q + r) * 8;
    const int fo = C::F_OFF + ((g * TN + (q >> 1)) * 4 + 2 * (c & 1)) * 1024 + (32 * (c >> 1) + 16 * (q & 1) + r) * 16;
    const int n = nk > g ? (nk - g + C::G - 1) / C::G : 0;
    u32x4 cw[2];
    floatx2 sb[2];
    int at = 0;  // the next phase to read
    auto read = [&](int set) {
      cw[set] = *reinterpret_cast<const u32x4*>(smem + co + at);
      sb[set] = *reinterpret_cast<const floatx2*>(smem + qo + at);
      at = at + C::CPHASE == R * C::CPHASE ? 0 : at + C::CPHASE;
    };
    auto phase = [&](int i, int set) {
      if (i + 1 < n) read(set ^ 1);
      __builtin_amdgcn_sched_barrier(0);
      if (i < n) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          u32x4 v;
#pragma unroll
          for (int e4 = 0; e4 < 2; ++e4) {
            const uint32_t cc = cw[set][2 * u + e4];
            float f[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) f[e] = __builtin_fmaf(sb[set].x, (float)((cc >> (8 * e)) & 0xFFu), sb[set].y);
            const bf16x2 lo = {(bf16)f[0], (bf16)f[1]}, hi = {(bf16)f[2], (bf16)f[3]};
            v[2 * e4] = __builtin_bit_cast(uint32_t, lo);
            v[2 * e4 + 1] = __builtin_bit_cast(uint32_t, hi);
          }
          *reinterpret_cast<u32x4*>(smem + fo + set * C::FRAGS + u * 1024) = v;
        }
      }
      __builtin_amdgcn_s_waitcnt((15) | (3 << 14) | (7 << 4));  // lgkmcnt(0): the fragments are written
      asm volatile("s_barrier" ::: "memory");
    };
    asm volatile("s_barrier" ::: "memory");
    if (n > 0) read(0);
    for (int i = 0; i < nph; i += 2) {
      phase(i, 0);
      if (i + 1 < nph) phase(i + 1, 1);
    }
  }

  // The tile row-major in LDS (a consumer's lane holds row 32 i + lane % 32,
  // columns 32 j + 8 q + 4 (lane / 32) + [0, 4)), stored by all waves.
  __syncthreads();
  if (w < C::NC) {
    char* st = smem + (32 * ci + c32) * C::PITCH + 128 * cj + 16 * hh;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<floatx4*>(st + 32 * q) = floatx4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
  }
  __syncthreads();
  if (vt_tile) {
    // V^T: 4 tokens of one column per thread (the waves' reads span columns);
    // rows past the utterance are finite filler, zeros past the tile up to
    // the attention's tile of 64 tokens
    const int t0 = m0 - seg * p.seg_T;
    bf16* VT = reinterpret_cast<bf16*>(p.vt) + (int64_t)seg * p.vt_Tpad;
    for (int id = tid; id < C::RUNS; id += C::NT) {
      const int c = id % C::BN, r = id / C::BN * 4, tok = t0 + r;
      if (tok >= p.vt_Tpad) continue;
      const float b = p.bias ? p.bias[n0 + c] : 0.f;
      bf16x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float s = round_to<bf16>(*reinterpret_cast<const float*>(smem + (r + e) * C::PITCH + c * 4));
        v[e] = (bf16)(p.bias ? s + b : s);
      }
      bf16* col = VT + (int64_t)(n0 + c - p.vt_col0) * p.vt_ld;
      *reinterpret_cast<bf16x4*>(col + tok) = v;
      if (C::BM % 64 && (tok & 32) == 0 && t0 + C::BM >= p.seg_T && tok + 32 < p.vt_Tpad)
        *reinterpret_cast<bf16x4*>(col + tok + 32) = bf16x4{};
    }
    return;
  }
#pragma unroll
  for (int it = 0; it < C::RIT; ++it) {
    const int id = it * C::NT + tid;
    if (C::RUNS % C::NT && id >= C::RUNS) break;
    const int r = id / (C::BN / 4), c = id % (C::BN / 4) * 4, row = m0 + r;
    if (row >= m_end) continue;
    bf16_store4(p, row, n0 + c, *reinterpret_cast<const floatx4*>(smem + r * C::PITCH + c * 4), bpre[it], rpre[it]);
  }
}

// One problem, or two independent ones in one launch: p1's tiles in
// workgroups [0, n1) (n1 a multiple of 8), p2's in those after them.
template <int TM, int TN, int R, bool QUANT>
__global__ __launch_bounds__((ChainTile<TM, TN, R, QUANT>::NT)) void gemm_chain_kernel(const GemmParams p1, int n1,
                                                                                    const GemmParams p2) {
  __shared__ __attribute__((aligned(1024))) char smem[ChainTile<TM, TN, R, QUANT>::LDS];
  const int block = (int)blockIdx.x;
  if (block < n1) chain_tile_body<TM, TN, R, QUANT>(p1, block, smem);
  else chain_tile_body<TM, TN, R, QUANT>(p2, block - n1, smem);
}
