// The bf16 GEMM of few output tiles, for the GEMM dispatcher. Included inside
// namespace mhsa { namespace { ... } } after common.hpp, kernels.hpp,
// quant.hpp and gemm_tile.hpp.
#pragma once

// bf16 projections with too few output tiles to fill the GPU (one utterance,
// a short position table). A 64 x 64 tile on 2 x 2 waves walks the whole
// contraction behind one barrier per 64 columns, a serial chain of 0.35 us a
// stage that bounds it however idle the chip is. Here the NW waves of a
// workgroup share the contraction instead: wave w takes 64-column stages w,
// w + NW, ... of the tile's rows of A and W into LDS of its own (direct-to-LDS
// loads, NS stages in flight, no barrier), multiplies them, and the NW
// partial tiles meet in LDS once, summed in wave order. What bounds it now is
// the latency of the first stage (about 2 us) and, past K = 1024, a CU's rate
// from L2 (384 KB of a quantised 32 x 32 tile at K = 4096 in 7 us). Measured,
// u8: 125 x 1024 x 1024 8.6 -> 4.4 us, 203 x 1024 x 4096 24.3 -> 9.1; bf16 5.8
// -> 4.1 and 14.2 -> 8.0. More of the measurements are at kw_form.
template <int TM, int TN, int NW_, int NS_, bool QUANT>
struct KwTile {
  static constexpr int NW = NW_, NS = NS_, NT = 64 * NW, BM = 32 * TM, BN = 32 * TN;
  static constexpr int BROW = QUANT ? 64 : 128;  // bytes of a W row per stage
  static constexpr int ABYTES = BM * 128, BBYTES = BN * BROW, SBYTES = QUANT ? BN * 8 : 0;
  static constexpr int STAGE = ABYTES + BBYTES + SBYTES;  // one wave's
  static constexpr int NA = ABYTES / 1024, NB = BBYTES / 1024, NQ = QUANT ? TN : 0;  // loads per stage
  static constexpr int NL = NA + NB + NQ;
  static constexpr int PITCH = BN * 4 + 16;  // partial tile row (bytes)
  static constexpr int PART = BM * PITCH;
  static constexpr int LDS = NW * (NS * STAGE > PART ? NS * STAGE : PART);
  static_assert((NS - 1) * NL < 64, "loads in flight");
};

// Waits until at most `n` of this wave's loads are in flight.
template <int N>
__device__ __forceinline__ void wait_loads() {
  static_assert(N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (15 << 8) | (7 << 4));
  asm volatile("" ::: "memory");
}

template <int TM, int TN, int NW, int NS, bool QUANT>
__device__ __forceinline__ void kw_tile_body(const GemmParams& p, int block, char* smem) {
  using C = KwTile<TM, TN, NW, NS, QUANT>;
  const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5, c32 = lane & 31;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);

  // contiguous tile ranges per XCD, walked down the rows 8 tiles at a time
  const int tilesM = (int)m_tiles<C::BM>(p), tilesN = p.N / C::BN, nt = tilesM * tilesN;
  const int per = (nt + 7) / 8;
  const int W = (int)((unsigned)block % 8u) * per + (int)((unsigned)block / 8u);
  if ((int)((unsigned)block / 8u) >= per || W >= nt) return;
  constexpr int GM = 8;
  const int gsz = GM * tilesN, first = W / gsz * GM, gm = min(tilesM - first, GM);
  const int n0 = (W % gsz) / gm * C::BN;
  int m0, m_end, seg;
  tile_rows<C::BM>(p, first + (W % gsz) % gm, m0, m_end, seg);

  // Stage rows as in the tile kernel: 128-byte rows of A and dense W with
  // chunk c at c ^ (row / 2 % 8), 64-byte rows of codes with chunk c at
  // c ^ (row / 4 % 4); rows of A past the matrix read as zero. {scale, bias}
  // of 32 rows are one 4-byte load, two lanes a row.
  const char* Ab = reinterpret_cast<const char*>(p.A) + (int64_t)m0 * p.lda * 2;
  const __amdgpu_buffer_rsrc_t ra =
      __builtin_amdgcn_make_buffer_rsrc((void*)Ab, (short)0, (int)((int64_t)(p.M - m0) * p.lda * 2), kRawBuffer);
  const char* Bb = reinterpret_cast<const char*>(p.W) + (int64_t)n0 * p.K * (QUANT ? 1 : 2);
  const __amdgpu_buffer_rsrc_t rb =
      __builtin_amdgcn_make_buffer_rsrc((void*)Bb, (short)0, (int)((int64_t)C::BN * p.K * (QUANT ? 1 : 2)), kRawBuffer);
  const int groups = p.K / 64;
  __amdgpu_buffer_rsrc_t rs;
  if constexpr (QUANT)
    rs = __builtin_amdgcn_make_buffer_rsrc((void*)(p.sb + 2 * (int64_t)n0 * groups), (short)0,
                                           (int)((int64_t)C::BN * groups * 8), kRawBuffer);
  // (8 g rows on keep the permutation: 16 g for codes likewise)
  const int arow = lane >> 3, brow = QUANT ? lane >> 2 : lane >> 3;
  int aoff[2];  // even and odd loads differ in bit 2 of row / 2
#pragma unroll
  for (int u = 0; u < 2; ++u)
    aoff[u] = (int)(arow * p.lda * 2) + 16 * ((lane & 7) ^ (((arow + 8 * u) >> 1) & 7));
  int boffd[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) boffd[u] = brow * p.K * 2 + 16 * ((lane & 7) ^ (((brow + 8 * u) >> 1) & 7));
  const int boff = brow * p.K + 16 * ((lane & 3) ^ ((brow >> 2) & 3));
  char* S0 = smem + w * (NS * C::STAGE);
  auto issue = [&](int kt, int buf) {
    char* S = S0 + buf * C::STAGE;
#pragma unroll
    for (int g = 0; g < C::NA; ++g)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void*)(S + g * 1024), 16, aoff[g & 1] + g * 16 * (int)p.lda,
                                               kt * 128, 0, 0);
#pragma unroll
    for (int g = 0; g < C::NB; ++g) {
      if constexpr (QUANT)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_void*)(S + C::ABYTES + g * 1024), 16, boff + g * 16 * p.K,
                                                 kt * 64, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_void*)(S + C::ABYTES + g * 1024), 16,
                                                 boffd[g & 1] + g * 16 * p.K, kt * 128, 0, 0);
    }
    if constexpr (QUANT) {
#pragma unroll
      for (int g = 0; g < C::NQ; ++g)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(S + C::ABYTES + C::BBYTES + g * 256), 4,
                                                 ((32 * g + (lane >> 1)) * groups) * 8 + 4 * (lane & 1), kt * 8, 0, 0);
    }
  };

  floatx16 acc[TN][TM];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i) acc[j][i] = floatx16{};

  // this wave's stages: w, w + NW, ...
  const int nk = p.K / 64, n = nk > w ? (nk - w + NW - 1) / NW : 0;
#pragma unroll
  for (int st = 0; st < NS; ++st)
    if (st < n) issue(w + st * NW, st);
  int buf = 0;
  for (int t = 0; t < n; ++t) {
    // stage t has landed; the stages after it may be in flight
    const int ahead = min(NS - 1, n - 1 - t);
    if (ahead == 0) wait_loads<0>();
    else if (NS == 2 || ahead == 1) wait_loads<C::NL>();
    else wait_loads<(NS > 2 ? 2 : 0) * C::NL>();
    __builtin_amdgcn_sched_barrier(0);
    const char* S = S0 + buf * C::STAGE;
    // fragments: lane l holds row l % 32, columns 16 s + 8 (l / 32) + [0, 8)
    // of sub-step s (quantized: 32 (l / 32) + 8 s + [0, 8))
    bf16x8 fa[4][TM], fb[4][TN];
    u32x4 cq[2][TN];
    floatx2 qs[TN];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int so = 16 * ((QUANT ? 4 * hh + s : 2 * s + hh) ^ ((lane >> 1) & 7));
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[s][i] = *reinterpret_cast<const bf16x8*>(S + (32 * i + c32) * 128 + so);
      if constexpr (!QUANT) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
          fb[s][j] = *reinterpret_cast<const bf16x8*>(S + C::ABYTES + (32 * j + c32) * 128 + so);
      }
    }
    if constexpr (QUANT) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
          cq[u][j] = *reinterpret_cast<const u32x4*>(S + C::ABYTES + (32 * j + c32) * 64 +
                                                     16 * ((2 * hh + u) ^ ((c32 >> 2) & 3)));
        qs[j] = *reinterpret_cast<const floatx2*>(S + C::ABYTES + C::BBYTES + (32 * j + c32) * 8);
      }
    }
    if (t + NS < n) {
      __builtin_amdgcn_s_waitcnt((15) | (3 << 14) | (7 << 4));  // lgkmcnt(0): the buffer is free again
      __builtin_amdgcn_sched_barrier(0);
      issue(w + (t + NS) * NW, buf);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if constexpr (QUANT) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          u32x4 v;
#pragma unroll
          for (int e4 = 0; e4 < 2; ++e4) {
            const uint32_t c = cq[s >> 1][j][2 * (s & 1) + e4];
            float f[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) f[e] = __builtin_fmaf(qs[j].x, (float)((c >> (8 * e)) & 0xFFu), qs[j].y);
            const bf16x2 lo = {(bf16)f[0], (bf16)f[1]}, hi = {(bf16)f[2], (bf16)f[3]};
            v[2 * e4] = __builtin_bit_cast(uint32_t, lo);
            v[2 * e4 + 1] = __builtin_bit_cast(uint32_t, hi);
          }
          fb[s][j] = __builtin_bit_cast(bf16x8, v);
        }
      }
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i) acc[j][i] = mma32(fb[s][j], fa[s][i], acc[j][i]);
    }
    buf = buf + 1 == NS ? 0 : buf + 1;
  }

  // The partial tiles row-major in LDS (a lane holds row 32 i + lane % 32,
  // columns 32 j + 8 q + 4 (lane / 32) + [0, 4)), summed in wave order.
  __syncthreads();
  {
    char* st = smem + w * C::PART + c32 * C::PITCH + 16 * hh;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<floatx4*>(st + i * 32 * C::PITCH + (32 * j + 8 * q) * 4) =
              floatx4{acc[j][i][4 * q], acc[j][i][4 * q + 1], acc[j][i][4 * q + 2], acc[j][i][4 * q + 3]};
  }
  __syncthreads();
  constexpr int RUNS = C::BM * C::BN / 4;
  if (p.vt && n0 >= p.vt_col0) {
    // V^T: 4 tokens of one column per thread (the waves' reads span columns);
    // rows past the utterance are finite filler, zeros past the tile up to
    // the attention's tile of 64 tokens
    const int t0 = m0 - seg * p.seg_T;
    bf16* VT = reinterpret_cast<bf16*>(p.vt) + (int64_t)seg * p.vt_Tpad;
    for (int id = tid; id < RUNS; id += C::NT) {
      const int c = id % C::BN, r = id / C::BN * 4, tok = t0 + r;
      if (tok >= p.vt_Tpad) continue;
      const float b = p.bias ? p.bias[n0 + c] : 0.f;
      bf16x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float s = *reinterpret_cast<const float*>(smem + (r + e) * C::PITCH + c * 4);
#pragma unroll
        for (int k = 1; k < NW; ++k) s += *reinterpret_cast<const float*>(smem + k * C::PART + (r + e) * C::PITCH + c * 4);
        s = round_to<bf16>(s);
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
  for (int it = 0; it < (RUNS + C::NT - 1) / C::NT; ++it) {
    const int id = it * C::NT + tid;
    if (RUNS % C::NT && id >= RUNS) break;
    const int r = id / (C::BN / 4), c = id % (C::BN / 4) * 4, row = m0 + r, col = n0 + c;
    if (row >= m_end) continue;
    const char* src = smem + r * C::PITCH + c * 4;
    floatx4 s = *reinterpret_cast<const floatx4*>(src);
#pragma unroll
    for (int k = 1; k < NW; ++k) s += *reinterpret_cast<const floatx4*>(src + k * C::PART);
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] = round_to<bf16>(s[e]);
    if (p.bias) {
      const floatx4 b = *reinterpret_cast<const floatx4*>(p.bias + col);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = round_to<bf16>(s[e] + b[e]);
    }
    if (p.act == kActSilu) {
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = silu_value<bf16>(s[e]);
    }
    if (p.R) {
      const bf16x4 rv = *reinterpret_cast<const bf16x4*>(reinterpret_cast<const bf16*>(p.R) + (int64_t)row * p.ldr + col);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = round_to<bf16>((float)rv[e] + p.res_scale * s[e]);
    }
    bf16x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = (bf16)s[e];
    *reinterpret_cast<bf16x4*>(reinterpret_cast<bf16*>(p.C) + row_offset(p, row) + col) = v;
  }
}

// One problem, or two independent ones in one launch: p1's tiles in
// workgroups [0, n1) (n1 a multiple of 8), p2's in those after them.
template <int TM, int TN, int NW, int NS, bool QUANT>
__global__ __launch_bounds__(64 * NW) void gemm_kw_kernel(const GemmParams p1, int n1, const GemmParams p2) {
  __shared__ __attribute__((aligned(1024))) char smem[KwTile<TM, TN, NW, NS, QUANT>::LDS];
  const int block = (int)blockIdx.x;
  if (block < n1) kw_tile_body<TM, TN, NW, NS, QUANT>(p1, block, smem);
  else kw_tile_body<TM, TN, NW, NS, QUANT>(p2, block - n1, smem);
}
