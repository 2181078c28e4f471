// The bf16 GEMM of a handful of output tiles, for the GEMM dispatcher.
// Included inside namespace mhsa { namespace { ... } } after common.hpp,
// kernels.hpp, quant.hpp, gemm_tile.hpp and gemm_chain_tile.hpp.
#pragma once

// bf16 projections of fewer than 16 tiles of 64 x 64 (a short utterance of a
// small model): each sum is that of its runs of 256 k-columns, every run one
// chain of 16x16x32 MFMAs, added in order. The runs are independent, so the
// eight waves of a workgroup take one each of a 32 x 32 tile: the 64-column
// stages of a run come to LDS of the wave's own (direct-to-LDS loads, two
// stages in flight, no barrier), and the runs' sums meet in LDS once per
// eight runs. It is bound by the latency of the first stage (about 2 us): 1 x
// 512 x 2048 takes 5.2 us, 5.8 with u8 weights, where runs on workgroups of
// their own and a second kernel to add them took 6.7 and 7.1.
template <bool QUANT>
struct KwTile {
  static constexpr int NW = 8, NS = 2, NT = 64 * NW, RUN = 256;
  static constexpr int BROW = QUANT ? 64 : 128;  // bytes of a W row per stage
  static constexpr int ABYTES = 32 * 128, BBYTES = 32 * BROW, STAGE = ABYTES + BBYTES + (QUANT ? 256 : 0);
  static constexpr int NA = 4, NB = QUANT ? 2 : 4, NL = NA + NB + (QUANT ? 1 : 0);  // loads per stage
  static constexpr int PART = 32 * 128;  // a run's sums of the tile
  static constexpr int P_OFF = NW * NS * STAGE, LDS = P_OFF + NW * PART;
  static_assert(LDS <= 160 * 1024, "limits");
};

template <bool QUANT>
__device__ __forceinline__ void kw_tile_body(const GemmParams& p, char* smem) {
  using C = KwTile<QUANT>;
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, kg = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tilesN = p.N / 32, m0 = (int)blockIdx.x / tilesN * 32, n0 = (int)blockIdx.x % tilesN * 32;

  // Stage rows as in the tile kernel: 128-byte rows of A and dense W with
  // chunk c at c ^ (row / 2 % 8), 64-byte rows of codes with chunk c at
  // c ^ (row / 4 % 4); rows of A past the matrix read as zero. {scale, bias}
  // of the 32 rows are one 4-byte load, two lanes a row.
  const char* Ab = reinterpret_cast<const char*>(p.A) + (int64_t)m0 * p.lda * 2;
  const __amdgpu_buffer_rsrc_t ra =
      __builtin_amdgcn_make_buffer_rsrc((void*)Ab, (short)0, (int)((int64_t)(p.M - m0) * p.lda * 2), kRawBuffer);
  const char* Bb = reinterpret_cast<const char*>(p.W) + (int64_t)n0 * p.K * (QUANT ? 1 : 2);
  const __amdgpu_buffer_rsrc_t rb =
      __builtin_amdgcn_make_buffer_rsrc((void*)Bb, (short)0, (int)((int64_t)32 * p.K * (QUANT ? 1 : 2)), kRawBuffer);
  const int groups = p.K / 64;
  __amdgpu_buffer_rsrc_t rs;
  if constexpr (QUANT)
    rs = __builtin_amdgcn_make_buffer_rsrc((void*)(p.sb + 2 * (int64_t)n0 * groups), (short)0, 32 * groups * 8,
                                           kRawBuffer);
  int aoff[C::NA], boff[C::NB];
#pragma unroll
  for (int i = 0; i < C::NA; ++i) {
    const int row = 8 * i + (lane >> 3);
    aoff[i] = (int)(row * p.lda * 2) + 16 * ((lane & 7) ^ ((row >> 1) & 7));
  }
#pragma unroll
  for (int i = 0; i < C::NB; ++i) {
    const int row = QUANT ? 16 * i + (lane >> 2) : 8 * i + (lane >> 3);
    boff[i] = QUANT ? row * p.K + 16 * ((lane & 3) ^ ((row >> 2) & 3))
                    : row * p.K * 2 + 16 * ((lane & 7) ^ ((row >> 1) & 7));
  }
  char* S0 = smem + w * (C::NS * C::STAGE);
  // this wave's runs are w, w + 8, ...; its stage t is stage t % 4 of run
  // w + 8 (t / 4)
  const int runs = p.K / C::RUN, n = runs > w ? (runs - w + C::NW - 1) / C::NW * 4 : 0;
  auto issue = [&](int t) {
    char* S = S0 + (t % C::NS) * C::STAGE;
    const int kt = (w + t / 4 * C::NW) * 4 + t % 4;
#pragma unroll
    for (int i = 0; i < C::NA; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void*)(S + i * 1024), 16, aoff[i], kt * 128, 0, 0);
#pragma unroll
    for (int i = 0; i < C::NB; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_void*)(S + C::ABYTES + i * 1024), 16, boff[i], kt * C::BROW, 0, 0);
    if constexpr (QUANT)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(S + C::ABYTES + C::BBYTES), 4,
                                               (lane >> 1) * groups * 8 + 4 * (lane & 1), kt * 8, 0, 0);
  };
  for (int t = 0; t < min(C::NS, n); ++t) issue(t);

  floatx4 sum{};  // threads 0-255: row tid / 8, columns 4 (tid % 8) + [0, 4)
  const int sr = tid >> 3 & 31, sc = tid & 7;
  for (int round = 0; round * C::NW < runs; ++round) {
    if (round * C::NW + w < runs) {
      floatx4 acc[2][2] = {};
      for (int t = 4 * round; t < 4 * round + 4; ++t) {
        if (t + 1 < n) wait_loads<C::NL>();  // stage t has landed; the one after it may be in flight
        else wait_loads<0>();
        __builtin_amdgcn_sched_barrier(0);
        // fragments: lane l holds row l % 16, columns 32 s + 8 (l / 16) + [0, 8)
        const char* S = S0 + (t % C::NS) * C::STAGE;
        bf16x8 fa[2][2], fb[2][2];
        u32x2 cq[2][2];
        floatx2 qs[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int row = 16 * i + l16;
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            fa[s][i] = *reinterpret_cast<const bf16x8*>(S + row * 128 + 16 * ((4 * s + kg) ^ ((row >> 1) & 7)));
            if constexpr (QUANT)
              cq[s][i] = *reinterpret_cast<const u32x2*>(S + C::ABYTES + row * 64 +
                                                         16 * ((2 * s + (kg >> 1)) ^ ((row >> 2) & 3)) + 8 * (kg & 1));
            else
              fb[s][i] =
                  *reinterpret_cast<const bf16x8*>(S + C::ABYTES + row * 128 + 16 * ((4 * s + kg) ^ ((row >> 1) & 7)));
          }
          if constexpr (QUANT) qs[i] = *reinterpret_cast<const floatx2*>(S + C::ABYTES + C::BBYTES + row * 8);
        }
        __builtin_amdgcn_s_waitcnt((15) | (3 << 14) | (7 << 4));  // lgkmcnt(0): the buffer is free again
        __builtin_amdgcn_sched_barrier(0);
        if (t + C::NS < n) issue(t + C::NS);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          if constexpr (QUANT) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              u32x4 v;
#pragma unroll
              for (int e4 = 0; e4 < 2; ++e4) {
                float f[4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                  f[e] = __builtin_fmaf(qs[j].x, (float)((cq[s][j][e4] >> (8 * e)) & 0xFFu), qs[j].y);
                const bf16x2 lo = {(bf16)f[0], (bf16)f[1]}, hi = {(bf16)f[2], (bf16)f[3]};
                v[2 * e4] = __builtin_bit_cast(uint32_t, lo);
                v[2 * e4 + 1] = __builtin_bit_cast(uint32_t, hi);
              }
              fb[s][j] = __builtin_bit_cast(bf16x8, v);
            }
          }
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = mma16(fa[s][i], fb[s][j], acc[i][j]);
        }
      }
      // (a lane holds rows 16 i + 4 (l / 16) + [0, 4) of column 16 j + l % 16;
      // 16-byte chunk c of a row at c ^ (row % 8))
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int row = 16 * i + 4 * kg + e, col = 16 * j + l16;
            *reinterpret_cast<float*>(smem + C::P_OFF + w * C::PART + row * 128 + 16 * ((col >> 2) ^ (row & 7)) +
                                      4 * (col & 3)) = acc[i][j][e];
          }
    }
    __syncthreads();
    if (tid < 256) {
      const int here = min(C::NW, runs - round * C::NW);
      for (int k = 0; k < here; ++k)
        sum += *reinterpret_cast<const floatx4*>(smem + C::P_OFF + k * C::PART + sr * 128 + 16 * (sc ^ (sr & 7)));
    }
    __syncthreads();
  }
  if (tid < 256 && m0 + sr < p.M) {
    const int row = m0 + sr, col = n0 + 4 * sc;
    floatx4 bias{};
    bf16x4 res{};
    if (p.bias) bias = *reinterpret_cast<const floatx4*>(p.bias + col);
    if (p.R) res = *reinterpret_cast<const bf16x4*>(reinterpret_cast<const bf16*>(p.R) + (int64_t)row * p.ldr + col);
    bf16_store4(p, row, col, sum, bias, res);
  }
}

template <bool QUANT>
__global__ __launch_bounds__(512) void gemm_kw_kernel(const GemmParams p) {
  __shared__ __attribute__((aligned(1024))) char smem[KwTile<QUANT>::LDS];
  kw_tile_body<QUANT>(p, smem);
}
