// The tile GEMM of fp32 activations on the bf16 matrix cores, for the GEMM
// dispatcher. Included inside namespace mhsa { namespace { ... } } after
// common.hpp, kernels.hpp, quant.hpp and gemm_tile.hpp.
#pragma once

enum WKind { kWF32 = 0, kWBF16 = 1, kWU8 = 2 };

// A[row, :] . W[col + c, :], c = 0..3, in plain fp32, four chains each (the
// epilogue's recomputation).
template <int WK>
__device__ __forceinline__ floatx4 f32_dot4(const GemmParams& p, int row, int col) {
  const float* a = reinterpret_cast<const float*>(p.A) + (int64_t)row * p.lda;
  const int64_t w0 = (int64_t)col * p.K;
  floatx4 s[4] = {};
#pragma unroll 1
  for (int k0 = 0; k0 < p.K; k0 += 64) {
    floatx2 sb[4];
    if constexpr (WK == kWU8) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        sb[c] = *reinterpret_cast<const floatx2*>(p.sb + 2 * ((int64_t)(col + c) * (p.K / 64) + k0 / 64));
    }
#pragma unroll 4
    for (int k = k0; k < k0 + 64; k += 4) {
      const floatx4 av = *reinterpret_cast<const floatx4*>(a + k);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int64_t at = w0 + (int64_t)c * p.K + k;
        floatx4 w;
        if constexpr (WK == kWF32) {
          w = *reinterpret_cast<const floatx4*>(reinterpret_cast<const float*>(p.W) + at);
        } else if constexpr (WK == kWBF16) {
          const bf16x4 wv = *reinterpret_cast<const bf16x4*>(reinterpret_cast<const bf16*>(p.W16) + at);
          w = floatx4{(float)wv[0], (float)wv[1], (float)wv[2], (float)wv[3]};
        } else {
          const uint32_t q = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const unsigned char*>(p.W) + at);
#pragma unroll
          for (int e = 0; e < 4; ++e) w[e] = __builtin_fmaf(sb[c].x, (float)((q >> (8 * e)) & 0xFFu), sb[c].y);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) s[c][e] = __builtin_fmaf(av[e], w[e], s[c][e]);
      }
    }
  }
  floatx4 r;
#pragma unroll
  for (int c = 0; c < 4; ++c) r[c] = (s[c][0] + s[c][1]) + (s[c][2] + s[c][3]);
  return r;
}

// Values under 2^-110 have parts below the smallest bf16, 2^-133, which are
// lost: up to 2^-134 of each. A sum of at least this, of up to 2^14 products
// with weights up to 2^8, is off by no more than 2^-26 of it. (A matrix of
// nothing else takes 10 to 15 times a launch, each weight read by every lane.)
constexpr float kF32Small = 0x1p-86f;

// A lane's sums that are not numbers of full precision, run by whole waves.
// Sums that are not finite come from leading parts alone (f32_sum), which
// carry an infinite value as it is, so what is left to know is the row's: with
// a NaN in it (whose leading part may be an infinity) every sum is NaN, with
// an infinity the sum stands, without either (an overflow, a weight that is
// not finite) it is recomputed, as small ones are. The wave reads a row once
// for all its lanes: recomputing each sum of rows with an infinity took up to
// 18 times a launch.
template <int WK>
__device__ __forceinline__ void f32_mend(const GemmParams& p, bool ok, int row, int col, floatx4& v) {
  bool odd = false;
#pragma unroll
  for (int e = 0; e < 4; ++e) odd = odd || (ok && !(__builtin_fabsf(v[e]) < INFINITY));
  bool has_nan = false, has_inf = false;
  for (uint64_t left = __ballot(odd); left;) {
    const int r = __builtin_amdgcn_readlane(row, __builtin_ctzll(left));
    const float* a = reinterpret_cast<const float*>(p.A) + (int64_t)r * p.lda;
    bool n = false, i = false;
    for (int k = 4 * (int)(threadIdx.x & 63); k < p.K; k += 256) {
      const floatx4 x = *reinterpret_cast<const floatx4*>(a + k);
#pragma unroll
      for (int e = 0; e < 4; ++e) n = n || x[e] != x[e], i = i || __builtin_fabsf(x[e]) == INFINITY;
    }
    n = __any(n), i = __any(i);
    if (row == r) has_nan = n, has_inf = i;
    left &= ~__ballot(row == r);
  }
  bool again[4], any = false;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const bool finite = __builtin_fabsf(v[e]) < INFINITY;
    again[e] = ok && (finite ? v[e] != 0.f && __builtin_fabsf(v[e]) < kF32Small : !has_nan && !has_inf);
    any = any || again[e];
    if (!finite && has_nan) v[e] = NAN;
  }
  if (any) {
    const floatx4 d = f32_dot4<WK>(p, row, col);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = again[e] ? d[e] : v[e];
  }
}

// The sum of a wave's accumulators: an infinite or NaN value's lower parts are
// NaN, and its leading products alone say what its sums are.
__device__ __forceinline__ float f32_sum(float lead, float rest) {
  return __builtin_fabsf(lead) < INFINITY ? lead + rest : lead;
}

// Columns [col, col + 4) of a row: the sums `v`, then the epilogue in the
// reference's order (bias, SiLU, scaled residual) and the store. Whole waves,
// `ok` where there is such a row.
template <int WK>
__device__ __forceinline__ void f32_store(const GemmParams& p, bool ok, int row, int col, floatx4 v) {
  auto whole = [](float x) { return __builtin_fabsf(x) >= kF32Small && __builtin_fabsf(x) < INFINITY; };
  if (__any(ok && !(whole(v[0]) && whole(v[1]) && whole(v[2]) && whole(v[3])))) f32_mend<WK>(p, ok, row, col, v);
  if (!ok) return;
  if (p.bias) v += *reinterpret_cast<const floatx4*>(p.bias + col);
  if (p.act == kActSilu) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = silu_value<float>(v[e]);
  }
  if (p.R) {
    const floatx4 r = *reinterpret_cast<const floatx4*>(reinterpret_cast<const float*>(p.R) + (int64_t)row * p.ldr + col);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = r[e] + p.res_scale * v[e];
  }
  float* dst;
  if (!p.C2) dst = reinterpret_cast<float*>(p.C) + row_offset(p, row) + col;
  else if (col < p.c2_col0) dst = reinterpret_cast<float*>(p.C) + (int64_t)row * p.ldc + col;
  else dst = reinterpret_cast<float*>(p.C2) + mapped_row(p, row) * p.ldc2 + col - p.c2_col0;
  *reinterpret_cast<floatx4*>(dst) = v;
}

// fp32 activations times fp32, bf16 or u8 weights. The fp32 MFMA is what
// bounded the kernels before (157 TFLOP/s, a sixteenth of the bf16 one), so
// the operands go through the bf16 MFMAs in three exact parts: three products
// per weight that is a bf16 value, eight per fp32 or dequantised one. Operands
// stream raw through NS LDS stages of 64 k-columns with direct-to-LDS loads
// (fp32 rows are 4 bytes a value there against 6 for their parts), and each
// wave splits its fragments in registers, one step ahead, between the MFMAs
// of the step before. The vector work is what bounds it now: the counters show
// 8 to 11 vector instructions per MFMA (the 64 x 64 and 32 x 64 tiles of fp32
// weights; 7.6 in the 64 x 128 ones of bf16 weights), whose 32 cycles hold 8,
// and MFMAs a third of the time (profiles/mfma_utilization.txt). The split of a
// fragment takes 44, so the waves share a tile along K first,
// where no fragment is split twice, and along M only with bf16 weights, which
// need no split; two workgroups per CU overlap each other's barriers.
// Measured (us before / now, MFMA rate now in bf16 products), 1500 rows:
// 4096 x 1024 bf16 weights 154 / 44 (860 TFLOP/s), fp32 155 / 108 (930), u8
// 157 / 106; 1024 x 4096 bf16 169 / 48, fp32 171 / 106; 224 rows: 4096 x 1024
// bf16 25.5 / 10.8, fp32 25.8 / 21.3, 1024 x 4096 bf16 30.5 / 15.0, fp32 30.6
// / 25.1. Its error against 64 bits is 0.9e-7 at K = 1024 (K-parallel kernel
// 1.6e-7, fp32 tiles before 5.3-6.4e-7) and 2.5e-8 for a single product, as
// fp32's. (Six products, without m l and l m, take 85 us on the first fp32
// shape, but a sum of one product is then up to 2.5e-7 off, not 6e-8.)
//
// MW x NW x KW waves: MW along the tile's rows, NW along its columns, KW
// along the contraction (each of those takes 4 / KW of a stage's four
// 16-column steps, and the partial tiles meet in LDS in the epilogue).
template <int BM, int BN, int MW, int NW, int KW, int WK, int NS_>
struct F32Tile {
  static constexpr int NS = NS_, NWV = MW * NW * KW, NT = 64 * NWV;
  static constexpr int WM = BM / MW, WN = BN / NW, TM = WM / 32, TN = WN / 32;
  static constexpr int KST = 4 / KW;               // 16-column steps per wave and stage
  static constexpr int PB = WK == kWBF16 ? 1 : 3;  // parts of a weight
  // a stage holds 64 k-columns: A rows of 256 bytes (fp32), B rows of 256
  // (fp32), 128 (bf16) or 64 bytes (codes, and 8 bytes of {scale, bias})
  static constexpr int BROW = WK == kWF32 ? 256 : WK == kWBF16 ? 128 : 64;
  static constexpr int ABYTES = BM * 256, BBYTES = BN * BROW, SBYTES = WK == kWU8 ? BN * 8 : 0;
  static constexpr int STAGE = ABYTES + BBYTES + SBYTES;
  static constexpr int NA = ABYTES / 1024 / NWV, NB = BBYTES / 1024 / NWV;  // 1 KB loads per wave and stage
  static constexpr int NQ = WK == kWU8 ? (BN / 32 + NWV - 1) / NWV : 0;     // 256 B scale loads per wave and stage
  static constexpr int NL = NA + NB + NQ;
  static constexpr int PITCH = WN * 4 + 16;        // epilogue staging row
  static constexpr int EPP = NWV * WM * PITCH <= 160 * 1024 ? 1 : TM;  // epilogue passes
  static constexpr int EROWS = WM / EPP;           // rows of a wave's block per pass
  static constexpr int EREG = EROWS * PITCH;
  static constexpr int LDS = NS * STAGE > NWV * EREG ? NS * STAGE : NWV * EREG;
  // waves per SIMD: two workgroups share a CU where LDS holds both
  static constexpr int OCC = NWV / 4 * (LDS <= 80 * 1024 ? 2 : 1);
  static_assert(NA * 1024 * NWV == ABYTES && NB * 1024 * NWV == BBYTES, "stage split");
  static_assert(LDS <= 160 * 1024 && (NS - 1) * NL < 64, "stage limits");
};

template <int BM, int BN, int MW, int NW, int KW, int WK, int NS>
__device__ __forceinline__ void f32_tile_body(const GemmParams& p, int splits, int block, char* smem) {
  using C = F32Tile<BM, BN, MW, NW, KW, WK, NS>;
  constexpr int TM = C::TM, TN = C::TN;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kw = w % KW, wn = w / KW % NW, wm = w / (KW * NW);
  const int hh = lane >> 5, c32 = lane & 31;

  // contiguous item ranges per XCD, 8 row tiles at a time (as the bf16 tile
  // kernel); the K splits are the slowest index
  const int tilesM = (p.M + BM - 1) / BM, tilesN = p.N / BN, nt = tilesM * tilesN;
  const int items = nt * splits, per = (items + 7) / 8;
  const int item = (int)((unsigned)block % 8u) * per + (int)((unsigned)block / 8u);
  if ((int)((unsigned)block / 8u) >= per || item >= items) return;
  const int z = item / nt, W = item % nt;
  constexpr int GM = 8;
  const int gsz = GM * tilesN, first = W / gsz * GM, gm = min(tilesM - first, GM);
  const int m0 = (first + (W % gsz) % gm) * BM, n0 = (W % gsz) / gm * BN;
  const int m_end = min(m0 + BM, p.M);
  const int nkt = p.K / 64, kt0 = (int)((int64_t)z * nkt / splits), nk = (int)((int64_t)(z + 1) * nkt / splits) - kt0;

  // A and fp32 B: 1 KB load g of wave w fills rows 4 (w NA + g) + [0, 4):
  // lane l stores row l / 16, 16-byte chunk l % 16, which holds chunk
  // (l % 16) ^ (row % 16), so the 16 rows an LDS read serves together hit
  // all 64 banks. bf16 and u8 rows as in the bf16 tile kernel.
  // (the tile's rows alone: all of A may be past 2 GiB)
  const char* Ab = reinterpret_cast<const char*>(p.A) + (int64_t)m0 * p.lda * 4;
  const __amdgpu_buffer_rsrc_t ra =
      __builtin_amdgcn_make_buffer_rsrc((void*)Ab, (short)0, (int)((int64_t)(m_end - m0) * p.lda * 4), kRawBuffer);
  int aoff[C::NA], boff[C::NB];
#pragma unroll
  for (int g = 0; g < C::NA; ++g) {
    const int row = (w * C::NA + g) * 4 + (lane >> 4);
    aoff[g] = (int)(row * p.lda * 4 + 16 * ((lane & 15) ^ (row & 15)));
  }
  constexpr int ES = WK == kWF32 ? 4 : WK == kWBF16 ? 2 : 1;
  const char* Bb = reinterpret_cast<const char*>(WK == kWBF16 ? p.W16 : p.W) + (int64_t)n0 * p.K * ES;
  const __amdgpu_buffer_rsrc_t rb =
      __builtin_amdgcn_make_buffer_rsrc((void*)Bb, (short)0, (int)((int64_t)BN * p.K * ES), kRawBuffer);
#pragma unroll
  for (int g = 0; g < C::NB; ++g) {
    if constexpr (WK == kWF32) {
      const int row = (w * C::NB + g) * 4 + (lane >> 4);
      boff[g] = row * p.K * 4 + 16 * ((lane & 15) ^ (row & 15));
    } else if constexpr (WK == kWBF16) {
      const int row = (w * C::NB + g) * 8 + (lane >> 3);
      boff[g] = row * p.K * 2 + 16 * ((lane & 7) ^ ((row >> 1) & 7));
    } else {
      const int row = (w * C::NB + g) * 16 + (lane >> 2);
      boff[g] = row * p.K + 16 * ((lane & 3) ^ ((row >> 2) & 3));
    }
  }
  // {scale, bias} of 32 rows per load (two lanes a row); waves past the
  // tile's rows load the same ones again, so every wave's count is the same
  const int groups = p.K / 64;
  __amdgpu_buffer_rsrc_t rs;
  int qoff[C::NQ ? C::NQ : 1], qrow[C::NQ ? C::NQ : 1];
  if constexpr (C::NQ > 0) {
    rs = __builtin_amdgcn_make_buffer_rsrc((void*)(p.sb + 2 * (int64_t)n0 * groups), (short)0,
                                           (int)((int64_t)BN * groups * 8), kRawBuffer);
#pragma unroll
    for (int g = 0; g < C::NQ; ++g) {
      qrow[g] = (w * C::NQ + g) * 32 % BN;
      qoff[g] = ((qrow[g] + (lane >> 1)) * groups) * 8 + 4 * (lane & 1);
    }
  }
  auto issue = [&](int kt, int buf) {
    char* S = smem + buf * C::STAGE;
    const int k = kt0 + min(kt, nk - 1);
#pragma unroll
    for (int g = 0; g < C::NA; ++g)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void*)(S + (w * C::NA + g) * 1024), 16, aoff[g], k * 256, 0, 0);
#pragma unroll
    for (int g = 0; g < C::NB; ++g)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_void*)(S + C::ABYTES + (w * C::NB + g) * 1024), 16, boff[g],
                                               k * C::BROW, 0, 0);
    if constexpr (C::NQ > 0) {
#pragma unroll
      for (int g = 0; g < C::NQ; ++g)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(S + C::ABYTES + C::BBYTES + qrow[g] * 8), 4, qoff[g],
                                                 k * 8, 0, 0);
    }
  };

  // Fragments of one 16-column step: lane l holds row l % 32, columns
  // 8 (l / 32) + [0, 8). Raw operands are read one step ahead, split into
  // parts during the step before their MFMAs.
  floatx4 xa[TM][2], xb[TN][2];
  u32x4 xw[TN];   // bf16 weights
  u32x2 xq[TN];   // codes
  floatx2 xs[TN];  // {scale, bias}
  u32x4 pa[2][TM][3], pb[2][TN][C::PB];
  auto rd = [&](const char* S, int s) {  // s: this wave's step in the stage
    const int ks = kw * C::KST + s;
    const char* A = S + (wm * C::WM + c32) * 256 + 16 * ((4 * ks + 2 * hh) ^ (lane & 15));
    const int x1 = 16 - 32 * ((lane & 1));  // chunk + 1 under the XOR
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      xa[i][0] = *reinterpret_cast<const floatx4*>(A + i * 8192);
      xa[i][1] = *reinterpret_cast<const floatx4*>(A + i * 8192 + x1);
    }
    const int brow = wn * C::WN + c32;
    const char* B = S + C::ABYTES + brow * C::BROW;
    if constexpr (WK == kWF32) {
      B += 16 * ((4 * ks + 2 * hh) ^ (lane & 15));
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        xb[j][0] = *reinterpret_cast<const floatx4*>(B + j * 8192);
        xb[j][1] = *reinterpret_cast<const floatx4*>(B + j * 8192 + x1);
      }
    } else if constexpr (WK == kWBF16) {
      B += 16 * ((2 * ks + hh) ^ ((lane >> 1) & 7));
#pragma unroll
      for (int j = 0; j < TN; ++j) xw[j] = *reinterpret_cast<const u32x4*>(B + j * 4096);
    } else {
      B += 16 * (ks ^ ((lane >> 2) & 3)) + 8 * hh;
      const char* Q = S + C::ABYTES + C::BBYTES + brow * 8;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        xq[j] = *reinterpret_cast<const u32x2*>(B + j * 2048);
        xs[j] = *reinterpret_cast<const floatx2*>(Q + j * 256);
      }
    }
  };
  // piece c of the conversion of the raw operands to set `b`: pair c % 4 of
  // fragment c / 4 (A's fragments, then B's)
  constexpr int NP = 4 * (TM + TN);
  auto cvt = [&](int c, int b) {
    const int f = c >> 2, q = c & 3;
    uint32_t h, m, l;
    if (f < TM) {
      split_pair(xa[f][q >> 1][2 * (q & 1)], xa[f][q >> 1][2 * (q & 1) + 1], h, m, l);
      pa[b][f][0][q] = h, pa[b][f][1][q] = m, pa[b][f][2][q] = l;
      return;
    }
    const int j = f - TM;
    if constexpr (WK == kWBF16) {
      pb[b][j][0][q] = xw[j][q];
    } else {
      float u, v;
      if constexpr (WK == kWF32) {
        u = xb[j][q >> 1][2 * (q & 1)], v = xb[j][q >> 1][2 * (q & 1) + 1];
      } else {
        const uint32_t cw = xq[j][q >> 1] >> (16 * (q & 1));
        u = __builtin_fmaf(xs[j].x, (float)(cw & 0xFFu), xs[j].y);
        v = __builtin_fmaf(xs[j].x, (float)((cw >> 8) & 0xFFu), xs[j].y);
      }
      split_pair(u, v, h, m, l);
      pb[b][j][0][q] = h, pb[b][j][C::PB / 2][q] = m, pb[b][j][C::PB - 1][q] = l;
    }
  };

  // The products kept (activation part, weight part), smallest first: all but
  // l l, which is below 2^-30 of a product. h h, exact in fp32, and the
  // others, 2^-6 of it and less, add up apart: the large sum is rounded once
  // per 16 columns instead of once per product, and a product that makes up a
  // sum by itself as if it were rounded from all its bits.
  floatx16 acc[2][TN][TM];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i) acc[0][j][i] = floatx16{}, acc[1][j][i] = floatx16{};
  constexpr int NPR = C::PB == 1 ? 3 : 8;
  constexpr int PRA[8] = {2, 1, 2, 0, 1, 0, 1, 0}, PRB[8] = {1, 2, 0, 0, 0, 2, 1, 1};
  constexpr int PRA1[3] = {2, 0, 1};
  constexpr int NM = NPR * TM * TN, LEAD = NM / 5;
  constexpr int CG = 2;  // MFMAs (and conversion pieces) scheduled together

#pragma unroll
  for (int st = 0; st < NS; ++st) issue(st, st);
  {
    constexpr int vm = (NS - 1) * C::NL;
    __builtin_amdgcn_s_waitcnt((vm & 15) | ((vm >> 4) << 14) | (7 << 4));
    asm volatile("s_barrier" ::: "memory");
  }
  // after the reads of this stage's last step: the next stage has landed in
  // every wave's share, and this stage's buffer takes stage kt + NS
  auto turn = [&](int kt) {
    constexpr int vm = (NS - 2) * C::NL;
    __builtin_amdgcn_s_waitcnt((vm & 15) | ((vm >> 4) << 14) | (7 << 4));  // lgkmcnt(0)
    asm volatile("s_barrier" ::: "memory");
    issue(kt + NS, kt % NS);
  };
  rd(smem, 0);
#pragma unroll
  for (int c = 0; c < NP; ++c) cvt(c, 0);
  if constexpr (C::KST == 1) {
    turn(0);
    rd(smem + (1 % NS) * C::STAGE, 0);
  } else {
    rd(smem, 1);
  }
  // step s of stage kt, parts in set b: its MFMAs with the conversion of the
  // next step's operands between them, then the reads of the step after it
  auto step = [&](int kt, int s, int b) {
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      const int pr = m / (TM * TN), t = m % (TM * TN), j = t / TM, i = t % TM;
      const int ia = C::PB == 1 ? PRA1[pr % 3] : PRA[pr], ib = C::PB == 1 ? 0 : PRB[pr];
      floatx16& d = acc[ia + ib == 0 ? 0 : 1][j][i];
      d = mma32(__builtin_bit_cast(bf16x8, pb[b][j][ib]), __builtin_bit_cast(bf16x8, pa[b][i][ia]), d);
#pragma unroll
      for (int c = 0; c < NP; ++c)
        if (LEAD + c / CG * CG * (NM - LEAD) / NP == m) cvt(c, b ^ 1);
      if (m % CG == CG - 1) __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (C::KST == 1) {
      turn(kt + 1);
      rd(smem + (kt + 2) % NS * C::STAGE, 0);
    } else if (s == C::KST - 2) {
      turn(kt);
      rd(smem + (kt + 1) % NS * C::STAGE, 0);
    } else {
      rd(smem + (s == C::KST - 1 ? kt + 1 : kt) % NS * C::STAGE, s == C::KST - 1 ? 1 : s + 2);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  if constexpr (C::KST == 1) {
    int kt = 0;
    for (; kt + 1 < nk; kt += 2) step(kt, 0, 0), step(kt + 1, 0, 1);
    if (kt < nk) step(kt, 0, 0);
  } else {
    for (int kt = 0; kt < nk; ++kt)
#pragma unroll
      for (int s = 0; s < C::KST; ++s) step(kt, s, s & 1);
  }

  if (p.acopy && z == 0) {
    // each column tile copies its share of the rows of A (the first tile's
    // workgroup alone took 3 us longer than the others at 64 x 3072 x 1024)
    const int total = (m_end - m0) * (p.K / 4), each = (total + tilesN - 1) / tilesN, tn = n0 / BN;
    for (int id = tn * each + tid; id < min((tn + 1) * each, total); id += C::NT) {
      const int row = m0 + id / (p.K / 4), c = id % (p.K / 4) * 4;
      *reinterpret_cast<floatx4*>(reinterpret_cast<float*>(p.acopy) + mapped_row(p, row) * p.acopy_ld + c) =
          *reinterpret_cast<const floatx4*>(reinterpret_cast<const float*>(p.A) + (int64_t)row * p.lda + c);
    }
  }

  // The partial tiles row-major in LDS (a lane holds row 32 i + lane % 32,
  // columns 32 j + 8 q + 4 (lane / 32) + [0, 4) of its block; the pitch puts
  // 16 rows of a store on all banks), then 16-byte runs summed over the KW
  // copies in order and stored.
  __builtin_amdgcn_s_waitcnt(0);
#pragma unroll
  for (int ep = 0; ep < C::EPP; ++ep) {
    __syncthreads();
    char* st = smem + w * C::EREG + c32 * C::PITCH + 16 * hh;
#pragma unroll
    for (int i = ep * (TM / C::EPP); i < (ep + 1) * (TM / C::EPP); ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<floatx4*>(st + (i - ep * (TM / C::EPP)) * 32 * C::PITCH + (32 * j + 8 * q) * 4) =
              floatx4{f32_sum(acc[0][j][i][4 * q], acc[1][j][i][4 * q]),
                      f32_sum(acc[0][j][i][4 * q + 1], acc[1][j][i][4 * q + 1]),
                      f32_sum(acc[0][j][i][4 * q + 2], acc[1][j][i][4 * q + 2]),
                      f32_sum(acc[0][j][i][4 * q + 3], acc[1][j][i][4 * q + 3])};
    __syncthreads();
    constexpr int CR = BN / 4, NCH = MW * C::EROWS * CR;  // runs per row, runs per pass
    static_assert(NCH % C::NT == 0, "runs per thread");
#pragma unroll 4
    for (int it = 0; it < NCH / C::NT; ++it) {
      const int id = it * C::NT + tid, er = id / CR, cc = id % CR * 4;
      const int bm = er / C::EROWS, r = er % C::EROWS, bn = cc / C::WN;
      const int row = m0 + bm * C::WM + ep * C::EROWS + r, col = n0 + cc;
      const char* src = smem + (bm * NW + bn) * KW * C::EREG + r * C::PITCH + (cc - bn * C::WN) * 4;
      floatx4 v = *reinterpret_cast<const floatx4*>(src);
#pragma unroll
      for (int k = 1; k < KW; ++k) v += *reinterpret_cast<const floatx4*>(src + k * C::EREG);
      if (splits > 1) {
        if (row < m_end) *reinterpret_cast<floatx4*>(p.partial + ((int64_t)z * p.M + row) * p.N + col) = v;
        continue;
      }
      f32_store<WK>(p, row < m_end, row, col, v);
    }
  }
}

template <int BM, int BN, int MW, int NW, int KW, int WK, int NS>
__global__ __launch_bounds__(64 * MW * NW * KW, (F32Tile<BM, BN, MW, NW, KW, WK, NS>::OCC))
void gemm_f32_tile_kernel(const GemmParams p, int splits) {
  __shared__ __attribute__((aligned(1024))) char smem[F32Tile<BM, BN, MW, NW, KW, WK, NS>::LDS];
  f32_tile_body<BM, BN, MW, NW, KW, WK, NS>(p, splits, (int)blockIdx.x, smem);
}

// Sums the K splits in order, then the epilogue: 4 columns per thread.
template <int WK>
__global__ __launch_bounds__(256) void gemm_f32_reduce_kernel(const GemmParams p, int splits) {
  const int64_t total = (int64_t)p.M * p.N;
  const int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  const bool ok = e < total;
  floatx4 v{};
  if (ok) {
    v = *reinterpret_cast<const floatx4*>(p.partial + e);
#pragma unroll 4
    for (int z = 1; z < splits; ++z) v += *reinterpret_cast<const floatx4*>(p.partial + z * total + e);
  }
  f32_store<WK>(p, ok, (int)(e / p.N), (int)(e % p.N), v);
}
