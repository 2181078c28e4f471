// Offline fp32 attention on the bf16 matrix cores, for the attention
// dispatcher. Included inside namespace mhsa { namespace { ... } } of
// attention.hip, after its query and key interval helpers.
#pragma once

// The fp32 form of the attention for inputs long enough to give the CUs a
// workgroup each. The fp32 MFMA bounded it (157 TFLOP/s; the kernel reached a
// quarter of that), so K, V, the position rows, the queries and the
// probabilities go through the bf16 MFMAs as three exact bf16 parts each
// (split_pair), eight products per pair of values: what is left out is below
// 2^-30 of a product. In the scores the product of the leading parts, exact in
// fp32, and the others add up apart, so a large sum is rounded once per 32
// terms, and one that a product makes up as the product of all its bits. (Six
// products leave out up to 2^-22: a score of one large product was then up to
// 2.5e-7 of it off, 6.0e-8 so.)
//
// A workgroup of 4 waves owns 64 queries of one (batch, head), 16 a wave, and
// walks the keys in tiles of 32. Rows are split once per workgroup, on their
// way to LDS: K as 32 rows and V^T as DK rows of 32 keys, each in three
// planes, and the position rows in a ring of three blocks of 32, of which a
// tile brings one (the 95 rows a tile reaches move on by 32). The next tile's
// rows load while this one computes, and are split between its PV products.
// V^T holds key 16 u + 4 g + r at 8 g + 4 u + r, the order in which a lane has
// the probabilities. Rows' 16-byte chunks are XOR-permuted by the row so that
// 16 rows of one fragment read cover all banks (V^T: an 80-byte pitch). The
// grid has the heads first, so a head's blocks share an XCD's L2.
// Measured, 4 x 375 frames, 8 heads of 128: 84.7 -> 61 us; a whole layer of 3 x
// 1500 frames 1305 -> 950 us, of 2 x 750 frames at 8 heads of 64 148 -> 120;
// error against 64 bits 9.8e-7 -> 3.6e-7 (4 x 375), 1.0e-6 -> 5.2e-7 (3 x 1500).
// What bounds it now at d_k = 128: LDS holds one workgroup per CU, so a SIMD
// has one wave, whose 224 products (3,600 cycles a tile), vector instructions
// (4.8 per product by the counters, 4,300 cycles) and LDS reads add up instead
// of overlapping.
template <int DK>
struct F32Attn {
  static constexpr int NT = 256, QB = 64, NK = 32;
  static constexpr int RB = DK * 2, VP = NK * 2 + 16;  // bytes of a K / position row and of a V^T row, per part
  static constexpr int KPART = NK * RB, VPART = DK * VP, PPART = 3 * NK * RB;
  static constexpr int V_OFF = 3 * KPART, P_OFF = V_OFF + 3 * VPART, R_OFF = P_OFF + 3 * PPART;
  static constexpr int RMP = NK + 20;  // remap row pitch (floats)
  static constexpr int LDS = R_OFF + 4 * 16 * RMP * 4;
  static constexpr int KC = NK * DK / 8 / NT;  // 8-value chunks of a 32-row block per thread
  static constexpr int VK = NK * DK / 4 / NT;  // keys of a thread's 4-column piece of V
  static constexpr int WPS = LDS <= 80 * 1024 ? 2 : 1;  // workgroups per CU
  static_assert(KC >= 1 && (VK == 2 || VK == 4) && LDS <= 160 * 1024, "tile split");
};

// V's values under 2^-110 have parts below the smallest bf16, 2^-133, which are
// lost: up to 2^-134 of each, and so of their mean, 2^-48 of this. (In the
// scores such values do not show.)
constexpr float kF32AttnSmall = 0x1p-86f;

// One query in plain fp32 by one wave (for the queries whose sums met a value
// that the parts cannot carry): 64 keys at a time, a key per lane for the
// scores, columns l and l + 64 per lane for the output. A NaN in the query or
// among the visible scores makes the output NaN and ends it.
template <int DK>
__device__ __forceinline__ void attn_f32_plain(const AttnParams& p, int bl, int h, int i, float sc_qk, float sc_bd) {
  constexpr int N = DK / 64;
  const int lane = threadIdx.x & 63, b = p.b0 + bl;
  const float* q = reinterpret_cast<const float*>(p.q) + (int64_t)b * p.q_bs + (int64_t)i * p.q_rs + h * DK;
  const float* kb = reinterpret_cast<const float*>(p.k) + (int64_t)b * p.kv_bs + h * DK;
  const float* vb = reinterpret_cast<const float*>(p.v) + (int64_t)b * p.kv_bs + h * DK + lane;
  const float* pb = reinterpret_cast<const float*>(p.p) + h * DK;
  float* orow = reinterpret_cast<float*>(p.o) + (int64_t)b * p.o_bs + (int64_t)i * p.o_rs + h * DK + lane;
  float o[N], m = -INFINITY, l = 0.f;
  bool nan = false;
#pragma unroll
  for (int n = 0; n < N; ++n) {
    const float x = q[lane + 64 * n];
    o[n] = 0.f;
    nan = nan || x != x;
  }
  const int2 iv = query_interval(p, bl, i);
  nan = __any(nan) && iv.x < iv.y;
#pragma unroll 1
  for (int j0 = iv.x; j0 < iv.y && !nan; j0 += 64) {
    const int j = min(j0 + lane, iv.y - 1), tp = p.center - p.qoff - i + j;
    const bool ok = tp >= 0 && tp < p.p_rows;
    const int64_t row = (int64_t)key_row(p, j) * p.kv_rs;
    const float* prow = pb + (int64_t)(ok ? tp : 0) * p.p_rs;
    floatx4 s{}, t{};
#pragma unroll 4
    for (int d = 0; d < DK; d += 4) {
      const floatx4 x = *reinterpret_cast<const floatx4*>(q + d);
      const floatx4 k = *reinterpret_cast<const floatx4*>(kb + row + d);
      const floatx4 r = *reinterpret_cast<const floatx4*>(prow + d);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[e] = __builtin_fmaf(x[e] + p.bias_u[h * DK + d + e], k[e], s[e]);
        t[e] = __builtin_fmaf(x[e] + p.bias_v[h * DK + d + e], ok ? r[e] : 0.f, t[e]);
      }
    }
    float v = ((s[0] + s[1]) + (s[2] + s[3])) * sc_qk + ((t[0] + t[1]) + (t[2] + t[3])) * sc_bd;
    if (j0 + lane >= iv.y) v = -INFINITY;
    float mn = fmaxf(m, v);
    for (int x = 32; x > 0; x >>= 1) mn = fmaxf(mn, __shfl_xor(mn, x, 64));
    const float mu = mn == -INFINITY ? 0.f : mn, alpha = __builtin_amdgcn_exp2f(m - mu);
    const float e = __builtin_amdgcn_exp2f(v - mu);
    m = mn;
    l = l * alpha + e;
    nan = __any(l != l);
    if (nan) break;
#pragma unroll
    for (int n = 0; n < N; ++n) o[n] *= alpha;
    const int keys = min(64, iv.y - j0);
    for (int x = 0; x < keys; ++x) {
      const float w = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, e), x));
      const float* vr = vb + (int64_t)key_row(p, j0 + x) * p.kv_rs;
#pragma unroll
      for (int n = 0; n < N; ++n) o[n] = __builtin_fmaf(w, vr[64 * n], o[n]);
    }
  }
  for (int x = 32; x > 0; x >>= 1) l += __shfl_xor(l, x, 64);
  const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
  for (int n = 0; n < N; ++n) orow[64 * n] = nan ? NAN : o[n] * inv;
}

// DEBUG: the position scores of the tiles it walks also go to dbg_bd.
template <int DK, bool DEBUG>
__global__ __launch_bounds__(256, F32Attn<DK>::WPS) void attn_f32_kernel(const AttnParams p) {
  using C = F32Attn<DK>;
  constexpr int NKF = DK / 32, ND = DK / 16, NK = C::NK, QB = C::QB;
  __shared__ __attribute__((aligned(16))) char smem[C::LDS];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, ql = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bl = blockIdx.z, b = p.b0 + bl, h = blockIdx.x, i0 = blockIdx.y * QB;
  const int qi = i0 + 16 * w + ql;
  float* Rm = reinterpret_cast<float*>(smem + C::R_OFF) + w * 16 * C::RMP;

  // the queries with the position biases, in parts: B operands
  u32x4 qu[NKF][3], qv[NKF][3];
  {
    const float* qrow = reinterpret_cast<const float*>(p.q) + (int64_t)b * p.q_bs + (int64_t)qi * p.q_rs + h * DK;
    const bool ok = qi < p.T;
#pragma unroll
    for (int kf = 0; kf < NKF; ++kf)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int d0 = kf * 32 + g * 8 + 4 * c;
        const floatx4 x = load16<floatx4>(qrow + d0, ok);
        const floatx4 u = *reinterpret_cast<const floatx4*>(p.bias_u + h * DK + d0);
        const floatx4 v = *reinterpret_cast<const floatx4*>(p.bias_v + h * DK + d0);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          uint32_t hh, mm, ll;
          split_pair(x[2 * e] + u[2 * e], x[2 * e + 1] + u[2 * e + 1], hh, mm, ll);
          qu[kf][0][2 * c + e] = hh, qu[kf][1][2 * c + e] = mm, qu[kf][2][2 * c + e] = ll;
          split_pair(x[2 * e] + v[2 * e], x[2 * e + 1] + v[2 * e + 1], hh, mm, ll);
          qv[kf][0][2 * c + e] = hh, qv[kf][1][2 * c + e] = mm, qv[kf][2][2 * c + e] = ll;
        }
      }
  }

  int jbeg, jend;
  key_range(p, bl, i0, min(i0 + QB, p.T), jbeg, jend);
  const int2 iv = query_interval(p, bl, qi);
  const float sc_qk = p.scale * kLog2e, sc_bd = p.scale_bd * kLog2e;
  const float* kbase = reinterpret_cast<const float*>(p.k) + (int64_t)b * p.kv_bs + h * DK;
  const float* vbase = reinterpret_cast<const float*>(p.v) + (int64_t)b * p.kv_bs + h * DK;
  const float* pbase = reinterpret_cast<const float*>(p.p) + h * DK;
  const int jfirst = jbeg / NK * NK, ntile = jend > jfirst ? (jend - jfirst + NK - 1) / NK : 0;
  const int pmin = p.center - p.qoff - (i0 + QB - 1) + jfirst;  // position row of ring block 0, row 0

  // Loads are unconditional: rows of keys that no query of the block sees
  // (padding may hold anything) or outside the table read row 0 and become
  // zeros. Chunk x of this thread: row and 8 columns.
  floatx4 kr[C::KC][2], pr[C::KC][2], vr[C::VK];
  const int vkq = tid % (NK / C::VK), vd = tid / (NK / C::VK) * 4;  // V: keys VK vkq + [0, VK), columns vd + [0, 4)
  auto crow = [&](int x) { return (tid + x * C::NT) / (DK / 8); };
  auto ccol = [&](int x) { return (tid + x * C::NT) % (DK / 8) * 8; };
  auto fetch_kv = [&](int j0) {
#pragma unroll
    for (int x = 0; x < C::KC; ++x) {
      const int j = j0 + crow(x);
      const bool ok = j >= jbeg && j < jend;
      const float* src = kbase + (int64_t)(ok ? key_row(p, j) : 0) * p.kv_rs + ccol(x);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const floatx4 v = *reinterpret_cast<const floatx4*>(src + 4 * c);
        kr[x][c] = ok ? v : floatx4{0.f, 0.f, 0.f, 0.f};
      }
    }
#pragma unroll
    for (int x = 0; x < C::VK; ++x) {
      const int j = j0 + C::VK * vkq + x;
      const bool ok = j >= jbeg && j < jend;
      const floatx4 v = *reinterpret_cast<const floatx4*>(vbase + (int64_t)(ok ? key_row(p, j) : 0) * p.kv_rs + vd);
      vr[x] = ok ? v : floatx4{0.f, 0.f, 0.f, 0.f};
    }
  };
  auto fetch_pos = [&](int blk) {
#pragma unroll
    for (int x = 0; x < C::KC; ++x) {
      const int tp = pmin + NK * blk + crow(x);
      const bool ok = tp >= 0 && tp < p.p_rows;
      const float* src = pbase + (int64_t)(ok ? tp : 0) * p.p_rs + ccol(x);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const floatx4 v = *reinterpret_cast<const floatx4*>(src + 4 * c);
        pr[x][c] = ok ? v : floatx4{0.f, 0.f, 0.f, 0.f};
      }
    }
  };
  u32x4 kp[C::KC][3], pp[C::KC][3];
  uint32_t vp[4][3][C::VK / 2];
  // piece c of the split of the fetched rows: position rows, K, then V, a pair at a time
  constexpr int NPIECE = 8 * C::KC + 2 * C::VK;
  auto split_piece = [&](int c) {
    if (c < 8 * C::KC) {
      const int x = c >> 2 & (C::KC - 1), e = c & 3;
      const floatx4(&r)[2] = c < 4 * C::KC ? pr[x] : kr[x];
      u32x4(&d)[3] = c < 4 * C::KC ? pp[x] : kp[x];
      uint32_t hh, mm, ll;
      split_pair(r[e >> 1][2 * (e & 1)], r[e >> 1][2 * (e & 1) + 1], hh, mm, ll);
      d[0][e] = hh, d[1][e] = mm, d[2][e] = ll;
    } else {
      const int e = (c - 8 * C::KC) & 3, x = (c - 8 * C::KC) >> 2;
      split_pair(vr[2 * x][e], vr[2 * x + 1][e], vp[e][0][x], vp[e][1][x], vp[e][2][x]);
    }
  };
  auto swz = [&](int row, int chunk) { return 16 * (chunk ^ (DK == 128 ? row & 15 : (row >> 1) & 7)); };
  auto store_pos = [&](int blk) {
#pragma unroll
    for (int x = 0; x < C::KC; ++x) {
      char* dst = smem + C::P_OFF + (blk % 3 * NK + crow(x)) * C::RB + swz(crow(x), ccol(x) >> 3);
#pragma unroll
      for (int t = 0; t < 3; ++t) *reinterpret_cast<u32x4*>(dst + t * C::PPART) = pp[x][t];
    }
  };
  auto store_kv = [&]() {
#pragma unroll
    for (int x = 0; x < C::KC; ++x) {
      char* dst = smem + crow(x) * C::RB + swz(crow(x), ccol(x) >> 3);
#pragma unroll
      for (int t = 0; t < 3; ++t) *reinterpret_cast<u32x4*>(dst + t * C::KPART) = kp[x][t];
    }
    const int key = C::VK * vkq, at = 8 * (key >> 2 & 3) + 4 * (key >> 4) + (key & 3);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        char* dst = smem + C::V_OFF + t * C::VPART + (vd + e) * C::VP + at * 2;
        if constexpr (C::VK == 4) *reinterpret_cast<u32x2*>(dst) = u32x2{vp[e][t][0], vp[e][t][C::VK / 2 - 1]};
        else *reinterpret_cast<uint32_t*>(dst) = vp[e][t][0];
      }
  };

  auto parts = [&](const char* at, int part_bytes, bf16x8 (&a)[3]) {
#pragma unroll
    for (int t = 0; t < 3; ++t) a[t] = *reinterpret_cast<const bf16x8*>(at + t * part_bytes);
  };
  // the eight products of two values in parts, smallest first (part of the
  // row, part of the query or probability)
  constexpr int NX = 8, PRA[NX] = {2, 1, 2, 0, 1, 1, 0, 0}, PRB[NX] = {1, 2, 0, 2, 1, 0, 1, 0};

  floatx4 o[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) o[d] = floatx4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;

  if (ntile > 0) {
#pragma unroll 1
    for (int blk = 0; blk < 2; ++blk) {
      fetch_pos(blk);
#pragma unroll
      for (int c = 0; c < 4 * C::KC; ++c) split_piece(c);
      store_pos(blk);
    }
    fetch_kv(jfirst);
    fetch_pos(2);
#pragma unroll
    for (int c = 0; c < NPIECE; ++c) split_piece(c);
  }
  for (int t = 0; t < ntile; ++t) {
    const int j0 = jfirst + NK * t;
    __syncthreads();  // the previous tile is consumed
    store_kv();
    store_pos(t + 2);
    __syncthreads();

    // S^T = K Qu^T and the wave's band B'^T = P' Qv^T: 16-row sub-tiles at
    // rows 48 - 16 w + 16 n of the tile's 95 position rows
    floatx4 sh[2], sl[2], bh[3], bl3[3];
#pragma unroll
    for (int u = 0; u < 2; ++u) sh[u] = sl[u] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int n = 0; n < 3; ++n) bh[n] = bl3[n] = floatx4{0.f, 0.f, 0.f, 0.f};
    int brow[3];
#pragma unroll
    for (int n = 0; n < 3; ++n) {
      const int r = 48 - 16 * w + 16 * n;
      brow[n] = (t + (r >> 5)) % 3 * NK + (r & 31);
    }
    // each kind's fragments are read while the other's products run
    bf16x8 ka[2][3], pa[3][3];
    auto read_k = [&](int kf) {
#pragma unroll
      for (int u = 0; u < 2; ++u) parts(smem + (16 * u + ql) * C::RB + swz(ql, 4 * kf + g), C::KPART, ka[u]);
    };
    read_k(0);
#pragma unroll
    for (int kf = 0; kf < NKF; ++kf) {
#pragma unroll
      for (int n = 0; n < 3; ++n)
        parts(smem + C::P_OFF + (brow[n] + ql) * C::RB + swz(ql, 4 * kf + g), C::PPART, pa[n]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < NX; ++x)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          floatx4& d = x < NX - 1 ? sl[u] : sh[u];
          d = mma16(ka[u][PRA[x]], __builtin_bit_cast(bf16x8, qu[kf][PRB[x]]), d);
        }
      __builtin_amdgcn_sched_barrier(0);
      if (kf + 1 < NKF) read_k(kf + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < NX; ++x)
#pragma unroll
        for (int n = 0; n < 3; ++n) {
          floatx4& d = x < NX - 1 ? bl3[n] : bh[n];
          d = mma16(pa[n][PRA[x]], __builtin_bit_cast(bf16x8, qv[kf][PRB[x]]), d);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
    fetch_kv(min(j0 + NK, jfirst + NK * (ntile - 1)));  // (the last tile loads itself again, unused)
    fetch_pos(t + 3);

    // rel_shift as an LDS remap: band row n of query column ql holds the
    // pair (i = 16 w + ql, j = n - 15 + ql)
#pragma unroll
    for (int n = 0; n < 3; ++n) *reinterpret_cast<floatx4*>(Rm + ql * C::RMP + 16 * n + 4 * g) = bh[n] + bl3[n];
    __builtin_amdgcn_wave_barrier();
    float sc[8], tmax = -INFINITY;
    const bool full = __all(iv.x <= j0 && iv.y >= j0 + NK);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int u = e >> 2, r = e & 3, jl = 16 * u + 4 * g + r;
      const float bd = Rm[ql * C::RMP + jl + 15 - ql];
      if (DEBUG && qi < p.T && j0 + jl < p.L)
        p.dbg_bd[(((int64_t)b * p.H + h) * p.T + qi) * p.L + j0 + jl] = p.scale_bd * bd;
      const float v = (sh[u][r] + sl[u][r]) * sc_qk + bd * sc_bd;
      sc[e] = full || in_interval(j0 + jl, iv) ? v : -INFINITY;
      tmax = fmaxf(tmax, sc[e]);
    }
    __builtin_amdgcn_wave_barrier();
    tmax = col_max(tmax);
    // lazy rescale, as in attn_kernel
    if (__any(tmax > m_run + 8.f)) {
      const float m_new = fmaxf(m_run, tmax);
      const float alpha = __builtin_amdgcn_exp2f(m_run - (m_new == -INFINITY ? 0.f : m_new));
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < ND; ++d) o[d] *= alpha;
    }
    const float m_use = m_run == -INFINITY ? 0.f : m_run;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      sc[e] = __builtin_amdgcn_exp2f(sc[e] - m_use);
      l_run += sc[e];
    }
    u32x4 pb[3];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t hh, mm, ll;
      split_pair(sc[2 * e], sc[2 * e + 1], hh, mm, ll);
      pb[0][e] = hh, pb[1][e] = mm, pb[2][e] = ll;
    }
    // O^T += V^T Pr^T two 16-row pieces at a time, the next pieces' reads
    // ahead of the products and the next tile's rows split between them
    bf16x8 va[2][2][3];
    auto read_v = [&](int d2) {
#pragma unroll
      for (int x = 0; x < 2; ++x)
        parts(smem + C::V_OFF + (32 * d2 + 16 * x + ql) * C::VP + 16 * g, C::VPART, va[d2 & 1][x]);
    };
    constexpr int NMM = NX * ND;
    read_v(0);
#pragma unroll
    for (int d2 = 0; d2 < ND / 2; ++d2) {
      if (d2 + 1 < ND / 2) read_v(d2 + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < NX; ++x) {
#pragma unroll
        for (int y = 0; y < 2; ++y)
          o[2 * d2 + y] = mma16(va[d2 & 1][y][PRA[x]], __builtin_bit_cast(bf16x8, pb[PRB[x]]), o[2 * d2 + y]);
        constexpr int LEAD = ND;  // (the rows' loads get a first part of the products to land)
        const int mm = 2 * NX * d2 + 2 * x;
#pragma unroll
        for (int c = 0; c < NPIECE; ++c)
          if (LEAD + c * (NMM - LEAD) / NPIECE / 2 * 2 == mm) split_piece(c);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  // normalise; a query that saw no key outputs zeros
  const float l_tot = col_sum(l_run);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  bool odd = false;
  float* orow = reinterpret_cast<float*>(p.o) + (int64_t)b * p.o_bs + (int64_t)qi * p.o_rs + h * DK;
#pragma unroll
  for (int d = 0; d < ND; ++d) {
    const floatx4 v = o[d] * inv;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float a = __builtin_fabsf(v[e]);
      odd = odd || !(a >= kF32AttnSmall || a == 0.f);
    }
    if (qi < p.T) *reinterpret_cast<floatx4*>(orow + 16 * d + 4 * g) = v;
  }
  // queries that met an infinite or NaN value, an overflow between parts or
  // values too small for them, again in plain fp32 (a layer of 4 x 375 frames, 8 heads of 128: 199 us, 230
  // with three items half padding of NaNs, 333 with a frame of infinities that
  // every query of an item sees)
  uint64_t redo = __ballot(odd && qi < p.T);
  redo |= redo >> 32, redo |= redo >> 16;
#pragma unroll 1
  for (uint32_t left = (uint32_t)redo & 0xFFFFu; left; left &= left - 1)
    attn_f32_plain<DK>(p, bl, h, i0 + 16 * w + __builtin_ctz(left), sc_qk, sc_bd);
}
