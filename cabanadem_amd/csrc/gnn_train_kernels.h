// gnn_train_kernels.h -- the training side of the surrogate's MLPs, included
// by gnn.hip: one MLP's backward rows pass, its parameter gradients, and the
// edge MLP's gradients at the nodes it gathered.
//
//   k_bwd_rows     dY' = dY + add[idx];  dH = (dY' W2^T) * [hid > 0];
//                  dX = dH W1^T for up to two input sources; dY' in BF16 and
//                  the FP32 column sums of dY' (db2)
//   k_wgrad_pair   partial dW1 = X^T dH, db1 and dW2 = hid^T dY' over row chunks
//   k_grad_reduce  the partials summed in chunk order into W1 | b1 | W2 | b2
//   k_edge_hidden_to_nodes
//                  dh[i] += sum over the edges e of i of dH[e] W1b^T
//                  + dH[rev[e]] W1c^T
#pragma once

constexpr int kBwdWaves = 8;
constexpr int kBiasCols = kLat; // a partial row of db2

struct BwdRowsArgs {
  int M, nout;
  const float* dY;    // [M][nout], or null (zeros, with add)
  const float* add;   // [.][128] rows added through idx, or null
  const int* idx;     // [M]
  const bf16* hid;    // [M][128] post-ReLU hidden of the forward pass
  const bf16* W2;     // [128][NO]
  const bf16* W1[2];  // [128][128] rows of W1 of the sources with a gradient
  float* dX[2];       // [M][128] their gradients
  int mode[2];        // 0: store, 1: += what is there, 2: dX = dY' + (dX is dY)
  bf16* dH;           // [M][128]
  bf16* dYb;          // [M][NO] BF16 of dY'
  float* bpart;       // [blocks][kBiasCols]
};

// One wave takes 16 rows at a time, persistent over the grid, weights in LDS
// for the block (rows in unit_of_row order) and transposed products, as the
// forward kernels: a lane's D fragments of dH^T are its B fragments of the
// dX^T product, so dH never goes through LDS, and a lane holds 8 contiguous
// channels of one row in every array it reads or writes.  The next tile's dY
// and hidden rows are in flight over the current tile's products.
//
// Bound: HBM, 16 + 8 s bytes per channel and row (dY, hid, dH, dY' in BF16,
// and 4 to 8 for each of the s dX).  The row-tiled kernel it replaces read its
// weights from L2 per wave, stored dH two bytes and dX four bytes per lane,
// took dX of the gathered sources to HBM as FP32 (two of the three of an edge
// MLP, 512 bytes per edge each, now k_edge_hidden_to_nodes) and left dY + add
// to a pass of its own.
template <int NO, int NX>
__global__ __launch_bounds__(64 * kBwdWaves, 1) void k_bwd_rows(BwdRowsArgs a) {
  constexpr int KS = NO == kLat ? 4 : 1; // k steps of dY' W2^T (NO = 16: one, padded to 32)
  constexpr int P2 = KS * 32 + 8;
  __shared__ bf16 sw2[kLat][P2];                      // W2: [row][n]
  __shared__ bf16 sw1[NX > 0 ? NX : 1][kLat][kWPitch]; // W1 of the sources: [row][u]
  for (int c = threadIdx.x; c < kLat * KS * 4; c += 64 * kBwdWaves) {
    const int r = c / (KS * 4), n8 = (c % (KS * 4)) * 8;
    bf16x8 v;
    if (n8 < NO) v = ld8(a.W2 + (long)unit_of_row(r) * NO + n8);
    else
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = (bf16)0.f;
    *reinterpret_cast<bf16x8*>(&sw2[r][n8]) = v;
  }
#pragma unroll
  for (int x = 0; x < NX; ++x)
    for (int c = threadIdx.x; c < kLat * 16; c += 64 * kBwdWaves) {
      const int r = c >> 4, k8 = (c & 15) * 8;
      *reinterpret_cast<bf16x8*>(&sw1[x][r][k8]) = ld8(a.W1[x] + (long)unit_of_row(r) * kLat + k8);
    }
  __syncthreads();
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lr = lane & 15, lg = lane >> 4, lk = 8 * lg;
  const int ntiles = (a.M + 15) / 16;
  const int stride = gridDim.x * kBwdWaves;
  float s2[KS][8]; // this lane's column sums of dY'
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
#pragma unroll
    for (int q = 0; q < 8; ++q) s2[ks][q] = 0.f;
  struct Rows {
    float y[KS][8];
    bf16x8 h[4];
  };
  auto load = [&](int t, Rows& R) {
    const int m = t * 16 + lr < a.M ? t * 16 + lr : a.M - 1; // clamped loads; stores are guarded
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) R.h[s4] = ld8(a.hid + (long)m * kLat + 32 * s4 + lk);
    if constexpr (NO == kLat) {
      const float* add = a.add ? a.add + (long)a.idx[m] * kLat + lk : nullptr;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        float4 u = make_float4(0.f, 0.f, 0.f, 0.f), v = u;
        if (a.dY) {
          const float* p = a.dY + (long)m * kLat + 32 * ks + lk;
          u = *reinterpret_cast<const float4*>(p);
          v = *reinterpret_cast<const float4*>(p + 4);
        }
        if (add) {
          const float4 b = *reinterpret_cast<const float4*>(add + 32 * ks);
          const float4 c = *reinterpret_cast<const float4*>(add + 32 * ks + 4);
          u.x += b.x; u.y += b.y; u.z += b.z; u.w += b.w;
          v.x += c.x; v.y += c.y; v.z += c.z; v.w += c.w;
        }
        R.y[ks][0] = u.x; R.y[ks][1] = u.y; R.y[ks][2] = u.z; R.y[ks][3] = u.w;
        R.y[ks][4] = v.x; R.y[ks][5] = v.y; R.y[ks][6] = v.z; R.y[ks][7] = v.w;
      }
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q) R.y[0][q] = lk + q < a.nout ? a.dY[(long)m * a.nout + lk + q] : 0.f;
    }
  };
  int t = blockIdx.x * kBwdWaves + w;
  Rows cur, nxt;
  if (t < ntiles) load(t, cur);
  for (; t < ntiles; t += stride) {
    const int tn = t + stride;
    if (tn < ntiles) load(tn, nxt);
    // keeps the weight fragments' LDS reads inside the loop
    __asm__ volatile("" ::: "memory");
    const int m = t * 16 + lr;
    const bool live = m < a.M;
    f32x4 acc[8];
#pragma unroll
    for (int ub = 0; ub < 8; ++ub) acc[ub] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      bf16x8 yb;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        yb[q] = (bf16)cur.y[ks][q];
        s2[ks][q] += live ? cur.y[ks][q] : 0.f;
      }
      if (live && 32 * ks + lk < NO) *reinterpret_cast<bf16x8*>(a.dYb + (long)m * NO + 32 * ks + lk) = yb;
#pragma unroll
      for (int ub = 0; ub < 8; ++ub)
        acc[ub] = mfma(*reinterpret_cast<const bf16x8*>(&sw2[ub * 16 + lr][ks * 32 + lk]), yb, acc[ub]);
    }
    bf16x8 g[4];
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const float v = q < 4 ? acc[2 * s4][q & 3] : acc[2 * s4 + 1][q & 3];
        g[s4][q] = (bf16)((float)cur.h[s4][q] > 0.f ? v : 0.f);
      }
      if (live) *reinterpret_cast<bf16x8*>(a.dH + (long)m * kLat + 32 * s4 + lk) = g[s4];
    }
#pragma unroll
    for (int x = 0; x < NX; ++x) {
#pragma unroll
      for (int ub = 0; ub < 8; ++ub) acc[ub] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int ub = 0; ub < 8; ++ub)
          acc[ub] = mfma(*reinterpret_cast<const bf16x8*>(&sw1[x][ub * 16 + lr][ks * 32 + lk]), g[ks], acc[ub]);
      if (!live) continue;
#pragma unroll
      for (int ub = 0; ub < 8; ++ub) {
        float* p = a.dX[x] + (long)m * kLat + 32 * (ub >> 1) + lk + 4 * (ub & 1);
        float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
        if (NO == kLat && a.mode[x] == 2) {
          const float* y = &cur.y[(ub >> 1) % KS][4 * (ub & 1)];
          o = make_float4(y[0], y[1], y[2], y[3]);
        } else if (a.mode[x]) {
          o = *reinterpret_cast<const float4*>(p);
        }
        if (a.mode[x]) {
          o.x += acc[ub][0]; o.y += acc[ub][1]; o.z += acc[ub][2]; o.w += acc[ub][3];
        } else {
          o = make_float4(acc[ub][0], acc[ub][1], acc[ub][2], acc[ub][3]);
        }
        *reinterpret_cast<float4*>(p) = o;
      }
    }
    if (tn < ntiles) cur = nxt;
  }
  // the block's column sums: over the 16 rows of each wave, then the waves in
  // order (the weights' LDS is free by then)
  __syncthreads();
  float* red = reinterpret_cast<float*>(&sw2[0][0]); // [kBwdWaves][kBiasCols], 4 KB
  static_assert(sizeof(float) * kBwdWaves * kBiasCols <= sizeof(bf16) * kLat * (32 + 8), "the sums fit in W2's tile");
  if (KS == 1 && lane < kLat / 2) red[w * kBiasCols + lane] = red[w * kBiasCols + kLat / 2 + lane] = 0.f;
  if (KS == 1) wave_lds_sync();
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      float v = s2[ks][q];
#pragma unroll
      for (int off = 1; off < 16; off <<= 1) v += __shfl_xor(v, off);
      if (lr == 0) red[w * kBiasCols + 32 * ks + lk + q] = v;
    }
  __syncthreads();
  if (threadIdx.x < kBiasCols) {
    float s = 0.f;
    for (int k = 0; k < kBwdWaves; ++k) s += red[k * kBiasCols + threadIdx.x];
    a.bpart[(long)blockIdx.x * kBiasCols + threadIdx.x] = s;
  }
}

struct WgradPairArgs {
  int M, K, NO, chunk;
  Segs in;            // X sources of W1
  const bf16* dH;     // [M][128]
  const bf16* hid;    // [M][128]: X of W2
  const bf16* dYb;    // [M][NO]
  float* part;        // [chunks][K 128 + 128 + 128 NO]: W1, b1, W2
};

__device__ inline unsigned dword_of(const uint4& v, int d) {
  return d == 0 ? v.x : (d == 1 ? v.y : (d == 2 ? v.z : v.w));
}

// Column f of a lane's block of 8 rows (one row of 8, or 2, BF16 columns per
// register group) as an MFMA fragment over the rows: one v_perm per two values.
__device__ inline bf16x8 column_fragment(const uint4 (&r)[8], int f) {
  uint4 o;
  const unsigned sel = f & 1 ? 0x07060302u : 0x05040100u;
  o.x = __builtin_amdgcn_perm(dword_of(r[1], f >> 1), dword_of(r[0], f >> 1), sel);
  o.y = __builtin_amdgcn_perm(dword_of(r[3], f >> 1), dword_of(r[2], f >> 1), sel);
  o.z = __builtin_amdgcn_perm(dword_of(r[5], f >> 1), dword_of(r[4], f >> 1), sel);
  o.w = __builtin_amdgcn_perm(dword_of(r[7], f >> 1), dword_of(r[6], f >> 1), sel);
  return __builtin_bit_cast(bf16x8, o);
}
__device__ inline bf16x8 column_fragment(const unsigned (&r)[8], int f) {
  uint4 o;
  const unsigned sel = f & 1 ? 0x07060302u : 0x05040100u;
  o.x = __builtin_amdgcn_perm(r[1], r[0], sel);
  o.y = __builtin_amdgcn_perm(r[3], r[2], sel);
  o.z = __builtin_amdgcn_perm(r[5], r[4], sel);
  o.w = __builtin_amdgcn_perm(r[7], r[6], sel);
  return __builtin_bit_cast(bf16x8, o);
}

constexpr int kWgWaves = 4; // one per SIMD: the 128 x 128 accumulators take 256 registers a wave

// Partial dW[k][n] = sum over the block's rows of X[m][k] G[m][n], for 16 CX
// columns of X and 16 CG of G (CX, CG columns per lane).  A wave walks 32 rows
// at a time; lane (lr, lg) loads rows 8 lg .. + 7 at its columns CX lr .. and
// CG lr .., whole rows being read by 16 neighbouring lanes, and turns them
// into fragments over the rows in registers (column_fragment), so nothing is
// transposed through LDS.  Fragment f of X holds column CX lr + f, so D row
// 4 lg + r of product (f, g) is column CX (4 lg + r) + f of X and its column lr
// is column CG lr + g of G.  The next rows load during the products.  The four
// waves' sums are added in wave order through LDS at the end.
//
// SUM: the column sums of G too (db), each lane its rows' in FP32.
//
// Bound: HBM (X, G once per 128 columns of X: 512 bytes a row) beside 64 MFMAs
// per 32 rows.
template <int CX, int CG, bool SUM>
__device__ __forceinline__ void wgrad_block(const bf16* X, const int* idx, int sx, const bf16* G, int sg, int m_begin,
                                   int m_end, float* out, int ldo, float* sum, f32x4* lds) {
  using XT = typename std::conditional<CX == 8, uint4, unsigned>::type;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lr = lane & 15, lg = lane >> 4;
  f32x4 acc[CX][CG];
#pragma unroll
  for (int f = 0; f < CX; ++f)
#pragma unroll
    for (int g = 0; g < CG; ++g) acc[f][g] = f32x4{0.f, 0.f, 0.f, 0.f};
  static_assert(!SUM || CG == 8, "column sums of 128 columns only");
  float cs[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  struct Raw {
    XT x[8];
    uint4 g8[CG == 8 ? 8 : 1];
    bf16 g1[CG == 8 ? 1 : 8];
  };
  auto load = [&](int m0, Raw& R) {
    const int mb = m0 + 8 * lg;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int m = mb + j < m_end ? mb + j : m_end - 1;
      const long row = idx ? idx[m] : m;
      R.x[j] = *reinterpret_cast<const XT*>(X + row * sx + CX * lr);
      if constexpr (CG == 8) R.g8[j] = *reinterpret_cast<const uint4*>(G + (long)m * sg + 8 * lr);
      else R.g1[j] = G[(long)m * sg + lr];
    }
    if (m0 + 32 > m_end) { // rows past the end count nothing
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (mb + j >= m_end) {
          R.x[j] = XT{};
          if constexpr (CG == 8) R.g8[j] = uint4{};
          else R.g1[j] = (bf16)0.f;
        }
    }
  };
  int m0 = m_begin + 32 * w;
  Raw cur, nxt;
  if (m0 < m_end) load(m0, cur);
  for (; m0 < m_end; m0 += 32 * kWgWaves) {
    const int mn = m0 + 32 * kWgWaves;
    if (mn < m_end) load(mn, nxt);
    bf16x8 gf[CG];
    if constexpr (CG == 8) {
#pragma unroll
      for (int g = 0; g < CG; ++g) gf[g] = column_fragment(cur.g8, g);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) gf[0][j] = cur.g1[j];
    }
#pragma unroll
    for (int f = 0; f < CX; ++f) {
      const bf16x8 xf = column_fragment(cur.x, f);
#pragma unroll
      for (int g = 0; g < CG; ++g) acc[f][g] = mfma(xf, gf[g], acc[f][g]);
    }
    if constexpr (SUM) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int g = 0; g < 8; ++g) {
          const unsigned d = dword_of(cur.g8[j], g >> 1);
          cs[g] += __uint_as_float(g & 1 ? d & 0xffff0000u : d << 16);
        }
    }
    if (mn < m_end) cur = nxt;
  }
  // the waves' sums, wave order, in rounds of up to four f (one per wave)
  constexpr int FR = CX < kWgWaves ? CX : kWgWaves;
  auto round = [&](auto first) {
    constexpr int f0 = decltype(first)::value;
    __syncthreads();
#pragma unroll
    for (int f = 0; f < FR; ++f)
#pragma unroll
      for (int g = 0; g < CG; ++g) lds[((w * FR + f) * CG + g) * 64 + lane] = acc[f0 + f][g];
    __syncthreads();
    if (w < FR) {
      const int f = f0 + w;
      float o[4][CG];
#pragma unroll
      for (int g = 0; g < CG; ++g) {
        f32x4 s = lds[((0 * FR + w) * CG + g) * 64 + lane];
#pragma unroll
        for (int k = 1; k < kWgWaves; ++k) s += lds[((k * FR + w) * CG + g) * 64 + lane];
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r][g] = s[r];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float* p = out + (long)(CX * (4 * lg + r) + f) * ldo + CG * lr;
        if constexpr (CG == 8) {
          *reinterpret_cast<float4*>(p) = make_float4(o[r][0], o[r][1], o[r][2], o[r][3]);
          *reinterpret_cast<float4*>(p + 4) = make_float4(o[r][4], o[r][5], o[r][6], o[r][7]);
        } else {
          *p = o[r][0];
        }
      }
    }
  };
  round(std::integral_constant<int, 0>{});
  if constexpr (CX > FR) round(std::integral_constant<int, FR>{});
  if constexpr (SUM) {
    float* ls = reinterpret_cast<float*>(lds); // [4 waves x 4 row groups][128]
    __syncthreads();
#pragma unroll
    for (int g = 0; g < 8; ++g) ls[(w * 4 + lg) * kLat + 8 * lr + g] = cs[g];
    __syncthreads();
    if (threadIdx.x < kLat) {
      float s = ls[threadIdx.x];
      for (int k = 1; k < 4 * kWgWaves; ++k) s += ls[k * kLat + threadIdx.x];
      sum[threadIdx.x] = s;
    }
  }
}

// Grid (chunks, 128-wide blocks of X + 1): the last row of blocks is W2.
// CX1: columns of X per lane for W1 (8: sources of 128, 2: one of 32);
// CG2: columns of dY' per lane (8: 128 outputs, 1: 16).
template <int CX1, int CG2>
__global__ __launch_bounds__(64 * kWgWaves, 1) void k_wgrad_pair(WgradPairArgs a) {
  __shared__ f32x4 lds[kWgWaves * kWgWaves * 8 * 64]; // 128 KB
  const int m_begin = blockIdx.x * a.chunk;
  const int m_end = min(a.M, m_begin + a.chunk);
  float* part = a.part + (long)blockIdx.x * ((long)(a.K + 1) * kLat + (long)kLat * a.NO);
  float* b1 = part + (long)a.K * kLat;
  if (blockIdx.y + 1 == gridDim.y) {
    wgrad_block<8, CG2, false>(a.hid, nullptr, kLat, a.dYb, a.NO, m_begin, m_end, b1 + kLat, a.NO, nullptr, lds);
  } else if (blockIdx.y == 0) {
    wgrad_block<CX1, 8, true>(a.in.src[0], a.in.idx[0], a.in.width[0], a.dH, kLat, m_begin, m_end, part, kLat, b1,
                              lds);
  } else {
    const int q = blockIdx.y;
    wgrad_block<CX1, 8, false>(a.in.src[q], a.in.idx[q], a.in.width[q], a.dH, kLat, m_begin, m_end,
                               part + (long)a.in.start[q] * kLat, kLat, nullptr, lds);
  }
}

// grad (W1 | b1 | W2 | b2) = the partials summed in chunk order.  A block
// takes 128 consecutive columns of one vector: 32 lanes of four columns by 8
// groups of consecutive chunks, the groups added in order at the end, so that
// eight chunks load at a time where one thread per column chained them all.
__global__ __launch_bounds__(kThreads) void k_grad_reduce(const float* part, int nch, const float* bpart, int nb,
                                                          int K, int NO, float* grad) {
  __shared__ float4 red[8][32];
  const int c = threadIdx.x & 31, g = threadIdx.x >> 5;
  const long cw = (long)(K + 1) * kLat + (long)kLat * NO;
  const long b = blockIdx.x * (long)kLat; // first column; b2 follows the others
  const bool b2 = b >= cw;
  const float* src = b2 ? bpart : part + b;
  const long stride = b2 ? kBiasCols : cw;
  const int count = b2 ? nb : nch, cols = b2 ? NO : kLat;
  const int per = (count + 7) / 8;
  const int k0 = g * per, k1 = min(count, k0 + per);
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 8
  for (int k = k0; k < k1; ++k) {
    const float4 v = *reinterpret_cast<const float4*>(src + k * stride + 4 * c);
    s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
  }
  red[g][c] = s;
  __syncthreads();
  if (g == 0 && 4 * c < cols) {
#pragma unroll
    for (int k = 1; k < 8; ++k) {
      const float4 v = red[k][c];
      s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
    *reinterpret_cast<float4*>(grad + b + 4 * c) = s;
  }
}

struct EdgeToNodesArgs {
  int N;
  const bf16* dH;     // [E][128]
  const int* row;     // [N + 1]
  const int* rev;     // [E]
  const bf16* W1;     // [384][128]: rows 128..255 the receiver's share, 256..383 the sender's
  float* dh;          // [N][128]
};

constexpr int kToNodesWaves = 4;
constexpr int kToNodesPitch = kLat + 4; // floats; rows 16 bytes aligned, banks skewed

// dh[i] += sum over the edges e of node i, in edge order, of the receiver's
// gradient dH[e] W1b^T and the sender's dH[rev[e]] W1c^T (each an FP32 sum over
// the hidden units, added one after the other).  A wave takes 16 consecutive
// nodes, whose edges are consecutive, and walks them 16 at a time: both
// products on the MFMA units from the BF16 rows, the 16 x 128 FP32 results of
// each into the wave's LDS tile, and from there every lane adds its two
// channels edge by edge into the running sum of the current node.  The edges'
// FP32 gradients (2 x 512 bytes per edge written and read back by the two
// kernels this replaces) never leave the chip: 2 x 256 bytes per edge are read.
__global__ __launch_bounds__(64 * kToNodesWaves, 1) void k_edge_hidden_to_nodes(EdgeToNodesArgs a) {
  __shared__ bf16 swb[kLat][kWPitch], swc[kLat][kWPitch]; // W1b, W1c: [row][u], rows in unit_of_row order
  __shared__ float st[kToNodesWaves][2][16][kToNodesPitch];
  for (int c = threadIdx.x; c < kLat * 16; c += 64 * kToNodesWaves) {
    const int r = c >> 4, k8 = (c & 15) * 8, u = unit_of_row(r);
    *reinterpret_cast<bf16x8*>(&swb[r][k8]) = ld8(a.W1 + (long)(kLat + u) * kLat + k8);
    *reinterpret_cast<bf16x8*>(&swc[r][k8]) = ld8(a.W1 + (long)(2 * kLat + u) * kLat + k8);
  }
  __syncthreads(); // the only block barrier: the loop below is per wave
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lr = lane & 15, lg = lane >> 4, lk = 8 * lg;
  const int groups = (a.N + 15) / 16;
  for (int grp = blockIdx.x * kToNodesWaves + w; grp < groups; grp += gridDim.x * kToNodesWaves) {
    // keeps the weight fragments' LDS reads inside the loop
    __asm__ volatile("" ::: "memory");
    const int n0 = grp * 16, n1 = min(a.N, n0 + 16);
    const int e_end = __builtin_amdgcn_readfirstlane(a.row[n1]);
    int e0 = __builtin_amdgcn_readfirstlane(a.row[n0]);
    int n = n0, end = __builtin_amdgcn_readfirstlane(a.row[n0 + 1]);
    float sx = 0.f, sy = 0.f;
    auto flush = [&]() { // node n is complete: add it and go to the next
      float2* p = reinterpret_cast<float2*>(a.dh + (long)n * kLat + 2 * lane);
      float2 v = *p;
      v.x += sx; v.y += sy;
      *p = v;
      sx = sy = 0.f;
      ++n;
      end = n < n1 ? __builtin_amdgcn_readfirstlane(a.row[n + 1]) : INT_MAX;
    };
    bf16x8 Br[4], Bs[4];
    auto load = [&](int e) {
      const int ee = e + lr < e_end ? e + lr : e_end - 1;
      const int er = a.rev[ee];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        Br[ks] = ld8(a.dH + (long)ee * kLat + 32 * ks + lk);
        Bs[ks] = ld8(a.dH + (long)er * kLat + 32 * ks + lk);
      }
    };
    if (e0 < e_end) load(e0);
    for (; e0 < e_end; e0 += 16) {
      f32x4 r[8], s[8];
#pragma unroll
      for (int ub = 0; ub < 8; ++ub) r[ub] = s[ub] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int ub = 0; ub < 8; ++ub) {
          r[ub] = mfma(*reinterpret_cast<const bf16x8*>(&swb[ub * 16 + lr][ks * 32 + lk]), Br[ks], r[ub]);
          s[ub] = mfma(*reinterpret_cast<const bf16x8*>(&swc[ub * 16 + lr][ks * 32 + lk]), Bs[ks], s[ub]);
        }
      if (e0 + 16 < e_end) load(e0 + 16);
#pragma unroll
      for (int ub = 0; ub < 8; ++ub) {
        const int c = 32 * (ub >> 1) + lk + 4 * (ub & 1);
        *reinterpret_cast<f32x4*>(&st[w][0][lr][c]) = r[ub];
        *reinterpret_cast<f32x4*>(&st[w][1][lr][c]) = s[ub];
      }
      wave_lds_sync();
      const int cnt = min(16, e_end - e0);
      for (int k = 0; k < cnt; ++k) {
        while (e0 + k >= end) flush();
        const float2 u = *reinterpret_cast<const float2*>(&st[w][0][k][2 * lane]);
        const float2 v = *reinterpret_cast<const float2*>(&st[w][1][k][2 * lane]);
        sx += u.x; sy += u.y;
        sx += v.x; sy += v.y;
      }
      wave_lds_sync(); // the next tile rewrites the sums
    }
    while (n < n1) flush();
  }
}
