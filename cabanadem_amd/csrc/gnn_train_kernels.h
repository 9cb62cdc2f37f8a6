// gnn_train_kernels.h -- the training side of the surrogate's MLPs, included
// by gnn.hip: one MLP's backward rows pass, its parameter gradients, and the
// edge MLP's gradients at the nodes it gathered.
//
//   k_bwd_rows     dY' = dY + add[idx];  dH = (dY' W2^T) * [hid > 0];
//                  dX = dH W1^T for up to two input sources
//   k_wgrad_pair   partial dW2 = hid^T dY', db2, dW1 = X^T dH and db1 over row
//                  chunks
//   k_grad_reduce  the partials summed in chunk order into W1 | b1 | W2 | b2
//   k_edge_hidden_to_nodes
//                  dh[i] += sum over the edges e of i of dH[e] W1b^T
//                  + dH[rev[e]] W1c^T
#pragma once

constexpr int kBwdWaves = 8;
constexpr int kBiasCols = kLat; // a partial row of db2
constexpr int kGradChunks = 64; // row chunks of the parameter gradients, of a multiple of 32 rows each

struct BwdRowsArgs {
  int M, nout;
  int per;            // tiles a block takes side by side (one per wave, at most its waves)
  const float* dY;    // [M][nout], or null (zeros, with add)
  const float* add;   // [.][128] rows added through idx, or null
  const int* idx;     // [M]
  const bf16* hid;    // [M][128] post-ReLU hidden of the forward pass
  const bf16* W2;     // [128][NO]
  const bf16* W1[2];  // [128][128] rows of W1 of the sources with a gradient
  float* dX[2];       // [M][128] their gradients
  int mode[2];        // 0: store, 1: += what is there, 2: dX = dY' + dH W1^T (dX may be dY)
  bf16* dH;           // [M][128]
  bf16* dYb;          // [M][NO] BF16 of dY', or null
};

// One wave takes 16 rows at a time, persistent over the grid, weights in LDS
// for the block (rows in unit_of_row order) and transposed products, as the
// forward kernels: a lane's D fragments of dH^T are its B fragments of the
// dX^T product, so dH never goes through LDS, and a lane holds 8 contiguous
// channels of one row in every array it reads or writes.  The next tile's dY
// and hidden rows are in flight over the current tile's products.
//
// Bound: HBM, 8 + 4 s bytes per channel and row (dY, hid, dH and the s dX; 8
// for a dX that adds).  The row-tiled kernel it replaces read its
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
  const int stride = gridDim.x * a.per;
  struct Rows {
    float y[KS][8];
    bf16x8 h[4];
  };
  // add's row of the tile that loads next: loads are waited for in the order of
  // their issue and stand outside branches (the last tile has a copy of the code
  // without them), so that a tile does not wait for the next one's rows
  int ai = 0;
  auto load_index = [&](int t) {
    if (a.add) ai = a.idx[t * 16 + lr < a.M ? t * 16 + lr : a.M - 1];
  };
  auto load = [&](int t, Rows& R) {
    const int m = t * 16 + lr < a.M ? t * 16 + lr : a.M - 1; // clamped loads; stores are guarded
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) R.h[s4] = ld8(a.hid + (long)m * kLat + 32 * s4 + lk);
    if constexpr (NO == kLat) {
      const float* add = a.add ? a.add + (long)ai * kLat + lk : nullptr;
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
  int t = blockIdx.x * a.per + w;
  if (w >= a.per || t >= ntiles) return;
  Rows cur, nxt;
  load_index(t);
  load(t, cur);
  load_index(min(t + stride, ntiles - 1));
  auto tile = [&](int t, auto more) {
    if constexpr (decltype(more)::value) {
      load(t + stride, nxt);
      load_index(min(t + 2 * stride, ntiles - 1));
    }
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
      for (int q = 0; q < 8; ++q) yb[q] = (bf16)cur.y[ks][q];
      if (a.dYb && live && 32 * ks + lk < NO) *reinterpret_cast<bf16x8*>(a.dYb + (long)m * NO + 32 * ks + lk) = yb;
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
  };
  for (; t + stride < ntiles; t += stride) {
    tile(t, std::true_type{});
    cur = nxt;
  }
  tile(t, std::false_type{});
}

struct WgradPairArgs {
  int M, K, NO, chunk;
  Segs in;            // X sources of W1
  const bf16* dH;     // [M][128]
  const bf16* hid;    // [M][128]: X of W2
  int nout;
  const float* dY;    // dY' = dY + add[idx], as k_bwd_rows forms it
  const float* add;
  const int* idx;
  float* part;        // [chunks][K 128 + 128 + 128 NO]: W1, b1, W2
  float* bpart;       // [chunks][kBiasCols]: b2
  int y0;             // the launch's first row of blocks: 0 for W2, 1 + q for source q of W1
};

// The parameter gradients are sums over all rows, added in one fixed order,
// that of gnn_weight_grad over 64 chunks: a chunk's rows go through the MFMA
// units 32 at a time into one accumulator, its column sums through 16 (or, for
// up to 16 outputs, 32) interleaved chains of FP32 adds, and the chunks are
// added in order.  Results are equal to gnn_weight_grad's bit for bit.  (An
// order of its own, for instance rows split over a block's waves, is as exact
// but differs in the last bits, and Adam's first steps turn a gradient that is
// all rounding into a step of full length.)

template <int C>
struct Cols { // C consecutive BF16 columns of a row
  unsigned d[C / 2];
};
// Features may start at any value of their array: a row's 32 go in pairs.
typedef unsigned pair2u __attribute__((aligned(2)));
template <int C>
__device__ inline Cols<C> load_cols(const bf16* p) {
  Cols<C> v;
  if constexpr (C == 8) {
    const uint4 u = *reinterpret_cast<const uint4*>(p);
    v.d[0] = u.x;
    v.d[1] = u.y;
    v.d[2] = u.z;
    v.d[3] = u.w;
  } else if constexpr (C == 4) {
    const uint2 u = *reinterpret_cast<const uint2*>(p);
    v.d[0] = u.x;
    v.d[1] = u.y;
  } else {
    v.d[0] = *reinterpret_cast<const pair2u*>(p);
  }
  return v;
}

// Column f of a lane's 8 rows as an MFMA fragment over the rows: one v_perm
// per two values.
template <int C>
__device__ inline bf16x8 column_fragment(const Cols<C> (&r)[8], int f) {
  const unsigned sel = f & 1 ? 0x07060302u : 0x05040100u;
  uint4 o;
  o.x = __builtin_amdgcn_perm(r[1].d[f >> 1], r[0].d[f >> 1], sel);
  o.y = __builtin_amdgcn_perm(r[3].d[f >> 1], r[2].d[f >> 1], sel);
  o.z = __builtin_amdgcn_perm(r[5].d[f >> 1], r[4].d[f >> 1], sel);
  o.w = __builtin_amdgcn_perm(r[7].d[f >> 1], r[6].d[f >> 1], sel);
  return __builtin_bit_cast(bf16x8, o);
}

// Row numbers m0 + 8 lg .. + 7 through idx (clamped to the chunk's last row):
// two loads where the step is whole, of any alignment of idx.
typedef int int4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ void load_rows(const int* idx, int m0, int lg, int m_end, int (&row)[8]) {
  const int mb = m0 + 8 * lg;
  if (m0 + 32 <= m_end) {
    const int4u u = *reinterpret_cast<const int4u*>(idx + mb), v = *reinterpret_cast<const int4u*>(idx + mb + 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      row[j] = u[j];
      row[4 + j] = v[j];
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) row[j] = idx[min(mb + j, m_end - 1)];
  }
}

constexpr int kWgWaves = 4;

// A wave's walk over the rows of a chunk, 32 at a time, D steps in flight.
// load(m0, slot) loads a step's rows (clamped to the chunk's last), use(m0,
// slot, tail) takes them; tail: some lie past the chunk's end.  The whole steps
// run D at a time without a branch between them, so that the wait for a step
// leaves the later ones in flight.
template <int D, class Slot, class Load, class Use>
__device__ __forceinline__ void walk_rows(int m_begin, int m_end, Slot (&buf)[D], Load load, Use use) {
#pragma unroll
  for (int d = 0; d < D; ++d) load(m_begin + 32 * d, buf[d]);
  int m0 = m_begin;
  for (; m0 + 32 * D <= m_end; m0 += 32 * D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      use(m0 + 32 * d, buf[d], false);
      load(m0 + 32 * (d + D), buf[d]);
    }
  }
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (m0 + 32 * d < m_end) use(m0 + 32 * d, buf[d], m0 + 32 * (d + 1) > m_end);
}

template <int CX, int CG>
__device__ __forceinline__ void store_product(const f32x4 (&acc)[CX][CG], float* out, int ldo, int lr, int lg) {
#pragma unroll
  for (int f = 0; f < CX; ++f)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float* p = out + (long)(CX * (4 * lg + r) + f) * ldo + CG * lr;
      if constexpr (CG == 4)
        *reinterpret_cast<float4*>(p) = make_float4(acc[f][0][r], acc[f][1][r], acc[f][2][r], acc[f][3][r]);
      else if constexpr (CG == 2) *reinterpret_cast<float2*>(p) = make_float2(acc[f][0][r], acc[f][1][r]);
      else *p = acc[f][0][r];
    }
}

// Column sums from the chains: 0..7 of lane group 0, then of the next groups.
template <int CG, int GROUPS>
__device__ __forceinline__ void store_sums(const float (&cs)[8][CG], float* sum, int lr, int lg) {
#pragma unroll
  for (int g = 0; g < CG; ++g) {
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < GROUPS; ++k) {
      if (k) s = __shfl(s, 16 * (k - 1) + lr);
#pragma unroll
      for (int j = 0; j < 8; ++j) s += cs[j][g];
    }
    if (lg == GROUPS - 1) sum[CG * lr + g] = s;
  }
}

// One wave of W1: dW[x0 ..][g0 ..], 16 CX columns of X by 16 CG of G = dH.  Lane
// (lr, lg) loads rows 8 lg .. + 7 at its columns CX lr .. and CG lr .. (a row's
// columns are read by 16 neighbouring lanes) and turns them into fragments over
// the rows in registers (column_fragment), so nothing is transposed through
// LDS.  Fragment f of X holds column CX lr + f, so D row 4 lg + r of product
// (f, g) is column CX (4 lg + r) + f of X and its column lr is column CG lr + g
// of G.  sum: the column sums of G too (db1).  A chain takes a step's rows r
// and r + 16, which are in lanes 32 apart; the lanes lg < 2 keep the chains.
//
// Waves split a block's columns, not its rows (the sums' order, above), and
// share rows through the CU's L1.  Bound: HBM beside 16 MFMAs per wave and
// step.  Four steps in flight (32 KB a wave of 64 x 64; 18 loads a step, and a
// wave can wait on 63).
template <bool IDX, int CX, int CG>
__device__ __forceinline__ void wgrad1_wave(const bf16* X, const int* idx, int sx, const bf16* G, int m_begin,
                                            int m_end, float* out, float* sum) {
  constexpr int D = 4;
  const int lane = threadIdx.x & 63;
  const int lr = lane & 15, lg = lane >> 4;
  f32x4 acc[CX][CG];
#pragma unroll
  for (int f = 0; f < CX; ++f)
#pragma unroll
    for (int g = 0; g < CG; ++g) acc[f][g] = f32x4{0.f, 0.f, 0.f, 0.f};
  float cs[8][CG];
#pragma unroll
  for (int j = 0; j < 8; ++j)
#pragma unroll
    for (int g = 0; g < CG; ++g) cs[j][g] = 0.f;
  struct Slot {
    Cols<CX> x[8];
    Cols<CG> g[8];
    int row[8]; // X's rows of the step that loads next into this slot
  } buf[D];
  if constexpr (IDX) {
#pragma unroll
    for (int d = 0; d < D; ++d) load_rows(idx, m_begin + 32 * d, lg, m_end, buf[d].row);
  }
  auto load = [&](int m0, Slot& R) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int m = min(m0 + 8 * lg + j, m_end - 1);
      R.x[j] = load_cols<CX>(X + (long)(IDX ? R.row[j] : m) * sx + CX * lr);
      R.g[j] = load_cols<CG>(G + (long)m * kLat + CG * lr);
    }
    if constexpr (IDX) load_rows(idx, m0 + 32 * D, lg, m_end, R.row);
  };
  auto use = [&](int m0, Slot& R, bool tail) {
    if (tail) { // rows past the end count nothing
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (m0 + 8 * lg + j >= m_end) {
          R.x[j] = Cols<CX>{};
          R.g[j] = Cols<CG>{};
        }
    }
    bf16x8 gf[CG];
#pragma unroll
    for (int g = 0; g < CG; ++g) gf[g] = column_fragment<CG>(R.g, g);
#pragma unroll
    for (int f = 0; f < CX; ++f) {
      const bf16x8 xf = column_fragment<CX>(R.x, f);
#pragma unroll
      for (int g = 0; g < CG; ++g) acc[f][g] = mfma(xf, gf[g], acc[f][g]);
    }
    if (sum) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int k = 0; k < CG / 2; ++k) {
          const unsigned u = R.g[j].d[k], v = __shfl_xor(u, 32);
          cs[j][2 * k] += __uint_as_float(u << 16);
          cs[j][2 * k] += __uint_as_float(v << 16);
          cs[j][2 * k + 1] += __uint_as_float(u & 0xffff0000u);
          cs[j][2 * k + 1] += __uint_as_float(v & 0xffff0000u);
        }
    }
  };
  walk_rows<D>(m_begin, m_end, buf, load, use);
  store_product<CX, CG>(acc, out, kLat, lr, lg);
  if (sum) store_sums<CG, 2>(cs, sum, lr, lg);
}

// One wave of W2: X = hid, G = dY' in FP32 (the products take it rounded to
// BF16, the column sums, db2, as it is).  128 outputs: a wave takes all of hid's
// columns by 32 of dY', so that dY' is read once; two steps in flight (32 KB).
// Up to 16 outputs (NARROW): 32 columns of hid by all of dY'; a step's 32 rows
// are 32 chains there.
template <bool NARROW, bool Y, bool ADD>
__device__ __forceinline__ void wgrad2_wave(const bf16* hid, const float* dY, const float* add, const int* idx,
                                            int nout, int m_begin, int m_end, float* out, float* sum) {
  constexpr int CX = NARROW ? 2 : 8, CG = NARROW ? 1 : 2, D = NARROW ? 3 : 2;
  const int lane = threadIdx.x & 63;
  const int lr = lane & 15, lg = lane >> 4;
  f32x4 acc[CX][CG];
#pragma unroll
  for (int f = 0; f < CX; ++f)
#pragma unroll
    for (int g = 0; g < CG; ++g) acc[f][g] = f32x4{0.f, 0.f, 0.f, 0.f};
  float cs[8][CG];
#pragma unroll
  for (int j = 0; j < 8; ++j)
#pragma unroll
    for (int g = 0; g < CG; ++g) cs[j][g] = 0.f;
  typedef float V __attribute__((ext_vector_type(CG)));
  struct Slot {
    Cols<CX> x[8];
    V y[8], z[8];
    int row[8]; // add's rows of the step that loads next into this slot
  } buf[D];
  if constexpr (ADD) {
#pragma unroll
    for (int d = 0; d < D; ++d) load_rows(idx, m_begin + 32 * d, lg, m_end, buf[d].row);
  }
  auto load = [&](int m0, Slot& R) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int m = min(m0 + 8 * lg + j, m_end - 1);
      R.x[j] = load_cols<CX>(hid + (long)m * kLat + CX * lr);
      if constexpr (NARROW) R.y[j] = V(dY[(long)m * nout + min(lr, nout - 1)]);
      else if constexpr (Y) R.y[j] = *reinterpret_cast<const V*>(dY + (long)m * kLat + CG * lr);
      if constexpr (ADD) R.z[j] = *reinterpret_cast<const V*>(add + (long)R.row[j] * kLat + CG * lr);
    }
    if constexpr (ADD) load_rows(idx, m0 + 32 * D, lg, m_end, R.row);
  };
  auto use = [&](int m0, Slot& R, bool tail) {
    V y[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      y[j] = V(0.f);
      if constexpr (NARROW) {
        if (lr < nout) y[j] = R.y[j];
      } else if constexpr (Y) {
        y[j] = R.y[j];
      }
      if constexpr (ADD) y[j] += R.z[j];
    }
    if (tail) { // rows past the end count nothing
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (m0 + 8 * lg + j >= m_end) {
          R.x[j] = Cols<CX>{};
          y[j] = V(0.f);
        }
    }
    bf16x8 gf[CG];
#pragma unroll
    for (int g = 0; g < CG; ++g)
#pragma unroll
      for (int j = 0; j < 8; ++j) gf[g][j] = (bf16)y[j][g];
#pragma unroll
    for (int f = 0; f < CX; ++f) {
      const bf16x8 xf = column_fragment<CX>(R.x, f);
#pragma unroll
      for (int g = 0; g < CG; ++g) acc[f][g] = mfma(xf, gf[g], acc[f][g]);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int g = 0; g < CG; ++g) {
        cs[j][g] += y[j][g];
        if constexpr (!NARROW) cs[j][g] += __shfl_xor(y[j][g], 32);
      }
  };
  walk_rows<D>(m_begin, m_end, buf, load, use);
  store_product<CX, CG>(acc, out, NARROW ? 16 : kLat, lr, lg);
  if (sum) store_sums<CG, NARROW ? 4 : 2>(cs, sum, lr, lg);
}

// What dY' is made of.
enum { kDyNarrow, kDyOnly, kAddOnly, kDyAndAdd };

// Grid (chunks padded to a multiple of 8, 128-wide blocks of W2 and X).  The
// blocks of a chunk read the same rows of dH, and with eight XCDs taking blocks
// in turn they share one's L2.  X128: sources of 128 columns (else one of 32).
//
// Measured: the edge MLP 38 us at 54,000 edges (44 with the rows split over the
// waves, one step in flight and the waves' sums added through 128 KB of LDS) and
// the node MLP 11 us at 9,240 nodes (19).  At 374,000 edges 250 us either way,
// but W2 now reads dY' itself, so that k_bwd_rows need not write it in BF16 (155
// -> 128 us) nor sum its columns.
template <bool X128, int DY>
__global__ __launch_bounds__(64 * kWgWaves, 1) void k_wgrad_pair(WgradPairArgs a) {
  const int m_begin = blockIdx.x * a.chunk;
  const int m_end = min(a.M, m_begin + a.chunk);
  if (m_begin >= m_end) return;
  float* part = a.part + (long)blockIdx.x * ((long)(a.K + 1) * kLat + (long)kLat * a.NO);
  float* b1 = part + (long)a.K * kLat;
  float* b2 = a.bpart + (long)blockIdx.x * kBiasCols;
  const int w = threadIdx.x >> 6;
  const int c32 = 32 * w;
  if (blockIdx.y + a.y0 == 0) {
    float* w2 = b1 + kLat;
    if constexpr (DY == kDyNarrow)
      wgrad2_wave<true, true, false>(a.hid + c32, a.dY, nullptr, nullptr, a.nout, m_begin, m_end, w2 + c32 * 16,
                                     w == 0 ? b2 : nullptr);
    else
      wgrad2_wave<false, DY != kAddOnly, DY != kDyOnly>(a.hid, a.dY + c32, a.add + c32, a.idx, kLat, m_begin, m_end,
                                                        w2 + c32, b2 + c32);
    return;
  }
  const int q = blockIdx.y + a.y0 - 1;
  float* out = part + (long)a.in.start[q] * kLat;
  if constexpr (X128) {
    const int x64 = 64 * (w >> 1), g64 = 64 * (w & 1);
    const bf16* X = a.in.src[q] + x64;
    float* o = out + x64 * kLat + g64;
    float* sum = q == 0 && x64 == 0 ? b1 + g64 : nullptr;
    if (a.in.idx[q]) wgrad1_wave<true, 4, 4>(X, a.in.idx[q], kLat, a.dH + g64, m_begin, m_end, o, sum);
    else wgrad1_wave<false, 4, 4>(X, nullptr, kLat, a.dH + g64, m_begin, m_end, o, sum);
  } else {
    if (a.in.idx[0])
      wgrad1_wave<true, 2, 2>(a.in.src[0], a.in.idx[0], 32, a.dH + c32, m_begin, m_end, out + c32, b1 + c32);
    else wgrad1_wave<false, 2, 2>(a.in.src[0], nullptr, 32, a.dH + c32, m_begin, m_end, out + c32, b1 + c32);
  }
}

// grad (W1 | b1 | W2 | b2) = the partials summed in chunk order: one column a
// thread, 32 chunks loading at a time.
__global__ __launch_bounds__(kThreads) void k_grad_reduce(const float* part, int nch, const float* bpart, int K,
                                                          int NO, float* grad) {
  const long cw = (long)(K + 1) * kLat + (long)kLat * NO;
  const long c = (long)blockIdx.x * kThreads + threadIdx.x;
  if (c >= cw + NO) return;
  const float* src = c < cw ? part + c : bpart + (c - cw); // b2 follows the others
  const long stride = c < cw ? cw : kBiasCols;
  float s = 0.f;
  for (int k0 = 0; k0 < nch; k0 += 32) {
    float v[32];
#pragma unroll
    for (int k = 0; k < 32; ++k) v[k] = src[min(k0 + k, nch - 1) * stride];
#pragma unroll
    for (int k = 0; k < 32; ++k)
      if (k0 + k < nch) s += v[k];
  }
  grad[c] = s;
}

struct EdgeToNodesArgs {
  int N;
  int per;            // groups of nodes a block takes side by side (one per wave, at most its waves)
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
// What a node needs besides (its dh row, its edges' end) and the reverse edges
// are loaded ahead: loaded when reached, each cost its wave a round trip per
// node (31 -> 25 us at 54,000 edges, 124 -> 98 at 374,000).
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
  if (w >= a.per) return;
  for (int grp = blockIdx.x * a.per + w; grp < groups; grp += gridDim.x * a.per) {
    // keeps the weight fragments' LDS reads inside the loop
    __asm__ volatile("" ::: "memory");
    const int n0 = grp * 16, n1 = min(a.N, n0 + 16);
    const int ends = a.row[min(n0 + lane, n1)]; // lane k: the first edge of node n0 + k
    const int e_end = __builtin_amdgcn_readlane(ends, n1 - n0);
    int e0 = __builtin_amdgcn_readlane(ends, 0);
    int n = n0, end = __builtin_amdgcn_readlane(ends, 1);
    float sx = 0.f, sy = 0.f;
    // this node's and the next one's dh, loaded two nodes ahead
    auto node_row = [&](int k) { return reinterpret_cast<float2*>(a.dh + (long)min(k, n1 - 1) * kLat + 2 * lane); };
    float2 d0 = *node_row(n0), d1 = *node_row(n0 + 1);
    auto flush = [&]() { // node n is complete: add it and go to the next
      d0.x += sx; d0.y += sy;
      *node_row(n) = d0;
      sx = sy = 0.f;
      ++n;
      d0 = d1;
      if (n + 1 < n1) d1 = *node_row(n + 1);
      end = n < n1 ? __builtin_amdgcn_readlane(ends, n - n0 + 1) : INT_MAX;
    };
    bf16x8 Br[4], Bs[4];
    int er = 0; // the reverse edge of the next tile's
    auto clamped = [&](int e) { return min(e + lr, e_end - 1); };
    auto load = [&](int e) {
      const int ee = clamped(e);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        Br[ks] = ld8(a.dH + (long)ee * kLat + 32 * ks + lk);
        Bs[ks] = ld8(a.dH + (long)er * kLat + 32 * ks + lk);
      }
      er = a.rev[clamped(e + 16)];
    };
    if (e0 < e_end) {
      er = a.rev[clamped(e0)];
      load(e0);
    }
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
      float2 u[16], v[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        u[k] = *reinterpret_cast<const float2*>(&st[w][0][k][2 * lane]);
        v[k] = *reinterpret_cast<const float2*>(&st[w][1][k][2 * lane]);
      }
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        if (e0 + k >= e_end) break;
        while (e0 + k >= end) flush();
        sx += u[k].x; sy += u[k].y;
        sx += v[k].x; sy += v[k].y;
      }
      wave_lds_sync(); // the next tile rewrites the sums
    }
    while (n < n1) flush();
  }
}
