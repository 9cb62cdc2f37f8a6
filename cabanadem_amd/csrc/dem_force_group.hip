// dem_force_group.hip -- the force pass with eight lanes per particle, for
// systems too small to fill the chip with one.
//
// With one lane per particle a small system's step is one wave's chain of
// dependent memory round trips (own state and row, neighbour positions, the
// row's tail, then per contact the old list, the partner and the FP64 block,
// one contact after the other): 10,000 spheres with three contacts each took
// 17 us on 158 waves, a sixth of the chip's SIMDs.  Here lane s of a particle's
// eight takes neighbour s of its row (then s + 8, ...), old contact s, wall s
// and, for the kicks, component s of (u, omega): everything that is needed is
// loaded in two round trips (own data, partner data, the partner's velocity
// and factors before it is known to touch), the contacts of a particle run
// side by side, and the chain ends in one FP64 block.  The shares of force and
// torque go through LDS and are added component by component in contact order,
// then wall order: the same operations in the same order as one lane walking
// its list, so the results are bitwise those of k_force.
#include "dem_force_kernels.h"

namespace demhip {
namespace {

constexpr int kGroup = 8;           // lanes per particle
constexpr int kGroupBlock = 128;    // threads per workgroup: 16 particles
static_assert(DEM_MAX_WALLS <= kGroup, "one lane per wall");

struct ContactParams {
  double c_eta_pp, c_eta_pw, fr_pp, fr_pw;
};

__device__ inline double pick3(int c, double x, double y, double z) { return c == 0 ? x : (c == 1 ? y : z); }

// ENS: the slot's system from a.sysid, its parameters and walls from a.sys.
// KICK as in force_tile.
template <bool REF, int KICK, bool ENS>
__global__ __launch_bounds__(kGroupBlock) void k_force_group(StepArgs a) {
  __shared__ double sh[kGroupBlock / kGroup][kGroup][6]; // shares of a round, by particle
  const int tid = threadIdx.x, s = tid & (kGroup - 1), lane = tid & 63;
  const int p = tid / kGroup;
  const long ld = a.ld;
  const int i0 = xcd_block(blockIdx.x, gridDim.x) * (kGroupBlock / kGroup) + p;
  const bool act = i0 < a.n;
  const int i = act ? i0 : a.n - 1; // clamped loads; nothing is stored
  // ---- first round trip: everything of the particle's own
  const int sys = ENS ? a.sysid[i] : 0;
  const double4 xi = a.xr_in[i];
  double ui[6];
  load6(a.uw_in + 6l * i, ui);
  const double uc = a.uw_in[6l * i + (s < 6 ? s : 0)]; // this lane's component
  const double2 mI = a.mI[i];
  const double4 mti = a.mat[i];
  const int meta = a.cmeta_in[i];
  const int nnb = act ? a.nn[i] : 0;
  // row entries 0..15, old contacts 0..7 and the wall histories are in bounds
  // whatever the counts, which mask them below
  int row0 = s < a.max_n ? a.nbr[s * ld + i] : i;
  int row1 = s + kGroup < a.max_n ? a.nbr[(s + kGroup) * ld + i] : i;
  int jo = INT_MAX;
  double ho[3] = {0., 0., 0.}, sw[3];
  if (s < a.max_c) {
    jo = a.cj_in[s * ld + i];
#pragma unroll
    for (int d = 0; d < 3; ++d) ho[d] = a.ch_in[(3 * s + d) * ld + i];
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) sw[d] = a.sw[(3 * s + d) * ld + i];
  const SysParams& SP = a.sys[sys];
  const WallConst W = SP.walls[s];
  const int n_walls = ENS ? SP.n_walls : a.sys0.n_walls;
  ContactParams P;
  P.c_eta_pp = ENS ? SP.c_eta_pp : a.sys0.c_eta_pp;
  P.c_eta_pw = ENS ? SP.c_eta_pw : a.sys0.c_eta_pw;
  P.fr_pp = ENS ? SP.fr_pp : a.sys0.fr_pp;
  P.fr_pw = ENS ? SP.fr_pw : a.sys0.fr_pw;
  const int oc = meta_count(meta);
  if (s >= oc) jo = INT_MAX;
  // force and torque: component s (0..2 force, 3..5 torque) in lane s
  double acc = 0.;
  if (s < 3) {
    acc = a.gravity_on ? mI.x * pick3(s, a.g[0], a.g[1], a.g[2]) : 0.;
    if (a.fext) acc += a.fext[3l * i + s];
  }
  // ---- particle contacts, eight row entries at a time
  int nc = 0;
  for (int k0 = 0; __any(k0 < nnb); k0 += kGroup) {
    const bool valid = k0 + s < nnb;
    const int e = k0 == 0 ? row0 : (k0 == kGroup ? row1 : (valid ? a.nbr[(k0 + s) * ld + i] : i));
    const int j = valid ? e : i;
    const double4 xj = a.xr_in[j];
    double uj[6];
    load6(a.uw_in + 6l * j, uj);
    const double4 mj = a.mat[j];
    const double d0 = xi.x - xj.x, d1 = xi.y - xj.y, d2 = xi.z - xj.z;
    const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
    const double sum = xi.w + xj.w;
    // as in force_tile: the margin never filters out a contact
    const bool hit = valid && r2 < sum * sum * (1. + 1e-12) && sum - sqrt(r2) > 0.;
    const unsigned hits = (unsigned)(__ballot(hit) >> (lane & ~(kGroup - 1))) & ((1u << kGroup) - 1);
    const int rank = __popc(hits & ((1u << s) - 1));
    const int m = nc + rank;
    const bool keep = hit && m < a.max_c;
    // the contact's slot in last step's list (src/CabanaDEM_Force.hpp:166-192)
    int po = -1;
#pragma unroll
    for (int t = 0; t < kGroup; ++t)
      if (__shfl(jo, t, kGroup) == j) po = t;
    double h[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double v = __shfl(ho[d], po >= 0 ? po : 0, kGroup);
      h[d] = po >= 0 ? v : 0.;
    }
    if (keep) {
      if (po < 0 && oc > kGroup) { // longer lists than eight: the rest from memory
        for (int t = kGroup; t < oc; ++t)
          if (a.cj_in[t * ld + i] == j) {
#pragma unroll
            for (int d = 0; d < 3; ++d) h[d] = a.ch_in[(3 * t + d) * ld + i];
            break;
          }
      }
      double F[3] = {-0., -0., -0.}, T[3] = {-0., -0., -0.};
      pp_contact<REF>(xi, ui, mti, xj, uj, mj, h, F, T, a, P);
      a.cj_out[m * ld + i] = j;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        a.ch_out[(3 * m + d) * ld + i] = h[d];
        sh[p][rank][d] = F[d];
        if (!REF) sh[p][rank][3 + d] = T[d];
      }
    }
    const int cnt = __popc(hits);
    const int kept = min(cnt, max(a.max_c - nc, 0));
    wave_lds_sync();
    if (s < (REF ? 3 : 6))
      for (int q = 0; q < kept; ++q) acc += sh[p][q][s];
    wave_lds_sync(); // the next round rewrites the shares
    nc += cnt;
  }
  if (nc > a.max_c) {
    if (act && s == 0) atomicMax(&a.flags->contact_overflow, nc);
    nc = a.max_c;
  }
  // ---- walls, one per lane
  double wx[3] = {W.x[0], W.x[1], W.x[2]};
  if (!REF)
#pragma unroll
    for (int d = 0; d < 3; ++d) wx[d] += W.u[d] * a.tw;
  const double q0 = xi.x - wx[0], q1 = xi.y - wx[1], q2 = xi.z - wx[2];  // src/CabanaDEM_Force.hpp:497-499
  const double tmp = q0 * W.n[0] + q1 * W.n[1] + q2 * W.n[2];            // :514
  const double overlap = xi.w - tmp;                                     // :515
  const bool wall = act && s < n_walls && overlap > 0.;                  // :556
  if (wall) {
    double hw[3] = {0., 0., 0.};
    if (meta_walls(meta) & (1 << s))
#pragma unroll
      for (int d = 0; d < 3; ++d) hw[d] = sw[d];
    double F[3] = {-0., -0., -0.}, T[3] = {-0., -0., -0.};
    pw_contact<REF>(xi, ui, mti, W, wx, overlap, hw, F, T, a, P);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      a.sw[(3 * s + d) * ld + i] = hw[d];
      sh[p][s][d] = F[d];
      sh[p][s][3 + d] = T[d];
    }
  }
  const unsigned wn = (unsigned)(__ballot(wall) >> (lane & ~(kGroup - 1))) & ((1u << kGroup) - 1);
  wave_lds_sync();
  if (s < 6)
    for (unsigned b = wn; b; b &= b - 1) acc += sh[p][__ffs(b) - 1][s];
  // ---- kicks and drift, component s in lane s
  double v = 0., xo = 0.;
  if (KICK != 0) {
    const double inv = 1. / (s < 3 ? mI.x : mI.y); // src/CabanaDEM_Integrator.hpp:42,48
    v = uc + a.hdt * acc * inv;                    // stage3 (:89-98)
    xo = pick3(s, xi.x, xi.y, xi.z);
    if (KICK == 2) {
      v = v + a.hdt * acc * inv;                   // stage1 of the next step (:42-51)
      xo = xo + a.dt * v;                          // stage2 (:67-69)
    }
  }
  if (act) {
    if (s == 0) a.cmeta_out[i] = make_meta(nc, (int)wn);
    if (KICK != 0) {
      if (s < 4) reinterpret_cast<double*>(a.xr_out)[4l * i + s] = s < 3 ? xo : xi.w;
      if (s < 6) a.uw_out[6l * i + s] = v;
    }
    if (KICK != 2 && s < 6) a.ft[6l * i + s] = acc;
  }
  if (KICK != 0 && a.disp) { // the displacement check's terms, summed as disp_terms does
    const double d = s < 3 ? xo - a.xb[3l * i + s] : 0.;
    const double dd = d * d, vv = v * v;
    double m2 = __shfl(dd, 0, kGroup) + __shfl(dd, 1, kGroup) + __shfl(dd, 2, kGroup);
    double s2 = __shfl(vv, 0, kGroup) + __shfl(vv, 1, kGroup) + __shfl(vv, 2, kGroup);
    m2 = act ? max_nan(0., m2) : 0.;
    s2 = act ? max_nan(0., s2) : 0.;
    disp_block_max<kGroupBlock>(m2, s2, a.disp);
  }
}

template <bool REF, bool ENS>
hipError_t launch_group(ForceKind kind, const StepArgs& a, hipStream_t s) {
  const int per = kGroupBlock / kGroup;
  const dim3 g((a.n + per - 1) / per), b(kGroupBlock);
  switch (kind) {
    case FK_PP_PW_FORCES: hipLaunchKernelGGL((k_force_group<REF, 0, ENS>), g, b, 0, s, a); break;
    case FK_STEP_LAST: hipLaunchKernelGGL((k_force_group<REF, 1, ENS>), g, b, 0, s, a); break;
    case FK_STEP_FUSED: hipLaunchKernelGGL((k_force_group<REF, 2, ENS>), g, b, 0, s, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

} // namespace

hipError_t launch_force_group(bool ref, ForceKind kind, const StepArgs& a, hipStream_t s) {
  if (a.sysid) return ref ? launch_group<true, true>(kind, a, s) : launch_group<false, true>(kind, a, s);
  return ref ? launch_group<true, false>(kind, a, s) : launch_group<false, false>(kind, a, s);
}

} // namespace demhip
