// k_hf_vol.hip - the flux form of the heat-flux pass in the volume mode
// (pgk_calforce_heatf and the MD loop's samples with z regions).
//
// calvirihf (calvirihf.F90:201-357) gives a pair with centres c_i, c_j and
// share s = f_i . v_i - f_j . v_j the weight of region [z1, z2]: the signed
// length of the segment c_j -> c_i inside the region.  With
// G_r(c) = clamp(c, z1, z2) - z1 that length is G_r(c_i) - G_r(c_j), so the
// sum over pairs separates into atoms,
//   sum_pairs s (G_r(c_i) - G_r(c_j)) = sum_atoms S_a G_r(c_a),
//   S_a = sum of s over the pairs where a comes first minus the others,
// and the pair pass does not look at regions at all: it adds a pair's energy
// and share to its two atoms, and one pass over the atoms puts them into the
// regions.  (Weighing every region a pair's segment crosses in the pair pass
// cost one LDS atomic per class, region and pair: 17.4 ms of a 26.5 ms call
// on 996,000 atoms with 300 one-A bins; now 4.6 ms, and the regions' sums
// 130 us instead of 1.5 ms.)
//
// The rule's one deviation from the segment's length is kept: a first atom
// whose centre lies exactly on a region's plane, with the second on the far
// side of it, counts the whole segment (a.z flag in the packed data, one
// branch; the regions' sums of these in jpart).
//
// Sums: per slot of the cluster list, FP64 in the FP64 and FP32 forms.  In the
// mixed form fixed point, so the result does not depend on the order of the
// additions: the energies in 2^-32 like the forces, the shares in two words
// (2^-10 and 2^-52), which hold as wide a range as FP64 sums need and resolve
// what a region's sum of cancelling shares keeps.
#include <type_traits>

#include "pgk_hf.h"

namespace {

// words of a slot: pairs between molecules e_elc e_vdw s_elc s_vdw (mixed: the
// s as 2^-10 words, then their 2^-52 words), then the same for pairs inside
// one molecule
template <class AH> struct VolAcc { static constexpr int N = 4; };
template <> struct VolAcc<unsigned long long> { static constexpr int N = 6; };

constexpr int kMolMole = 1 << 30;    // mt.x: molecule id, MOLE centre
constexpr int kTypPlane = 1 << 30;   // mt.y: 0-based type, centre on a region's plane

__device__ __forceinline__ unsigned long long vol_hi(double v) {
  return (unsigned long long)__double2ll_rn(v * 1024.0);
}
__device__ __forceinline__ unsigned long long vol_lo(double v) {
  const double r = v - (double)__double2ll_rn(v * 1024.0) * (1.0 / 1024.0);
  return (unsigned long long)__double2ll_rn(r * 0x1p52);
}

// value `k` (0 e_elc, 1 e_vdw, 2 s_elc, 3 s_vdw) of a slot's group w; half:
// 0 the whole value or its high word, 1 the low word (mixed shares)
__device__ __forceinline__ void vol_add(double *w, int k, int half, double v) {
  if (half == 0) atomicAdd(&w[k], v);
}
__device__ __forceinline__ void vol_add(unsigned long long *w, int k, int half, double v) {
  if (k < 2) {
    if (half == 0) acc_add(&w[k], v);
  } else {
    atomicAdd(&w[k + 2 * half], half ? vol_lo(v) : vol_hi(v));
  }
}
// a share in two adjacent words (mixed: high and low)
__device__ __forceinline__ void share_add(double *w, double v) { atomicAdd(w, v); }
__device__ __forceinline__ void share_add(unsigned long long *w, double v) {
  atomicAdd(w, vol_hi(v));
  atomicAdd(w + 1, vol_lo(v));
}
__device__ __forceinline__ double share_load(const double *w) { return *w; }
__device__ __forceinline__ double share_load(const unsigned long long *w) {
  return (double)(long long)w[0] * (1.0 / 1024.0) + (double)(long long)w[1] * 0x1p-52;
}

// the 4 sums of a cluster's slot over the 8 lanes that share it, added by
// lanes jj = 0..3 (4, 5: the low words of the mixed shares).  Mixed energies
// are rounded to fixed point per lane, as every addition to a sum is.
__device__ __forceinline__ void vol_add_i(double *w, const double (&v)[4], int jj) {
  double t[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    t[k] = v[k];
#pragma unroll
    for (int o = 8; o < 64; o <<= 1) t[k] += __shfl_xor(t[k], o, 64);
  }
  const double x = jj == 0 ? t[0] : jj == 1 ? t[1] : jj == 2 ? t[2] : t[3];
  if (jj < 4 && x != 0.0) atomicAdd(&w[jj], x);
}
__device__ __forceinline__ void vol_add_i(unsigned long long *w, const double (&v)[4], int jj) {
  unsigned long long t[6] = {acc_val<unsigned long long>(v[0]), acc_val<unsigned long long>(v[1]),
                             vol_hi(v[2]), vol_hi(v[3]), vol_lo(v[2]), vol_lo(v[3])};
#pragma unroll
  for (int k = 0; k < 6; k++)
#pragma unroll
    for (int o = 8; o < 64; o <<= 1) t[k] += __shfl_xor(t[k], o, 64);
  const unsigned long long x = jj == 0   ? t[0]
                               : jj == 1 ? t[1]
                               : jj == 2 ? t[2]
                               : jj == 3 ? t[3]
                               : jj == 4 ? t[4]
                                         : t[5];
  if (jj < 6 && x != 0) atomicAdd(&w[jj], x);
}
__device__ __forceinline__ double vol_load(const double *w, int k) { return w[k]; }
__device__ __forceinline__ double vol_load(const unsigned long long *w, int k) {
  if (k < 2) return acc_load(&w[k]);
  return (double)(long long)w[k] * (1.0 / 1024.0) + (double)(long long)w[k + 2] * 0x1p-52;
}

// per slot: position and charge, collision-part velocity and centre z,
// molecule and type with their flags; the slot's sums start at zero
template <class AH>
__global__ __launch_bounds__(256) void k_hf_vol_pack(int nslot,
                                                     const int32_t *__restrict__ cl_atom,
                                                     HfDev h, const double *__restrict__ q,
                                                     const int32_t *__restrict__ ct,
                                                     double4 *__restrict__ xq,
                                                     double4 *__restrict__ vc,
                                                     int2 *__restrict__ mt,
                                                     AH *__restrict__ acc) {
  constexpr int NW = 2 * VolAcc<AH>::N;
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  // the block's slots hold NW * 256 consecutive words
  const int w0 = blockIdx.x * 256 * NW, w1 = min(w0 + 256 * NW, nslot * NW);
  for (int k = w0 + (int)threadIdx.x; k < w1; k += 256) acc[k] = (AH)0;
  if (s >= nslot) return;
  const int a = cl_atom[s];
  if (a < 0) {
    xq[s] = vc[s] = make_double4(0.0, 0.0, 0.0, 0.0);
    mt[s] = make_int2(0, 0);
    return;
  }
  xq[s] = make_double4(h.pos[3 * a], h.pos[3 * a + 1], h.pos[3 * a + 2], q[a]);
  double c[3];
  const int atomc = hf_centre(h, a, false, c);
  bool plane = false;
  int r0, r1;
  hf_region_window(h, c[2], c[2], r0, r1);
  for (int r = r0; r <= r1; r++) plane = plane || h.z1[r] == c[2] || h.z2[r] == c[2];
  vc[s] = make_double4(h.vel[3 * a], h.vel[3 * a + 1], h.vel[3 * a + 2], c[2]);
  mt[s] = make_int2(h.molid[a] | (atomc ? 0 : kMolMole), ct[s] | (plane ? kTypPlane : 0));
}

struct HfVolArgs {
  const int32_t *ci_start, *cj;   // cj: half-cluster index of each entry
  const uint32_t *mask;
  const int32_t *witem;           // chunked form: work items (cluster * 32 + chunk of 64 entries)
  int ncl, nwi, ntype;
  const double4 *xq, *vc;
  const int2 *mt;
  const double *lj;               // ntype^2 x (eps, 0 unless INTTYPE_VDW; rmin^2)
  double sqcut, sqcut2, rrsq;
  double L[3], Li[3];
};

// One wave per cluster, or per 64 entries of one (CH); lane = ii + 8 jq + 32 hs
// as in the pair kernel, whose scheme of a chunk's entries in registers and
// the next pass's j data in flight it follows (the pass waits for memory: 72
// bytes per j slot and about 100 FP64 instructions per 64 pairs).  The i
// atoms' sums stay in registers; a j atom's four sums over its 8 lanes leave
// as one atomic each to adjacent words of its slot.
template <class AH, bool CH, bool LJLDS>
__global__ __launch_bounds__(256) void k_hf_pairs_vol(HfVolArgs p, HfDev h,
                                                      AH *__restrict__ acc) {
  using R = typename std::conditional<std::is_same<AH, unsigned long long>::value, float,
                                      double>::type;
  constexpr int NG = VolAcc<AH>::N, NW = 2 * NG;
  extern __shared__ double s_lj[];
  if (LJLDS) {
    for (int k = threadIdx.x; k < 2 * p.ntype * p.ntype; k += 256) s_lj[k] = p.lj[k];
    __syncthreads();
  }
  const double *lj = LJLDS ? s_lj : p.lj;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  int ci = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + wave), chunk = 0;
  if (CH) {
    const int w = ci;
    ci = p.ncl;
    if (w < p.nwi) {
      const int item = __builtin_amdgcn_readfirstlane(p.witem[w]);
      ci = item >> 5;
      chunk = item & 31;
    }
  }
  if (ci >= p.ncl) return;
  const int ii = lane & 7, jq = (lane >> 3) & 3, hs = lane >> 5;
  const int islot = ci * PGK_CL + ii;
  const double4 xi = p.xq[islot], vi = p.vc[islot];
  const int2 mi = p.mt[islot];
  const int typi = mi.y & ~kTypPlane;
  const bool plane = (mi.y & kTypPlane) != 0;
  // the i atom's sums over this lane's pairs: between molecules, inside one
  double si[4] = {0.0, 0.0, 0.0, 0.0}, sin[4] = {0.0, 0.0, 0.0, 0.0};
  int e0 = __builtin_amdgcn_readfirstlane(p.ci_start[ci]),
      e1 = __builtin_amdgcn_readfirstlane(p.ci_start[ci + 1]);
  if (CH) {
    e0 += 64 * chunk;
    e1 = min(e1, e0 + 64);
  }
  struct Ent {
    int js;
    uint32_t m;   // this lane's entry's mask
    double4 xj, vj;
    int2 mj;
  };
  const int nent = e1 - e0;
  bool any_inner = false, far = false;
  for (int cb = 0; cb < nent; cb += 64) {
    const int nin = min(64, nent - cb);
    const int c_hc = (lane < nin) ? p.cj[e0 + cb + lane] : 0;
    const uint32_t c_m = (lane < nin) ? p.mask[e0 + cb + lane] : 0u;
    auto fetch = [&](Ent &d, int k) {   // entries k and k + 1 (mask 0 past the end)
      const int kk = min(k, 62);
      const int ha = __builtin_amdgcn_readlane(c_hc, kk);
      const int hb = __builtin_amdgcn_readlane(c_hc, kk + 1);
      const uint32_t ma = (k < nin) ? (uint32_t)__builtin_amdgcn_readlane((int)c_m, kk) : 0u;
      const uint32_t mb =
          (k + 1 < nin) ? (uint32_t)__builtin_amdgcn_readlane((int)c_m, kk + 1) : 0u;
      d.m = hs ? mb : ma;
      d.js = (hs ? hb : ha) * 4 + jq;
      d.xj = p.xq[d.js];
      d.vj = p.vc[d.js];
      d.mj = p.mt[d.js];
    };
    auto pass = [&](const Ent &d) {
      double sj[4] = {0.0, 0.0, 0.0, 0.0};   // e_elc, e_vdw, s_elc, s_vdw of the j atom
      bool same = false;
      if ((d.m >> (lane & 31)) & 1u) {
        double r[3] = {xi.x - d.xj.x, xi.y - d.xj.y, xi.z - d.xj.z};
        for (int k = 0; k < 3; k++) r[k] = r[k] - p.L[k] * rint(r[k] * p.Li[k]);
        const double r2 = hf_r2_exact(r);
        if (r2 <= p.sqcut) {
          // the cutoff tests stay exact FP64 decisions; the pair terms are in
          // the compute type R (FP32 in the mixed form: one hardware rsqrt)
          const R rinv1 = hf_rinv<R>(r2);
          const R rinv2 = rinv1 * rinv1;
          same = ((mi.x ^ d.mj.x) & ~kMolMole) == 0;
          const double dz = vi.w - d.vj.w;
          const bool seg = !(same && (mi.x & d.mj.x & kMolMole)) && fabs(dz) * p.Li[2] < 0.5;
          // s / 2 per unit force coefficient (fi . v_i - fj . v_j, fj = -fi)
          const double w[3] = {vi.x + d.vj.x, vi.y + d.vj.y, vi.z + d.vj.z};
          const double rw = seg ? 0.5 * (r[0] * w[0] + r[1] * w[1] + r[2] * w[2]) : 0.0;
          R ec = R(0), ev = R(0), fc = R(0), fv = R(0);
          if (r2 <= p.rrsq) {
            ec = (R)xi.w * (R)d.xj.w * rinv1;
            fc = ec * rinv2;
          }
          if (r2 <= p.sqcut2) {
            const int tp = typi + p.ntype * (d.mj.y & ~kTypPlane);
            const R ep = (R)lj[2 * tp];   // 0 unless INTTYPE_VDW
            const R t2 = rinv2 * (R)lj[2 * tp + 1];
            const R t6 = t2 * t2 * t2;
            const R t12 = t6 * t6;
            ev = ep * (t12 - (R)2 * t6);
            fv = (R)12 * ep * (t12 - t6) * rinv2;
          }
          const double v[4] = {0.5 * (double)ec, 0.5 * (double)ev, (double)fc * rw,
                               (double)fv * rw};
#pragma unroll
          for (int k = 0; k < 4; k++) {
            if (same) sin[k] += v[k];
            else si[k] += v[k];
            sj[k] = k < 2 ? v[k] : -v[k];
          }
          if (plane && rw != 0.0 && dz != 0.0) {
            for (int q = 0; q < h.nreg; q++)
              if (dz > 0.0 ? h.z1[q] == vi.w : h.z2[q] == vi.w) {
                AH *pw = reinterpret_cast<AH *>(h.jpart) + ((size_t)q * 4 + (same ? 0 : 2)) * 2;
                share_add(pw, v[2] * dz);
                share_add(pw + 2, v[3] * dz);
              }
          }
        }
      }
      // lanes ii and ii ^ 1 hold sum (ii >> 1) of j slot js; the even lane adds
      // the value (or its high word), the odd one a mixed share's low word
      const bool inner = __ballot(same) != 0;   // pairs inside one molecule are few
      double so[4];
#pragma unroll
      for (int k = 0; k < 4; k++) so[k] = inner && same ? 0.0 : sj[k];
      const double t = hf_sum4x8(so, ii);
      far = far || !(fabs(t) < 0x1p52);
      if (t != 0.0) vol_add(acc + (size_t)d.js * NW, ii >> 1, ii & 1, t);
      if (inner) {
        any_inner = true;
#pragma unroll
        for (int k = 0; k < 4; k++) so[k] = same ? sj[k] : 0.0;
        const double u = hf_sum4x8(so, ii);
        far = far || !(fabs(u) < 0x1p52);
        if (u != 0.0) vol_add(acc + (size_t)d.js * NW + NG, ii >> 1, ii & 1, u);
      }
    };
    Ent A, B;
    fetch(A, 0);
    for (int k = 0; k < nin; k += 4) {
      fetch(B, k + 2);
      pass(A);
      fetch(A, k + 4);
      pass(B);
    }
  }
  vol_add_i(acc + (size_t)islot * NW, si, lane >> 3);
  if (any_inner) vol_add_i(acc + (size_t)islot * NW + NG, sin, lane >> 3);
  // a share that fixed point cannot hold (infinite, NaN): flagged for the
  // regions' sums, which FP64 sums would carry it into
  if (std::is_same<AH, unsigned long long>::value && __ballot(far) != 0 && lane == 0)
    atomicOr(reinterpret_cast<unsigned long long *>(h.jpart) + 8 * (size_t)h.nreg, 1ull);
}

// one item's (slot's or atom's) contributions
struct VolItem {
  double cz;             // transport centre z, wrapped into [0, Lz)
  double c;              // collision centre z
  double vz;             // the centre's velocity
  double e[1 + PGK_NHF]; // kinetic energy, potential energies by class
  double s[4];           // collision shares ELIN, LJIN, ELC, VDW
};

template <class AH>
__device__ __forceinline__ bool vol_item(const HfBinArgs &a, int k, VolItem &o) {
  const int i = a.order ? a.order[k] : k;
  if (i < 0) return false;
  const bool mole = a.hftyp[i] == PGK_HFTYP_MOLE;
  const int m = a.molid[i] - 1;
  double z = mole ? a.molecom[3 * (size_t)m + 2] : a.pos[3 * (size_t)i + 2];
  o.c = z;
  if (z < 0.0) z = z + a.Lz;
  else if (z >= a.Lz) z = z - a.Lz;
  o.cz = z;
  if (!mole) o.c = z;
  o.vz = mole ? a.molevel[3 * (size_t)m + 2] : a.vel[3 * (size_t)i + 2];
  // kinetic energy relative to the streaming velocity (calheatf.F90:368-369,
  // 677-681); the transported centre velocity stays lab-frame
  double v[3] = {a.vel[3 * (size_t)i], a.vel[3 * (size_t)i + 1], a.vel[3 * (size_t)i + 2]};
  if (a.vstrm)
    for (int d = 0; d < 3; d++) v[d] = v[d] - a.vstrm[3 * (size_t)i + d];
  o.e[0] = 0.5 * a.mass[i] * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
  const AH *pe = reinterpret_cast<const AH *>(a.pe);
#pragma unroll
  for (int q = 0; q < PGK_HF_ELIN; q++)
    o.e[1 + q] = pe ? acc_load(&pe[(size_t)q * a.natom + i]) : 0.0;
  constexpr int NG = VolAcc<AH>::N;
  const AH *w = a.acc ? reinterpret_cast<const AH *>(a.acc) + (size_t)k * 2 * NG : nullptr;
#pragma unroll
  for (int g = 0; g < 2; g++)
#pragma unroll
    for (int q = 0; q < 2; q++) {   // g 0: inside one molecule (ELIN, LJIN), 1: ELC, VDW
      const AH *wg = g ? w : w + NG;
      o.e[1 + PGK_HF_ELIN + 2 * g + q] = w ? vol_load(wg, q) : 0.0;
      o.s[2 * g + q] = w ? vol_load(wg, 2 + q) : 0.0;
    }
  return true;
}

// Regions that tile their range (h.tiled): one wave per part of the items,
// every region's sums in LDS.  An atom adds its transport values to the
// region (or, on a plane, the two) it lies in, and its shares S to region ka
// (the last with z1 <= c) as S (min(c, z2) - z1); the regions below ka take
// S times their whole width, kept as a sum per ka and summed from above at
// the end.  Record per region and part: 9 transport sums, 4 collision sums.
// 64-thread blocks: additions of one wave to one address happen in lane
// order, so the sums do not depend on timing.
template <class AH>
__global__ __launch_bounds__(64) void k_hf_vol_bins(HfBinArgs a, double *__restrict__ part) {
  extern __shared__ double sm[];   // [17][nreg]: 9 transport, 4 partial, 4 whole-width
  const int nreg = a.nreg, lane = threadIdx.x;
  for (int k = lane; k < 17 * nreg; k += 64) sm[k] = 0.0;
  __syncthreads();
  double *sp = sm + 9 * nreg, *sd = sm + 13 * nreg;
  const int i0 = blockIdx.x * a.per, i1 = min(a.nitem, i0 + a.per);
  auto region_of = [&](double z) {   // the last region with z1 <= z, -1: none
    int k = min(nreg - 1, max(-1, (int)floor((z - a.ubz0) * a.ubwi)));
    while (k + 1 < nreg && a.z1[k + 1] <= z) k++;
    while (k >= 0 && a.z1[k] > z) k--;
    return k;
  };
  for (int k = i0 + lane; k < i1; k += 64) {
    VolItem it;
    if (!vol_item<AH>(a, k, it)) continue;
    const int kt = region_of(it.cz);
#pragma unroll
    for (int b = 0; b < 2; b++) {   // region kt, and kt - 1 where its upper plane is met
      const int r = kt - b;
      if (r < 0 || it.cz > a.z2[r]) continue;
#pragma unroll
      for (int t = 0; t < 1 + PGK_NHF; t++)
        if (it.e[t] != 0.0) atomicAdd(&sm[t * nreg + r], it.e[t] * it.vz);
    }
    const int kc = region_of(it.c);
    if (kc >= 0) {
      const double len = fmin(it.c, a.z2[kc]) - a.z1[kc];
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (it.s[q] != 0.0) {
          atomicAdd(&sp[q * nreg + kc], it.s[q] * len);
          atomicAdd(&sd[q * nreg + kc], it.s[q]);
        }
    }
  }
  __syncthreads();
  // shares of the regions above, per class: each lane a run of regions
  const int run = (nreg + 63) / 64, r0 = min(nreg, lane * run), r1 = min(nreg, r0 + run);
#pragma unroll
  for (int q = 0; q < 4; q++) {
    double own = 0.0;
    for (int r = r0; r < r1; r++) own += sd[q * nreg + r];
    double above = own;   // inclusive sum of the lanes from here up
    for (int o = 1; o < 64; o <<= 1) {
      const double t = __shfl_down(above, o, 64);
      if (lane + o < 64) above += t;
    }
    above -= own;
    for (int r = r1 - 1; r >= r0; r--) {
      sp[q * nreg + r] += (a.z2[r] - a.z1[r]) * above;
      above += sd[q * nreg + r];
    }
  }
  __syncthreads();
  for (int k = lane; k < 13 * nreg; k += 64) {
    const int r = k / 13, t = k - 13 * r;
    part[((size_t)r * a.nsplit + blockIdx.x) * 13 + t] = sm[t * nreg + r];
  }
}

// any regions (few, or not tiling their range): block (part of the items,
// region), the same record
template <class AH>
__global__ __launch_bounds__(256) void k_hf_vol_regions(HfBinArgs a, double *__restrict__ part) {
  const int r = blockIdx.y;
  const double z1 = a.z1[r], z2 = a.z2[r];
  double v[13];
#pragma unroll
  for (int t = 0; t < 13; t++) v[t] = 0.0;
  const int i0 = blockIdx.x * a.per, i1 = min(a.nitem, i0 + a.per);
  for (int k = i0 + (int)threadIdx.x; k < i1; k += 256) {
    VolItem it;
    if (!vol_item<AH>(a, k, it)) continue;
    if (z1 <= it.cz && it.cz <= z2)
#pragma unroll
      for (int t = 0; t < 9; t++) v[t] += it.e[t] * it.vz;
    const double len = fmin(fmax(it.c, z1), z2) - z1;
#pragma unroll
    for (int q = 0; q < 4; q++) v[9 + q] += it.s[q] * len;
  }
  block_record<13, 4>(v, part + ((size_t)r * a.nsplit + blockIdx.x) * 13);
}

// the parts' records in a fixed order, the bonded terms' sums (jcol), the
// volume factor and the total (calheatf.F90:1334-1436): one block per region
template <class AH>
__global__ __launch_bounds__(256) void k_hf_vol_final(HfBinArgs a, const double *__restrict__ part,
                                                      const AH *__restrict__ jcol,
                                                      const AH *__restrict__ plane,
                                                      double *__restrict__ out) {
#pragma clang fp contract(off)
  constexpr int G = 19;   // 19 groups of 13 threads
  __shared__ double s[G][13], fin[PGK_HFJ_TOT];
  const int r = blockIdx.x, g = threadIdx.x / 13, t = threadIdx.x - 13 * g;
  if (g < G) {
    double v = 0.0;
    for (int k = g; k < a.nsplit; k += G) v += part[((size_t)r * a.nsplit + k) * 13 + t];
    s[g][t] = v;
  }
  __syncthreads();
  const double vol_inv = ((1.0 / a.Lx) * (1.0 / a.Ly)) / (a.z2[r] - a.z1[r]);
  if (threadIdx.x < PGK_HFJ_TOT) {
    const int k = threadIdx.x;   // 0 kinetic, 1..8 potential, 9..16 collision classes
    double v = 0.0;
    const int src = k < 9 ? k : (k - 9 >= PGK_HF_ELIN ? k - PGK_HF_ELIN : -1);
    if (src >= 0)
      for (int q = 0; q < G; q++) v += s[q][src];
    if (src >= 9) v += share_load(plane + ((size_t)r * 4 + (src - 9)) * 2);
    if (src >= 9 && plane[8 * (size_t)a.nreg] != (AH)0) v = __builtin_nan("");
    if (k >= 9) v += acc_load(&jcol[3 * ((size_t)(k - 9) * a.nreg + r) + 2]);
    fin[k] = v * vol_inv;
  }
  __syncthreads();
  double *o = out + (size_t)r * PGK_NHFJ * 3;
  for (int k = threadIdx.x; k < PGK_HFJ_TOT * 3; k += 256) o[k] = k % 3 == 2 ? fin[k / 3] : 0.0;
  if (threadIdx.x < 3) {
    double tot = threadIdx.x == 2 ? fin[0] : 0.0;
    if (threadIdx.x == 2)
      for (int k = 1; k < PGK_HFJ_TOT; k++) tot = tot + fin[k];
    o[3 * PGK_HFJ_TOT + threadIdx.x] = tot;
  }
}

template <class AH>
int launch_pairs_vol(pgk_ctx *c) {
  constexpr int NW = 2 * VolAcc<AH>::N;
  hipStream_t st = c->stream;
  const HfDev &h = c->hfdev;
  const int nslot = c->ncl * PGK_CL;
  int rc;
  if ((rc = grow_dev((void **)&c->d_hfw_xq, &c->hfw_xq_bytes, sizeof(double4) * nslot)) ||
      (rc = grow_dev((void **)&c->d_hfw_v, &c->hfw_v_bytes, sizeof(double4) * nslot)) ||
      (rc = grow_dev((void **)&c->d_hfv_mt, &c->hfv_mt_bytes, sizeof(int2) * nslot)) ||
      (rc = grow_dev(&c->d_hfv_acc, &c->hfv_acc_bytes, sizeof(AH) * NW * (size_t)nslot)))
    return rc;
  AH *acc = reinterpret_cast<AH *>(c->d_hfv_acc);
  k_hf_vol_pack<AH><<<pgk_grid_blocks(nslot, 256), 256, 0, st>>>(
      nslot, c->d_cl_atom, h, c->d_q, c->d_ct, c->d_hfw_xq, c->d_hfw_v,
      reinterpret_cast<int2 *>(c->d_hfv_mt), acc);
  HIP_CHECK(hipGetLastError());
  HfVolArgs p;
  p.ci_start = c->d_ci_start;
  p.cj = c->d_cj;
  p.mask = c->d_mask;
  p.witem = c->d_witem;
  p.ncl = c->ncl;
  p.nwi = c->nwi;
  p.ntype = c->ntype;
  p.xq = c->d_hfw_xq;
  p.vc = c->d_hfw_v;
  p.mt = reinterpret_cast<const int2 *>(c->d_hfv_mt);
  p.lj = c->d_ljp64;
  const double sq = c->rrcut * c->rrcut, sq2 = c->rcut * c->rcut;
  p.sqcut = sq2 > sq ? sq2 : sq;
  p.sqcut2 = sq2;
  p.rrsq = c->rrsq_cut;
  for (int d = 0; d < 3; d++) {
    p.L[d] = h.L[d];
    p.Li[d] = h.Li[d];
  }
  const int nblk = pgk_grid_blocks(pgk_pair_waves(c), 4);
  const bool ch = pgk_pair_chunked(c);
  // the LJ table in LDS up to 16 KiB (32 atom types)
  const size_t ljb = sizeof(double) * 2 * (size_t)c->ntype * c->ntype;
  const bool ll = ljb <= 16384;
  auto kf = ch ? (ll ? k_hf_pairs_vol<AH, true, true> : k_hf_pairs_vol<AH, true, false>)
               : (ll ? k_hf_pairs_vol<AH, false, true> : k_hf_pairs_vol<AH, false, false>);
  kf<<<nblk, 256, ll ? ljb : 0, st>>>(p, h, acc);
  HIP_CHECK(hipGetLastError());
  c->hfdev.vol_pairs = 1;
  return PGK_OK;
}

template <class AH>
int launch_bins(pgk_ctx *c, HfBinArgs &a, double *part, double *out) {
  hipStream_t st = c->stream;
  if (a.tiled) {
    const size_t lds = sizeof(double) * 17 * (size_t)a.nreg;
    const int lr = pgk_lds_limit((const void *)k_hf_vol_bins<AH>, lds);
    if (lr) return lr;
    k_hf_vol_bins<AH><<<a.nsplit, 64, lds, st>>>(a, part);
  } else {
    k_hf_vol_regions<AH><<<dim3(a.nsplit, a.nreg), 256, 0, st>>>(a, part);
  }
  HIP_CHECK(hipGetLastError());
  k_hf_vol_final<AH><<<a.nreg, 256, 0, st>>>(
      a, part, reinterpret_cast<const AH *>(c->hfdev.jcol),
      reinterpret_cast<const AH *>(c->hfdev.jpart), out);
  HIP_CHECK(hipGetLastError());
  return PGK_OK;
}

}  // namespace

// Queue the packing and the pair pass; the slots' sums are in d_hfv_acc.
int pgk_hf_vol_launch(pgk_ctx *c) {
  return c->precision == PGK_PREC_MIXED ? launch_pairs_vol<unsigned long long>(c)
                                        : launch_pairs_vol<double>(c);
}

// Queue the regions' sums over the slots (over the atoms when no pair pass
// ran) into out, nregion x PGK_NHFJ x 3 doubles.
int pgk_hf_vol_bins_launch(pgk_ctx *c, HfBinArgs a, double *out) {
  const HfDev &h = c->hfdev;
  a.natom = c->natom;
  a.nreg = h.nreg;
  a.tiled = h.tiled;
  a.ubz0 = h.ubz0;
  a.ubwi = h.ubwi;
  a.z1 = h.z1;
  a.z2 = h.z2;
  a.hftyp = h.hftyp;
  a.molid = h.molid;
  a.molecom = h.molecom;
  a.pos = h.pos;
  a.Lx = h.L[0];
  a.Ly = h.L[1];
  a.Lz = h.L[2];
  a.pe = pgk_has_bonded(c) ? h.pe : nullptr;
  a.acc = h.vol_pairs ? c->d_hfv_acc : nullptr;
  a.order = h.vol_pairs ? c->d_cl_atom : nullptr;
  a.nitem = h.vol_pairs ? c->ncl * PGK_CL : c->natom;
  // tiled: parts of 256 items up to 1024 waves; otherwise about 2048 blocks in
  // all, at least 256 items each
  int ns = (a.nitem + 255) / 256;
  ns = std::max(1, std::min(ns, a.tiled ? 1024 : (2048 + a.nreg - 1) / a.nreg));
  a.nsplit = ns;
  a.per = (a.nitem + ns - 1) / ns;
  int rc;
  if ((rc = grow_dev((void **)&c->d_hj_part, &c->hj_part_cap,
                     sizeof(double) * 13 * (size_t)a.nreg * ns)))
    return rc;
  return c->precision == PGK_PREC_MIXED
             ? launch_bins<unsigned long long>(c, a, c->d_hj_part, out)
             : launch_bins<double>(c, a, c->d_hj_part, out);
}
