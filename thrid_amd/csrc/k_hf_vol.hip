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
// on 996,000 atoms with 300 one-A bins; now 4.9 ms, and the regions' sums
// 0.21 ms instead of 1.5.)
//
// The atoms' sums cancel where the pairs' did not: every region below a pair
// takes s from one atom and -s from the other.  So the shares are whole
// numbers of a unit, rounded once per pair, and summed exactly: two words of
// 64 bits, multiples of 2^-16 and of 2^-58 of a typical velocity times the
// force (vol_unit).  The pairs above a region then leave exactly nothing in
// it, a region that no segment meets is exactly zero, and the rounding of a
// region's sum is that of its own pairs (2^-59 each).  The products with
// lengths inside a region and the regions' sums of them carry two doubles.
// (With FP64 sums per atom instead the pair pass took 4.6 ms there, and 98 us
// against 117 on an 18,000-atom slab in FP64.)
//
// Three kinds of pair are weighed region by region instead, into jpart:
// - a first atom whose centre lies exactly on a region's plane, with the
//   second on the far side of it: there the reference's rule counts the whole
//   segment (kTypPlane; the atoms' shares count the rest);
// - a share of 2^24 units and more, infinite or NaN (atoms on top of each
//   other): it reaches the regions its segment meets and no other;
// - every pair, if a region's bounds are the wrong way round (h.reversed).
//
// Energies per slot of the cluster list: FP64 in the FP64 and FP32 forms, 2^-32
// fixed point like the forces in the mixed form.
#include <type_traits>

#include "pgk_hf.h"

namespace {

// words of a slot: pairs between molecules e_elc e_vdw, the shares' high words
// s_elc s_vdw and their low words, then the same for pairs inside one molecule
constexpr int kVolN = 6, kVolNW = 2 * kVolN;
using vol_word = unsigned long long;

constexpr int kMolMole = 1 << 30;    // mt.x: molecule id, MOLE centre
constexpr int kTypPlane = 1 << 30;   // mt.y: 0-based type, centre on a region's plane

// Adding 1.5 x 2^(52 - b) to a number rounds it to a multiple of 2^-b, and
// leaves that multiple as an integer in the low bits of the sum: |v| < 2^35
// for the high words (b = 16), 2^-7 for the low ones (b = 58).  A lane sums at
// most 1024 pairs (2048 entries of a cluster, two a pass) before it converts.
constexpr double kVolHi = 0x1.8p36, kVolLo = 0x1.8p-6, kVolMax = 0x1p24;
__device__ __forceinline__ vol_word vol_int(double v, double k) {
  return (vol_word)(__double_as_longlong(v + k) - __double_as_longlong(k));
}
__device__ __forceinline__ void vol_split(double s, double &hi, double &lo) {
  hi = (s + kVolHi) - kVolHi;
  lo = ((s - hi) + kVolLo) - kVolLo;
}
__device__ __forceinline__ double vol_val_hi(vol_word w) { return (double)(long long)w * 0x1p-16; }
__device__ __forceinline__ double vol_val_lo(vol_word w) { return (double)(long long)w * 0x1p-58; }

// jpart in this mode: per region and pair class a high word, a low word and a
// double for what they cannot hold; then the sum of the velocities' exponents
// and their count
__device__ __host__ __forceinline__ size_t vol_jw(int reg, int cls) {
  return ((size_t)reg * 4 + cls) * 3;
}
__device__ __forceinline__ void vol_region_add(const HfDev &h, int reg, int cls, double v) {
  double *w = h.jpart + vol_jw(reg, cls);
  if (fabs(v) < 0x1p32) {
    const double hi = rint(v * 0x1p16);
    atomicAdd(reinterpret_cast<vol_word *>(w), (vol_word)(long long)hi);
    atomicAdd(reinterpret_cast<vol_word *>(w) + 1,
              (vol_word)__double2ll_rn((v - hi * 0x1p-16) * 0x1p58));
  } else {
    atomicAdd(w + 2, v);
  }
}

// The unit of the shares: the power of two at the mean exponent of the atoms'
// velocities (their largest components; zeros, infinities and NaN aside), so
// that the words hold as many digits of a cold system's shares as of a hot
// one's, and one atom of extreme velocity does not shift it.
__device__ __forceinline__ int vol_unit_exp(const double *jpart, int nreg) {
  const vol_word *w = reinterpret_cast<const vol_word *>(jpart + vol_jw(nreg, 0));
  const vol_word n = w[1];
  if (n == 0) return 0;
  const int e = (int)rint((double)w[0] / (double)n) - 1023;
  return max(-1000, min(1000, e));
}
__device__ __forceinline__ double vol_pow2(int e) {
  return __longlong_as_double((long long)(1023 + e) << 52);
}

// Sums to a slot's words.  Mixed: energies in fixed point, shares as integers.
// FP64: doubles, in which the shares' multiples add exactly as well (an atom's
// high words below 2^37 units, its low ones below 2^-5: residues of some
// thousand pairs), so that all words take one kind of addition.
template <class AH>
__device__ __forceinline__ void vol_add_word(vol_word *w, int k, double t, double kc) {
  if constexpr (std::is_same<AH, double>::value)
    atomicAdd(reinterpret_cast<double *>(w + k), t);
  else
    atomicAdd(w + k, k < 2 ? acc_val<AH>(t) : vol_int(t, kc));
}
// the sums of a cluster's slot over the 8 lanes that share it, added by lanes
// jj = 0..5.  Mixed energies are rounded to fixed point per lane, as every
// addition to a sum is.
template <class AH>
__device__ __forceinline__ void vol_add_i(vol_word *w, const double (&v)[kVolN], int jj) {
  AH s[kVolN];
#pragma unroll
  for (int k = 0; k < kVolN; k++) {
    if constexpr (std::is_same<AH, double>::value) s[k] = v[k];
    else s[k] = k < 2 ? acc_val<AH>(v[k]) : vol_int(v[k], k < 4 ? kVolHi : kVolLo);
#pragma unroll
    for (int o = 8; o < 64; o <<= 1) s[k] += __shfl_xor(s[k], o, 64);
  }
  const AH x = jj == 0   ? s[0]
               : jj == 1 ? s[1]
               : jj == 2 ? s[2]
               : jj == 3 ? s[3]
               : jj == 4 ? s[4]
                         : s[5];
  if (jj < kVolN && x != (AH)0) atomicAdd(reinterpret_cast<AH *>(w + jj), x);
}
// a slot's share words as integers
__device__ __forceinline__ vol_word vol_word_of(double w, double scale) {
  return (vol_word)__double2ll_rn(w * scale);
}
__device__ __forceinline__ vol_word vol_word_of(unsigned long long w, double) { return w; }

// v[0..5] summed over each aligned group of 8 lanes (k = lane & 7) in six
// exchanges, as hf_sum4x8: afterwards lanes 0, 1, 2 hold the sums 0, 1, 2 and
// lanes 4, 5, 6 the sums 3, 4, 5.  The group's whole wave must be active.
__device__ __forceinline__ double vol_sum6x8(const double (&v)[kVolN], int k) {
  const bool hi = (k & 4) != 0, b1 = (k & 2) != 0, odd = (k & 1) != 0;
  double a[3];
#pragma unroll
  for (int m = 0; m < 3; m++)
    a[m] = (hi ? v[3 + m] : v[m]) + dpp8d<0x141>(hi ? v[m] : v[3 + m]);
  const double b = (b1 ? a[2] : a[0]) + dpp8d<0x4E>(b1 ? a[0] : a[2]);
  const double c = a[1] + dpp8d<0x4E>(a[1]);
  return (odd ? c : b) + dpp8d<0xB1>(odd ? b : c);
}

// a pair weighed region by region: shares sc (class qc) and sv (class qc + 1)
// times the reference's weight (whole), or times the whole segment in the
// regions whose plane the first centre lies on with the second on its far side
__device__ __forceinline__ void vol_regions(const HfDev &h, bool whole, int qc, double ci,
                                            double cj, double sc, double sv) {
  const double dz = ci - cj, lo = fmin(ci, cj), hi = fmax(ci, cj);
  int r0, r1;
  hf_region_window(h, lo, hi, r0, r1);
  for (int r = r0; r <= r1; r++) {
    const double z1 = h.z1[r], z2 = h.z2[r];
    if (hi < z1 || lo > z2) continue;   // the segment misses the region
    const double ff = whole ? hf_volume_weight_z(z1, z2, ci, cj, dz, fabs(dz), 1.0)
                            : ((dz > 0.0 ? z1 == ci : z2 == ci) ? dz : 0.0);
    if (ff == 0.0) continue;
    if (sc != 0.0) vol_region_add(h, r, qc, ff * sc);
    if (sv != 0.0) vol_region_add(h, r, qc + 1, ff * sv);
  }
}

// per slot: position and charge, collision-part velocity and centre z,
// molecule and type with their flags; the slot's sums start at zero
__global__ __launch_bounds__(256) void k_hf_vol_pack(int nslot,
                                                     const int32_t *__restrict__ cl_atom,
                                                     HfDev h, const double *__restrict__ q,
                                                     const int32_t *__restrict__ ct,
                                                     double4 *__restrict__ xq,
                                                     double4 *__restrict__ vc,
                                                     int2 *__restrict__ mt,
                                                     vol_word *__restrict__ acc) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  // the block's slots hold kVolNW * 256 consecutive words
  const size_t w0 = (size_t)blockIdx.x * 256 * kVolNW, w1 = min(w0 + 256 * kVolNW,
                                                                (size_t)nslot * kVolNW);
  for (size_t k = w0 + threadIdx.x; k < w1; k += 256) acc[k] = 0;
  int ex = 0;   // biased exponent of the velocity's largest component
  if (s < nslot) {
    const int a = cl_atom[s];
    if (a < 0) {
      xq[s] = vc[s] = make_double4(0.0, 0.0, 0.0, 0.0);
      mt[s] = make_int2(0, 0);
    } else {
      xq[s] = make_double4(h.pos[3 * a], h.pos[3 * a + 1], h.pos[3 * a + 2], q[a]);
      double c[3];
      const int atomc = hf_centre(h, a, false, c);
      bool plane = false;
      int r0, r1;
      hf_region_window(h, c[2], c[2], r0, r1);
      for (int r = r0; r <= r1; r++) plane = plane || h.z1[r] == c[2] || h.z2[r] == c[2];
      const double v[3] = {h.vel[3 * a], h.vel[3 * a + 1], h.vel[3 * a + 2]};
      vc[s] = make_double4(v[0], v[1], v[2], c[2]);
      mt[s] = make_int2(h.molid[a] | (atomc ? 0 : kMolMole), ct[s] | (plane ? kTypPlane : 0));
#pragma unroll
      for (int d = 0; d < 3; d++)
        ex = max(ex, (int)((__double_as_longlong(v[d]) >> 52) & 2047));
    }
  }
  __shared__ int s_e[4], s_n[4];
  const bool in = ex > 0 && ex < 2047;
  int e = in ? ex : 0;
  for (int o = 32; o >= 1; o >>= 1) e += __shfl_xor(e, o, 64);
  if ((threadIdx.x & 63) == 0) s_e[threadIdx.x >> 6] = e;
  const int n = (int)__popcll(__ballot(in));
  if ((threadIdx.x & 63) == 0) s_n[threadIdx.x >> 6] = n;
  __syncthreads();
  if (threadIdx.x < 2) {
    const int *p = threadIdx.x ? s_n : s_e;
    atomicAdd(reinterpret_cast<vol_word *>(h.jpart + vol_jw(h.nreg, 0)) + threadIdx.x,
              (vol_word)(p[0] + p[1] + p[2] + p[3]));
  }
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
// atoms' sums stay in registers; a j atom's six sums over its 8 lanes leave
// as one atomic each to adjacent words of its slot.
template <class AH, bool CH, bool LJLDS>
__global__ __launch_bounds__(256) void k_hf_pairs_vol(HfVolArgs p, HfDev h,
                                                      vol_word *__restrict__ acc) {
  using R = typename std::conditional<std::is_same<AH, unsigned long long>::value, float,
                                      double>::type;
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
  double si[kVolN] = {}, sin[kVolN] = {};
  const double half_unit = 0.5 * vol_pow2(-vol_unit_exp(h.jpart, h.nreg));
  // the word of a j slot this lane adds to (lanes 3 and 7: none)
  const int jw = ii < 4 ? ii : ii - 1;
  const double jk = jw < 4 ? kVolHi : kVolLo;
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
  bool any_inner = false;
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
      double sj[kVolN] = {};   // of the j atom
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
          const double rw = half_unit * (r[0] * w[0] + r[1] * w[1] + r[2] * w[2]);
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
            if (ep != R(0)) {   // (0 x infinity at a contact of atoms without LJ is nothing)
              ev = ep * (t12 - (R)2 * t6);
              fv = (R)12 * ep * (t12 - t6) * rinv2;
            }
          }
          double sc = seg ? (double)fc * rw : 0.0, sv = seg ? (double)fv * rw : 0.0;
          const bool whole = h.reversed || !(fabs(sc) < kVolMax && fabs(sv) < kVolMax);
          if (__builtin_expect(whole || (plane && dz != 0.0), 0)) {
            vol_regions(h, whole, same ? 0 : 2, vi.w, d.vj.w, sc, sv);
            if (whole) sc = sv = 0.0;
          }
          double v[kVolN] = {0.5 * (double)ec, 0.5 * (double)ev};
          vol_split(sc, v[2], v[4]);
          vol_split(sv, v[3], v[5]);
#pragma unroll
          for (int k = 0; k < kVolN; k++) {
            if (same) sin[k] += v[k];
            else si[k] += v[k];
            sj[k] = k < 2 ? v[k] : -v[k];
          }
        }
      }
      const bool inner = __ballot(same) != 0;   // pairs inside one molecule are few
      auto add_j = [&](const double (&v)[kVolN], int at) {
        const double t = vol_sum6x8(v, ii);
        if (t != 0.0 && (ii & 3) != 3)
          vol_add_word<AH>(acc + (size_t)d.js * kVolNW + at, jw, t, jk);
      };
      if (!inner) {
        add_j(sj, 0);
      } else {
        any_inner = true;
        double so[kVolN];
#pragma unroll
        for (int k = 0; k < kVolN; k++) so[k] = same ? 0.0 : sj[k];
        add_j(so, 0);
#pragma unroll
        for (int k = 0; k < kVolN; k++) so[k] = same ? sj[k] : 0.0;
        add_j(so, kVolN);
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
  vol_add_i<AH>(acc + (size_t)islot * kVolNW, si, lane >> 3);
  if (any_inner) vol_add_i<AH>(acc + (size_t)islot * kVolNW + kVolN, sin, lane >> 3);
}

// What the regions take from one item (slot or atom).  Transport: the centre's
// z wrapped into [0, Lz), its velocity, kinetic energy and potential energies
// by class.  Collision: the centre's z and the shares ELIN, LJIN, ELC, VDW as
// their words.
struct VolTr {
  double z, vz, e[1 + PGK_NHF];
};
struct VolCol {
  double z;
  vol_word hi[4], lo[4];
};

template <class AH>
__device__ __forceinline__ bool vol_tr(const HfBinArgs &a, int k, VolTr &o) {
  const int i = a.order ? a.order[k] : k;
  if (i < 0) return false;
  const bool mole = a.hftyp[i] == PGK_HFTYP_MOLE;
  const int m = a.molid[i] - 1;
  double z = mole ? a.molecom[3 * (size_t)m + 2] : a.pos[3 * (size_t)i + 2];
  if (z < 0.0) z = z + a.Lz;
  else if (z >= a.Lz) z = z - a.Lz;
  o.z = z;
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
  const AH *w = reinterpret_cast<const AH *>(a.acc);
#pragma unroll
  for (int g = 0; g < 2; g++)   // g 0: inside one molecule (ELIN, LJIN), 1: ELC, VDW
#pragma unroll
    for (int q = 0; q < 2; q++)
      o.e[1 + PGK_HF_ELIN + 2 * g + q] =
          w ? acc_load(&w[(size_t)k * kVolNW + (g ? 0 : kVolN) + q]) : 0.0;
  return true;
}

template <class AH>
__device__ __forceinline__ bool vol_col(const HfBinArgs &a, int k, VolCol &o) {
  const int i = a.order ? a.order[k] : k;
  if (i < 0 || !a.acc) return false;
  const bool mole = a.hftyp[i] == PGK_HFTYP_MOLE;
  double z = mole ? a.molecom[3 * (size_t)(a.molid[i] - 1) + 2] : a.pos[3 * (size_t)i + 2];
  if (!mole) {
    if (z < 0.0) z = z + a.Lz;
    else if (z >= a.Lz) z = z - a.Lz;
  }
  o.z = z;
  const AH *w = reinterpret_cast<const AH *>(a.acc) + (size_t)k * kVolNW;
#pragma unroll
  for (int g = 0; g < 2; g++)
#pragma unroll
    for (int q = 0; q < 2; q++) {
      o.hi[2 * g + q] = vol_word_of(w[(g ? 0 : kVolN) + 2 + q], 0x1p16);
      o.lo[2 * g + q] = vol_word_of(w[(g ? 0 : kVolN) + 4 + q], 0x1p58);
    }
  return true;
}

// sums in two doubles (value h + l)
struct Dd {
  double h, l;
};
__device__ __forceinline__ Dd dd_diff(double a, double b) {   // a - b, exactly
  const double s = a - b, t = a - s;
  return {s, (a - (s + t)) + (t - b)};
}
__device__ __forceinline__ void dd_add(Dd &x, const Dd &y) {
  const double s = x.h + y.h, t = s - x.h;
  const double e = (x.h - (s - t)) + (y.h - t);
  x.h = s;
  x.l += y.l + e;
}
// a share (its two words) times a length
__device__ __forceinline__ Dd vol_times(vol_word hi, vol_word lo, const Dd &len) {
  const double s = vol_val_hi(hi), p = s * len.h;
  return {p, __builtin_fma(s, len.h, -p) + (s * len.l + vol_val_lo(lo) * len.h)};
}

// Record of a region and part of the items: 9 transport sums; 4 collision sums
// of the atoms inside, first then second double; the shares of the atoms above
// the region, 4 high and 4 low words.
constexpr int kVolRec = 25;

// Regions that tile their range (h.tiled): one wave per part of the items,
// every region's sums in LDS; blockIdx.y 0 the transport part, 1 the collision
// part.  An atom adds its transport values to the region (or, on a plane, the
// two) it lies in; the product of its shares S with c - z1 to the region it
// lies in, in multiples of 2^-10 (kLen: summed exactly below 2^43) and the
// rest; and S itself once, for the regions below, where the integers are
// summed from above at the end.
// 64-thread blocks: additions of one wave to one address happen in lane
// order, so the sums do not depend on timing.
template <class AH>
__global__ __launch_bounds__(64) void k_hf_vol_bins(HfBinArgs a, double *__restrict__ part) {
  extern __shared__ double sm[];   // [9][nreg], or [8][nreg] and words [8][nreg + 1]
  constexpr double kLen = 0x1.8p42;
  const int nreg = a.nreg, lane = threadIdx.x;
  const int i0 = blockIdx.x * a.per, i1 = min(a.nitem, i0 + a.per);
  auto region_of = [&](double z) {   // the last region with z1 <= z, -1: none
    int k = min(nreg - 1, max(-1, (int)floor((z - a.ubz0) * a.ubwi)));
    while (k + 1 < nreg && a.z1[k + 1] <= z) k++;
    while (k >= 0 && a.z1[k] > z) k--;
    return k;
  };
  auto rec = [&](int r) { return part + ((size_t)r * a.nsplit + blockIdx.x) * kVolRec; };
  if (blockIdx.y == 0) {
    for (int k = lane; k < 9 * nreg; k += 64) sm[k] = 0.0;
    __syncthreads();
    for (int k = i0 + lane; k < i1; k += 64) {
      VolTr it;
      if (!vol_tr<AH>(a, k, it)) continue;
      const int kt = region_of(it.z);
#pragma unroll
      for (int b = 0; b < 2; b++) {   // region kt, and kt - 1 where its upper plane is met
        const int r = kt - b;
        if (r < 0 || it.z > a.z2[r]) continue;
#pragma unroll
        for (int t = 0; t < 1 + PGK_NHF; t++)
          if (it.e[t] != 0.0) atomicAdd(&sm[t * nreg + r], it.e[t] * it.vz);
      }
    }
    __syncthreads();
    for (int k = lane; k < 9 * nreg; k += 64) {
      const int r = k / 9, t = k - 9 * r;
      rec(r)[t] = sm[t * nreg + r];
    }
    return;
  }
  const int ns = nreg + 1;   // shares by the first region above the atom's
  vol_word *sd = reinterpret_cast<vol_word *>(sm + 8 * nreg);
  for (int k = lane; k < 8 * nreg; k += 64) sm[k] = 0.0;
  for (int k = lane; k < 8 * ns; k += 64) sd[k] = 0;
  __syncthreads();
  for (int k = i0 + lane; k < i1; k += 64) {
    VolCol it;
    if (!vol_col<AH>(a, k, it)) continue;
    const int kc = region_of(it.z);
    if (kc < 0) continue;
    const bool past = it.z >= a.z2[kc];   // beyond the last region
    const Dd len = dd_diff(it.z, a.z1[kc]);
#pragma unroll
    for (int q = 0; q < 4; q++)
      if ((it.hi[q] | it.lo[q]) != 0) {
        atomicAdd(&sd[q * ns + kc + past], it.hi[q]);
        atomicAdd(&sd[(4 + q) * ns + kc + past], it.lo[q]);
        if (past) continue;
        const Dd x = vol_times(it.hi[q], it.lo[q], len);
        const double h = (x.h + kLen) - kLen;
        atomicAdd(&sm[q * nreg + kc], h);
        atomicAdd(&sm[(4 + q) * nreg + kc], (x.h - h) + x.l);
      }
  }
  __syncthreads();
  // shares of the atoms above region r: entries r + 1 .. nreg.  Each lane a
  // run of regions.
  const int run = (nreg + 63) / 64, r0 = min(nreg, lane * run), r1 = min(nreg, r0 + run);
#pragma unroll
  for (int q = 0; q < 8; q++) {
    vol_word own = 0;
    for (int r = r0; r < r1; r++) own += sd[q * ns + r + 1];
    vol_word above = own;   // inclusive sum of the lanes from here up
    for (int o = 1; o < 64; o <<= 1) {
      const vol_word t = __shfl_down(above, o, 64);
      if (lane + o < 64) above += t;
    }
    above -= own;
    for (int r = r1 - 1; r >= r0; r--) {
      above += sd[q * ns + r + 1];
      reinterpret_cast<vol_word *>(rec(r))[17 + q] = above;
    }
  }
  for (int k = lane; k < 8 * nreg; k += 64) {
    const int r = k >> 3, t = k & 7;
    rec(r)[9 + t] = sm[t * nreg + r];
  }
}

// any regions (one, or not tiling their range): block (part of the items,
// region, 0 the transport and 1 the collision part), the same record
template <class AH>
__global__ __launch_bounds__(256) void k_hf_vol_regions(HfBinArgs a, double *__restrict__ part) {
  const int r = blockIdx.y, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const double z1 = a.z1[r], z2 = a.z2[r];
  const int i0 = blockIdx.x * a.per, i1 = min(a.nitem, i0 + a.per);
  double *rec = part + ((size_t)r * a.nsplit + blockIdx.x) * kVolRec;
  if (blockIdx.z == 0) {
    double v[9];
#pragma unroll
    for (int t = 0; t < 9; t++) v[t] = 0.0;
    for (int k = i0 + (int)threadIdx.x; k < i1; k += 256) {
      VolTr it;
      if (!vol_tr<AH>(a, k, it)) continue;
      if (z1 <= it.z && it.z <= z2)
#pragma unroll
        for (int t = 0; t < 9; t++) v[t] += it.e[t] * it.vz;
    }
    block_record<9, 4>(v, rec);
    return;
  }
  Dd in[4];
  vol_word up[8];
#pragma unroll
  for (int q = 0; q < 4; q++) in[q].h = in[q].l = 0.0;
#pragma unroll
  for (int q = 0; q < 8; q++) up[q] = 0;
  for (int k = i0 + (int)threadIdx.x; k < i1; k += 256) {
    VolCol it;
    if (!vol_col<AH>(a, k, it) || !(it.z > z1)) continue;
    const bool past = it.z >= z2;
    const Dd len = dd_diff(it.z, z1);
#pragma unroll
    for (int q = 0; q < 4; q++) {
      if (past) {
        up[q] += it.hi[q];
        up[4 + q] += it.lo[q];
      } else {
        dd_add(in[q], vol_times(it.hi[q], it.lo[q], len));
      }
    }
  }
  __shared__ Dd s_in[4][4];
  __shared__ vol_word s_up[4][8];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
#pragma unroll
    for (int q = 0; q < 4; q++)
      dd_add(in[q], {__shfl_xor(in[q].h, o, 64), __shfl_xor(in[q].l, o, 64)});
#pragma unroll
    for (int q = 0; q < 8; q++) up[q] += __shfl_xor(up[q], o, 64);
  }
  if (lane == 0) {
#pragma unroll
    for (int q = 0; q < 4; q++) s_in[wave][q] = in[q];
#pragma unroll
    for (int q = 0; q < 8; q++) s_up[wave][q] = up[q];
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    Dd x = s_in[0][threadIdx.x];
    for (int w = 1; w < 4; w++) dd_add(x, s_in[w][threadIdx.x]);
    rec[9 + threadIdx.x] = x.h;
    rec[13 + threadIdx.x] = x.l;
  } else if (threadIdx.x < 12) {
    const int q = threadIdx.x - 4;
    reinterpret_cast<vol_word *>(rec)[17 + q] =
        s_up[0][q] + s_up[1][q] + s_up[2][q] + s_up[3][q];
  }
}

// the parts' records in a fixed order, the pairs weighed on their own (jpart),
// the bonded terms' sums (jcol), the volume factor and the total
// (calheatf.F90:1334-1436): one block per region
template <class AH>
__global__ __launch_bounds__(512) void k_hf_vol_final(HfBinArgs a, const double *__restrict__ part,
                                                      const AH *__restrict__ jcol,
                                                      const double *__restrict__ jpart,
                                                      double *__restrict__ out) {
#pragma clang fp contract(off)
  // 30 groups of 17 threads: 9 transport sums, 4 collision sums inside, 4
  // shares from above
  constexpr int G = 30;
  __shared__ Dd s[G][13];
  __shared__ vol_word s_up[G][8];
  __shared__ double fin[PGK_HFJ_TOT];
  const int r = blockIdx.x, g = threadIdx.x / 17, t = threadIdx.x - 17 * g;
  if (g < G) {
    const double *rec = part + (size_t)r * a.nsplit * kVolRec;
    if (t < 13) {
      Dd v = {0.0, 0.0};
      for (int k = g; k < a.nsplit; k += G) {
        const double *p = rec + (size_t)k * kVolRec;
        if (t < 9) v.h += p[t];
        else dd_add(v, {p[t], p[t + 4]});
      }
      s[g][t] = v;
    } else {
      vol_word hi = 0, lo = 0;
      for (int k = g; k < a.nsplit; k += G) {
        const vol_word *p = reinterpret_cast<const vol_word *>(rec + (size_t)k * kVolRec);
        hi += p[t + 4];
        lo += p[t + 8];
      }
      s_up[g][t - 13] = hi;
      s_up[g][t - 9] = lo;
    }
  }
  __syncthreads();
  const double vol_inv = ((1.0 / a.Lx) * (1.0 / a.Ly)) / (a.z2[r] - a.z1[r]);
  if (threadIdx.x < PGK_HFJ_TOT) {
    const int k = threadIdx.x;   // 0 kinetic, 1..8 potential, 9..16 collision classes
    const int q = k - 9 - PGK_HF_ELIN;
    double v = 0.0;
    if (k < 9) {
      for (int i = 0; i < G; i++) v += s[i][k].h;
    } else if (q >= 0) {
      Dd x = {0.0, 0.0};
      vol_word hi = 0, lo = 0;
      for (int i = 0; i < G; i++) {
        dd_add(x, s[i][9 + q]);
        hi += s_up[i][q];
        lo += s_up[i][4 + q];
      }
      dd_add(x, vol_times(hi, lo, dd_diff(a.z2[r], a.z1[r])));
      const double *w = jpart + vol_jw(r, q);
      const vol_word *wi = reinterpret_cast<const vol_word *>(w);
      dd_add(x, {vol_val_hi(wi[0]), vol_val_lo(wi[1])});
      v = ((x.h + x.l) + w[2]) * vol_pow2(vol_unit_exp(jpart, a.nreg));
    }
    if (k >= 9) v += acc_load(&jcol[3 * ((size_t)(k - 9) * a.nreg + r) + 2]);
    fin[k] = v * vol_inv;
  }
  __syncthreads();
  double *o = out + (size_t)r * PGK_NHFJ * 3;
  for (int k = threadIdx.x; k < PGK_HFJ_TOT * 3; k += 512) o[k] = k % 3 == 2 ? fin[k / 3] : 0.0;
  if (threadIdx.x < 3) {
    double tot = threadIdx.x == 2 ? fin[0] : 0.0;
    if (threadIdx.x == 2)
      for (int k = 1; k < PGK_HFJ_TOT; k++) tot = tot + fin[k];
    o[3 * PGK_HFJ_TOT + threadIdx.x] = tot;
  }
}

template <class AH>
int launch_pairs_vol(pgk_ctx *c) {
  hipStream_t st = c->stream;
  const HfDev &h = c->hfdev;
  const int nslot = c->ncl * PGK_CL;
  int rc;
  if ((rc = grow_dev((void **)&c->d_hfw_xq, &c->hfw_xq_bytes, sizeof(double4) * nslot)) ||
      (rc = grow_dev((void **)&c->d_hfw_v, &c->hfw_v_bytes, sizeof(double4) * nslot)) ||
      (rc = grow_dev((void **)&c->d_hfv_mt, &c->hfv_mt_bytes, sizeof(int2) * nslot)) ||
      (rc = grow_dev(&c->d_hfv_acc, &c->hfv_acc_bytes, sizeof(vol_word) * kVolNW * (size_t)nslot)))
    return rc;
  vol_word *acc = reinterpret_cast<vol_word *>(c->d_hfv_acc);
  k_hf_vol_pack<<<pgk_grid_blocks(nslot, 256), 256, 0, st>>>(
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
    const size_t lds = sizeof(double) * 8 * (2 * (size_t)a.nreg + 1);
    const int lr = pgk_lds_limit((const void *)k_hf_vol_bins<AH>, lds);
    if (lr) return lr;
    k_hf_vol_bins<AH><<<dim3(a.nsplit, 2), 64, lds, st>>>(a, part);
  } else {
    k_hf_vol_regions<AH><<<dim3(a.nsplit, a.nreg, 2), 256, 0, st>>>(a, part);
  }
  HIP_CHECK(hipGetLastError());
  k_hf_vol_final<AH><<<a.nreg, 512, 0, st>>>(
      a, part, reinterpret_cast<const AH *>(c->hfdev.jcol), c->hfdev.jpart, out);
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
  // tiled: parts of 256 items up to 512 (1024 waves with both halves; the LDS of
  // 300 regions holds four on a CU); otherwise about 2048 blocks of a half in
  // all, at least 256 items each
  int ns = (a.nitem + 255) / 256;
  ns = std::max(1, std::min(ns, a.tiled ? 512 : (2048 + a.nreg - 1) / a.nreg));
  a.nsplit = ns;
  a.per = (a.nitem + ns - 1) / ns;
  int rc;
  if ((rc = grow_dev((void **)&c->d_hj_part, &c->hj_part_cap,
                     sizeof(double) * kVolRec * (size_t)a.nreg * ns)))
    return rc;
  return c->precision == PGK_PREC_MIXED
             ? launch_bins<unsigned long long>(c, a, c->d_hj_part, out)
             : launch_bins<double>(c, a, c->d_hj_part, out);
}
