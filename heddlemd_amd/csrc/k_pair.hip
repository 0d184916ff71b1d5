// Fused Lennard-Jones + real-space Ewald pair forces over the row lists and
// the per-atom lists, and the bonded terms (gfx950, wave64).
//
// Reference: the JIT-composed packed pair kernel
// (src/forces/jit_composed.rs:1490-1838) with the LJ functor
// (src/forces/lj.rs:225-335) and the SPME real-space functor
// (src/forces/spme.rs:708-783).  Kept: per-pair arithmetic (f32, Hastings
// erfc A&S 7.1.26, optional cubic LJ switch), f32 partial sums folded into
// i64 fixed point at 2^48 with truncation, per-atom energy and virial split
// half/half.  Exclusions (|key_i - key_j| <= span) are applied when the
// lists are built.
//
// MI355X design: every pair is evaluated from both sides, which costs twice
// the useful pairs but leaves no j-side sums to rotate, reduce or add with
// atomics, and lets a list hold exactly the pairs within the search radius:
// (r_search / r_c)^3 x 2 slots per useful pair and the rows' padding, 3.4 on
// water at a 0.14 nm skin where packed 64 x 64 tiles evaluated 5.2.  The
// gather that such lists need runs out of LDS: the i-atoms of a 64-atom
// block share one neighbourhood (about 1,700 j-atoms of water at that skin,
// 27 KB), staged once per block; 16-bit list entries are LDS byte offsets.
#include "hd_device.h"
#include "hd_kernels.h"

#define PAIR_WAVES 4
#define PAIR_MAXT 4

struct PairParams {
  float c6[PAIR_MAXT * PAIR_MAXT];   // 4 eps sigma^6
  float c12[PAIR_MAXT * PAIR_MAXT];  // 4 eps sigma^12
  float ljcut2[PAIR_MAXT * PAIR_MAXT];
  float rsw2[PAIR_MAXT * PAIR_MAXT];
  float inv_delta[PAIR_MAXT * PAIR_MAXT];  // 1/(rc^2 - rs^2), 0 when no switch
  int ntypes;
  float kc, alpha, coul_rc2;  // coul_rc2 < 0 disables the Coulomb term
  int ortho;  // the box has no tilt
  float reach;  // of a list beyond its block's box, with what atoms move
  int active_type;  // the LJ-active type when there is only one
  // 1: one cutoff for every interacting type pair and Coulomb, no switch;
  // 2: LJ only (no Coulomb), one cutoff for every interacting type pair, no
  // switch; 0: neither (the general loop)
  int uniform;
  float uc_rc2;  // the shared cutoff^2 of modes 1 and 2
  float cg;  // -alpha^2 log2(e): exp(-(alpha r)^2) = exp2(cg r^2)
  float pa;  // 0.3275911 alpha, the Hastings t = 1 / (1 + pa r)
};

// The i-atom's row of the LJ type-pair table, held in VGPRs for the whole
// kernel.  NT = table width (1, 2 or 4).  Each value passes through an
// empty asm that pins it to a register: otherwise the compiler folds the
// per-pair select chain back into an indexed load from a private array,
// which lands in scratch memory inside the inner loop.
template <int NT>
struct LjRow {
  float c6[NT], c12[NT], f6[NT], f12[NT], cut2[NT], rsw2[NT], idl[NT];
};

// NT = 0: more than four types.  The type-pair table sits in LDS (copied
// in by every workgroup) and a lane keeps pointers to its i-type's row:
// a[t] = (12 c12, 6 c6, c12, c6), b[t] = (cut^2, r_switch^2, 1/(cut^2 -
// r_switch^2), 0) for j-type t.  One LDS read per pair replaces the
// register select chain.
#define PAIR_TAB_TYPES 32
template <>
struct LjRow<0> {
  const float4* a;
  const float4* b;
  bool valid;
};

template <int NT>
struct PairTab {
  float4 a[1], b[1];
};
template <>
struct PairTab<0> {
  float4 a[PAIR_TAB_TYPES * PAIR_TAB_TYPES], b[PAIR_TAB_TYPES * PAIR_TAB_TYPES];
};

template <int NT>
__device__ __forceinline__ float pick(const float (&v)[NT], unsigned t) {
  if (NT == 1) return v[0];
  if (NT == 2) return t ? v[1] : v[0];
  float r = v[0];
  r = (t == 1u) ? v[1] : r;
  r = (t == 2u) ? v[2] : r;
  r = (t == 3u) ? v[3] : r;
  return r;
}

// Per-pair LJ coefficients of the i-row against j-type t.
template <int NT>
__device__ __forceinline__ float lj_f12(const LjRow<NT>& R, unsigned t) {
  if constexpr (NT == 0) return R.a[t].x; else return pick<NT>(R.f12, t);
}
template <int NT>
__device__ __forceinline__ float lj_f6(const LjRow<NT>& R, unsigned t) {
  if constexpr (NT == 0) return R.a[t].y; else return pick<NT>(R.f6, t);
}
template <int NT>
__device__ __forceinline__ float lj_c12(const LjRow<NT>& R, unsigned t) {
  if constexpr (NT == 0) return R.a[t].z; else return pick<NT>(R.c12, t);
}
template <int NT>
__device__ __forceinline__ float lj_c6(const LjRow<NT>& R, unsigned t) {
  if constexpr (NT == 0) return R.a[t].w; else return pick<NT>(R.c6, t);
}
template <int NT>
__device__ __forceinline__ float lj_cut2(const LjRow<NT>& R, unsigned t) {
  if constexpr (NT == 0) return R.valid ? R.b[t].x : -1.0f; else return pick<NT>(R.cut2, t);
}
template <int NT>
__device__ __forceinline__ float lj_rsw2(const LjRow<NT>& R, unsigned t) {
  if constexpr (NT == 0) return R.b[t].y; else return pick<NT>(R.rsw2, t);
}
template <int NT>
__device__ __forceinline__ float lj_idl(const LjRow<NT>& R, unsigned t) {
  if constexpr (NT == 0) return R.b[t].z; else return pick<NT>(R.idl, t);
}

__device__ __forceinline__ void pin(float& x) { __asm__("" : "+v"(x)); }

// Copy the type-pair table (2 float4 per pair, nt <= PAIR_TAB_TYPES) into
// LDS; the caller synchronises before the first read.
__device__ __forceinline__ void load_tab(PairTab<0>& T, const float4* __restrict__ lj_tab,
                                         int nt) {
  for (unsigned k = threadIdx.x; k < (unsigned)(nt * nt); k += blockDim.x) {
    T.a[k] = lj_tab[2 * k];
    T.b[k] = lj_tab[2 * k + 1];
  }
}

template <int NT>
__device__ __forceinline__ LjRow<NT> load_row(const PairParams& P, unsigned itype, bool ivalid,
                                              const PairTab<NT>& T) {
  LjRow<NT> r;
  if constexpr (NT == 0) {
    r.a = &T.a[itype * (unsigned)P.ntypes];
    r.b = &T.b[itype * (unsigned)P.ntypes];
    r.valid = ivalid;
    return r;
  } else {
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    int k = (t < P.ntypes) ? (int)itype * P.ntypes + t : 0;
    r.c6[t] = P.c6[k];
    r.c12[t] = P.c12[k];
    r.f6[t] = 6.0f * P.c6[k];
    r.f12[t] = 12.0f * P.c12[k];
    r.cut2[t] = ivalid ? P.ljcut2[k] : -1.0f;
    r.rsw2[t] = P.rsw2[k];
    r.idl[t] = P.inv_delta[k];
    pin(r.c6[t]); pin(r.c12[t]); pin(r.f6[t]); pin(r.f12[t]);
    pin(r.cut2[t]); pin(r.rsw2[t]); pin(r.idl[t]);
  }
  return r;
  }
}

// One axis of a minimum-image pair displacement in an orthorhombic box.
// Within the box the f32 difference of the two coordinates is exact or
// rounds at the pair's own scale; across a face it would round at the
// box's scale (an error of up to half an ulp of L, ~1e-6 of a contact
// distance, which the r^-13 of the LJ repulsion multiplies), so such pairs
// take the difference in FP64 and round once.
__device__ __forceinline__ float pair_axis_disp(float a, float b, float len, float ilen) {
  float d = a - b;
  float k = rintf(d * ilen);
  if (k != 0.f) d = (float)(((double)a - (double)b) - (double)len * (double)k);
  return d;
}

// The same for a tilted cell: the image triple from the f32 fractional
// rounding of hd_min_image_rcp, and, when it is not (0, 0, 0), the
// difference and the lattice shift formed in FP64 and rounded once.
__device__ __forceinline__ void pair_tri_disp(float pix, float piy, float piz, float pjx,
                                              float pjy, float pjz, const HdLattice& L,
                                              float ilx, float ily, float ilz, float& dx,
                                              float& dy, float& dz) {
  dx = pix - pjx;
  dy = piy - pjy;
  dz = piz - pjz;
  float sc = dz * ilz;
  float sb = (dy - sc * L.yz) * ily;
  float sa = (dx - sb * L.xy - sc * L.xz) * ilx;
  float ka = floorf(sa + 0.5f), kb = floorf(sb + 0.5f), kc = floorf(sc + 0.5f);
  if (ka == 0.f && kb == 0.f && kc == 0.f) return;
  double a = ka, b = kb, c = kc;
  dx = (float)(((double)pix - (double)pjx) - (a * L.lx + b * L.xy + c * L.xz));
  dy = (float)(((double)piy - (double)pjy) - (b * L.ly + c * L.yz));
  dz = (float)(((double)piz - (double)pjz) - c * L.lz);
}

// ---- row lists -----------------------------------------------------------

// What one lane needs of its i-atom and of the pair terms.
struct RowI {
  int x, y, z;                // offset from the block centre in 1 / scale
  float kq, inv2;             // k_C q_i; 1 / scale^2
  float f12, f6, c12, c6;     // KIND 0: coefficients against the one active type
  const float4 *ta, *tb;      // KIND 1, 2: the i-type's table rows (LDS)
  const unsigned char* jt;    // KIND 1, 2: j types (LDS)
  float rc2, cg, pa, k2;      // KIND 0, 1: shared cutoff^2, see PairParams
  float alpha, coul_rc2;      // KIND 2
};

struct RowSum {
  float fx, fy, fz, e, w;
};

// One pair of a row.  KIND 0: one cutoff for LJ and Coulomb, no switch, one
// LJ-active type; 1: the same with several active types (table row of the
// i-type, one LDS read per pair); 2: per-type cutoffs and the cubic switch.
// LJ = false: the j-atom's type has no LJ interaction.  Terms of KIND 0 and
// 1 are regrouped for fewer instructions: exp(-(alpha r)^2) as exp2(cg r^2);
// the Ewald force factor erfc(alpha r)/r^3 + 2 alpha/sqrt(pi)
// exp(-(alpha r)^2)/r^2 as gauss * (poly(t) t / r + 2 alpha/sqrt(pi)) / r^2;
// one 1/r^2 and one cutoff select for the sum.  The force arithmetic is the
// same for every EV, so energy steps move atoms as force-only steps do.
template <int EV, int KIND, bool COUL, bool LJ>
__device__ __forceinline__ void row_pair(const RowI& I, const int4* __restrict__ jrec,
                                         unsigned off, RowSum& S) {
  const int4 jr = *reinterpret_cast<const int4*>(reinterpret_cast<const char*>(jrec) + off);
  const float jq = __int_as_float(jr.w);
  float4 ta = make_float4(0.f, 0.f, 0.f, 0.f), tb = ta;
  if (KIND != 0 && LJ) {
    unsigned jt = I.jt[off >> 4];
    ta = I.ta[jt];
    if (KIND == 2) tb = I.tb[jt];
  }
  const float dx = (float)(I.x - jr.x), dy = (float)(I.y - jr.y), dz = (float)(I.z - jr.z);
  const float r2 = (dx * dx + dy * dy + dz * dz) * I.inv2;
  float factor, energy = 0.f;
  if (KIND < 2) {
    const float f12 = KIND == 0 ? I.f12 : ta.x, f6 = KIND == 0 ? I.f6 : ta.y;
    // LJ only: 1/r^2 from one reciprocal (half the rounding of squaring a
    // reciprocal square root, and one instruction fewer)
    const float inv_r = COUL ? __builtin_amdgcn_rsqf(r2) : 0.f;
    const float inv_r2 = COUL ? inv_r * inv_r : __builtin_amdgcn_rcpf(r2);
    float lj = 0.f, ir6 = 0.f;
    if (LJ) {
      ir6 = inv_r2 * inv_r2 * inv_r2;
      lj = ir6 * (f12 * ir6 - f6);
    }
    if (COUL) {
      const float r = r2 * inv_r;
      const float gauss = __builtin_amdgcn_exp2f(I.cg * r2);
      const float tt = __builtin_amdgcn_rcpf(fmaf(I.pa, r, 1.0f));
      const float poly =
          (0.254829592f +
           (-0.284496736f + (1.421413741f + (-1.453152027f + 1.061405429f * tt) * tt) * tt) * tt) *
          tt;
      const float ci = gauss * fmaf(poly, inv_r, I.k2);
      const float qq = I.kq * jq;
      factor = LJ ? inv_r2 * fmaf(qq, ci, lj) : inv_r2 * (qq * ci);
      if (EV == 1) energy = qq * gauss * (poly * inv_r);
    } else {
      factor = inv_r2 * lj;
    }
    if (EV == 1 && LJ) {
      const float c12 = KIND == 0 ? I.c12 : ta.z, c6 = KIND == 0 ? I.c6 : ta.w;
      energy += ir6 * (c12 * ir6 - c6);
    }
    const bool on = r2 <= I.rc2;
    factor = on ? factor : 0.f;
    if (EV == 1) energy = on ? energy : 0.f;
  } else {
    const float inv_r = __builtin_amdgcn_rsqf(r2);
    const float inv_r2 = inv_r * inv_r;
    factor = 0.f;
    if (LJ) {
      // LJ (lj.rs:237-247) and the cubic switch (lj.rs:250-287); without a
      // switch tb.z = 0, tau = 0 and the factors below are exactly 1 and 0
      const float ir6 = inv_r2 * inv_r2 * inv_r2;
      float flj = inv_r2 * ir6 * (ta.x * ir6 - ta.y);
      float elj = ir6 * (ta.z * ir6 - ta.w);
      const float tau = fmaxf((r2 - tb.y) * tb.z, 0.0f), omt = 1.0f - tau;
      const float s = omt * omt * (1.0f + 2.0f * tau), chain = 12.0f * tau * omt * tb.z;
      flj = s * flj + chain * elj;
      elj = s * elj;
      const bool on = r2 <= tb.x;
      factor = on ? flj : 0.f;
      if (EV == 1) energy = on ? elj : 0.f;
    }
    if (COUL) {
      // real-space Coulomb, f32 Hastings erfc (spme.rs:744-770)
      const float r = r2 * inv_r, qq = I.kq * jq, ar = I.alpha * r;
      const float gauss = __expf(-(ar * ar));
      const float tt = __builtin_amdgcn_rcpf(1.0f + 0.3275911f * ar);
      const float erfc_ar =
          (0.254829592f +
           (-0.284496736f + (1.421413741f + (-1.453152027f + 1.061405429f * tt) * tt) * tt) * tt) *
          tt * gauss;
      const bool on = r2 <= I.coul_rc2;
      const float fc = qq * inv_r2 * (erfc_ar * inv_r + I.k2 * gauss);
      factor += on ? fc : 0.f;
      if (EV == 1) energy += on ? qq * erfc_ar * inv_r : 0.f;
    }
  }
  S.fx = fmaf(factor, dx, S.fx);
  S.fy = fmaf(factor, dy, S.fy);
  S.fz = fmaf(factor, dz, S.fz);
  if (EV == 1) S.e += energy;
  if (EV) S.w = fmaf(factor, r2, S.w);
}

// A lane's sums in fixed point at 2^48.
struct RowTotal {
  long long fx, fy, fz, e, w;
};

// Adds a lane's f32 sums to its totals and clears them.  The force factors
// multiplied displacements in 1 / scale = inv; each side of a pair carries
// half of its energy and virial.
template <int EV>
__device__ __forceinline__ void row_fold(RowSum& S, RowTotal& T, float inv) {
  T.fx += hd_to_fixed48(inv * S.fx);
  T.fy += hd_to_fixed48(inv * S.fy);
  T.fz += hd_to_fixed48(inv * S.fz);
  if (EV == 1) T.e += hd_to_fixed48(0.5f * S.e);
  if (EV) T.w += hd_to_fixed48(0.5f * S.w);
  S = RowSum{0.f, 0.f, 0.f, 0.f, 0.f};
}

// Chunks [k0, k1) of the wave's rows, the next chunk's load in flight while
// one is evaluated.  An f32 sum runs over at most 64 entries (16 chunks) of
// a lane, as in the atom lists, so that its rounding does not grow with the
// length of the rows (a lane's whole share of a 2,400-entry row lost 2.6e-6
// of its largest term where this loses 1.2e-6).  The folds cost 1 % of a
// step: 10,000 argon atoms 1,505 to 1,527 us per 50 steps.
template <int EV, int KIND, bool COUL, bool LJ>
__device__ __forceinline__ void row_chunks(const RowI& I, const int4* __restrict__ jrec,
                                           const uint2* __restrict__ rp, unsigned k0,
                                           unsigned k1, float inv, RowTotal& T) {
  if (k0 >= k1) return;
  RowSum S = {0.f, 0.f, 0.f, 0.f, 0.f};
  uint2 nx = rp[k0 * (HD_ROW_CHUNK / 4u)];
  for (unsigned k = k0; k < k1; ++k) {
    const uint2 c = nx;
    if (k + 1 < k1) nx = rp[(k + 1) * (HD_ROW_CHUNK / 4u)];
    row_pair<EV, KIND, COUL, LJ>(I, jrec, c.x & 0xFFFFu, S);
    row_pair<EV, KIND, COUL, LJ>(I, jrec, c.x >> 16, S);
    row_pair<EV, KIND, COUL, LJ>(I, jrec, c.y & 0xFFFFu, S);
    row_pair<EV, KIND, COUL, LJ>(I, jrec, c.y >> 16, S);
    if (((k - k0) & 15u) == 15u) row_fold<EV>(S, T, inv);
  }
  row_fold<EV>(S, T, inv);
}

// sum over the 8 lanes that share an i-atom (lane bits 0..2), in every lane
template <int CTRL>
__device__ __forceinline__ long long row_dpp(long long v) {
  const int lo = __builtin_amdgcn_mov_dpp((int)(unsigned)v, CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(v >> 32), CTRL, 0xF, 0xF, true);
  return (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ long long row_sum8(long long v) {
  v += row_dpp<0xB1>(v);
  v += row_dpp<0x4E>(v);
  v += row_dpp<0x141>(v);
  return v;
}

// One workgroup of 8 waves per unit of the row lists (k_build_rows): the
// unit's j-atoms are staged once in LDS, relative to the block centre in
// their own image; wave w holds i-atoms 8 w .. 8 w + 7, eight lanes each,
// lane 8 r + s taking entries s of row r.  Both sides of every pair are
// evaluated, so nothing is added to the j-atoms: the lanes' f32 sums (64
// entries at most) go to fixed point at 2^48, are added over the 8 lanes and
// once per i-atom to its accumulator (one coalesced 64-bit atomic
// instruction per wave).
//
// Positions are whole numbers of a power-of-two step relative to the block
// centre (hd_rel_fixed): f32 offsets rounded the displacement of a pair at
// the block's size, and the error of a force (rms, 64-bit reference) was
// 8.2e-7 of the rms force in a tilted cell where it is now 5.7e-7.
//
// Bound by the vector ALU (about 34 instructions a slot of an LJ-active
// j-atom, 27 of another, plus one LDS read): listing the active j-atoms
// first lets a wave drop the LJ half for whole chunks.  The rows and j-atoms
// are not far behind: 396 MB a launch at 196,608 atoms of water, 84 us of
// its 118 alone at a large copy's 4.72 TB/s.  54 VGPRs, so the LDS of the
// j-list sets the occupancy.  Measured, us per launch (the packed tiles it
// replaced): 196,608 atoms of water 129 beside the SPME pipeline (209);
// 24,576 atoms 29 (76); 7,938 atoms 13.5 (69); 267 atoms 5.1 (16).
template <int EV, int KIND, bool COUL>
__global__ void __launch_bounds__(HD_ROW_THREADS) k_pair_rows(
    PairParams P, const float* __restrict__ lattice, const float4* __restrict__ tile_posq,
    const unsigned* __restrict__ tile_type, const unsigned char* __restrict__ tile_img,
    const float4* __restrict__ center, const float4* __restrict__ half,
    const unsigned* __restrict__ jslot, const unsigned* __restrict__ jcount,
    const unsigned* __restrict__ rowhdr,
    const unsigned short* __restrict__ rows, const unsigned* __restrict__ order, unsigned parts,
    unsigned jcap, unsigned rcap, unsigned n, unsigned long long* __restrict__ fpj,
    unsigned long long* __restrict__ fpj_ew, const float4* __restrict__ lj_tab, unsigned* status,
    unsigned* rebuild_count) {
  // End of a rebuild with few units: the request is cleared and counted here
  // (nothing that runs beside this launch reads it).  A launch of its own cost
  // 2.5 us of every step (10,000 argon atoms); a ticket in the build, whose
  // units then wait for the returned count, 30 us of every rebuild.
  if (status && blockIdx.x == 0 && threadIdx.x == 0) {
    const unsigned s = *(volatile unsigned*)status;
    if (s & (NB_STATUS_REBUILD | NB_STATUS_FORCE)) {
      atomicAnd(status, ~(NB_STATUS_REBUILD | NB_STATUS_FORCE));
      *rebuild_count += 1u;
    }
  }
  extern __shared__ float4 lds[];
  int4* jrec = reinterpret_cast<int4*>(lds);
  const unsigned nt2 = (unsigned)(P.ntypes * P.ntypes);
  float4* tab_a = lds + jcap + 1;
  float4* tab_b = tab_a + (KIND != 0 ? nt2 : 0u);
  unsigned char* jt = reinterpret_cast<unsigned char*>(tab_b + (KIND == 2 ? nt2 : 0u));
  const unsigned t = threadIdx.x, lane = t & 63u, w = t >> 6;
  const unsigned unit = order[blockIdx.x];  // heaviest first
  const unsigned b = unit / parts;
  const HdLattice L = hd_load_lattice(lattice);
  const float4 cb = center[b];
  // scale: offsets reach the block's half extent, the search radius and what
  // atoms moved since; 2^23 or 2^24 for a dense block (2^-24 Bohr is 1/8 of
  // the rounding of a 4 Bohr displacement)
  const float4 hb = half[b];
  const int se = 28 - ilogbf(fmaxf(hb.x, fmaxf(hb.y, hb.z)) + P.reach);
  const double scale = ldexp(1.0, se);
  const float inv = ldexpf(1.0f, -se);
  const unsigned jc = jcount[unit], nja = jc & 0xFFFFu;
  const unsigned hdr = rowhdr[unit * HD_ROW_WAVES + w];
  const unsigned islot = b * 64u + w * HD_ROW_I + (lane >> 3);
  const bool ivalid = islot < n;
  const float4 pi = tile_posq[islot];  // npad entries
  const unsigned itype = ivalid ? tile_type[islot] : 0u;
  // without Coulomb the j-atoms of inactive types are not read
  const unsigned nj = nja + (COUL ? jc >> 16 : 0u);
  for (unsigned q = t; q < nj; q += HD_ROW_THREADS) {
    const unsigned k = q < nja ? q : jcap - 1u - (q - nja);
    const unsigned js = jslot[(size_t)unit * jcap + k];
    const unsigned s = js & (HD_ROW_SLOTS - 1u), code = js >> HD_ROW_SLOT_BITS;
    const float4 p = tile_posq[s];
    const int3 f = hd_rel_fixed(p.x, p.y, p.z, cb, code, tile_img[s], L, scale);
    jrec[k] = make_int4(f.x, f.y, f.z, __float_as_int(p.w));
    if (KIND != 0) jt[k] = (unsigned char)tile_type[s];
  }
  if (t == 0) {
    jrec[jcap] = make_int4(HD_FIXED_FAR, 0, 0, 0);
    if (KIND != 0) jt[jcap] = 0;
  }
  if (KIND != 0)
    for (unsigned k = t; k < nt2; k += HD_ROW_THREADS) {
      tab_a[k] = lj_tab[2 * k];
      if (KIND == 2) tab_b[k] = lj_tab[2 * k + 1];
    }
  RowI I;
  const int3 fi = hd_rel_fixed(pi.x, pi.y, pi.z, cb, HD_IMAGE_NONE, tile_img[islot], L, scale);
  // a slot without atom, or an atom out of reach, on the other side of the
  // far j-atoms
  I.x = !ivalid || fi.x == HD_FIXED_FAR ? -HD_FIXED_FAR : fi.x;
  I.y = fi.y;
  I.z = fi.z;
  I.inv2 = inv * inv;
  I.kq = P.kc * pi.w;
  if (KIND == 0) {
    const float4 c = lj_tab[2 * (itype * (unsigned)P.ntypes + (unsigned)P.active_type)];
    I.f12 = c.x;
    I.f6 = c.y;
    I.c12 = c.z;
    I.c6 = c.w;
  } else {
    I.ta = tab_a + itype * (unsigned)P.ntypes;
    I.tb = tab_b + itype * (unsigned)P.ntypes;
    I.jt = jt;
  }
  I.rc2 = P.uc_rc2;
  I.cg = P.cg;
  I.pa = P.pa;
  I.k2 = 2.0f * P.alpha * 0.5641895835477563f;
  I.alpha = P.alpha;
  I.coul_rc2 = P.coul_rc2;
  __syncthreads();
  const uint2* rp = reinterpret_cast<const uint2*>(
                        rows + ((size_t)unit * 64u + w * HD_ROW_I + (lane >> 3)) *
                                   rcap) +
                    (lane & 7u);
  RowTotal T = {0, 0, 0, 0, 0};
  const unsigned hu = (unsigned)__builtin_amdgcn_readfirstlane((int)hdr);
  row_chunks<EV, KIND, COUL, true>(I, jrec, rp, 0u, hu & 0xFFFFu, inv, T);
  // without Coulomb the j-atoms of inactive types contribute nothing
  if (COUL) row_chunks<EV, KIND, COUL, false>(I, jrec, rp, hu & 0xFFFFu, hu >> 16, inv, T);
  const long long fx = row_sum8(T.fx), fy = row_sum8(T.fy), fz = row_sum8(T.fz);
  long long v = (lane & 7u) == 0u ? fx : ((lane & 7u) == 1u ? fy : fz);
  unsigned long long* dst = fpj + (size_t)islot * 4 + (lane & 7u);
  bool mine = ivalid && (lane & 7u) < 3u;
  if (EV) {
    const long long e = row_sum8(T.e), wv = row_sum8(T.w);
    if ((lane & 7u) >= 3u) {
      v = (lane & 7u) == 3u ? e : wv;
      dst = fpj_ew + (size_t)islot * 2 + ((lane & 7u) - 3u);
    }
    mine = ivalid && (lane & 7u) < 5u && (EV == 1 || (lane & 7u) != 3u);
  }
  if (mine && v) atomicAdd(dst, (unsigned long long)v);
}

// Atom-list mode: one workgroup of 4 waves per 64-atom i-block, lane =
// i-atom; wave w walks rows w, w + 4, ... of the block's list region (row
// k = the k-th neighbour of every lane: coalesced index loads, gathered j
// positions).  Each wave issues the loads of ALIST_U rows before it
// evaluates them, so ALIST_U gathers per lane are in flight at once.
// Every pair is evaluated from both sides, so there is no j-side partial
// and no atomic: the i-side f32 sums are folded into i64 fixed point at
// 2^48 every 64 neighbours (the reference's per-entry fold), combined over
// the 4 waves in LDS (integer sums, so the order does not matter) and
// stored once.  Each side of a pair carries half of its energy and virial.
// Exclusions were applied when the lists were built.  The displacement takes
// a per-pair minimum image (ORTHO: one rint per axis).
#define ALIST_U 4

template <int EV, int NT, bool SW, bool ORTHO>
__device__ __forceinline__ void alist_pair(const PairParams& P, const HdLattice& L, float ilx,
                                           float ily, float ilz, const LjRow<NT>& R, float4 pi,
                                           float kqi, float4 pj, unsigned jtype, float& efx,
                                           float& efy, float& efz, float& ee, float& ew) {
  const float two_a_sqrtpi = 2.0f * P.alpha * 0.5641895835477563f;
  float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
  if (ORTHO) {
    dx = pair_axis_disp(pi.x, pj.x, L.lx, ilx);
    dy = pair_axis_disp(pi.y, pj.y, L.ly, ily);
    dz = pair_axis_disp(pi.z, pj.z, L.lz, ilz);
  } else {
    pair_tri_disp(pi.x, pi.y, pi.z, pj.x, pj.y, pj.z, L, ilx, ily, ilz, dx, dy, dz);
  }
  float r2 = dx * dx + dy * dy + dz * dz;
  float inv_r = __builtin_amdgcn_rsqf(r2);
  float inv_r2 = inv_r * inv_r;
  float ir6 = inv_r2 * inv_r2 * inv_r2;
  float flj = inv_r2 * ir6 * (lj_f12(R, jtype) * ir6 - lj_f6(R, jtype));
  float elj = 0.f;
  if (EV == 1 || SW) elj = ir6 * (lj_c12(R, jtype) * ir6 - lj_c6(R, jtype));
  if (SW) {
    float rs2 = lj_rsw2(R, jtype), idl = lj_idl(R, jtype);
    float tau = fmaxf((r2 - rs2) * idl, 0.0f);
    float omt = 1.0f - tau;
    float sw = omt * omt * (1.0f + 2.0f * tau);
    float chain = 12.0f * tau * omt * idl;
    flj = sw * flj + chain * elj;
    elj = sw * elj;
  }
  bool lj_on = r2 <= lj_cut2(R, jtype);
  float r = r2 * inv_r;
  float qq = kqi * pj.w;
  float ar = P.alpha * r;
  float gauss = __expf(-(ar * ar));
  float tt = __builtin_amdgcn_rcpf(1.0f + 0.3275911f * ar);
  float erfc_ar =
      (0.254829592f +
       (-0.284496736f + (1.421413741f + (-1.453152027f + 1.061405429f * tt) * tt) * tt) * tt) *
      tt * gauss;
  float ec = qq * erfc_ar * inv_r;
  float fc = qq * inv_r2 * (erfc_ar * inv_r + two_a_sqrtpi * gauss);
  bool c_on = r2 <= P.coul_rc2;
  float factor = lj_on ? flj : 0.f;
  factor += c_on ? fc : 0.f;
  efx += factor * dx;
  efy += factor * dy;
  efz += factor * dz;
  if (EV == 1) {
    float energy = lj_on ? elj : 0.f;
    energy += c_on ? ec : 0.f;
    ee += 0.5f * energy;
  }
  if (EV) ew += 0.5f * factor * r2;
}

template <int EV, int NT, bool SW, bool ORTHO>
__global__ void __launch_bounds__(256) k_pair_alist(
    PairParams P, const float* __restrict__ lattice, const float4* __restrict__ tile_posq,
    const unsigned* __restrict__ tile_type, const unsigned* __restrict__ rows_in,
    const unsigned* __restrict__ row_count, unsigned cap, unsigned n, unsigned nblocks,
    long long* __restrict__ fpi, long long* __restrict__ fpi_ew,
    const float4* __restrict__ lj_tab) {
  __shared__ long long red[PAIR_WAVES][5][64];
  __shared__ PairTab<NT> tab;
  if constexpr (NT == 0) {
    load_tab(tab, lj_tab, P.ntypes);
    __syncthreads();
  }
  unsigned w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  unsigned b = blockIdx.x;
  HdLattice L = hd_load_lattice(lattice);
  const float ilx = 1.0f / L.lx, ily = 1.0f / L.ly, ilz = 1.0f / L.lz;
  unsigned islot = b * 64 + lane;
  bool ivalid = islot < n;
  float4 pi = tile_posq[ivalid ? islot : 0u];
  unsigned itype = ivalid ? tile_type[islot] : 0u;
  LjRow<NT> R = load_row<NT>(P, itype, ivalid, tab);
  const float kqi = P.kc * (ivalid ? pi.w : 0.f);
  const unsigned rows = row_count[b];
  const unsigned* list = rows_in + (size_t)b * cap * 64 + lane;
  long long ax = 0, ay = 0, az = 0, ae = 0, aw = 0;
  float efx = 0.f, efy = 0.f, efz = 0.f, ee = 0.f, ew = 0.f;
  unsigned since_fold = 0;
  for (unsigned k = w; k < rows; k += PAIR_WAVES * ALIST_U) {
    unsigned js[ALIST_U];
#pragma unroll
    for (int u = 0; u < ALIST_U; ++u) {
      unsigned kk = k + u * PAIR_WAVES;
      js[u] = kk < rows ? list[(size_t)kk * 64] : HD_SENTINEL;
    }
    float4 pj[ALIST_U];
    unsigned tj[ALIST_U];
#pragma unroll
    for (int u = 0; u < ALIST_U; ++u) {
      unsigned jsafe = js[u] < n ? js[u] : 0u;
      pj[u] = tile_posq[jsafe];
      tj[u] = (NT != 1) ? tile_type[jsafe] : 0u;
    }
#pragma unroll
    for (int u = 0; u < ALIST_U; ++u)
      if (js[u] < n)
        alist_pair<EV, NT, SW, ORTHO>(P, L, ilx, ily, ilz, R, pi, kqi, pj[u], tj[u], efx, efy,
                                      efz, ee, ew);
    since_fold += ALIST_U;
    if (since_fold >= 64) {
      ax += hd_to_fixed48(efx);
      ay += hd_to_fixed48(efy);
      az += hd_to_fixed48(efz);
      if (EV) {
        ae += hd_to_fixed48(ee);
        aw += hd_to_fixed48(ew);
      }
      efx = efy = efz = ee = ew = 0.f;
      since_fold = 0;
    }
  }
  ax += hd_to_fixed48(efx);
  ay += hd_to_fixed48(efy);
  az += hd_to_fixed48(efz);
  if (EV) {
    ae += hd_to_fixed48(ee);
    aw += hd_to_fixed48(ew);
  }
  red[w][0][lane] = ax;
  red[w][1][lane] = ay;
  red[w][2][lane] = az;
  if (EV) {
    red[w][3][lane] = ae;
    red[w][4][lane] = aw;
  }
  __syncthreads();
  if (w == 0 && ivalid) {
    long long sm[5] = {0, 0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < PAIR_WAVES; ++q) {
      sm[0] += red[q][0][lane];
      sm[1] += red[q][1][lane];
      sm[2] += red[q][2][lane];
      if (EV) {
        sm[3] += red[q][3][lane];
        sm[4] += red[q][4][lane];
      }
    }
    reinterpret_cast<longlong2*>(fpi)[2 * islot] = make_longlong2(sm[0], sm[1]);
    reinterpret_cast<longlong2*>(fpi)[2 * islot + 1] = make_longlong2(sm[2], 0);
    if (EV) reinterpret_cast<longlong2*>(fpi_ew)[islot] = make_longlong2(sm[3], sm[4]);
  }
}

// Harmonic angles (src/forces/angle.rs:258-313 functor, composed kernel
// src/forces/jit_composed.rs:2300-2345): one thread per angle i-j-k with
// minimum-image bond vectors, theta = atan2(|r_ij||r_kj| sin, dot),
// F_i, F_k from g = -k (theta - theta_0) / sin theta, F_j = -(F_i + F_k),
// energy and virial split in thirds.  The three forces are folded into the
// j-side fixed-point accumulators at 2^48 (integer sums, so the total is
// independent of the order in which angles land).
__global__ void k_angles(const float4* __restrict__ posq, const float* __restrict__ lattice,
                         const unsigned* __restrict__ ijk, const double* __restrict__ kth,
                         const double* __restrict__ th0, const unsigned* __restrict__ slot_of,
                         unsigned long long* __restrict__ fpj,
                         unsigned long long* __restrict__ fpj_ew, unsigned n_angles, int ev) {
  unsigned m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= n_angles) return;
  HdLattice L = hd_load_lattice(lattice);
  unsigned ai = ijk[3 * m], aj = ijk[3 * m + 1], ak = ijk[3 * m + 2];
  float4 pi = posq[ai], pj = posq[aj], pk = posq[ak];
  // FP64 throughout: the force is proportional to theta - theta0, a small
  // difference of two angles near 2 rad that f32 would resolve only to
  // ~1e-7 rad, i.e. to a relative 1e-4 of the force for a 1e-3 rad strain
  double ui[3] = {(double)pi.x - (double)pj.x, (double)pi.y - (double)pj.y,
                  (double)pi.z - (double)pj.z};
  double uk[3] = {(double)pk.x - (double)pj.x, (double)pk.y - (double)pj.y,
                  (double)pk.z - (double)pj.z};
  hd_min_image_f64(ui[0], ui[1], ui[2], L);
  hd_min_image_f64(uk[0], uk[1], uk[2], L);
  double li2 = ui[0] * ui[0] + ui[1] * ui[1] + ui[2] * ui[2];
  double lk2 = uk[0] * uk[0] + uk[1] * uk[1] + uk[2] * uk[2];
  double gi[3] = {0.0, 0.0, 0.0}, gk[3] = {0.0, 0.0, 0.0}, u = 0.0, w = 0.0;
  if (li2 > 0.0 && lk2 > 0.0) {
    double li = sqrt(li2), lk = sqrt(lk2);
    double cr[3] = {ui[1] * uk[2] - ui[2] * uk[1], ui[2] * uk[0] - ui[0] * uk[2],
                    ui[0] * uk[1] - ui[1] * uk[0]};
    double sn_l = sqrt(cr[0] * cr[0] + cr[1] * cr[1] + cr[2] * cr[2]);  // |ui||uk| sin
    double dt_l = ui[0] * uk[0] + ui[1] * uk[1] + ui[2] * uk[2];        // |ui||uk| cos
    if (sn_l > 1e-12 * li * lk) {
      double theta = atan2(sn_l, dt_l);
      double dth = theta - th0[m];
      double kf = kth[m];
      // dtheta/dx_i = (cos ui/|ui|^2 - uk/(|ui||uk|)) / sin, and for k
      // alike; F = -k dth dtheta/dx
      double cs = dt_l / (li * lk), sn = sn_l / (li * lk);
      double g = -kf * dth / sn, inv_ik = 1.0 / (li * lk);
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        gi[d] = g * (cs * ui[d] / li2 - uk[d] * inv_ik);
        gk[d] = g * (cs * uk[d] / lk2 - ui[d] * inv_ik);
      }
      u = 0.5 * kf * dth * dth;
      w = ui[0] * gi[0] + ui[1] * gi[1] + ui[2] * gi[2] + uk[0] * gk[0] + uk[1] * gk[1] +
          uk[2] * gk[2];
    }
  }
  float fix = (float)gi[0], fiy = (float)gi[1], fiz = (float)gi[2];
  float fkx = (float)gk[0], fky = (float)gk[1], fkz = (float)gk[2];
  float fjx = (float)-(gi[0] + gk[0]), fjy = (float)-(gi[1] + gk[1]),
        fjz = (float)-(gi[2] + gk[2]);
  unsigned si = slot_of[ai], sj = slot_of[aj], sk = slot_of[ak];
  const float f3[3][3] = {{fix, fiy, fiz}, {fjx, fjy, fjz}, {fkx, fky, fkz}};
  const unsigned sl[3] = {si, sj, sk};
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      long long v = hd_to_fixed48(f3[a][d]);
      if (v) atomicAdd(fpj + (size_t)sl[a] * 4 + d, (unsigned long long)v);
    }
  if (ev) {
    long long e3 = hd_to_fixed48((float)(u / 3.0)), w3 = hd_to_fixed48((float)(w / 3.0));
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      if (e3) atomicAdd(fpj_ew + (size_t)sl[a] * 2, (unsigned long long)e3);
      if (w3) atomicAdd(fpj_ew + (size_t)sl[a] * 2 + 1, (unsigned long long)w3);
    }
  }
}

void hd_launch_angles(hipStream_t st, const float4* posq, const float* lattice,
                      const unsigned* ijk, const double* kth, const double* th0,
                      const unsigned* slot_of, long long* fpj, long long* fpj_ew,
                      unsigned n_angles, bool ev) {
  if (n_angles == 0) return;
  hipLaunchKernelGGL(k_angles, dim3((n_angles + 255) / 256), dim3(256), 0, st, posq, lattice,
                     ijk, kth, th0, slot_of, (unsigned long long*)fpj,
                     (unsigned long long*)fpj_ew, n_angles, ev ? 1 : 0);
}

// Per-atom scatter of a bonded term's force, energy share and virial share
// into the j-side fixed-point accumulators (slot order).
__device__ __forceinline__ void bonded_scatter(unsigned long long* __restrict__ fpj,
                                               unsigned long long* __restrict__ fpj_ew,
                                               unsigned slot, double fx, double fy, double fz,
                                               long long e_share, long long w_share, int ev) {
  const float f3[3] = {(float)fx, (float)fy, (float)fz};
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    long long v = hd_to_fixed48(f3[d]);
    if (v) atomicAdd(fpj + (size_t)slot * 4 + d, (unsigned long long)v);
  }
  if (ev) {
    if (e_share) atomicAdd(fpj_ew + (size_t)slot * 2, (unsigned long long)e_share);
    if (w_share) atomicAdd(fpj_ew + (size_t)slot * 2 + 1, (unsigned long long)w_share);
  }
}

__device__ __forceinline__ void disp_f64(const float4& a, const float4& b, const HdLattice& L,
                                         double d[3]) {
  d[0] = (double)a.x - (double)b.x;
  d[1] = (double)a.y - (double)b.y;
  d[2] = (double)a.z - (double)b.z;
  hd_min_image_f64(d[0], d[1], d[2], L);
}

// Two-body bonded terms in FP64 (src/forces/harmonic_bond.rs:288-330,
// src/forces/morse.rs:290-320): U = k/2 (r - r0)^2, or
// U = De (1 - exp(-a (r - re)))^2; F_i = -dU/dr (r_i - r_j)/r, F_j = -F_i;
// W = F_i . (r_i - r_j); energy and virial shared half and half.
__global__ void k_bonds(const float4* __restrict__ posq, const float* __restrict__ lattice,
                        const unsigned* __restrict__ ij, const int* __restrict__ kind,
                        const double* __restrict__ prm, const unsigned* __restrict__ slot_of,
                        unsigned long long* __restrict__ fpj,
                        unsigned long long* __restrict__ fpj_ew, unsigned n_bonds, int ev) {
  unsigned m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= n_bonds) return;
  HdLattice L = hd_load_lattice(lattice);
  unsigned ai = ij[2 * m], aj = ij[2 * m + 1];
  double d[3];
  disp_f64(posq[ai], posq[aj], L, d);
  double r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
  double r = sqrt(r2);
  double dudr = 0.0, u = 0.0;
  const double* p = prm + 3 * (size_t)m;
  if (r > 1e-7) {
    if (kind[m] == 0) {
      double dr = r - p[1];
      dudr = p[0] * dr;
      u = 0.5 * p[0] * dr * dr;
    } else {
      double e = exp(-p[1] * (r - p[2]));
      dudr = 2.0 * p[0] * p[1] * (1.0 - e) * e;
      u = p[0] * (1.0 - e) * (1.0 - e);
    }
  }
  double g = r > 1e-7 ? -dudr / r : 0.0;
  long long e2 = 0, w2 = 0;
  if (ev) {
    e2 = hd_to_fixed48((float)(0.5 * u));
    w2 = hd_to_fixed48((float)(0.5 * g * r2));
  }
  bonded_scatter(fpj, fpj_ew, slot_of[ai], g * d[0], g * d[1], g * d[2], e2, w2, ev);
  bonded_scatter(fpj, fpj_ew, slot_of[aj], -g * d[0], -g * d[1], -g * d[2], e2, w2, ev);
}

void hd_launch_bonds(hipStream_t st, const float4* posq, const float* lattice, const unsigned* ij,
                     const int* kind, const double* prm, const unsigned* slot_of, long long* fpj,
                     long long* fpj_ew, unsigned n_bonds, bool ev) {
  if (n_bonds == 0) return;
  hipLaunchKernelGGL(k_bonds, dim3((n_bonds + 255) / 256), dim3(256), 0, st, posq, lattice, ij,
                     kind, prm, slot_of, (unsigned long long*)fpj, (unsigned long long*)fpj_ew,
                     n_bonds, ev ? 1 : 0);
}

// Periodic dihedral U = k (1 + cos(n phi - phi0)) (src/forces/dihedral.rs:23,
// 360-460) in FP64.  With F = r_i - r_j, G = r_j - r_k, H = r_l - r_k,
// A = F x G and B = H x G: cos phi = A.B / (|A||B|) and, since B.G = 0,
// sin phi = (B x A).G / (|A||B||G|) = -|G| F.B / (|A||B|), the same angle
// and sign as the reference's atan2(|b2| b1.n, m.n); the gradients are
// those of Blondel and Karplus (J. Comput. Chem. 17, 1132 (1996)):
//   dphi/dr_i = -|G|/|A|^2 A,  dphi/dr_l = |G|/|B|^2 B,
//   dphi/dr_j = |G|/|A|^2 A + (F.G)/(|A|^2 |G|) A - (H.G)/(|B|^2 |G|) B,
//   dphi/dr_k = -|G|/|B|^2 B - (F.G)/(|A|^2 |G|) A + (H.G)/(|B|^2 |G|) B.
// W = sum_a (r_a - r_j) . F_a; energy and virial shared in quarters.
__global__ void k_dihedrals(const float4* __restrict__ posq, const float* __restrict__ lattice,
                            const unsigned* __restrict__ ijkl, const double* __restrict__ prm,
                            const unsigned* __restrict__ slot_of,
                            unsigned long long* __restrict__ fpj,
                            unsigned long long* __restrict__ fpj_ew, unsigned n_dih, int ev) {
  unsigned m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= n_dih) return;
  HdLattice L = hd_load_lattice(lattice);
  unsigned a0 = ijkl[4 * m], a1 = ijkl[4 * m + 1], a2 = ijkl[4 * m + 2], a3 = ijkl[4 * m + 3];
  float4 p0 = posq[a0], p1 = posq[a1], p2 = posq[a2], p3 = posq[a3];
  double F[3], G[3], H[3];
  disp_f64(p0, p1, L, F);
  disp_f64(p1, p2, L, G);
  disp_f64(p3, p2, L, H);
  double A[3] = {F[1] * G[2] - F[2] * G[1], F[2] * G[0] - F[0] * G[2], F[0] * G[1] - F[1] * G[0]};
  double B[3] = {H[1] * G[2] - H[2] * G[1], H[2] * G[0] - H[0] * G[2], H[0] * G[1] - H[1] * G[0]};
  double a2n = A[0] * A[0] + A[1] * A[1] + A[2] * A[2];
  double b2n = B[0] * B[0] + B[1] * B[1] + B[2] * B[2];
  double g2 = G[0] * G[0] + G[1] * G[1] + G[2] * G[2];
  double fi[3] = {0, 0, 0}, fj[3] = {0, 0, 0}, fk[3] = {0, 0, 0}, fl[3] = {0, 0, 0};
  double u = 0.0, w = 0.0;
  if (a2n >= 1e-14 && b2n >= 1e-14 && g2 >= 1e-14) {
    double gl = sqrt(g2);
    double fb = F[0] * B[0] + F[1] * B[1] + F[2] * B[2];
    double ab = A[0] * B[0] + A[1] * B[1] + A[2] * B[2];
    double phi = atan2(-gl * fb, ab);
    const double* p = prm + 3 * (size_t)m;
    double k = p[0], nm = p[1], phi0 = p[2];
    double delta = nm * phi - phi0;
    double sd, cd;
    sincos(delta, &sd, &cd);
    u = k * (1.0 + cd);
    double mdu = k * nm * sd;  // -dU/dphi
    double fg = F[0] * G[0] + F[1] * G[1] + F[2] * G[2];
    double hg = H[0] * G[0] + H[1] * G[1] + H[2] * G[2];
    double ca = gl / a2n, cb = gl / b2n;
    double sa = fg / (a2n * gl), sb = hg / (b2n * gl);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      double gi = -ca * A[d], gl_ = cb * B[d];
      double gj = ca * A[d] + sa * A[d] - sb * B[d];
      double gk = -cb * B[d] - sa * A[d] + sb * B[d];
      fi[d] = mdu * gi;
      fj[d] = mdu * gj;
      fk[d] = mdu * gk;
      fl[d] = mdu * gl_;
    }
    // positions relative to r_j: r_i - r_j = F, r_k - r_j = -G, r_l - r_j = H - G
    for (int d = 0; d < 3; ++d) w += F[d] * fi[d] - G[d] * fk[d] + (H[d] - G[d]) * fl[d];
  }
  long long e4 = 0, w4 = 0;
  if (ev) {
    e4 = hd_to_fixed48((float)(0.25 * u));
    w4 = hd_to_fixed48((float)(0.25 * w));
  }
  bonded_scatter(fpj, fpj_ew, slot_of[a0], fi[0], fi[1], fi[2], e4, w4, ev);
  bonded_scatter(fpj, fpj_ew, slot_of[a1], fj[0], fj[1], fj[2], e4, w4, ev);
  bonded_scatter(fpj, fpj_ew, slot_of[a2], fk[0], fk[1], fk[2], e4, w4, ev);
  bonded_scatter(fpj, fpj_ew, slot_of[a3], fl[0], fl[1], fl[2], e4, w4, ev);
}

void hd_launch_dihedrals(hipStream_t st, const float4* posq, const float* lattice,
                         const unsigned* ijkl, const double* prm, const unsigned* slot_of,
                         long long* fpj, long long* fpj_ew, unsigned n_dih, bool ev) {
  if (n_dih == 0) return;
  hipLaunchKernelGGL(k_dihedrals, dim3((n_dih + 255) / 256), dim3(256), 0, st, posq, lattice,
                     ijkl, prm, slot_of, (unsigned long long*)fpj, (unsigned long long*)fpj_ew,
                     n_dih, ev ? 1 : 0);
}

// Scaled exclusions (src/forces/jit_composed.rs:1445-1458 with the LJ and
// SPME-real fragments' own scale tables, lj.rs:295-321, spme.rs:723-762):
// the pair kernel applies weight 1 to every pair within the cutoff whose
// keys differ by more than the span and 0 to the rest; this pass adds
// (scale - that weight) times each term, evaluated in FP64 with the same
// Hastings erfc and cubic LJ switch, so the pair ends at its scale.
__global__ void k_excl_scaled(const float4* __restrict__ posq, const float* __restrict__ lattice,
                              const HdExclPair* __restrict__ pairs, unsigned n_pairs, double kc,
                              double alpha, double coul_rc2, const unsigned* __restrict__ slot_of,
                              unsigned long long* __restrict__ fpj,
                              unsigned long long* __restrict__ fpj_ew, int ev) {
  unsigned m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= n_pairs) return;
  HdLattice L = hd_load_lattice(lattice);
  HdExclPair P = pairs[m];
  float4 pi = posq[P.i], pj = posq[P.j];
  double d[3];
  disp_f64(pi, pj, L, d);
  double r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
  double factor = 0.0, energy = 0.0;
  if (r2 > 0.0) {
    double inv_r2 = 1.0 / r2, inv_r = sqrt(inv_r2), r = r2 * inv_r;
    if (P.w_lj != 0.0 && r2 <= P.cut2 && P.eps != 0.0) {
      double sr2 = P.sigma * P.sigma * inv_r2;
      double sr6 = sr2 * sr2 * sr2;
      double f = 24.0 * P.eps * inv_r2 * (2.0 * sr6 * sr6 - sr6);
      double e = 4.0 * P.eps * (sr6 * sr6 - sr6);
      double delta = P.cut2 - P.rsw2;
      if (delta > 0.0 && r2 > P.rsw2) {
        double tau = (r2 - P.rsw2) / delta, omt = 1.0 - tau;
        double s = omt * omt * (1.0 + 2.0 * tau);
        f = s * f + 12.0 * tau * omt / delta * e;
        e = s * e;
      }
      factor += P.w_lj * f;
      energy += P.w_lj * e;
    }
    if (P.w_coul != 0.0 && coul_rc2 > 0.0 && r2 <= coul_rc2) {
      double qq = kc * (double)pi.w * (double)pj.w;
      double ar = alpha * r;
      double gauss = exp(-ar * ar);
      double t = 1.0 / (1.0 + 0.3275911 * ar);
      double ec = (0.254829592 +
                   (-0.284496736 + (1.421413741 + (-1.453152027 + 1.061405429 * t) * t) * t) * t) *
                  t * gauss;
      factor += P.w_coul * qq * inv_r2 * (ec * inv_r + 2.0 * alpha * 0.5641895835477563 * gauss);
      energy += P.w_coul * qq * ec * inv_r;
    }
  }
  long long e2 = 0, w2 = 0;
  if (ev) {
    e2 = hd_to_fixed48((float)(0.5 * energy));
    w2 = hd_to_fixed48((float)(0.5 * factor * r2));
  }
  bonded_scatter(fpj, fpj_ew, slot_of[P.i], factor * d[0], factor * d[1], factor * d[2], e2, w2,
                 ev);
  bonded_scatter(fpj, fpj_ew, slot_of[P.j], -factor * d[0], -factor * d[1], -factor * d[2], e2,
                 w2, ev);
}

void hd_launch_excl_scaled(hipStream_t st, const float4* posq, const float* lattice,
                           const HdExclPair* pairs, unsigned n_pairs, double kc, double alpha,
                           double coul_rc2, const unsigned* slot_of, long long* fpj,
                           long long* fpj_ew, bool ev) {
  if (n_pairs == 0) return;
  hipLaunchKernelGGL(k_excl_scaled, dim3((n_pairs + 255) / 256), dim3(256), 0, st, posq, lattice,
                     pairs, n_pairs, kc, alpha, coul_rc2, slot_of, (unsigned long long*)fpj,
                     (unsigned long long*)fpj_ew, ev ? 1 : 0);
}

// Diagnostic: number of distinct pairs of the current list with
// r^2 <= r_max^2 (the "useful" pairs).  Every pair is in both atoms' rows:
// counted from the lower slot.
__global__ void __launch_bounds__(HD_ROW_THREADS) k_count_rows(
    float rmax2, const float* __restrict__ lattice, const float4* __restrict__ tile_posq,
    const unsigned char* __restrict__ tile_img, const float4* __restrict__ center,
    const unsigned* __restrict__ jslot,
    const unsigned* __restrict__ rowhdr,
    const unsigned short* __restrict__ rows, unsigned parts, unsigned jcap, unsigned rcap,
    unsigned n, unsigned long long* __restrict__ out) {
  const unsigned unit = blockIdx.x, b = unit / parts;
  const unsigned lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
  const unsigned islot = b * 64u + w * HD_ROW_I + (lane >> 3);
  if (islot >= n) return;
  const HdLattice L = hd_load_lattice(lattice);
  const float4 cb = center[b], pi = tile_posq[islot];
  float ix, iy, iz;
  hd_rel_image(pi.x, pi.y, pi.z, cb, HD_IMAGE_NONE, tile_img[islot], L, ix, iy, iz);
  const unsigned nk = rowhdr[unit * HD_ROW_WAVES + w] >> 16;
  const unsigned short* rp =
      rows + ((size_t)unit * 64u + w * HD_ROW_I + (lane >> 3)) * rcap;
  unsigned long long cnt = 0;
  for (unsigned k = 0; k < nk; ++k)
    for (unsigned u = 0; u < 4; ++u) {
      unsigned j = rp[k * HD_ROW_CHUNK + (lane & 7u) * 4u + u] >> 4;
      if (j >= jcap) continue;
      const unsigned code = jslot[(size_t)unit * jcap + j] >> HD_ROW_SLOT_BITS;
      const unsigned js = jslot[(size_t)unit * jcap + j] & (HD_ROW_SLOTS - 1u);
      if (js <= islot) continue;
      float4 pj = tile_posq[js];
      float jx, jy, jz;
      hd_rel_image(pj.x, pj.y, pj.z, cb, code, tile_img[js], L, jx, jy, jz);
      float dx = ix - jx, dy = iy - jy, dz = iz - jz;
      if (dx * dx + dy * dy + dz * dz <= rmax2) ++cnt;
    }
  atomicAdd(out, cnt);
}

// Atom-list mode: each pair is in both atoms' lists; count it from the
// lower slot.
__global__ void __launch_bounds__(64) k_count_pairs_alist(
    float rmax2, const float* __restrict__ lattice, const float4* __restrict__ tile_posq,
    const unsigned* __restrict__ rows_in, const unsigned* __restrict__ row_count, unsigned cap,
    unsigned n, unsigned long long* __restrict__ out) {
  unsigned b = blockIdx.x, lane = threadIdx.x;
  unsigned islot = b * 64 + lane;
  if (islot >= n) return;
  HdLattice L = hd_load_lattice(lattice);
  float4 pi = tile_posq[islot];
  const unsigned* list = rows_in + (size_t)b * cap * 64 + lane;
  unsigned long long cnt = 0;
  for (unsigned k = 0; k < row_count[b]; ++k) {
    unsigned js = list[(size_t)k * 64];
    if (js >= n || js <= islot) continue;
    float4 pj = tile_posq[js];
    float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
    hd_min_image(dx, dy, dz, L);
    if (dx * dx + dy * dy + dz * dz <= rmax2) ++cnt;
  }
  atomicAdd(out, cnt);
}

void hd_launch_count_pairs(hipStream_t st, const HdPairArgs& a, unsigned long long* out) {
  unsigned nblocks = a.npad / 64;
  if (a.atom_lists)
    hipLaunchKernelGGL(k_count_pairs_alist, dim3(nblocks), dim3(64), 0, st,
                       (float)(a.rmax * a.rmax), a.lattice, a.tile_posq, a.entry_atoms,
                       a.entry_count, a.cap, a.n, out);
  else
    hipLaunchKernelGGL(k_count_rows, dim3(nblocks * a.parts), dim3(HD_ROW_THREADS), 0, st,
                       (float)(a.rmax * a.rmax), a.lattice, a.tile_posq, a.tile_img, a.center,
                       a.jslot, a.rowhdr, a.rows, a.parts, a.jcap, a.rcap, a.n, out);
}

template <int EV, int NT, bool SW>
static void launch_alist_t(hipStream_t st, const HdPairArgs& a, const PairParams& P) {
  unsigned nblocks = a.npad / 64;
  dim3 grid(nblocks);
  if (P.ortho)
    hipLaunchKernelGGL((k_pair_alist<EV, NT, SW, true>), grid, dim3(64 * PAIR_WAVES), 0, st, P,
                       a.lattice, a.tile_posq, a.tile_type, a.entry_atoms, a.entry_count,
                       a.cap, a.n, nblocks, a.fpi, a.fpi_ew, a.lj_tab);
  else
    hipLaunchKernelGGL((k_pair_alist<EV, NT, SW, false>), grid, dim3(64 * PAIR_WAVES), 0, st,
                       P, a.lattice, a.tile_posq, a.tile_type, a.entry_atoms, a.entry_count,
                       a.cap, a.n, nblocks, a.fpi, a.fpi_ew, a.lj_tab);
}

// LDS beside the j records: the dummy record; KIND 1 and 2 also the type-pair
// table (two float4 a pair in KIND 2) and the j types
static unsigned rows_lds(int kind, int nt, unsigned jcap) {
  return 16u + (kind ? (kind == 2 ? 32u : 16u) * (unsigned)(nt * nt) + jcap + 1u : 0u);
}

unsigned hd_pair_rows_lds(int nt, unsigned jcap) { return rows_lds(2, nt, jcap); }

template <int EV, int KIND>
static void launch_rows_c(hipStream_t st, const HdPairArgs& a, const PairParams& P) {
  dim3 grid(a.npad / 64 * a.parts), wg(HD_ROW_THREADS);
  const size_t lds = (size_t)a.jcap * sizeof(float4) + rows_lds(KIND, P.ntypes, a.jcap);
  if (P.coul_rc2 > 0.f)
    hipLaunchKernelGGL((k_pair_rows<EV, KIND, true>), grid, wg, lds, st, P, a.lattice,
                       a.tile_posq, a.tile_type, a.tile_img, a.center, a.half, a.jslot, a.jcount,
                       a.rowhdr, a.rows, a.block_order, a.parts, a.jcap, a.rcap, a.n,
                       (unsigned long long*)a.fpj, (unsigned long long*)a.fpj_ew, a.lj_tab,
                       a.status, a.rebuild_count);
  else
    hipLaunchKernelGGL((k_pair_rows<EV, KIND, false>), grid, wg, lds, st, P, a.lattice,
                       a.tile_posq, a.tile_type, a.tile_img, a.center, a.half, a.jslot, a.jcount,
                       a.rowhdr, a.rows, a.block_order, a.parts, a.jcap, a.rcap, a.n,
                       (unsigned long long*)a.fpj, (unsigned long long*)a.fpj_ew, a.lj_tab,
                       a.status, a.rebuild_count);
}

template <int EV, int NT>
static void launch_alist_nt(hipStream_t st, const HdPairArgs& a, const PairParams& P, bool sw) {
  if (sw) launch_alist_t<EV, NT, true>(st, a, P);
  else launch_alist_t<EV, NT, false>(st, a, P);
}

template <int EV>
static void launch_pair_ev(hipStream_t st, const HdPairArgs& a, const PairParams& P, bool sw) {
  if (!a.atom_lists) {
    // one cutoff and no switch: the regrouped terms, with the coefficients
    // in registers when a single type interacts
    if (!P.uniform) launch_rows_c<EV, 2>(st, a, P);
    else if (P.active_type < 0) launch_rows_c<EV, 1>(st, a, P);
    else launch_rows_c<EV, 0>(st, a, P);
    return;
  }
  if (P.ntypes <= 1) launch_alist_nt<EV, 1>(st, a, P, sw);
  else if (P.ntypes == 2) launch_alist_nt<EV, 2>(st, a, P, sw);
  else if (P.ntypes <= PAIR_MAXT) launch_alist_nt<EV, 4>(st, a, P, sw);
  else launch_alist_nt<EV, 0>(st, a, P, sw);
}

// f32 coefficients of one type pair, as every pair kernel form uses them
struct PairCoef {
  float c6, c12, cut2, rsw2, idl;
  bool sw;  // a switch region on an interacting pair
};
static PairCoef pair_coef(double s, double e, double rc, double rs) {
  PairCoef q;
  double s6 = s * s * s * s * s * s;
  q.c6 = (float)(4.0 * e * s6);
  q.c12 = (float)(4.0 * e * s6 * s6);
  q.cut2 = (e != 0.0) ? (float)(rc * rc) : -1.0f;
  q.rsw2 = (float)(rs * rs);
  double d = rc * rc - rs * rs;
  q.idl = d > 0.0 ? (float)(1.0 / d) : 0.0f;
  q.sw = d > 0.0 && e != 0.0;
  return q;
}

int hd_pair_table_max_types() { return PAIR_TAB_TYPES; }

unsigned hd_pair_active_types(int nt, const double* sigma, const double* eps) {
  unsigned m = 0;
  for (int k = 0; k < nt * nt; ++k)
    if (sigma[k] != 0.0 && eps[k] != 0.0) m |= 1u << (k / nt);
  return m;
}

void hd_pair_lj_table(int nt, const double* sigma, const double* eps, const double* cut,
                      const double* rsw, float* out) {
  for (int k = 0; k < nt * nt; ++k) {
    PairCoef q = pair_coef(sigma[k], eps[k], cut[k], rsw[k]);
    float* o = out + 8 * (size_t)k;
    o[0] = 12.0f * q.c12; o[1] = 6.0f * q.c6; o[2] = q.c12; o[3] = q.c6;
    o[4] = q.cut2; o[5] = q.rsw2; o[6] = q.idl; o[7] = 0.0f;
  }
}

void hd_launch_pair(hipStream_t st, const HdPairArgs& a, int ev) {
  PairParams P;
  memset(&P, 0, sizeof(P));
  P.ntypes = a.ntypes;
  bool any_switch = false;
  const int nt2 = a.ntypes * a.ntypes;
  PairCoef q[PAIR_TAB_TYPES * PAIR_TAB_TYPES];
  for (int k = 0; k < nt2; ++k) {
    q[k] = pair_coef(a.sigma[k], a.eps[k], a.cut[k], a.rsw[k]);
    if (q[k].sw) any_switch = true;
  }
  // atom lists: up to four types the rows travel in the kernel arguments;
  // beyond that, and in the row-list kernel, a.lj_tab (hd_pair_lj_table)
  if (a.ntypes <= PAIR_MAXT)
    for (int k = 0; k < nt2; ++k) {
      P.c6[k] = q[k].c6;
      P.c12[k] = q[k].c12;
      P.ljcut2[k] = q[k].cut2;
      P.rsw2[k] = q[k].rsw2;
      P.inv_delta[k] = q[k].idl;
    }
  P.kc = (float)a.kc;
  P.alpha = (float)a.alpha;
  P.coul_rc2 = a.coul_rc > 0.0 ? (float)(a.coul_rc * a.coul_rc) : -1.0f;
  P.ortho = a.ortho;
  P.reach = (float)(a.rmax + 2.0 * a.r_skin + 1.0);
  const unsigned act = hd_pair_active_types(a.ntypes, a.sigma, a.eps);
  P.active_type = __builtin_popcount(act) <= 1 ? (act ? __builtin_ctz(act) : 0) : -1;
  bool uniform = P.coul_rc2 > 0.f && !any_switch;
  for (int k = 0; k < nt2; ++k)
    if (!(q[k].c6 == 0.f && q[k].c12 == 0.f) && q[k].cut2 != P.coul_rc2) uniform = false;
  // LJ only: the interacting type pairs share one cutoff
  float ljc = -1.f;
  bool lj_uniform = !(P.coul_rc2 > 0.f) && !any_switch;
  for (int k = 0; k < nt2; ++k) {
    if (q[k].c6 == 0.f && q[k].c12 == 0.f) continue;
    if (ljc < 0.f) ljc = q[k].cut2;
    else if (q[k].cut2 != ljc) lj_uniform = false;
  }
  if (!(ljc > 0.f)) lj_uniform = false;
  P.uniform = uniform ? 1 : (lj_uniform ? 2 : 0);
  P.uc_rc2 = uniform ? P.coul_rc2 : ljc;
  P.cg = (float)(-a.alpha * a.alpha * 1.4426950408889634);
  P.pa = (float)(0.3275911 * a.alpha);
  if (ev == 1) launch_pair_ev<1>(st, a, P, any_switch);
  else if (ev == 2) launch_pair_ev<2>(st, a, P, any_switch);
  else launch_pair_ev<0>(st, a, P, any_switch);
}
