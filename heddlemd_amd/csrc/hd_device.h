// Device-side helpers shared by every HeddleMD HIP kernel (gfx950, wave64).
//
// Conventions (all kernels):
//   * Hartree atomic units; k_B = 1, k_C = 1.
//   * Lattice [lx, ly, lz, xy, xz, yz] (lower-triangular box), kept on the
//     device as float[6] so that a barostat can rescale it without a host
//     round trip.
//   * posq float4 (x, y, z, q) per atom; velocities/forces are SoA float.
//   * "slot" = position of an atom in the spatially sorted order built by
//     the neighbour list (sorted_id[slot] = atom id).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define HD_WAVE 64
#define HD_SENTINEL 0xFFFFFFFFu

struct HdLattice {
  float lx, ly, lz, xy, xz, yz;
};

// Workgroup index remap for the 8 XCDs of MI355X, which receive
// workgroups in turn (b to XCD b % 8): the result gives XCD x the
// contiguous range [x * per, (x + 1) * per) with per = nb / 8, and leaves
// the nb % 8 tail in place.  A bijection on [0, nb).
__device__ __forceinline__ unsigned hd_xcd_block(unsigned b, unsigned nb) {
  unsigned per = nb >> 3;
  return b < (per << 3) ? (b & 7u) * per + (b >> 3) : b;
}

__device__ __forceinline__ HdLattice hd_load_lattice(const float* L) {
  HdLattice l;
  l.lx = L[0]; l.ly = L[1]; l.lz = L[2];
  l.xy = L[3]; l.xz = L[4]; l.yz = L[5];
  return l;
}

// Cartesian -> fractional by back substitution (same operation order as
// the reference, kernels/pbc.cuh:18-27).
__device__ __forceinline__ void hd_cart_to_frac(float x, float y, float z, const HdLattice& L,
                                                float& sa, float& sb, float& sc) {
  sc = z / L.lz;
  sb = (y - sc * L.yz) / L.ly;
  sa = (x - sb * L.xy - sc * L.xz) / L.lx;
}

// In-place minimum image (kernels/pbc.cuh:30-43).
__device__ __forceinline__ void hd_min_image(float& dx, float& dy, float& dz, const HdLattice& L) {
  float sa, sb, sc;
  hd_cart_to_frac(dx, dy, dz, L, sa, sb, sc);
  float ka = floorf(sa + 0.5f), kb = floorf(sb + 0.5f), kc = floorf(sc + 0.5f);
  dx -= ka * L.lx + kb * L.xy + kc * L.xz;
  dy -= kb * L.ly + kc * L.yz;
  dz -= kc * L.lz;
}

// The same minimum image in FP64 (the lattice's f32 values widened): exact
// differences of f32 coordinates, for the constraint solvers.
__device__ __forceinline__ void hd_min_image_f64(double& dx, double& dy, double& dz,
                                                 const HdLattice& L) {
  double lx = L.lx, ly = L.ly, lz = L.lz, xy = L.xy, xz = L.xz, yz = L.yz;
  double sc = dz / lz;
  double sb = (dy - sc * yz) / ly;
  double sa = (dx - sb * xy - sc * xz) / lx;
  double ka = floor(sa + 0.5), kb = floor(sb + 0.5), kc = floor(sc + 0.5);
  dx -= ka * lx + kb * xy + kc * xz;
  dy -= kb * ly + kc * yz;
  dz -= kc * lz;
}

// Minimum image with the reciprocal box lengths precomputed (inv = 1/lx,
// 1/ly, 1/lz).  It differs from hd_min_image only by the rounding of the
// fractional coordinate, i.e. only for separations within an ulp of half a
// box length, which lie far beyond any cutoff (setup requires r_search <
// L/2).  Used by the pair kernel's general-cell path.
__device__ __forceinline__ void hd_min_image_rcp(float& dx, float& dy, float& dz,
                                                 const HdLattice& L, float ilx, float ily,
                                                 float ilz) {
  float sc = dz * ilz;
  float sb = (dy - sc * L.yz) * ily;
  float sa = (dx - sb * L.xy - sc * L.xz) * ilx;
  float ka = floorf(sa + 0.5f), kb = floorf(sb + 0.5f), kc = floorf(sc + 0.5f);
  dx -= ka * L.lx + kb * L.xy + kc * L.xz;
  dy -= kb * L.ly + kc * L.yz;
  dz -= kc * L.lz;
}

// In-place wrap into the primary cell returning the image triple
// (kernels/pbc.cuh:74-92).
__device__ __forceinline__ void hd_wrap_with_image(float& x, float& y, float& z, int& ka_o,
                                                   int& kb_o, int& kc_o, const HdLattice& L) {
  float sa, sb, sc;
  hd_cart_to_frac(x, y, z, L, sa, sb, sc);
  float ka = floorf(sa + 0.5f), kb = floorf(sb + 0.5f), kc = floorf(sc + 0.5f);
  x -= ka * L.lx + kb * L.xy + kc * L.xz;
  y -= kb * L.ly + kc * L.yz;
  z -= kc * L.lz;
  ka_o = (int)ka;
  kb_o = (int)kb;
  kc_o = (int)kc;
}

// Shift (x,y,z) to the periodic image nearest the centre (cx,cy,cz)
// (kernels/pbc.cuh:54-72).
__device__ __forceinline__ void hd_wrap_against_center(float& x, float& y, float& z, float cx,
                                                       float cy, float cz, const HdLattice& L) {
  float dx = x - cx, dy = y - cy, dz = z - cz;
  float sa, sb, sc;
  hd_cart_to_frac(dx, dy, dz, L, sa, sb, sc);
  float ka = floorf(sa + 0.5f), kb = floorf(sb + 0.5f), kc = floorf(sc + 0.5f);
  x -= ka * L.lx + kb * L.xy + kc * L.xz;
  y -= kb * L.ly + kc * L.yz;
  z -= kc * L.lz;
}

// Position relative to a centre, shifted to the nearest periodic image,
// evaluated in FP64 and rounded once: the result is small (|d| <~ r_cut +
// block extent), so it keeps ~1e-7 relative precision where the f32
// difference of two wrapped absolute coordinates would carry the rounding
// error of the large absolute value.  Orthorhombic cells only.
__device__ __forceinline__ void hd_rel_to_center(float x, float y, float z, float cx, float cy,
                                                 float cz, const HdLattice& L, float& rx,
                                                 float& ry, float& rz) {
  double dx = (double)x - (double)cx, dy = (double)y - (double)cy, dz = (double)z - (double)cz;
  double lx = L.lx, ly = L.ly, lz = L.lz;
  dx -= lx * floor(dx / lx + 0.5);
  dy -= ly * floor(dy / ly + 0.5);
  dz -= lz * floor(dz / lz + 0.5);
  rx = (float)dx;
  ry = (float)dy;
  rz = (float)dz;
}

// The same with the reciprocal box lengths (FP64) precomputed: a multiply
// instead of a correctly rounded FP64 division per axis.  The nearest image
// can differ from hd_rel_to_center only for a separation within an ulp of
// half a box length, far beyond any search radius.
__device__ __forceinline__ void hd_rel_to_center_rcp(float x, float y, float z, float cx,
                                                     float cy, float cz, const HdLattice& L,
                                                     double ilx, double ily, double ilz,
                                                     float& rx, float& ry, float& rz) {
  double dx = (double)x - (double)cx, dy = (double)y - (double)cy, dz = (double)z - (double)cz;
  dx -= (double)L.lx * floor(dx * ilx + 0.5);
  dy -= (double)L.ly * floor(dy * ily + 0.5);
  dz -= (double)L.lz * floor(dz * ilz + 0.5);
  rx = (float)dx;
  ry = (float)dy;
  rz = (float)dz;
}

// Periodic images within one box vector per axis, as a code 0..26:
// (ka + 1) + 3 (kb + 1) + 9 (kc + 1).
#define HD_IMAGE_NONE 13u
#define HD_FIXED_FAR 1073741824  // hd_rel_fixed: out of every list's reach

// An atom's position relative to a centre c: x - c + the lattice vectors of
// two image codes (the list's image of the j-atom's cell, and the atom's own
// return to the cell it was listed in).  Without a shift the f32 difference
// is rounded once; with one the sum is formed in FP64 and rounded once.
__device__ __forceinline__ void hd_rel_image(float x, float y, float z, float4 c, unsigned code,
                                             unsigned own, const HdLattice& L, float& rx,
                                             float& ry, float& rz) {
  if (code == HD_IMAGE_NONE && own == HD_IMAGE_NONE) {
    rx = x - c.x;
    ry = y - c.y;
    rz = z - c.z;
    return;
  }
  double ka = (double)((int)(code % 3u + own % 3u) - 2),
         kb = (double)((int)((code / 3u) % 3u + (own / 3u) % 3u) - 2),
         kc = (double)((int)(code / 9u + own / 9u) - 2);
  rx = (float)(((double)x - (double)c.x) +
               (ka * (double)L.lx + kb * (double)L.xy + kc * (double)L.xz));
  ry = (float)(((double)y - (double)c.y) + (kb * (double)L.ly + kc * (double)L.yz));
  rz = (float)(((double)z - (double)c.z) + kc * (double)L.lz);
}

// The same in units of 1 / scale (a power of two), rounded to a whole
// number: differences of two such offsets are exact, so a pair's
// displacement is rounded once, at its own size, in whatever image.  The
// caller's scale keeps offsets within 2^29; a position that is not (or is
// not a number) goes to 2^30 along x, out of everything's reach.
__device__ __forceinline__ int3 hd_rel_fixed(float x, float y, float z, float4 c, unsigned code,
                                             unsigned own, const HdLattice& L, double scale) {
  double dx = (double)x - (double)c.x, dy = (double)y - (double)c.y, dz = (double)z - (double)c.z;
  if (code != HD_IMAGE_NONE || own != HD_IMAGE_NONE) {
    const double ka = (double)((int)(code % 3u + own % 3u) - 2),
                 kb = (double)((int)((code / 3u) % 3u + (own / 3u) % 3u) - 2),
                 kc = (double)((int)(code / 9u + own / 9u) - 2);
    dx += ka * (double)L.lx + kb * (double)L.xy + kc * (double)L.xz;
    dy += kb * (double)L.ly + kc * (double)L.yz;
    dz += kc * (double)L.lz;
  }
  const double lim = 536870912.0;
  dx *= scale;
  dy *= scale;
  dz *= scale;
  if (!(fabs(dx) <= lim && fabs(dy) <= lim && fabs(dz) <= lim))
    return make_int3(HD_FIXED_FAR, 0, 0);
  return make_int3(__double2int_rn(dx), __double2int_rn(dy), __double2int_rn(dz));
}

// The code of the lattice vector that takes a wrapped position p back to
// the image nearest its wrapped position `ref` at the last rebuild (an atom
// that has crossed a face since then was wrapped to the other side).
__device__ __forceinline__ unsigned hd_own_image(float4 p, float4 ref, const HdLattice& L) {
  float sa, sb, sc;
  hd_cart_to_frac(p.x - ref.x, p.y - ref.y, p.z - ref.z, L, sa, sb, sc);
  int ka = (int)floorf(sa + 0.5f), kb = (int)floorf(sb + 0.5f), kc = (int)floorf(sc + 0.5f);
  ka = min(max(ka, -1), 1);
  kb = min(max(kb, -1), 1);
  kc = min(max(kc, -1), 1);
  return (unsigned)(1 - ka) + 3u * (unsigned)(1 - kb) + 9u * (unsigned)(1 - kc);
}

// SPME spline origin of one atom: wrap into the primary cell, fractional
// coordinate + 1/2, u = s * n, primary bin floor(u) (mod n) and offset
// t = u - floor(u) (the geometry of kernels/spme_spread_gather.cuh:90-126).
// Evaluated in FP64 and rounded once, so the offset t keeps ~1e-7
// precision on 128^3 grids (f32 would lose log2(n) bits of it).
__device__ __forceinline__ void hd_spline_origin(float x, float y, float z, const HdLattice& L,
                                                 unsigned na, unsigned nb, unsigned nc,
                                                 float& ta, float& tb, float& tc, int& ga,
                                                 int& gb, int& gc) {
  double sc = (double)z / (double)L.lz;
  double sb = ((double)y - sc * (double)L.yz) / (double)L.ly;
  double sa = ((double)x - sb * (double)L.xy - sc * (double)L.xz) / (double)L.lx;
  sa -= floor(sa + 0.5);
  sb -= floor(sb + 0.5);
  sc -= floor(sc + 0.5);
  double ua = (sa + 0.5) * (double)na, ub = (sb + 0.5) * (double)nb, uc = (sc + 0.5) * (double)nc;
  double fa = floor(ua), fb = floor(ub), fc = floor(uc);
  ta = (float)(ua - fa);
  tb = (float)(ub - fb);
  tc = (float)(uc - fc);
  int la = (int)fa, lb = (int)fb, lc = (int)fc;
  ga = ((la % (int)na) + (int)na) % (int)na;
  gb = ((lb % (int)nb) + (int)nb) % (int)nb;
  gc = ((lc % (int)nc) + (int)nc) % (int)nc;
}

// Per-slot SPME spline record of a gathered position: (t_a, t_b, t_c, q)
// and the packed origin cell g_a | g_b << 10 | g_c << 20, or HD_SPME_NO_CELL
// for an uncharged atom (nothing written to spl then).
#define HD_SPME_NO_CELL 0xFFFFFFFFu
__device__ __forceinline__ void hd_spline_record(float4 pq, const HdLattice& L, unsigned na,
                                                 unsigned nb, unsigned nc, float4* spl,
                                                 unsigned* sg, unsigned s) {
  if (pq.w == 0.f) {
    sg[s] = HD_SPME_NO_CELL;
    return;
  }
  float ta, tb, tc;
  int ga, gb, gc;
  hd_spline_origin(pq.x, pq.y, pq.z, L, na, nb, nc, ta, tb, tc, ga, gb, gc);
  spl[s] = make_float4(ta, tb, tc, pq.w);
  sg[s] = (unsigned)ga | ((unsigned)gb << 10) | ((unsigned)gc << 20);
}

// Wave64 rotation through DPP: every lane receives the value held by lane
// (lane + 1) mod 64 ("wave_rol:1"; a full-rate VALU move, no LDS traffic).
__device__ __forceinline__ int hd_rot1_i(int v) {
  // every lane is written (no row or bank masked, no lane out of range), so
  // the "old" operand is never observed and bound_ctrl is irrelevant
  return __builtin_amdgcn_mov_dpp(v, 0x134, 0xF, 0xF, true);
}

// f32 -> i64 fixed point at scale 2^48, truncating toward zero; the scale
// is applied as two exact power-of-two products so no intermediate
// rounding occurs (src/forces/jit_composed.rs:1462-1475).
__device__ __forceinline__ long long hd_to_fixed48(float f) {
  float s = f * 16777216.0f;
  s *= 16777216.0f;
  return (long long)s;
}
// i64 -> f32 (round to nearest) then * 2^-48 (kernels/neighbor.cu:744-758).
__device__ __forceinline__ float hd_from_fixed48(long long v) {
  const float inv = (1.0f / 16777216.0f) / 16777216.0f;
  return (float)v * inv;
}

// Set bits of a wave mask below this lane.
__device__ __forceinline__ unsigned hd_rank(unsigned long long m) {
  return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                   __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

// Orders one wave's LDS accesses: what its lanes wrote before is what its
// lanes read after.
__device__ __forceinline__ void hd_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Two words that may alias anything (16-bit list entries moved four at a time).
typedef unsigned hd_u32x2 __attribute__((ext_vector_type(2), may_alias));
