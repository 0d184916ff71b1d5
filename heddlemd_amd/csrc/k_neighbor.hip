// Neighbour maintenance for the row lists and the per-atom lists (gfx950).
//
// Reference behaviour (what is kept):
//   * displacement check |x - x_ref|^2 > (r_skin/2)^2 sets bit 0 of a status
//     word (kernels/neighbor.cu:50-75);
//   * i-blocks of consecutive sorted atoms, each with the list of the
//     individual j-atoms within r_search of it
//     (kernels/neighbor.cu:416-631);
//   * capacity overflow / high-water bits in the same status word
//     (kernels/neighbor.cu:643-671).
// MI355X design (what changes):
//   * blocks are 64 atoms; a block's j-atoms are listed once (they are
//     staged in LDS by the pair kernel) and every i-atom has a row of
//     16-bit indices into that list, both sides of every pair, exclusions
//     applied (k_build_rows);
//   * atoms are ordered along a Hilbert curve over a fixed voxel grid
//     (voxel = fractional-coordinate cell, so the order survives box
//     rescaling) instead of by particle id inside r_search cells, which
//     makes a block spatially compact;
//   * each block owns fixed-capacity regions, written in a fixed order (no
//     atomics, no scatter pass), so the list is deterministic;
//   * every kernel here is gated on the status word on the device, so the
//     whole rebuild lives inside a captured step and needs no host sync.
#include "hd_device.h"
#include "hd_kernels.h"


// r_search^2 margins: the box tests and the row test are done in f32 on
// block-relative coordinates; a relative 1e-5 (boxes) and 4e-6 (pairs)
// covers their rounding, so no pair within r_search is ever lost
#define NB_BOX_MARGIN 1.00001f
#define NB_ROW_MARGIN 1.000004f

__device__ __forceinline__ bool nb_rebuild_due(const unsigned* status) {
  return (*(volatile const unsigned*)status & (NB_STATUS_REBUILD | NB_STATUS_FORCE)) != 0u;
}
// The same in a kernel during which the request cannot change before every
// workgroup has read it: one scalar load through the caches.
__device__ __forceinline__ bool nb_rebuild_due_now(const unsigned* status) {
  return (*status & (NB_STATUS_REBUILD | NB_STATUS_FORCE)) != 0u;
}

// One atomic per launch in the main: waves that find the request set leave
// it (device atomics on one word queue up, about 20 ns each).
__device__ __forceinline__ void nb_request_rebuild(unsigned* status, bool over) {
  if (__any(over) && (threadIdx.x & 63u) == 0 &&
      !(*(volatile unsigned*)status & NB_STATUS_REBUILD))
    atomicOr(status, NB_STATUS_REBUILD);
}

// Displacement check against the positions of the last rebuild.  A box
// change since the rebuild (barostat) moves every minimum-image pair
// vector by at most sqrt(3) * max|dL|, which is added to each atom's
// displacement so that |x - x_ref| + sqrt(3) max|dL| <= r_skin/2 still
// bounds every pair-distance change by r_skin.
__global__ void k_disp_check(const float4* __restrict__ posq, const float4* __restrict__ ref,
                             const float* __restrict__ lattice,
                             const float* __restrict__ ref_lattice, float half_skin,
                             unsigned* status, unsigned n) {
  unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  bool over = false;
  if (i < n) {
    HdLattice L = hd_load_lattice(lattice);
    float dl = 0.f;
#pragma unroll
    for (int k = 0; k < 6; ++k) dl = fmaxf(dl, fabsf(lattice[k] - ref_lattice[k]));
    float4 p = posq[i], r = ref[i];
    float dx = p.x - r.x, dy = p.y - r.y, dz = p.z - r.z;
    hd_min_image(dx, dy, dz, L);
    over = sqrtf(dx * dx + dy * dy + dz * dz) + 1.7320508f * dl > half_skin;
  }
  nb_request_rebuild(status, over);
}

// Curve rank of the fractional voxel that holds the atom (wrapped into the
// primary cell).
__device__ __forceinline__ unsigned nb_voxel_key(float4 p, const HdLattice& L,
                                                 const unsigned* __restrict__ voxel_rank,
                                                 unsigned nva, unsigned nvb, unsigned nvc) {
  float x = p.x, y = p.y, z = p.z;
  int ia, ib, ic;
  hd_wrap_with_image(x, y, z, ia, ib, ic, L);
  float sa, sb, sc;
  hd_cart_to_frac(x, y, z, L, sa, sb, sc);
  int va = (int)floorf((sa + 0.5f) * (float)nva);
  int vb = (int)floorf((sb + 0.5f) * (float)nvb);
  int vc = (int)floorf((sc + 0.5f) * (float)nvc);
  va = min(max(va, 0), (int)nva - 1);
  vb = min(max(vb, 0), (int)nvb - 1);
  vc = min(max(vc, 0), (int)nvc - 1);
  return voxel_rank[((unsigned)va * nvb + (unsigned)vb) * nvc + (unsigned)vc];
}

// Voxel key = curve rank of the atom's fractional voxel; histogram.
// Also records the positions and lattice of this rebuild, against which the
// displacement check measures (positions do not change within a force
// evaluation, so the copy can be taken here, with the keys).
__global__ void k_voxel_keys(const float4* __restrict__ posq, const float* __restrict__ lattice,
                             const unsigned* __restrict__ voxel_rank, unsigned nva, unsigned nvb,
                             unsigned nvc, unsigned* __restrict__ atom_key,
                             unsigned* __restrict__ voxel_count, float4* __restrict__ ref,
                             float* __restrict__ ref_lattice, const unsigned* status,
                             unsigned n) {
  if (!nb_rebuild_due(status)) return;
  HdLattice L = hd_load_lattice(lattice);
  if (blockIdx.x == 0 && threadIdx.x < 6) ref_lattice[threadIdx.x] = lattice[threadIdx.x];
  for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    float4 p = posq[i];
    ref[i] = p;
    unsigned key = nb_voxel_key(p, L, voxel_rank, nva, nvb, nvc);
    atom_key[i] = key;
    atomicAdd(&voxel_count[key], 1u);
  }
}

// Exclusive scan of voxel_count -> voxel_off (and cleared scatter
// cursors) over chunks of NB_SCAN_CHUNK voxels: chunk sums, then a
// workgroup scan per chunk.  Up to NB_SCAN_FUSED_MAX chunks (16 M atoms),
// each workgroup sums the chunk sums before its own; beyond that a
// one-workgroup pass turns them into offsets first (k_voxel_scan_parts).
#define NB_SCAN_CHUNK 2048u  // 256 threads x 8 voxels
#define NB_SCAN_FUSED_MAX 4096u

__device__ __forceinline__ unsigned nb_block_excl_scan256(unsigned v, unsigned* tmp,
                                                          unsigned& total) {
  unsigned t = threadIdx.x;
  tmp[t] = v;
  __syncthreads();
  for (unsigned off = 1; off < 256u; off <<= 1) {
    unsigned u = (t >= off) ? tmp[t - off] : 0u;
    __syncthreads();
    tmp[t] += u;
    __syncthreads();
  }
  total = tmp[255];
  unsigned r = tmp[t] - v;
  __syncthreads();
  return r;
}

__global__ void __launch_bounds__(256) k_voxel_scan_reduce(const unsigned* __restrict__ count,
                                                           unsigned* __restrict__ part,
                                                           const unsigned* status, unsigned nvox) {
  if (!nb_rebuild_due(status)) return;
  __shared__ unsigned tmp[256];
  unsigned base = blockIdx.x * NB_SCAN_CHUNK;
  unsigned s = 0;
#pragma unroll
  for (unsigned k = 0; k < NB_SCAN_CHUNK / 256u; ++k) {
    unsigned i = base + k * 256u + threadIdx.x;
    if (i < nvox) s += count[i];
  }
  unsigned total;
  (void)nb_block_excl_scan256(s, tmp, total);
  if (threadIdx.x == 0) part[blockIdx.x] = total;
}


__global__ void __launch_bounds__(1024) k_voxel_scan_parts(unsigned* __restrict__ part,
                                                           const unsigned* status,
                                                           unsigned nparts) {
  if (!nb_rebuild_due(status)) return;
  __shared__ unsigned tmp[1024];
  unsigned t = threadIdx.x, carry = 0;
  for (unsigned base = 0; base < nparts; base += 1024u) {
    unsigned i = base + t;
    unsigned v = (i < nparts) ? part[i] : 0u;
    tmp[t] = v;
    __syncthreads();
    for (unsigned off = 1; off < 1024u; off <<= 1) {
      unsigned u = (t >= off) ? tmp[t - off] : 0u;
      __syncthreads();
      tmp[t] += u;
      __syncthreads();
    }
    if (i < nparts) part[i] = carry + tmp[t] - v;
    carry += tmp[1023];
    __syncthreads();
  }
  if (t == 0) part[nparts] = carry;
}
__global__ void __launch_bounds__(256) k_voxel_scan_apply(const unsigned* __restrict__ count,
                                                          const unsigned* __restrict__ part,
                                                          unsigned* __restrict__ voxel_off,
                                                          unsigned* __restrict__ voxel_cursor,
                                                          const unsigned* status, unsigned nvox,
                                                          unsigned nparts) {
  if (!nb_rebuild_due(status)) return;
  __shared__ unsigned tmp[256];
  const unsigned per = NB_SCAN_CHUNK / 256u;
  unsigned b0 = blockIdx.x * NB_SCAN_CHUNK + threadIdx.x * per;
  unsigned c[NB_SCAN_CHUNK / 256u];
  unsigned s = 0;
#pragma unroll
  for (unsigned k = 0; k < per; ++k) {
    c[k] = (b0 + k < nvox) ? count[b0 + k] : 0u;
    s += c[k];
  }
  unsigned before, all;
  if (nparts <= NB_SCAN_FUSED_MAX) {
    // offset of this chunk: the sum of the chunk sums before it; chunk 0
    // also sums them all, for voxel_off[nvox]
    unsigned lim = blockIdx.x == 0 ? nparts : blockIdx.x;
    unsigned o = 0;
    for (unsigned k = threadIdx.x; k < lim; k += 256u) o += part[k];
    (void)nb_block_excl_scan256(o, tmp, before);
    all = before;
    if (blockIdx.x == 0) before = 0u;
  } else {
    // offsets from k_voxel_scan_parts
    before = part[blockIdx.x];
    all = part[nparts];
  }
  unsigned total;
  unsigned run = before + nb_block_excl_scan256(s, tmp, total);
#pragma unroll
  for (unsigned k = 0; k < per; ++k) {
    if (b0 + k < nvox) {
      voxel_off[b0 + k] = run;
      voxel_cursor[b0 + k] = 0u;
    }
    run += c[k];
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) voxel_off[nvox] = all;
}

__global__ void k_voxel_scatter(const unsigned* __restrict__ atom_key,
                                const unsigned* __restrict__ voxel_off,
                                unsigned* __restrict__ voxel_cursor,
                                unsigned* __restrict__ sorted_id, const unsigned* status,
                                unsigned n) {
  if (!nb_rebuild_due(status)) return;
  for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    unsigned k = atom_key[i];
    unsigned slot = voxel_off[k] + atomicAdd(&voxel_cursor[k], 1u);
    sorted_id[slot] = i;
  }
}

__device__ __forceinline__ void nb_sort_voxel(unsigned v, const unsigned* __restrict__ voxel_off,
                                              unsigned* __restrict__ sorted_id,
                                              unsigned* __restrict__ slot_of) {
  unsigned b = voxel_off[v], e = voxel_off[v + 1];
  for (unsigned k = b + 1; k < e; ++k) {
    unsigned key = sorted_id[k];
    int pos = (int)k - 1;
    while (pos >= (int)b && sorted_id[pos] > key) {
      sorted_id[pos + 1] = sorted_id[pos];
      --pos;
    }
    sorted_id[pos + 1] = key;
  }
  for (unsigned k = b; k < e; ++k) slot_of[sorted_id[k]] = k;
}

// Per voxel: sort its atom ids ascending (a voxel holds a handful of
// atoms) so the slot order is independent of atomic arrival order; then
// clear the voxel histogram for the next rebuild and record slot_of[id].
__global__ void k_voxel_sort(const unsigned* __restrict__ voxel_off,
                             unsigned* __restrict__ voxel_count, unsigned* __restrict__ sorted_id,
                             unsigned* __restrict__ slot_of, const unsigned* status,
                             unsigned nvox) {
  if (!nb_rebuild_due(status)) return;
  for (unsigned v = blockIdx.x * blockDim.x + threadIdx.x; v < nvox;
       v += gridDim.x * blockDim.x) {
    nb_sort_voxel(v, voxel_off, sorted_id, slot_of);
    voxel_count[v] = 0u;
  }
}

// Per-slot static data refreshed at a rebuild: type and exclusion key in
// slot order, padding lanes marked with sentinels.

// Every step: gather positions into slot order (wrapped into the primary
// cell) and clear the j-side fixed-point accumulators of the pair kernel.
// Slot-order copy of the positions (wrapped into the cell) and clearing of
// the j-side accumulators, every step.  On rebuild steps (status given and
// the request set) it also fills the slots' types and keys and each 64-slot
// block's bounding box (one wave per block), from the same positions, and
// keeps those positions (tile_ref): on the other steps an atom that has
// crossed a face since is marked with the image that takes it back
// (tile_img), which the row lists' image codes assume.
// One slot s < npad; the wave's 64 lanes hold the 64 slots of one block
// (the bounding-box reduction is a wave reduction).
__device__ __forceinline__ void nb_gather_slot(unsigned s, bool rebuild,
                                               const float4* __restrict__ posq,
                                               const unsigned* __restrict__ sorted_id,
                                               const float* __restrict__ lattice,
                                               float4* __restrict__ tile_posq,
                                               long long* __restrict__ fpj,
                                               long long* __restrict__ fpj_ew, unsigned n,
                                               const unsigned* __restrict__ type,
                                               const unsigned* __restrict__ key,
                                               unsigned* __restrict__ tile_type,
                                               unsigned* __restrict__ tile_key,
                                               float4* __restrict__ center,
                                               float4* __restrict__ half,
                                               float4* __restrict__ tile_ref,
                                               unsigned char* __restrict__ tile_img) {
  float4 out = make_float4(0.f, 0.f, 0.f, 0.f);
  unsigned id = 0u, img = HD_IMAGE_NONE;
  if (s < n) {
    HdLattice L = hd_load_lattice(lattice);
    id = sorted_id[s];
    float4 p = posq[id];
    int a, b, c;
    hd_wrap_with_image(p.x, p.y, p.z, a, b, c, L);
    out = p;
    if (!rebuild) img = hd_own_image(p, tile_ref[s], L);
  }
  tile_posq[s] = out;
  tile_img[s] = (unsigned char)img;
  if (rebuild) tile_ref[s] = out;
  longlong2 z = make_longlong2(0, 0);
  reinterpret_cast<longlong2*>(fpj)[2 * s] = z;
  reinterpret_cast<longlong2*>(fpj)[2 * s + 1] = z;
  if (fpj_ew) reinterpret_cast<longlong2*>(fpj_ew)[s] = z;
  if (!rebuild) return;
  bool v = s < n;
  tile_type[s] = v ? type[id] : 0u;
  tile_key[s] = v ? key[id] : HD_SENTINEL - 1u;
  float lox = v ? out.x : 3.0e38f, loy = v ? out.y : 3.0e38f, loz = v ? out.z : 3.0e38f;
  float hix = v ? out.x : -3.0e38f, hiy = v ? out.y : -3.0e38f, hiz = v ? out.z : -3.0e38f;
  for (int off = 32; off > 0; off >>= 1) {
    lox = fminf(lox, __shfl_xor(lox, off));
    loy = fminf(loy, __shfl_xor(loy, off));
    loz = fminf(loz, __shfl_xor(loz, off));
    hix = fmaxf(hix, __shfl_xor(hix, off));
    hiy = fmaxf(hiy, __shfl_xor(hiy, off));
    hiz = fmaxf(hiz, __shfl_xor(hiz, off));
  }
  if ((threadIdx.x & 63u) == 0) {
    // the centre is rounded to 1/16 Bohr: the offset of an atom from it is
    // then exact in f32 whenever the coordinate is at least as large as the
    // offset (the pair kernel works with those offsets)
    unsigned blk = s >> 6;
    float cx = 0.0625f * rintf(8.0f * (lox + hix)), cy = 0.0625f * rintf(8.0f * (loy + hiy)),
          cz = 0.0625f * rintf(8.0f * (loz + hiz));
    center[blk] = make_float4(cx, cy, cz, 0.f);
    half[blk] = make_float4(fmaxf(hix - cx, cx - lox), fmaxf(hiy - cy, cy - loy),
                            fmaxf(hiz - cz, cz - loz), 0.f);
  }
}

__global__ void k_tile_gather(const float4* __restrict__ posq, const unsigned* __restrict__ sorted_id,
                              const float* __restrict__ lattice, float4* __restrict__ tile_posq,
                              long long* __restrict__ fpj, long long* __restrict__ fpj_ew,
                              unsigned n, unsigned npad, const unsigned* status,
                              const unsigned* __restrict__ type, const unsigned* __restrict__ key,
                              unsigned* __restrict__ tile_type, unsigned* __restrict__ tile_key,
                              float4* __restrict__ center, float4* __restrict__ half,
                              float4* __restrict__ tile_ref,
                              unsigned char* __restrict__ tile_img, float4* __restrict__ spl,
                              unsigned* __restrict__ sg, unsigned gna, unsigned gnb,
                              unsigned gnc) {
  unsigned s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= npad) return;  // whole waves: npad is a multiple of 64
  nb_gather_slot(s, status && nb_rebuild_due(status), posq, sorted_id, lattice, tile_posq, fpj,
                 fpj_ew, n, type, key, tile_type, tile_key, center, half, tile_ref, tile_img);
  // the SPME spline record of the slot the thread has just written
  if (spl && s < n)
    hd_spline_record(tile_posq[s], hd_load_lattice(lattice), gna, gnb, gnc, spl, sg, s);
}


// Per-block axis-aligned bounding box: centre and half extents (one wave
// per block).  Padding lanes are ignored.

// Closest approach of two boxes under the minimum image (per axis; exact
// for orthorhombic cells), as kernels/neighbor.cu:364-388.  In a tilted
// cell a pair's own minimum image (fractional rounding of its separation)
// can differ by one lattice vector per axis from the one the box centres
// round to, so the 27 images around the centres' are all tried there.
__device__ __forceinline__ float nb_box_gap2(float dx, float dy, float dz, float4 ha, float4 hb) {
  float ex = fmaxf(fabsf(dx) - (ha.x + hb.x), 0.f);
  float ey = fmaxf(fabsf(dy) - (ha.y + hb.y), 0.f);
  float ez = fmaxf(fabsf(dz) - (ha.z + hb.z), 0.f);
  return ex * ex + ey * ey + ez * ez;
}
__device__ __forceinline__ float nb_box_dist2(float4 ca, float4 ha, float4 cb, float4 hb,
                                              const HdLattice& L) {
  float dx = ca.x - cb.x, dy = ca.y - cb.y, dz = ca.z - cb.z;
  hd_min_image(dx, dy, dz, L);
  if (L.xy == 0.f && L.xz == 0.f && L.yz == 0.f) return nb_box_gap2(dx, dy, dz, ha, hb);
  float best = 3.0e38f;
  for (int kc = -1; kc <= 1; ++kc)
    for (int kb = -1; kb <= 1; ++kb)
      for (int ka = -1; ka <= 1; ++ka) {
        float sx = dx + (float)ka * L.lx + (float)kb * L.xy + (float)kc * L.xz;
        float sy = dy + (float)kb * L.ly + (float)kc * L.yz;
        float sz = dz + (float)kc * L.lz;
        best = fminf(best, nb_box_gap2(sx, sy, sz, ha, hb));
      }
  return best;
}

// Block-pair candidates: bit (jb % 64) of mask[b * nchunks + jb / 64] is
// set when j-block jb's box lies within r_search of block b's.  Each wave handles (b, chunk of 64 j-blocks) items in
// a grid-stride loop, so the box tests of a rebuild run at full width
// instead of as a dependent loop inside each block's wave, while the launch
// stays small on the steps where the rebuild gate closes it at once.
#define NB_PAIR_WAVES 4096
// One (block, chunk of 64 j-blocks) item, one wave.
__device__ __forceinline__ void nb_block_pair_item(unsigned wv, const float4* __restrict__ center,
                                                   const float4* __restrict__ half,
                                                   const HdLattice& L, float rs2,
                                                   unsigned long long* __restrict__ mask,
                                                   unsigned nblocks, unsigned nchunks) {
  unsigned lane = threadIdx.x & 63;
  unsigned b = wv / nchunks, c = wv % nchunks;
  unsigned jb = c * 64 + lane;
  bool cand = false;
  if (jb < nblocks)
    cand = nb_box_dist2(center[b], half[b], center[jb], half[jb], L) <= rs2;
  unsigned long long m = __ballot(cand);
  if (lane == 0) mask[wv] = m;
}
__global__ void __launch_bounds__(256) k_block_pairs(const float4* __restrict__ center,
                                                     const float4* __restrict__ half,
                                                     const float* __restrict__ lattice, float rs2,
                                                     unsigned long long* __restrict__ mask,
                                                     unsigned nblocks, unsigned nchunks,
                                                     const unsigned* status) {
  if (!nb_rebuild_due(status)) return;
  unsigned nwaves = gridDim.x * (blockDim.x >> 6);
  HdLattice L = hd_load_lattice(lattice);
  for (unsigned wv = (blockIdx.x * blockDim.x + threadIdx.x) >> 6; wv < nblocks * nchunks;
       wv += nwaves)
    nb_block_pair_item(wv, center, half, L, rs2, mask, nblocks, nchunks);
}

// Systems of at most NB_SMALL_ATOMS atoms and NB_SMALL_VOX voxels: the
// displacement check and the rebuild's voxel binning (keys, histogram, scan,
// scatter, per-voxel sort) run in one workgroup, with barriers between the
// phases in place of the general path's six launches.  Up to NB_SMALL_GATHER
// atoms the tile gather (with the SPME spline records when asked) runs there
// too; beyond that one CU takes longer over it than a launch of its own
// costs (7,938 atoms: 29 us for everything in one workgroup, 7.4 + 4.2 apart).  The histogram and the scatter cursors live in LDS (the
// global voxel_count stays zero, as the general path leaves it).  Results
// are those of the general path: the per-atom arithmetic is shared with its
// kernels, the scan is exact and the per-voxel sort makes the slot order
// independent of the order of the atomics.
#define NB_SMALL_THREADS 1024u
#define NB_SMALL_ATOMS 16384u
#define NB_SMALL_GATHER 1024u
#define NB_SMALL_VOX 8192u

__global__ void __launch_bounds__(NB_SMALL_THREADS) k_nb_small(HdNeighborArgs a, int check,
                                                               long long* __restrict__ fpj,
                                                               long long* __restrict__ fpj_ew,
                                                               float4* __restrict__ spl,
                                                               unsigned* __restrict__ sg,
                                                               unsigned gna, unsigned gnb,
                                                               unsigned gnc) {
  __shared__ unsigned cnt[NB_SMALL_VOX];
  __shared__ unsigned scan[NB_SMALL_THREADS];
  __shared__ int s_over;
  const unsigned t = threadIdx.x;
  HdLattice L = hd_load_lattice(a.lattice);
  if (t == 0) s_over = 0;
  __syncthreads();
  if (check) {
    // k_disp_check's test per atom
    float dl = 0.f;
#pragma unroll
    for (int k = 0; k < 6; ++k) dl = fmaxf(dl, fabsf(a.lattice[k] - a.ref_lattice[k]));
    bool over = false;
#pragma unroll 4
    for (unsigned i = t; i < a.n; i += NB_SMALL_THREADS) {
      float4 p = a.posq[i], r = a.ref_pos[i];
      float dx = p.x - r.x, dy = p.y - r.y, dz = p.z - r.z;
      hd_min_image(dx, dy, dz, L);
      over |= sqrtf(dx * dx + dy * dy + dz * dz) + 1.7320508f * dl > a.half_skin;
    }
    nb_request_rebuild(a.status, over);
    if (over) s_over = 1;
  }
  __syncthreads();
  // one thread decides and every thread reads its decision, so the
  // barriers of the rebuild phases are reached by the whole workgroup
  if (t == 0) s_over = (s_over != 0 || nb_rebuild_due(a.status)) ? 1 : 0;
  __syncthreads();
  const bool rebuild = s_over != 0;
  if (rebuild) {
    if (t < 6) a.ref_lattice[t] = a.lattice[t];
    for (unsigned v = t; v < a.nvox; v += NB_SMALL_THREADS) cnt[v] = 0u;
    __syncthreads();
    for (unsigned i = t; i < a.n; i += NB_SMALL_THREADS) {
      float4 p = a.posq[i];
      a.ref_pos[i] = p;
      unsigned key = nb_voxel_key(p, L, a.voxel_rank, a.nv[0], a.nv[1], a.nv[2]);
      a.atom_key[i] = key;
      atomicAdd(&cnt[key], 1u);
    }
    __syncthreads();
    // exclusive scan: thread t owns voxels [t per, (t + 1) per)
    const unsigned per = (a.nvox + NB_SMALL_THREADS - 1u) / NB_SMALL_THREADS;
    const unsigned b0 = t * per;
    unsigned sum = 0u;
    for (unsigned k = 0; k < per; ++k)
      if (b0 + k < a.nvox) sum += cnt[b0 + k];
    scan[t] = sum;
    __syncthreads();
    for (unsigned off = 1; off < NB_SMALL_THREADS; off <<= 1) {
      unsigned u = t >= off ? scan[t - off] : 0u;
      __syncthreads();
      scan[t] += u;
      __syncthreads();
    }
    unsigned run = scan[t] - sum;
    for (unsigned k = 0; k < per; ++k) {
      unsigned v = b0 + k;
      if (v < a.nvox) {
        unsigned c = cnt[v];
        a.voxel_off[v] = run;
        cnt[v] = run;  // the scatter cursor
        run += c;
      }
    }
    if (t == NB_SMALL_THREADS - 1u) a.voxel_off[a.nvox] = scan[t];
    __syncthreads();
    for (unsigned i = t; i < a.n; i += NB_SMALL_THREADS)
      a.sorted_id[atomicAdd(&cnt[a.atom_key[i]], 1u)] = i;
    __syncthreads();
    for (unsigned v = t; v < a.nvox; v += NB_SMALL_THREADS)
      nb_sort_voxel(v, a.voxel_off, a.sorted_id, a.slot_of);
    __syncthreads();
  }
  if (a.n > NB_SMALL_GATHER) return;  // k_tile_gather follows
  // npad is a multiple of 64 and so is the stride: each wave covers whole
  // blocks in every pass
  for (unsigned s = t; s < a.npad; s += NB_SMALL_THREADS)
    nb_gather_slot(s, rebuild, a.posq, a.sorted_id, a.lattice, a.tile_posq, fpj, fpj_ew, a.n,
                   a.type, a.key, a.tile_type, a.tile_key, a.center, a.half, a.tile_ref, a.tile_img);
  if (spl) {
    // SPME spline records from the gathered positions (each thread reads
    // back the slots it wrote)
    for (unsigned s = t; s < a.n; s += NB_SMALL_THREADS)
      hd_spline_record(a.tile_posq[s], L, gna, gnb, gnc, spl, sg, s);
  }
}

bool hd_neighbor_small(const HdNeighborArgs& a) {
  return a.n <= NB_SMALL_ATOMS && a.nvox <= NB_SMALL_VOX;
}

void hd_launch_neighbor_small(hipStream_t st, const HdNeighborArgs& a, bool check, long long* fpj,
                              long long* fpj_ew, float4* spl, unsigned* sg, unsigned na,
                              unsigned nb, unsigned nc) {
  hipLaunchKernelGGL(k_nb_small, dim3(1), dim3(NB_SMALL_THREADS), 0, st, a, check ? 1 : 0, fpj,
                     fpj_ew, spl, sg, na, nb, nc);
  if (a.n > NB_SMALL_GATHER)
    hd_launch_tile_gather_rebuild(st, a, fpj, fpj_ew, spl, sg, na, nb, nc);
}

#define NB_CAND_MAX 1024

// The candidate j-blocks of block b in increasing order, from the chunk
// masks, into an LDS list (at most NB_CAND_MAX; *too_many flags more).
__device__ __forceinline__ unsigned nb_collect(const unsigned long long* __restrict__ mask,
                                               unsigned b, unsigned nchunks, unsigned lane,
                                               unsigned* cand, bool* too_many) {
  unsigned ncand = 0;
  for (unsigned c0 = 0; c0 < nchunks; c0 += 64) {
    unsigned c = c0 + lane;
    unsigned long long mk = c < nchunks ? mask[(size_t)b * nchunks + c] : 0ull;
    unsigned cnt = __popcll(mk);
    unsigned inc = cnt;
#pragma unroll
    for (unsigned off = 1; off < 64; off <<= 1) {
      unsigned v = __shfl_up(inc, off);
      if (lane >= off) inc += v;
    }
    unsigned base = ncand + inc - cnt;
    while (mk) {
      unsigned bit = __builtin_ctzll(mk);
      mk &= mk - 1;
      if (base < NB_CAND_MAX) cand[base] = c * 64 + bit;
      ++base;
    }
    ncand += __shfl(inc, 63);
  }
  __builtin_amdgcn_wave_barrier();
  if (ncand > NB_CAND_MAX) {
    *too_many = true;
    ncand = NB_CAND_MAX;
  }
  return ncand;
}

#define NB_WAVES 4  // waves (i-blocks) per workgroup of the atom-list build

// Row lists.  A unit is one part of one i-block's neighbourhood: the
// block's candidate (j-block, periodic image) pairs are dealt out to
// `parts` units in pieces of 8 atoms, so that small systems still fill the
// chip.  One workgroup of 8 waves per unit:
//   1. the candidates from the block-pair mask, each expanded into the
//      images (of -1, 0, 1 box vectors per axis) whose box lies within
//      r_search: with an image per j-atom the pair kernel needs no minimum
//      image, in narrow and tilted boxes too;
//   2. the j-atoms within r_search of the box of one of the block's 16-atom
//      quarters (of one of its atoms where the box is wide), in a fixed
//      order, to the unit's j-list and to LDS: those of Lennard-Jones-active
//      types from the front of the list, the others from its back;
//   3. rows: wave w owns i-atoms 8 w .. 8 w + 7, octet w (coordinates in
//      scalar registers), queues the j-atoms within r_search of the octet's
//      box and tests 64 of them at a time against each i-atom; the ballot of
//      the hits gives every hit its place in the row.  A row
//      holds the hits' LDS byte offsets (16 index) among the active
//      j-atoms, padded to a multiple of 32 entries common to the wave's 8
//      rows, then those among the others, padded alike; padding points to
//      a dummy record past the list.
// The pair kernel's lane 8 r + s reads entries 4 s .. 4 s + 3 of a 32-entry
// chunk of row r as one 8-byte load: 64 contiguous bytes per row.
// Bound by instruction issue (two 8-wave workgroups per CU; a unit's waves
// spend 55 % of their cycles listing j-atoms and 45 % on the rows): 79 us at
// 24,576 atoms and a 0.27 nm skin, 190 for the packed tiles' build; 294 us
// at 196,608 atoms and 0.14 nm beside the SPME kernels, where that took 170.
// The list is a pure function of the positions.
#define NB_PER_WAVE 2u
// Up to this many mask words per block (512 blocks, one pass over them) a
// unit tests every block's box itself: the mask's launch costs more than it
// saves there (24,576 atoms, a frame with its rebuild: 417 us, 440 with the
// mask; 10,000 argon atoms, a step: 29.5 and 31.7)
#define NB_MASK_CHUNKS 8u
#define NB_ROUND (HD_ROW_WAVES * NB_PER_WAVE)
#define NB_STAGE 96u         // entries of a row staged in LDS: a rest below 32 and 64 hits
#define NB_WORDS_MAX 512u    // mask words (64 blocks each) with candidates
#define NB_IMAGES_MAX 1024u  // images of 512 blocks listed at a time

__device__ __forceinline__ unsigned nb_scan512(unsigned v, unsigned* wsum, unsigned& total) {
  const unsigned lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
  unsigned inc = v;
#pragma unroll
  for (unsigned off = 1; off < 64; off <<= 1) {
    unsigned u = __shfl_up(inc, off);
    if (lane >= off) inc += u;
  }
  __syncthreads();  // wsum free for reuse
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  unsigned before = 0;
  total = 0;
#pragma unroll
  for (unsigned k = 0; k < HD_ROW_WAVES; ++k) {
    unsigned c = wsum[k];
    before += k < w ? c : 0u;
    total += c;
  }
  return before + inc - v;
}

// Images (bit = code) of j-block box (cj, hj) within r_search of the
// i-block's.  Orthorhombic: the images of each axis that are close enough
// along it, then (almost always one per axis) their combinations.
__device__ __forceinline__ unsigned nb_images(float4 ci, float4 hi, float4 cj, float4 hj,
                                              const HdLattice& L, float rs2) {
  const float dx = cj.x - ci.x, dy = cj.y - ci.y, dz = cj.z - ci.z;
  unsigned m = 0;
  if (L.xy == 0.f && L.xz == 0.f && L.yz == 0.f) {
    float ex[3], ey[3], ez[3];
    unsigned ok = 0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      ex[k] = fmaxf(fabsf(dx + (float)(k - 1) * L.lx) - (hi.x + hj.x), 0.f);
      ey[k] = fmaxf(fabsf(dy + (float)(k - 1) * L.ly) - (hi.y + hj.y), 0.f);
      ez[k] = fmaxf(fabsf(dz + (float)(k - 1) * L.lz) - (hi.z + hj.z), 0.f);
      ex[k] *= ex[k];
      ey[k] *= ey[k];
      ez[k] *= ez[k];
      ok |= (ex[k] <= rs2 ? 1u << k : 0u) | (ey[k] <= rs2 ? 8u << k : 0u) |
            (ez[k] <= rs2 ? 64u << k : 0u);
    }
    for (int c = 0; c < 3; ++c) {
      if (!((ok >> (6 + c)) & 1u)) continue;
      const float zc = c == 0 ? ez[0] : (c == 1 ? ez[1] : ez[2]);
      for (int b = 0; b < 3; ++b) {
        if (!((ok >> (3 + b)) & 1u)) continue;
        const float yz = zc + (b == 0 ? ey[0] : (b == 1 ? ey[1] : ey[2]));
#pragma unroll
        for (int a = 0; a < 3; ++a)
          if (ex[a] + yz <= rs2) m |= 1u << (a + 3 * b + 9 * c);
      }
    }
    return m;
  }
  unsigned code = 0;
  for (int c = -1; c <= 1; ++c)
    for (int b = -1; b <= 1; ++b)
      for (int a = -1; a <= 1; ++a, ++code) {
        float sx = dx + (float)a * L.lx + (float)b * L.xy + (float)c * L.xz;
        float sy = dy + (float)b * L.ly + (float)c * L.yz;
        float sz = dz + (float)c * L.lz;
        if (nb_box_gap2(sx, sy, sz, hi, hj) <= rs2) m |= 1u << code;
      }
  return m;
}

__global__ void __launch_bounds__(HD_ROW_THREADS, 4) k_build_rows(HdNeighborArgs a,
                                                                  unsigned nchunks) {
  if (!nb_rebuild_due_now(a.status)) return;
  extern __shared__ float4 jrec[];  // x, y, z relative to the block centre; key
  __shared__ unsigned words[NB_WORDS_MAX];
  __shared__ unsigned images[NB_IMAGES_MAX];  // j-block * 32 + image code
  __shared__ unsigned wsum[HD_ROW_WAVES];
  __shared__ unsigned wcnt[2][HD_ROW_WAVES];
  __shared__ unsigned s_cost, s_need;
  __shared__ float4 quart[4][2];  // centre, half; half.w: its atoms are tested one by one
  __shared__ float ipos[3][64];   // the block's atoms relative to its centre
  __shared__ unsigned short ring[HD_ROW_WAVES][128];
  __shared__ __align__(16) unsigned short stage[HD_ROW_WAVES][HD_ROW_I][NB_STAGE];
  const unsigned t = threadIdx.x, lane = t & 63u, w = t >> 6;
  const unsigned unit = blockIdx.x;
  const unsigned b = unit / a.parts, part = unit - b * a.parts;
  HdLattice L = hd_load_lattice(a.lattice);
  const float4 cb = a.center[b], hb = a.half[b];
  const float rs2 = a.rs2 * NB_BOX_MARGIN, rs2p = a.rs2 * NB_ROW_MARGIN;
  if (t == 0) s_cost = s_need = 0u;
  // 1. the mask words with candidates (few blocks have no mask: all of them)
  const bool all = nchunks <= NB_MASK_CHUNKS;
  unsigned nw = 0;
  for (unsigned base = 0; base < nchunks; base += HD_ROW_THREADS) {
    const unsigned c = base + t;
    const bool nz = c < nchunks && (all || a.block_mask[(size_t)b * nchunks + c] != 0ull);
    unsigned total;
    const unsigned o = nw + nb_scan512(nz ? 1u : 0u, wsum, total);
    if (nz && o < NB_WORDS_MAX) words[o] = c;
    nw += total;
  }
  bool too_many = nw > NB_WORDS_MAX;
  nw = min(nw, NB_WORDS_MAX);
  // boxes, relative to the block centre, of the block's 16-atom quarters
  // (which j-atoms to list) and of this wave's 8-atom octet (which of them
  // to test); lane = atom
  float4 oc, oh;
  {
    const unsigned islot = b * 64u + lane;
    float4 p = a.tile_posq[islot];
    hd_rel_image(p.x, p.y, p.z, cb, HD_IMAGE_NONE, HD_IMAGE_NONE, L, p.x, p.y, p.z);
    const bool v = islot < a.n;
    float lx = v ? p.x : 3.0e18f, ly = v ? p.y : 3.0e18f, lz = v ? p.z : 3.0e18f;
    float hx = v ? p.x : -3.0e18f, hy = v ? p.y : -3.0e18f, hz = v ? p.z : -3.0e18f;
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) {
      if (off == 8) {
        // octet w's box (no atoms: lo > hi, a negative half that nothing
        // reaches)
        const int src = (int)(w * 8u);
        const float ax = __shfl(lx, src), bx = __shfl(hx, src), ay = __shfl(ly, src),
                    by = __shfl(hy, src), az = __shfl(lz, src), bz = __shfl(hz, src);
        oc = make_float4(0.5f * (ax + bx), 0.5f * (ay + by), 0.5f * (az + bz), 0.f);
        oh = make_float4(0.5f * (bx - ax), 0.5f * (by - ay), 0.5f * (bz - az), 0.f);
      }
      lx = fminf(lx, __shfl_xor(lx, off)); hx = fmaxf(hx, __shfl_xor(hx, off));
      ly = fminf(ly, __shfl_xor(ly, off)); hy = fmaxf(hy, __shfl_xor(hy, off));
      lz = fminf(lz, __shfl_xor(lz, off)); hz = fmaxf(hz, __shfl_xor(hz, off));
    }
    if (w == 0) {
      ipos[0][lane] = v ? p.x : 3.0e18f;
      ipos[1][lane] = v ? p.y : 3.0e18f;
      ipos[2][lane] = v ? p.z : 3.0e18f;
      if ((lane & 15u) == 0u) {
        const float qx = 0.5f * (hx - lx), qy = 0.5f * (hy - ly), qz = 0.5f * (hz - lz);
        quart[lane >> 4][0] =
            make_float4(0.5f * (lx + hx), 0.5f * (ly + hy), 0.5f * (lz + hz), 0.f);
        // wide: half a diagonal beyond the search radius.  In a liquid no
        // quarter is (24,576 water atoms: 0 of 1,536); beside a void a
        // quarter of a few vapour atoms has a box that spans the liquid
        // (24,603 atoms in a slab: 24,196 j-atoms by the boxes, 2,920 so)
        quart[lane >> 4][1] = make_float4(
            qx, qy, qz, qx > 0.f && qx * qx + qy * qy + qz * qz > a.rs2 ? 1.f : 0.f);
      }
    }
  }
  __syncthreads();
  // 2. j-atoms.  Eight mask words at a time (thread = block): the candidate
  // blocks' images are listed, and the unit takes the 8-atom pieces
  // 8 e + (lane / 8) of the images e that are `part` modulo parts (a power
  // of two).  Rounds of 16 images, two per wave and the next two in flight;
  // the list keeps the images' order, active types from the front, the
  // others from the back.
  const unsigned pm = a.parts - 1u;
  unsigned nact = 0, nina = 0, e0 = 0, buf = 0;
  // the wide quarters (bit = quarter) and the limit of their pairs, whose
  // terms reach across the block
  const unsigned wide = (unsigned)__builtin_amdgcn_readfirstlane(
      (quart[0][1].w > 0.f ? 1 : 0) | (quart[1][1].w > 0.f ? 2 : 0) |
      (quart[2][1].w > 0.f ? 4 : 0) | (quart[3][1].w > 0.f ? 8 : 0));
  const float reach = sqrtf(rs2) + hb.x + hb.y + hb.z, rs2w = rs2 + 2.0e-6f * reach * reach;
  for (unsigned w0 = 0; w0 < nw; w0 += HD_ROW_WAVES) {
    unsigned total, m = 0, jb = 0;
    if (w0 + w < nw) {
      const unsigned c = words[w0 + w];
      jb = c * 64u + lane;
      if (all ? jb < a.npad / 64u : (a.block_mask[(size_t)b * nchunks + c] >> lane) & 1ull) {
        const float4 cj = a.center[jb], hj = a.half[jb];
        // without a mask its test comes first: most waves end there
        if (!all || nb_box_dist2(cb, hb, cj, hj, L) <= rs2) m = nb_images(cb, hb, cj, hj, L, rs2);
      }
    }
    const unsigned o0 = nb_scan512((unsigned)__popc(m), wsum, total);
    // almost always one pass: a block that spans a narrow box meets most
    // blocks in several images
    for (unsigned l0 = 0; l0 < total; l0 += NB_IMAGES_MAX) {
      const unsigned ne = min(total - l0, NB_IMAGES_MAX);
      unsigned o = o0 - l0;  // wraps before the pass
      for (unsigned k = m; k; k &= k - 1u, ++o)
        if (o < NB_IMAGES_MAX) images[o] = jb * 32u + (unsigned)__builtin_ctz(k);
      __syncthreads();  // after it every wave is done with the pass before
      float4 np[NB_PER_WAVE];
      unsigned nt[NB_PER_WAVE], nk[NB_PER_WAVE];
      auto load = [&](unsigned r0) {
#pragma unroll
        for (unsigned u = 0; u < NB_PER_WAVE; ++u) {
          const unsigned it = r0 + w * NB_PER_WAVE + u;
          // past the end: block 0, not used
          const unsigned sl = (it < ne ? images[it] >> 5 : 0u) * 64u + lane;  // < npad
          np[u] = a.tile_posq[sl];
          nt[u] = a.tile_type[sl];
          nk[u] = a.tile_key[sl];
        }
      };
      load(0u);
      for (unsigned r0 = 0; r0 < ne; r0 += NB_ROUND) {
        float4 p[NB_PER_WAVE];
        unsigned js[NB_PER_WAVE], ca = 0, ci = 0;
        unsigned long long ma[NB_PER_WAVE], mi[NB_PER_WAVE];
#pragma unroll
        for (unsigned u = 0; u < NB_PER_WAVE; ++u) {
          const unsigned it = r0 + w * NB_PER_WAVE + u;
          const unsigned img = it < ne ? images[it] : HD_IMAGE_NONE, slot = (img >> 5) * 64u + lane;
          hd_rel_image(np[u].x, np[u].y, np[u].z, cb, img & 31u, HD_IMAGE_NONE, L, p[u].x, p[u].y,
                       p[u].z);
          p[u].w = __uint_as_float(nk[u]);
          js[u] = slot | ((img & 31u) << HD_ROW_SLOT_BITS);
          unsigned hit = 0u;  // bit = quarter
#pragma unroll
          for (int o = 0; o < 4; ++o) {
            const float4 qc = quart[o][0], qh = quart[o][1];
            hit |= nb_box_gap2(p[u].x - qc.x, p[u].y - qc.y, p[u].z - qc.z, qh,
                               make_float4(0.f, 0.f, 0.f, 0.f)) <= rs2
                       ? 1u << o
                       : 0u;
          }
          if (wide && hit && !(hit & ~wide)) {
            float d2 = 3.0e38f;
            for (unsigned i = 0; i < 64u; ++i) {
              if (!((hit >> (i >> 4)) & 1u)) continue;
              const float dx = p[u].x - ipos[0][i], dy = p[u].y - ipos[1][i],
                          dz = p[u].z - ipos[2][i];
              d2 = fminf(d2, dx * dx + dy * dy + dz * dz);
            }
            hit = d2 <= rs2w ? hit : 0u;
          }
          bool near = hit != 0u;
          near = near && it < ne && slot < a.n && (((e0 + it) * 8u + (lane >> 3)) & pm) == part;
          const unsigned long long mn = __ballot(near),
                                   mt = __ballot((a.active_types >> nt[u]) & 1u);
          ma[u] = mn & mt;
          mi[u] = mn & ~mt;
          ca += (unsigned)__popcll(ma[u]);
          ci += (unsigned)__popcll(mi[u]);
        }
        load(r0 + NB_ROUND);
        if (lane == 0) wcnt[buf][w] = ca | (ci << 16);
        __syncthreads();  // two buffers: the next round's counts land elsewhere
        unsigned before = 0, all = 0;
#pragma unroll
        for (unsigned v = 0; v < HD_ROW_WAVES; ++v) {
          const unsigned cv = wcnt[buf][v];
          if (v < w) before += cv;
          all += cv;
        }
        buf ^= 1u;
        unsigned ja = nact + (before & 0xFFFFu), ji = nina + (before >> 16);
#pragma unroll
        for (unsigned u = 0; u < NB_PER_WAVE; ++u) {
          const bool act = __builtin_amdgcn_inverse_ballot_w64(ma[u]);
          if (__builtin_amdgcn_inverse_ballot_w64(ma[u] | mi[u])) {
            const unsigned k = act ? ja + hd_rank(ma[u]) : ji + hd_rank(mi[u]);
            if (k < a.jcap) {
              const unsigned o = act ? k : a.jcap - 1u - k;
              jrec[o] = p[u];
              a.jslot[(size_t)unit * a.jcap + o] = js[u];
            }
          }
          ja += (unsigned)__popcll(ma[u]);
          ji += (unsigned)__popcll(mi[u]);
        }
        nact += all & 0xFFFFu;
        nina += all >> 16;
      }
      e0 += ne;
    }
  }
  __syncthreads();
  const unsigned need_j = nact + nina;
  nact = min(nact, a.jcap);
  nina = min(nina, a.jcap - nact);  // less on overflow, flagged below
  // 3. rows
  const unsigned rcap = a.rcap;
  unsigned short* rows = a.rows + ((size_t)unit * 64u + w * HD_ROW_I) * rcap;
  const unsigned short dummy = (unsigned short)(a.jcap << 4);
  // r^2 <= rs^2 as j.(j - 2 i) <= rs^2 - i.i: three multiply-adds per pair.
  // The terms reach (r_search + half extent)^2, so the test is wider by
  // their rounding.
  float sx[HD_ROW_I], sy[HD_ROW_I], sz[HD_ROW_I], sr[HD_ROW_I];
  unsigned sk[HD_ROW_I], cnt[HD_ROW_I];
  {
    unsigned islot = b * 64u + w * HD_ROW_I + (lane & 7u);
    float4 p = a.tile_posq[islot];
    unsigned key = a.tile_key[islot];
    hd_rel_image(p.x, p.y, p.z, cb, HD_IMAGE_NONE, HD_IMAGE_NONE, L, p.x, p.y, p.z);
    // no j-atom is within reach of a slot without atom
    float lim = islot < a.n ? rs2p + 2.0e-6f * reach * reach - (p.x * p.x + p.y * p.y + p.z * p.z)
                            : -3.0e38f;
#pragma unroll
    for (int q = 0; q < HD_ROW_I; ++q) {
      sx[q] = -2.0f * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p.x), q));
      sy[q] = -2.0f * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p.y), q));
      sz[q] = -2.0f * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p.z), q));
      sr[q] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(lim), q));
      sk[q] = (unsigned)__builtin_amdgcn_readlane((int)key, q);
      cnt[q] = 0u;
    }
  }
  unsigned done = 0;  // entries of every row so far (a multiple of 32)
  unsigned nact_chunks = 0;
  // the j-atoms near this wave's octet are queued, and tested 64 at a time
  // (lane = queue position) against its 8 i-atoms
  unsigned short* queue = ring[w];
  unsigned short(*st)[NB_STAGE] = stage[w];
  const unsigned fq = lane >> 3, fs = (lane & 7u) * 4u;  // row and entries of the lane's stores
  unsigned short* frow = rows + fq * rcap + fs;
  // Hits are staged in LDS behind the row's rest (cnt mod 32 entries) and
  // leave in whole chunks of 32, eight lanes of 8 bytes per row: storing
  // each hit by itself, a 2-byte store per lane, took as long as all the
  // rest of the build together.
  auto flush = [&](unsigned before, unsigned pops) {
    // lane q < 8: row q's entries before the group, and those added
    const unsigned c0 = __shfl(before, fq), add = __shfl(pops, fq);
    const unsigned rest = c0 & (HD_ROW_CHUNK - 1u), nf = (rest + add) / HD_ROW_CHUNK;
    const unsigned base = c0 - rest;
    hd_wave_sync();
#pragma unroll
    for (unsigned c = 0; c < 2; ++c)
      if (c < nf && base + c * HD_ROW_CHUNK < rcap)
        *reinterpret_cast<hd_u32x2*>(frow + base + c * HD_ROW_CHUNK) =
            *reinterpret_cast<const hd_u32x2*>(&st[fq][c * HD_ROW_CHUNK + fs]);
    hd_u32x2 tail = {0u, 0u};
    if (nf) tail = *reinterpret_cast<const hd_u32x2*>(&st[fq][nf * HD_ROW_CHUNK + fs]);
    hd_wave_sync();
    if (nf) *reinterpret_cast<hd_u32x2*>(&st[fq][fs]) = tail;
    hd_wave_sync();
  };
  unsigned cntv = 0u;  // lane q < 8: row q's entries
  auto test = [&](unsigned nq) {
    const bool kv = lane < nq;
    const unsigned k = queue[kv ? lane : 0u];  // idle lanes: a written record, too far off below
    const float4 r = jrec[k];
    const float j2 = kv ? r.x * r.x + r.y * r.y + r.z * r.z : 3.0e38f;
    const unsigned jkey = __float_as_uint(r.w);
    const unsigned before = cntv;
    unsigned pops = 0u;
#pragma unroll
    for (int q = 0; q < HD_ROW_I; ++q) {
      const float d = fmaf(r.x, sx[q], fmaf(r.y, sy[q], fmaf(r.z, sz[q], j2)));
      const unsigned long long m =
          __ballot(d <= sr[q]) & __ballot((jkey - sk[q] + a.excl_span) > 2u * a.excl_span);
      if (__builtin_amdgcn_inverse_ballot_w64(m))
        st[q][(cnt[q] & (HD_ROW_CHUNK - 1u)) + hd_rank(m)] = (unsigned short)(k << 4);
      const unsigned add = (unsigned)__popcll(m);
      pops = lane == (unsigned)q ? add : pops;
      cnt[q] += add;
    }
    cntv += pops;
    flush(before, pops);
  };
  for (int seg = 0; seg < 2; ++seg) {
    const unsigned nk = seg ? nina : nact;
    unsigned nq = 0;
    for (unsigned k0 = 0; k0 < nk; k0 += 64u) {
      const unsigned k = k0 + lane, o = seg ? a.jcap - 1u - k : k;
      bool near = false;
      if (k < nk) {
        const float4 p = jrec[o];
        near = nb_box_gap2(p.x - oc.x, p.y - oc.y, p.z - oc.z, oh,
                           make_float4(0.f, 0.f, 0.f, 0.f)) <= rs2;
      }
      const unsigned long long m = __ballot(near);
      if (near) queue[nq + hd_rank(m)] = (unsigned short)o;
      nq += (unsigned)__popcll(m);
      hd_wave_sync();
      if (nq >= 64u) {
        test(64u);
        const unsigned short rest = queue[64u + lane];
        hd_wave_sync();
        nq -= 64u;
        if (lane < nq) queue[lane] = rest;
        hd_wave_sync();
      }
    }
    if (nq) test(nq);
    unsigned mx = 0;
#pragma unroll
    for (int q = 0; q < HD_ROW_I; ++q) mx = max(mx, cnt[q]);
    done = max(done, (mx + HD_ROW_CHUNK - 1u) / HD_ROW_CHUNK * HD_ROW_CHUNK);
    // the rows' rests padded to a chunk, then whole chunks of padding
    {
      const unsigned before = cntv;
      cntv = done;
#pragma unroll
      for (int q = 0; q < HD_ROW_I; ++q) {
        const unsigned rest = cnt[q] & (HD_ROW_CHUNK - 1u);
        if (lane >= rest && lane < HD_ROW_CHUNK) st[q][lane] = dummy;
        cnt[q] = done;
      }
      hd_wave_sync();
      const unsigned c0 = __shfl(before, fq), rest = c0 & (HD_ROW_CHUNK - 1u);
      unsigned base = c0 - rest;
      if (rest && base < rcap)
        *reinterpret_cast<hd_u32x2*>(frow + base) = *reinterpret_cast<const hd_u32x2*>(&st[fq][fs]);
      base += rest ? HD_ROW_CHUNK : 0u;
      const unsigned d2 = (unsigned)dummy * 0x10001u;
      for (; base < min(done, rcap); base += HD_ROW_CHUNK)
        *reinterpret_cast<hd_u32x2*>(frow + base) = hd_u32x2{d2, d2};
      hd_wave_sync();
    }
    if (seg == 0) nact_chunks = done / HD_ROW_CHUNK;
  }
  const unsigned cap_chunks = a.rcap / HD_ROW_CHUNK;
  const unsigned nchunk = done / HD_ROW_CHUNK;
  if (lane == 0) {
    a.rowhdr[unit * HD_ROW_WAVES + w] =
        min(nact_chunks, cap_chunks) | (min(nchunk, cap_chunks) << 16);
    atomicAdd(&s_cost, nchunk);
    atomicMax(&s_need, done);
  }
  __syncthreads();
  if (t == 0) {
    a.entry_count[unit] = s_cost;
    a.jcount[unit] = nact | (nina << 16);
    // global maxima: device atomics on one word queue up (about 20 ns each,
    // a millisecond for every wave of a large system), so a unit reads the
    // word first and only raises it
    const unsigned need_r = s_need;
    if (need_r > *(volatile unsigned*)a.max_count) atomicMax(a.max_count, need_r);
    if (need_j > *(volatile unsigned*)a.max_j) atomicMax(a.max_j, need_j);
    unsigned bits = 0u;
    if (need_r > rcap || need_j > a.jcap || too_many) bits = NB_STATUS_OVERFLOW;
    else if (4u * need_r > 3u * rcap || need_j > a.jmark) bits = NB_STATUS_HIGHWATER;
    if (bits & ~*(volatile unsigned*)a.status) atomicOr(a.status, bits);
  }
}

// Per-atom full lists (the atom-list mode): one wave per i-block, lane =
// i-atom.  The wave reads its candidate j-blocks (every j-block whose box
// lies within r_search, not only j >= i) into an LDS list, then stages the
// candidates' atoms in LDS one block at a time, loading the next block
// while it tests the current one.  Each lane appends the j-atoms within
// r_search of its own atom that are neither itself nor excluded by the key
// rule.  Row k of block b holds the k-th neighbour of every lane
// (column-major, so the pair kernel's index loads are coalesced); rows past
// a lane's count up to the block's longest list hold HD_SENTINEL.  Each
// pair appears once in each atom's list, so the pair kernel needs no j-side
// accumulation.  The order is j-block by j-block, then j-slot: the lists
// are a pure function of the positions.

__device__ __forceinline__ void alist_stage(const float4* __restrict__ tile_posq,
                                            const unsigned* __restrict__ tile_key, unsigned jb,
                                            unsigned lane, unsigned n, float4& p, unsigned& key) {
  unsigned jslot = jb * 64 + lane;
  bool jvalid = jslot < n;
  p = tile_posq[jvalid ? jslot : 0u];
  key = jvalid ? tile_key[jslot] : 0u;
}

__global__ void __launch_bounds__(256) k_build_alist(
    const float4* __restrict__ tile_posq, const unsigned* __restrict__ tile_key,
    unsigned excl_span, const float4* __restrict__ center, const float4* __restrict__ half,
    const float* __restrict__ lattice, float rs2, const unsigned long long* __restrict__ mask,
    unsigned nchunks, unsigned* __restrict__ rows_out, unsigned* __restrict__ row_count,
    unsigned cap, unsigned* __restrict__ max_count, unsigned* status, unsigned n,
    unsigned nblocks) {
  if (!nb_rebuild_due(status)) return;
  __shared__ float4 jpos[NB_WAVES][64];
  __shared__ unsigned jkey[NB_WAVES][64];
  __shared__ unsigned cand[NB_WAVES][NB_CAND_MAX];
  unsigned w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  unsigned b = blockIdx.x * NB_WAVES + w;
  if (b >= nblocks) return;
  HdLattice L = hd_load_lattice(lattice);
  unsigned islot = b * 64 + lane;
  bool ivalid = islot < n;
  float4 pi = tile_posq[ivalid ? islot : 0u];
  unsigned ikey = ivalid ? tile_key[islot] : 0u;
  float4 cb = center[b], hb = half[b];
  float rsearch = sqrtf(rs2);
  // far from every periodic boundary (orthorhombic box): i and j relative
  // to the block centre, the periodic shift applied once per staged atom
  bool rel = (L.xy == 0.f && L.xz == 0.f && L.yz == 0.f) && (0.5f * L.lx - hb.x >= rsearch) &&
             (0.5f * L.ly - hb.y >= rsearch) && (0.5f * L.lz - hb.z >= rsearch);
  float ix = pi.x, iy = pi.y, iz = pi.z;
  if (rel) hd_rel_to_center(pi.x, pi.y, pi.z, cb.x, cb.y, cb.z, L, ix, iy, iz);
  bool too_many = false;
  unsigned ncand = nb_collect(mask, b, nchunks, lane, cand[w], &too_many);
  const double ilx = 1.0 / (double)L.lx, ily = 1.0 / (double)L.ly, ilz = 1.0 / (double)L.lz;
  unsigned cnt = 0;
  unsigned* out = rows_out + (size_t)b * cap * 64;
  float4 pn = make_float4(0.f, 0.f, 0.f, 0.f);
  unsigned kn = 0;
  if (ncand) alist_stage(tile_posq, tile_key, cand[w][0], lane, n, pn, kn);
  for (unsigned c = 0; c < ncand; ++c) {
    unsigned jb = cand[w][c];
    float4 pj = pn;
    if (rel) {
      float jx, jy, jz;
      hd_rel_to_center_rcp(pj.x, pj.y, pj.z, cb.x, cb.y, cb.z, L, ilx, ily, ilz, jx, jy, jz);
      pj.x = jx; pj.y = jy; pj.z = jz;
    }
    jpos[w][lane] = pj;
    jkey[w][lane] = kn;
    __builtin_amdgcn_wave_barrier();
    if (c + 1 < ncand) alist_stage(tile_posq, tile_key, cand[w][c + 1], lane, n, pn, kn);
    unsigned nj = min(64u, n - jb * 64);
    if (ivalid) {
#pragma unroll 8
      for (unsigned m = 0; m < 64; ++m) {
        float4 a = jpos[w][m];
        float dx = ix - a.x, dy = iy - a.y, dz = iz - a.z;
        if (!rel) hd_min_image(dx, dy, dz, L);
        float r2 = dx * dx + dy * dy + dz * dz;
        unsigned js = jb * 64 + m;
        bool ok = (jkey[w][m] - ikey + excl_span) > 2u * excl_span;
        if (r2 <= rs2 && ok && js != islot && m < nj) {
          if (cnt < cap) out[(size_t)cnt * 64 + lane] = js;
          ++cnt;
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  unsigned mx = cnt;
  for (int off = 32; off > 0; off >>= 1) mx = max(mx, (unsigned)__shfl_xor((int)mx, off));
  unsigned rows = min(mx, cap);
  for (unsigned k = cnt; k < rows; ++k) out[(size_t)k * 64 + lane] = HD_SENTINEL;
  if (lane == 0) {
    row_count[b] = rows;
    atomicMax(max_count, mx);
    if (mx > cap || too_many) atomicOr(status, NB_STATUS_OVERFLOW);
    else if (4 * mx > 3 * cap) atomicOr(status, NB_STATUS_HIGHWATER);
  }
}

// End of a rebuild: remember the reference positions and clear the
// rebuild request bits (sticky overflow/high-water bits stay for the host).

// Clears the rebuild request and, on rebuild steps, orders the pair
// kernel's work units (blocks in the atom-list mode, whose kernel takes them
// in index order) by row chunks, heaviest first: unit costs vary about
// twofold, and a heavy unit dispatched last runs alone at the end of the
// launch.  One workgroup: a histogram of the counts, suffix
// sums, a scatter (the order among equal counts is arbitrary; the forces do
// not depend on it, their sums being integer).
#define NB_ORDER_BINS 1024u
__global__ void __launch_bounds__(NB_ORDER_BINS) k_rebuild_clear(
    unsigned* status, unsigned* rebuild_count, const unsigned* __restrict__ entry_count,
    unsigned nblocks, unsigned* __restrict__ order) {
  __shared__ unsigned hist[NB_ORDER_BINS], cur[NB_ORDER_BINS];
  unsigned s = *status;  // read by every thread before thread 0 rewrites it
  if (!(s & (NB_STATUS_REBUILD | NB_STATUS_FORCE))) return;
  unsigned t = threadIdx.x;
  hist[t] = 0u;
  __syncthreads();
  for (unsigned i = t; i < nblocks; i += NB_ORDER_BINS)
    atomicAdd(&hist[min(entry_count[i], NB_ORDER_BINS - 1u)], 1u);
  __syncthreads();
  // hist[c] <- number of blocks whose count is >= c
  for (unsigned d = 1; d < NB_ORDER_BINS; d <<= 1) {
    unsigned v = (t + d < NB_ORDER_BINS) ? hist[t + d] : 0u;
    __syncthreads();
    hist[t] += v;
    __syncthreads();
  }
  // the blocks with count c take positions [hist[c + 1], hist[c])
  cur[t] = (t + 1 < NB_ORDER_BINS) ? hist[t + 1] : 0u;
  __syncthreads();
  for (unsigned i = t; i < nblocks; i += NB_ORDER_BINS) {
    unsigned pos = atomicAdd(&cur[min(entry_count[i], NB_ORDER_BINS - 1u)], 1u);
    order[pos] = i;
  }
  if (t == 0) {
    *status = s & ~(NB_STATUS_REBUILD | NB_STATUS_FORCE);
    *rebuild_count += 1u;
  }
}

// ---------------------------------------------------------------------
// Host launch wrappers
// ---------------------------------------------------------------------
static inline unsigned cdiv(unsigned a, unsigned b) { return (a + b - 1) / b; }

unsigned hd_voxel_scan_parts(unsigned nvox) { return cdiv(nvox, NB_SCAN_CHUNK); }

// Kernels gated by the rebuild flag run grid-stride loops over a modest grid
// (NB_GATED_WGS workgroups): on the steps where the gate closes them they
// retire quickly, and on rebuild steps the loops cover the work.
#define NB_GATED_WGS 512u

void hd_launch_disp_check(hipStream_t st, const HdNeighborArgs& a) {
  const unsigned T = 256;
  hipLaunchKernelGGL(k_disp_check, dim3(cdiv(a.n, T) ? cdiv(a.n, T) : 1), dim3(T), 0, st,
                     a.posq, a.ref_pos, a.lattice, a.ref_lattice, a.half_skin, a.status, a.n);
}

void hd_launch_neighbor_update(hipStream_t st, const HdNeighborArgs& a, bool check) {
  const unsigned T = 256;
  unsigned gridN = min(cdiv(a.n, T), NB_GATED_WGS);
  if (gridN == 0) gridN = 1;
  if (check)
    hipLaunchKernelGGL(k_disp_check, dim3(cdiv(a.n, T) ? cdiv(a.n, T) : 1), dim3(T), 0, st,
                       a.posq, a.ref_pos, a.lattice, a.ref_lattice, a.half_skin, a.status, a.n);
  hipLaunchKernelGGL(k_voxel_keys, dim3(gridN), dim3(T), 0, st, a.posq, a.lattice, a.voxel_rank,
                     a.nv[0], a.nv[1], a.nv[2], a.atom_key, a.voxel_count, a.ref_pos,
                     a.ref_lattice, a.status, a.n);
  unsigned nparts = hd_voxel_scan_parts(a.nvox);
  hipLaunchKernelGGL(k_voxel_scan_reduce, dim3(nparts), dim3(256), 0, st, a.voxel_count,
                     a.voxel_part, a.status, a.nvox);
  if (nparts > NB_SCAN_FUSED_MAX)
    hipLaunchKernelGGL(k_voxel_scan_parts, dim3(1), dim3(1024), 0, st, a.voxel_part, a.status,
                       nparts);
  hipLaunchKernelGGL(k_voxel_scan_apply, dim3(nparts), dim3(256), 0, st, a.voxel_count,
                     a.voxel_part, a.voxel_off, a.voxel_cursor, a.status, a.nvox, nparts);
  hipLaunchKernelGGL(k_voxel_scatter, dim3(gridN), dim3(T), 0, st, a.atom_key, a.voxel_off,
                     a.voxel_cursor, a.sorted_id, a.status, a.n);
  unsigned gridV = min(cdiv(a.nvox, T), NB_GATED_WGS);
  hipLaunchKernelGGL(k_voxel_sort, dim3(gridV), dim3(T), 0, st, a.voxel_off, a.voxel_count,
                     a.sorted_id, a.slot_of, a.status, a.nvox);
}

void hd_launch_tile_gather(hipStream_t st, const float4* posq, const unsigned* sorted_id,
                           const float* lattice, float4* tile_posq, long long* fpj,
                           long long* fpj_ew, unsigned n, unsigned npad, float4* tile_ref,
                           unsigned char* tile_img) {
  hipLaunchKernelGGL(k_tile_gather, dim3(cdiv(npad, 256)), dim3(256), 0, st, posq, sorted_id,
                     lattice, tile_posq, fpj, fpj_ew, n, npad, nullptr, nullptr, nullptr,
                     nullptr, nullptr, nullptr, nullptr, tile_ref, tile_img, nullptr, nullptr,
                     0u, 0u, 0u);
}

void hd_launch_tile_gather_rebuild(hipStream_t st, const HdNeighborArgs& a, long long* fpj,
                                   long long* fpj_ew, float4* spl, unsigned* sg, unsigned na,
                                   unsigned nb, unsigned nc) {
  hipLaunchKernelGGL(k_tile_gather, dim3(cdiv(a.npad, 256)), dim3(256), 0, st, a.posq,
                     a.sorted_id, a.lattice, a.tile_posq, fpj, fpj_ew, a.n, a.npad, a.status,
                     a.type, a.key, a.tile_type, a.tile_key, a.center, a.half, a.tile_ref,
                     a.tile_img, spl, sg, na, nb, nc);
}

unsigned hd_block_pair_chunks(unsigned nblocks) { return cdiv(nblocks, 64); }

void hd_launch_neighbor_build(hipStream_t st, const HdNeighborArgs& a, bool clear) {
  unsigned nblocks = a.npad / 64;
  const unsigned units = a.atom_lists ? nblocks : nblocks * a.parts;
  const size_t lds = (size_t)a.jcap * sizeof(float4);
  unsigned nchunks = hd_block_pair_chunks(nblocks);
  unsigned pair_waves = min(nblocks * nchunks, (unsigned)NB_PAIR_WAVES);
  if (a.atom_lists || nchunks > NB_MASK_CHUNKS)
    hipLaunchKernelGGL(k_block_pairs, dim3(cdiv(pair_waves * 64, 256)), dim3(256), 0, st,
                       a.center, a.half, a.lattice, a.rs2 * NB_BOX_MARGIN, a.block_mask, nblocks,
                       nchunks, a.status);
  if (a.atom_lists)
    hipLaunchKernelGGL(k_build_alist, dim3(cdiv(nblocks, NB_WAVES)), dim3(64 * NB_WAVES), 0, st,
                       a.tile_posq, a.tile_key, a.excl_span, a.center, a.half, a.lattice, a.rs2,
                       a.block_mask, nchunks, a.entry_atoms, a.entry_count, a.cap, a.max_count,
                       a.status, a.n, nblocks);
  else
    hipLaunchKernelGGL(k_build_rows, dim3(units), dim3(HD_ROW_THREADS), lds, st, a, nchunks);
  if (clear)
    hipLaunchKernelGGL(k_rebuild_clear, dim3(1), dim3(NB_ORDER_BINS), 0, st, a.status,
                       a.rebuild_count, a.entry_count, units, a.block_order);
}
