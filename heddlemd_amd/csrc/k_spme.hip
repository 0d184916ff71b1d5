// SPME reciprocal space on gfx950: charge spread, an own 3D real FFT in
// LDS, the influence-function multiply with its virial/energy reduction,
// and the force gather.
//
// Reference pipeline (src/forces/spme.rs:403-502):
//   influence (kernels/spme_recip.cu:34-115) -> spread, i64 fixed point at
//   2^32 with round-to-nearest (kernels/spme_spread_gather.cuh:151-221) ->
//   f32 conversion (spme_recip.cu:237-253) -> cuFFT R2C -> influence
//   multiply + per-block virial tree (spme_recip.cu:296-342) -> cuFFT C2R
//   -> reduce (spme_recip.cu:376-403) -> gather (spme_spread_gather.cuh:
//   223-334).
// MI355X design:
//   * no cuFFT/rocFFT: R2C along c (packed half-length complex FFT + post
//     twiddle), then b, then a, all radix-2 in LDS with per-axis twiddle
//     tables;
//   * the a-axis pass fuses forward FFT, influence multiply (G(k) and the
//     virial factor are evaluated in registers from the live lattice, so no
//     G/vf arrays are stored or re-read), the energy/virial partial sums in
//     FP64 and the inverse a-axis FFT: one read and one write of the
//     complex grid instead of five;
//   * the c-axis forward pass reads the i64 spread grid directly (the
//     fixed-point -> f32 conversion is fused);
//   * the gather is fused into the force finalize kernel (k_integrate.hip).
#include "hd_device.h"
#include "hd_kernels.h"

#define FFT_THREADS 256
#define FFT_TILE 2048  // complex elements staged per workgroup

// Cardinal B-spline by Cox-de Boor at order P (spme_spread_gather.cuh:36-54);
// the spread and the gather are built for P = 4 and 5.
template <int P>
__device__ __forceinline__ float bspline_w(float x) {
  float v[P];
#pragma unroll
  for (int i = 0; i < P; ++i) {
    float xi = x - (float)i;
    v[i] = (xi >= 0.f && xi < 1.f) ? 1.f : 0.f;
  }
#pragma unroll
  for (int order = 2; order <= P; ++order) {
    float inv = 1.0f / (float)(order - 1);
#pragma unroll
    for (int i = 0; i < P - order + 1; ++i) {
      float xi = x - (float)i;
      v[i] = xi * inv * v[i] + ((float)order - xi) * inv * v[i + 1];
    }
  }
  return v[0];
}

// Spline records, once per step in slot order, written with the tile gather
// (k_neighbor.hip): the FP64 spline origin (hd_spline_origin) of every
// charged atom, as (t_a, t_b, t_c, q) plus the packed origin cell
// g_a | g_b << 10 | g_c << 20 (SPME_NO_CELL for uncharged atoms).  Read by
// the spread and by the force gather.
#define SPME_NO_CELL HD_SPME_NO_CELL

// Spread: the reference accumulates each atom's p^3 contributions with
// i64 atomics at 2^32, rounded to nearest (spme_spread_gather.cuh:151-221).
// Here every workgroup owns one brick of grid cells and computes it
// completely: it gathers the atoms of the neighbour list's voxels that can
// reach the brick, adds their in-brick contributions into LDS with 64-bit
// LDS atomics, and stores the brick with plain coalesced stores.  No global
// atomics (device-scope atomics on MI355X are resolved past the per-XCD L2)
// and no clearing pass.  The per-cell values are the same integers in any
// order, so the grid equals per-atom global accumulation bit for bit.
//
// Which atoms can reach a brick: cells [c0, c1) receive contributions from
// atoms whose origin cell lies in [c0, c1 + p - 1), i.e. whose fractional
// coordinate (+1/2) lies in [c0/n, (c1 + p - 1)/n).  Atoms sit in the voxel
// they were binned into at the last rebuild, and have moved less than half
// the skin since (the rebuild criterion), so the window is widened by that
// distance in voxel units on each side.  The voxels shrink and grow with the
// box, whose present lattice is read here: a captured step goes on while a
// barostat scales it.
//
// The work of a brick is a chain of dependent loads (voxel -> slots ->
// origin cells -> records), so every stage is spread over all threads: the
// window's slots are listed, the ones that touch the brick are collected,
// their 3 p weights are evaluated one per thread into LDS, and a thread adds
// one c-layer of one atom (p lanes of an atom on neighbouring cells).
// Measured, us per launch (one atom per thread on bricks of 2,048 cells,
// before): 267 atoms, 32^3 cells 6.2 (16); 7,938 atoms, 40^3 8.9 (25);
// 24,576 atoms, 64^3 12 (33); 196,608 atoms, 128^3 43 (46) beside the pair kernel, bound by
// the LDS atomics of the atoms that several bricks visit.
#define SPREAD_THREADS 512
#define SPREAD_BRICK_MAX 1024   // cells per brick (8 KiB of i64)
#define SPREAD_VOX 2            // voxels of a window per thread at a time
#define SPREAD_LIST 2048u       // window atoms listed at a time
#define SPREAD_HITS 256u        // atoms whose weights are in LDS at a time

// round(x) as i64 for an integer-valued or rounded f32 x, the value
// __float2ll_rn gives: one conversion through i32 when |x| < 2^31 (every
// contribution below 0.5 e at the 2^32 scale), the general conversion
// otherwise.
__device__ __forceinline__ long long spread_fixed(float x) {
  float r = rintf(x);
  if (fabsf(r) < 2147483648.0f) return (long long)(int)r;
  return __float2ll_rn(r);
}

template <int SPME_P>
__global__ void __launch_bounds__(SPREAD_THREADS) k_spread(
    const float4* __restrict__ spl, const unsigned* __restrict__ sg, unsigned na, unsigned nb,
    unsigned nc, unsigned ba, unsigned bb, unsigned bc, const unsigned* __restrict__ voxel_rank,
    const unsigned* __restrict__ voxel_off, unsigned nva, unsigned nvb, unsigned nvc,
    const float* __restrict__ lattice, float reach, unsigned long long* __restrict__ rho) {
  __shared__ unsigned long long acc[SPREAD_BRICK_MAX];
  __shared__ unsigned list[SPREAD_LIST];
  __shared__ uint2 hits[SPREAD_LIST];  // slot; first stencil cell per axis, 8 bits each
  __shared__ float wgt[SPREAD_HITS * 3 * SPME_P];
  __shared__ unsigned wsum[SPREAD_THREADS / 64];
  __shared__ unsigned nhit;
  const unsigned t = threadIdx.x, lane = t & 63u, w = t >> 6;
  const unsigned nbb = nb / bb, nbc = nc / bc;
  const unsigned bi = blockIdx.x;
  const unsigned bic = bi % nbc, bib = (bi / nbc) % nbb, bia = bi / (nbc * nbb);
  const int c0a = (int)(bia * ba), c0b = (int)(bib * bb), c0c = (int)(bic * bc);
  const unsigned vol = ba * bb * bc;
  for (unsigned k = t; k < vol; k += SPREAD_THREADS) acc[k] = 0ull;
  // the reach along the axes' fractional coordinates, in voxels, and 1/64 of
  // one for the binning's rounding
  const HdLattice L = hd_load_lattice(lattice);
  const float ia = 1.0f / L.lx, ib = 1.0f / L.ly, ic = 1.0f / L.lz;
  const float ab = L.xy * ia * ib, ac = (L.xy * L.yz - L.xz * L.ly) * ia * ib * ic,
              bc_ = L.yz * ib * ic;
  const float mva = reach * (float)nva * sqrtf(ia * ia + ab * ab + ac * ac) + 0.015625f,
              mvb = reach * (float)nvb * sqrtf(ib * ib + bc_ * bc_) + 0.015625f,
              mvc = reach * (float)nvc * ic + 0.015625f;
  // voxel window per axis (periodic), at most one full period
  auto low = [](int c, unsigned nv, unsigned n, float m) {
    return (int)floorf((float)c * (float)nv / (float)n - m);
  };
  const int vla = low(c0a, nva, na, mva), vlb = low(c0b, nvb, nb, mvb), vlc = low(c0c, nvc, nc, mvc);
  const unsigned wa_n = (unsigned)min(low(c0a + (int)ba + SPME_P - 1, nva, na, -mva) - vla + 1, (int)nva);
  const unsigned wb_n = (unsigned)min(low(c0b + (int)bb + SPME_P - 1, nvb, nb, -mvb) - vlb + 1, (int)nvb);
  const unsigned wc_n = (unsigned)min(low(c0c + (int)bc + SPME_P - 1, nvc, nc, -mvc) - vlc + 1, (int)nvc);
  const unsigned nwin = wa_n * wb_n * wc_n;
  for (unsigned v0 = 0; v0 < nwin; v0 += SPREAD_VOX * SPREAD_THREADS) {
    // the slot ranges of the thread's voxels and their places in the list
    unsigned s0[SPREAD_VOX], cnt[SPREAD_VOX], my = 0;
#pragma unroll
    for (unsigned j = 0; j < SPREAD_VOX; ++j) {
      const unsigned k = v0 + j * SPREAD_THREADS + t;
      s0[j] = cnt[j] = 0u;
      if (k < nwin) {
        const unsigned kc = k % wc_n, kab = k / wc_n;
        const unsigned kb = kab % wb_n, ka = kab / wb_n;
        // periodic wrap; the voxel grid sides are powers of two
        const unsigned va = (unsigned)((vla + (int)ka) & ((int)nva - 1));
        const unsigned vb = (unsigned)((vlb + (int)kb) & ((int)nvb - 1));
        const unsigned vc = (unsigned)((vlc + (int)kc) & ((int)nvc - 1));
        const unsigned r = voxel_rank[(va * nvb + vb) * nvc + vc];
        s0[j] = voxel_off[r];
        cnt[j] = voxel_off[r + 1] - s0[j];
      }
    }
#pragma unroll
    for (unsigned j = 0; j < SPREAD_VOX; ++j) my += cnt[j];
    unsigned inc = my;
#pragma unroll
    for (unsigned off = 1; off < 64; off <<= 1) {
      const unsigned u = __shfl_up(inc, off);
      if (lane >= off) inc += u;
    }
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    unsigned run = inc - my, total = 0;
#pragma unroll
    for (unsigned k = 0; k < SPREAD_THREADS / 64; ++k) {
      const unsigned c = wsum[k];
      run += k < w ? c : 0u;
      total += c;
    }
    for (unsigned l0 = 0; l0 < total; l0 += SPREAD_LIST) {
      const unsigned nl = min(total - l0, SPREAD_LIST);
      unsigned o = run - l0;  // place of the thread's next atom; wraps before the chunk
#pragma unroll
      for (unsigned j = 0; j < SPREAD_VOX; ++j)
        for (unsigned i = 0; i < cnt[j]; ++i, ++o)
          if (o < nl) list[o] = s0[j] + i;
      if (t == 0) nhit = 0u;
      __syncthreads();
      for (unsigned k = t; k < nl; k += SPREAD_THREADS) {
        const unsigned s = list[k], g = sg[s];
        // brick-relative index of the stencil's first cell per axis; cell
        // (g - d) mod n lies in the brick when 0 <= rel - d < extent (g and
        // the brick origin both lie in [0, n), so one conditional add is
        // mod n); where the brick fills a small axis the stencil comes round
        // to it again, which the conditional adds below take in
        int rla = (int)(g & 1023u) - c0a, rlb = (int)((g >> 10) & 1023u) - c0b,
            rlc = (int)(g >> 20) - c0c;
        rla += rla < 0 ? (int)na : 0;
        rlb += rlb < 0 ? (int)nb : 0;
        rlc += rlc < 0 ? (int)nc : 0;
        const bool hit = g != SPME_NO_CELL && rla < (int)ba + SPME_P - 1 &&
                         rlb < (int)bb + SPME_P - 1 && rlc < (int)bc + SPME_P - 1;
        const unsigned long long m = __ballot(hit);
        if (hit) {
          const unsigned rank = hd_rank(m);
          unsigned base = 0;
          if (rank == 0u) base = atomicAdd(&nhit, (unsigned)__popcll(m));
          base = (unsigned)__builtin_amdgcn_readlane((int)base, (int)__builtin_ctzll(m));
          hits[base + rank] =
              make_uint2(s, (unsigned)rla | ((unsigned)rlb << 8) | ((unsigned)rlc << 16));
        }
      }
      __syncthreads();
      const unsigned nh = nhit;
      for (unsigned h0 = 0; h0 < nh; h0 += SPREAD_HITS) {
        const unsigned nr = min(nh - h0, SPREAD_HITS);
        for (unsigned k = t; k < nr * 3u * SPME_P; k += SPREAD_THREADS) {
          const unsigned h = k / (3u * SPME_P), e = k - h * (3u * SPME_P);
          const unsigned axis = e / SPME_P, d = e - axis * SPME_P;
          const float4 r = spl[hits[h0 + h].x];
          const float x = axis == 0u ? r.x : (axis == 1u ? r.y : r.z);
          float v = bspline_w<SPME_P>((float)d + x);
          // the 2^32 scale is a power of two: applying it to q w_c first
          // gives the same products as applying it last
          if (axis == 2u) v = (r.w * v) * 4294967296.0f;
          wgt[k] = v;
        }
        __syncthreads();
        for (unsigned k = t; k < nr * SPME_P; k += SPREAD_THREADS) {
          const unsigned h = k / SPME_P, iz = k - h * SPME_P;
          const unsigned rel = hits[h0 + h].y;
          const int rla = (int)(rel & 255u), rlb = (int)((rel >> 8) & 255u);
          int oc = (int)(rel >> 16) - (int)iz;
          oc += oc < 0 ? (int)nc : 0;
          if (oc >= (int)bc) continue;
          const float* wr = &wgt[h * 3u * SPME_P];
          const float dz = wr[2 * SPME_P + iz];
          float wb[SPME_P];
#pragma unroll
          for (int db = 0; db < SPME_P; ++db) wb[db] = wr[SPME_P + db];
#pragma unroll
          for (int da = 0; da < SPME_P; ++da) {
            int oa = rla - da;
            oa += oa < 0 ? (int)na : 0;
            if (oa >= (int)ba) continue;
            const float dzda = dz * wr[da];
#pragma unroll
            for (int db = 0; db < SPME_P; ++db) {
              int ob = rlb - db;
              ob += ob < 0 ? (int)nb : 0;
              if (ob >= (int)bb) continue;
              const long long vf = spread_fixed(dzda * wb[db]);
              if (vf != 0)
                atomicAdd(&acc[((unsigned)oa * bb + (unsigned)ob) * bc + (unsigned)oc],
                          (unsigned long long)vf);
            }
          }
        }
        __syncthreads();
      }
    }
    __syncthreads();
  }
  for (unsigned k = t; k < vol; k += SPREAD_THREADS) {
    const unsigned kc = k % bc, kab = k / bc;
    const unsigned kb = kab % bb, ka = kab / bb;
    rho[((size_t)(c0a + ka) * nb + (c0b + kb)) * nc + (c0c + kc)] = acc[k];
  }
}

// the largest divisor of n that is at most cap
static unsigned divisor_at_most(unsigned n, unsigned cap) {
  for (unsigned d = cap < n ? cap : n; d > 1; --d)
    if (n % d == 0) return d;
  return 1;
}

unsigned hd_spread_bricks(unsigned na, unsigned nb, unsigned nc, unsigned brick[3]) {
  // up to 8 x 8 x 16 cells, each side a divisor of the grid's; smaller while
  // that leaves a quarter of the CUs without a brick (an atom is then
  // visited by more of them: 2.2 at 8 x 8 x 16, 4.2 at 4 x 4 x 8).  8 x 16 x
  // 16 cells, visited 1.9 times, took 20,120 us per pass against 20,270 at
  // 196,608 atoms but 7,100 against 7,030 at 24,576 and 9,040 against 8,940
  // at 52,773.
  static const unsigned caps[4][3] = {{8, 8, 16}, {8, 8, 8}, {4, 8, 8}, {4, 4, 8}};
  unsigned count = 0;
  for (const auto& cap : caps) {
    brick[0] = divisor_at_most(na, cap[0]);
    brick[1] = divisor_at_most(nb, cap[1]);
    brick[2] = divisor_at_most(nc, cap[2]);
    count = (na / brick[0]) * (nb / brick[1]) * (nc / brick[2]);
    if (count >= 192u) break;
  }
  return count;
}

__global__ void k_zero_u64(unsigned long long* __restrict__ p, size_t count) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < count; i += stride) p[i] = 0ull;
}

// ---------------------------------------------------------------------
// Radix-2 complex FFT over `nlines` lines of length n held contiguously in
// LDS, input already in bit-reversed order.  tw[k] = exp(-2 pi i k / twn),
// k < twn/2, staged in LDS by the caller (fft_stage_twiddles) so that no
// butterfly waits on a global load; sign = -1 forward, +1 inverse
// (unnormalised).
// ---------------------------------------------------------------------
#define FFT_TW_MAX 256  // twn / 2 for the largest axis (nc <= 512)

__device__ __forceinline__ void fft_stage_twiddles(float2* stw, const float2* __restrict__ tw,
                                                   unsigned twn) {
  for (unsigned i = threadIdx.x; i < twn / 2; i += blockDim.x) stw[i] = tw[i];
}
__device__ __forceinline__ float2 cmul(float2 b, float2 w) {
  return make_float2(b.x * w.x - b.y * w.y, b.x * w.y + b.y * w.x);
}

// Two radix-2 stages per LDS pass (a radix-4 unit of 4 elements per thread:
// the same butterflies in the same order, half the passes and barriers),
// a last radix-2 pass when log2n is odd.
__device__ __forceinline__ void lds_fft(float2* d, unsigned n, unsigned log2n, unsigned nlines,
                                        unsigned lstride, int sign, const float2* tw,
                                        unsigned twn) {
  unsigned s = 1;
  for (; s + 1 <= log2n; s += 2) {
    unsigned h = 1u << (s - 1);         // half of stage s
    unsigned t1 = twn >> s, t2 = twn >> (s + 1);
    unsigned qn = n >> 2;                // radix-4 units per line
    unsigned nu = nlines * qn;
    for (unsigned idx = threadIdx.x; idx < nu; idx += blockDim.x) {
      unsigned line = idx >> (log2n - 2), u = idx & (qn - 1);
      unsigned j = u & (h - 1);
      unsigned i0 = ((u >> (s - 1)) << (s + 1)) + j;
      float2 w1 = tw[j * t1], w2 = tw[j * t2], w3 = tw[(j + h) * t2];
      if (sign > 0) { w1.y = -w1.y; w2.y = -w2.y; w3.y = -w3.y; }
      float2* row = d + line * lstride;
      float2 a0 = row[i0], a1 = row[i0 + h], a2 = row[i0 + 2 * h], a3 = row[i0 + 3 * h];
      float2 b1 = cmul(a1, w1), b3 = cmul(a3, w1);
      float2 y0 = make_float2(a0.x + b1.x, a0.y + b1.y), y1 = make_float2(a0.x - b1.x, a0.y - b1.y);
      float2 y2 = make_float2(a2.x + b3.x, a2.y + b3.y), y3 = make_float2(a2.x - b3.x, a2.y - b3.y);
      float2 c2 = cmul(y2, w2), c3 = cmul(y3, w3);
      row[i0] = make_float2(y0.x + c2.x, y0.y + c2.y);
      row[i0 + 2 * h] = make_float2(y0.x - c2.x, y0.y - c2.y);
      row[i0 + h] = make_float2(y1.x + c3.x, y1.y + c3.y);
      row[i0 + 3 * h] = make_float2(y1.x - c3.x, y1.y - c3.y);
    }
    __syncthreads();
  }
  if (s == log2n) {
    unsigned half = 1u << (s - 1);
    unsigned tstr = twn >> s;
    unsigned hn = n >> 1;
    unsigned nbf = nlines * hn;
    for (unsigned idx = threadIdx.x; idx < nbf; idx += blockDim.x) {
      unsigned line = idx >> (log2n - 1);
      unsigned k = idx & (hn - 1);
      unsigned j = k & (half - 1);
      unsigned i0 = ((k >> (s - 1)) << s) + j;
      unsigned i1 = i0 + half;
      float2 w = tw[j * tstr];
      if (sign > 0) w.y = -w.y;
      float2* row = d + line * lstride;
      float2 a = row[i0], bw = cmul(row[i1], w);
      row[i0] = make_float2(a.x + bw.x, a.y + bw.y);
      row[i1] = make_float2(a.x - bw.x, a.y - bw.y);
    }
    __syncthreads();
  }
}

// Decimation-in-frequency twin: natural-order input, bit-reversed output;
// stages log2n .. 1, two per pass (the radix-2 DIF butterflies in order).
__device__ __forceinline__ void lds_fft_dif(float2* d, unsigned n, unsigned log2n,
                                            unsigned nlines, unsigned lstride, int sign,
                                            const float2* tw, unsigned twn) {
  unsigned s = log2n;
  for (; s >= 2; s -= 2) {
    unsigned H = 1u << (s - 2);          // half of stage s - 1
    unsigned t1 = twn >> s, t2 = twn >> (s - 1);
    unsigned qn = n >> 2;
    unsigned nu = nlines * qn;
    for (unsigned idx = threadIdx.x; idx < nu; idx += blockDim.x) {
      unsigned line = idx >> (log2n - 2), u = idx & (qn - 1);
      unsigned j = u & (H - 1);
      unsigned i0 = ((u >> (s - 2)) << s) + j;
      float2 w1 = tw[j * t1], w1b = tw[(j + H) * t1], w2 = tw[j * t2];
      if (sign > 0) { w1.y = -w1.y; w1b.y = -w1b.y; w2.y = -w2.y; }
      float2* row = d + line * lstride;
      float2 x0 = row[i0], x1 = row[i0 + H], x2 = row[i0 + 2 * H], x3 = row[i0 + 3 * H];
      float2 y0 = make_float2(x0.x + x2.x, x0.y + x2.y);
      float2 y2 = cmul(make_float2(x0.x - x2.x, x0.y - x2.y), w1);
      float2 y1 = make_float2(x1.x + x3.x, x1.y + x3.y);
      float2 y3 = cmul(make_float2(x1.x - x3.x, x1.y - x3.y), w1b);
      row[i0] = make_float2(y0.x + y1.x, y0.y + y1.y);
      row[i0 + H] = cmul(make_float2(y0.x - y1.x, y0.y - y1.y), w2);
      row[i0 + 2 * H] = make_float2(y2.x + y3.x, y2.y + y3.y);
      row[i0 + 3 * H] = cmul(make_float2(y2.x - y3.x, y2.y - y3.y), w2);
    }
    __syncthreads();
  }
  if (s == 1) {
    unsigned hn = n >> 1;
    unsigned nbf = nlines * hn;
    for (unsigned idx = threadIdx.x; idx < nbf; idx += blockDim.x) {
      unsigned line = idx >> (log2n - 1);
      unsigned k = idx & (hn - 1);
      unsigned i0 = k << 1, i1 = i0 + 1;
      float2 w = tw[0];
      if (sign > 0) w.y = -w.y;
      float2* row = d + line * lstride;
      float2 a = row[i0], b = row[i1];
      float2 dlt = make_float2(a.x - b.x, a.y - b.y);
      row[i0] = make_float2(a.x + b.x, a.y + b.y);
      row[i1] = cmul(dlt, w);
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------
// Mixed-radix line FFT for lengths n = 2^a 3^b 5^c that are not powers of
// two (the reference sizes its grids for cuFFT's small primes, e.g.
// 48 x 48 x 96 and 20 x 20 x 80).  Self-sorting (Stockham) stages of radix
// 4, then 2, 3, 5: natural order in and out, so no bit reversal.  A stage
// of radix R with span ns (the product of the earlier radices) takes, for
// every j < n/R, the R values x[j + r n/R], multiplies value r by
// w^(r k) with w = exp(sign 2 pi i / (ns R)) and k = j mod ns, applies the
// R-point DFT and stores output r at (j div ns) ns R + k + r ns.  Each
// thread holds its butterflies' outputs in registers across a barrier, so
// the stage runs in place in LDS.
// ---------------------------------------------------------------------
#define FFT_MR_PER_THREAD 8  // butterflies per thread: nlines * n / R <= 2048 at 256 threads

// exp(sign * 2 pi i t / twn) for 0 <= t < twn from the half-circle table
// stw[t] = exp(-2 pi i t / twn), t < twn / 2
__device__ __forceinline__ float2 tw_full(const float2* stw, unsigned t, unsigned twn, int sign) {
  unsigned half = twn >> 1;
  float2 w = (t < half) ? stw[t] : make_float2(-stw[t - half].x, -stw[t - half].y);
  if (sign > 0) w.y = -w.y;
  return w;
}

__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cscale(float2 a, float f) { return make_float2(a.x * f, a.y * f); }
// a * (i f)
__device__ __forceinline__ float2 cmul_if(float2 a, float f) { return make_float2(-a.y * f, a.x * f); }

// R-point DFT with exp(sign 2 pi i jk / R), in place
template <int R>
__device__ __forceinline__ void small_dft(float2 (&a)[R], int sign) {
  const float sg = (float)sign;
  if constexpr (R == 2) {
    float2 t = a[0];
    a[0] = cadd(t, a[1]);
    a[1] = csub(t, a[1]);
  } else if constexpr (R == 4) {
    float2 t0 = cadd(a[0], a[2]), t1 = csub(a[0], a[2]);
    float2 t2 = cadd(a[1], a[3]), t3 = cmul_if(csub(a[1], a[3]), sg);
    a[0] = cadd(t0, t2);
    a[2] = csub(t0, t2);
    a[1] = cadd(t1, t3);
    a[3] = csub(t1, t3);
  } else if constexpr (R == 3) {
    const float h3 = 0.86602540378443865f;  // sin(2 pi / 3)
    float2 t = cadd(a[1], a[2]);
    float2 u = cmul_if(csub(a[1], a[2]), sg * h3);
    float2 m = csub(a[0], cscale(t, 0.5f));
    a[0] = cadd(a[0], t);
    a[1] = cadd(m, u);
    a[2] = csub(m, u);
  } else {  // R == 5
    const float c1 = 0.30901699437494742f, c2 = -0.80901699437494742f;  // cos 2pi/5, cos 4pi/5
    const float s1 = 0.95105651629515357f, s2 = 0.58778525229247313f;   // sin 2pi/5, sin 4pi/5
    float2 b1 = cadd(a[1], a[4]), b2 = cadd(a[2], a[3]);
    float2 d1 = csub(a[1], a[4]), d2 = csub(a[2], a[3]);
    float2 e1 = cadd(a[0], cadd(cscale(b1, c1), cscale(b2, c2)));
    float2 e2 = cadd(a[0], cadd(cscale(b1, c2), cscale(b2, c1)));
    float2 f1 = cmul_if(cadd(cscale(d1, s1), cscale(d2, s2)), sg);
    float2 f2 = cmul_if(csub(cscale(d1, s2), cscale(d2, s1)), sg);
    a[0] = cadd(a[0], cadd(b1, b2));
    a[1] = cadd(e1, f1);
    a[4] = csub(e1, f1);
    a[2] = cadd(e2, f2);
    a[3] = csub(e2, f2);
  }
}

template <int R>
__device__ __forceinline__ void mr_stage(float2* d, unsigned n, unsigned nlines, unsigned lstride,
                                         unsigned ns, int sign, const float2* stw, unsigned twn) {
  const unsigned m = n / R, total = nlines * m;
  const unsigned tstep = twn / (ns * R);
  float2 v[FFT_MR_PER_THREAD][R];
  unsigned dst[FFT_MR_PER_THREAD];
#pragma unroll
  for (int b = 0; b < FFT_MR_PER_THREAD; ++b) {
    unsigned idx = threadIdx.x + (unsigned)b * blockDim.x;
    dst[b] = 0xFFFFFFFFu;
    if (idx < total) {
      unsigned line = idx / m, j = idx - line * m;
      unsigned k = j % ns;
      const float2* row = d + line * lstride;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        float2 x = row[j + (unsigned)r * m];
        v[b][r] = r ? cmul(x, tw_full(stw, (unsigned)r * k * tstep, twn, sign)) : x;
      }
      small_dft<R>(v[b], sign);
      dst[b] = line * lstride + (j / ns) * ns * R + k;
    }
  }
  __syncthreads();
#pragma unroll
  for (int b = 0; b < FFT_MR_PER_THREAD; ++b)
    if (dst[b] != 0xFFFFFFFFu) {
#pragma unroll
      for (int r = 0; r < R; ++r) d[dst[b] + (unsigned)r * ns] = v[b][r];
    }
  __syncthreads();
}

// Complex FFT of `nlines` LDS lines of length n (2^a 3^b 5^c), natural
// order in and out; stw: exp(-2 pi i t / twn), t < twn / 2, with n | twn.
__device__ __forceinline__ void lds_fft_mixed(float2* d, unsigned n, unsigned nlines,
                                              unsigned lstride, int sign, const float2* stw,
                                              unsigned twn) {
  unsigned ns = 1, rem = n;
  while (rem > 1) {
    if (rem % 4 == 0) {
      mr_stage<4>(d, n, nlines, lstride, ns, sign, stw, twn);
      ns *= 4; rem /= 4;
    } else if (rem % 2 == 0) {
      mr_stage<2>(d, n, nlines, lstride, ns, sign, stw, twn);
      ns *= 2; rem /= 2;
    } else if (rem % 3 == 0) {
      mr_stage<3>(d, n, nlines, lstride, ns, sign, stw, twn);
      ns *= 3; rem /= 3;
    } else {
      mr_stage<5>(d, n, nlines, lstride, ns, sign, stw, twn);
      ns *= 5; rem /= 5;
    }
  }
}

__device__ __forceinline__ unsigned bitrev(unsigned k, unsigned log2n) {
  return log2n ? (__brev(k) >> (32 - log2n)) : 0u;
}

// c-axis forward R2C: rows of nc reals read from the i64 spread grid
// (converted to f32 exactly as spme_recip.cu:237-253), packed as nc/2
// complex values, FFT'd, then untangled into nc/2+1 spectrum values.
// twc: twiddles for length nc (exp(-2 pi i k/nc), k < nc/2).
template <bool MIXED>
__global__ void __launch_bounds__(FFT_THREADS) k_fft_c_fwd(
    const long long* __restrict__ rho, float2* __restrict__ cgrid, unsigned nrows, unsigned nc,
    unsigned log2h, const float2* __restrict__ twc) {
  __shared__ float2 d[FFT_TILE];
  __shared__ float2 stw[FFT_TW_MAX];
  unsigned h = nc >> 1, nch = h + 1;
  unsigned rows = FFT_TILE / h;
  unsigned r0 = blockIdx.x * rows;
  unsigned nr = min(rows, nrows - r0);
  const float inv = 1.0f / 4294967296.0f;
  fft_stage_twiddles(stw, twc, nc);
  for (unsigned e = threadIdx.x; e < nr * h; e += blockDim.x) {
    unsigned r = e / h, m = e - r * h;
    longlong2 v = reinterpret_cast<const longlong2*>(rho + (size_t)(r0 + r) * nc)[m];
    d[r * h + (MIXED ? m : bitrev(m, log2h))] = make_float2((float)v.x * inv, (float)v.y * inv);
  }
  __syncthreads();
  if (MIXED)
    lds_fft_mixed(d, h, nr, h, -1, stw, nc);
  else
    lds_fft(d, h, log2h, nr, h, -1, stw, nc);
  for (unsigned e = threadIdx.x; e < nr * nch; e += blockDim.x) {
    unsigned r = e / nch, k = e - r * nch;
    float2 zk = d[r * h + (k % h)];
    float2 zc = d[r * h + ((h - k) % h)];
    zc.y = -zc.y;  // conj(Z[h-k])
    float2 E = make_float2(0.5f * (zk.x + zc.x), 0.5f * (zk.y + zc.y));
    // O = (Z[k] - conj(Z[h-k])) / (2i)
    float2 O = make_float2(0.5f * (zk.y - zc.y), -0.5f * (zk.x - zc.x));
    float2 w = (k < h) ? stw[k] : make_float2(-1.f, 0.f);  // exp(-2 pi i k / nc)
    float2 wO = make_float2(w.x * O.x - w.y * O.y, w.x * O.y + w.y * O.x);
    cgrid[(size_t)(r0 + r) * nch + k] = make_float2(E.x + wO.x, E.y + wO.y);
  }
}

// c-axis inverse C2R: nc/2+1 spectrum values per row -> nc reals,
// unnormalised (round trip = nc * x).
// 256 threads; se, sw: 256 doubles of LDS each
static_assert(FFT_THREADS == 256, "the inverse c pass runs the 256-thread reduction");
__device__ __forceinline__ void recip_reduce_block(const double2* __restrict__ partials,
                                                   unsigned np, double* __restrict__ recip,
                                                   float* __restrict__ w_share, unsigned n,
                                                   double* se, double* sw) {
  double e = 0.0, w = 0.0;
  for (unsigned i = threadIdx.x; i < np; i += 256) {
    double2 p = partials[i];
    e += p.x;
    w += p.y;
  }
  se[threadIdx.x] = e;
  sw[threadIdx.x] = w;
  __syncthreads();
  for (unsigned s = 1; s < 256; s <<= 1) {
    if ((threadIdx.x % (2 * s)) == 0) {
      se[threadIdx.x] += se[threadIdx.x + s];
      sw[threadIdx.x] += sw[threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    recip[0] = 0.5 * se[0];
    recip[1] = 0.5 * sw[0];
    w_share[0] = n ? (float)(0.5 * sw[0] / (double)n) : 0.f;
  }
}

template <bool MIXED>
__global__ void __launch_bounds__(FFT_THREADS) k_fft_c_inv(
    const float2* __restrict__ cgrid, float* __restrict__ vgrid, unsigned nrows, unsigned nc,
    unsigned log2h, const float2* __restrict__ twc, const double2* __restrict__ partials,
    unsigned np, double* __restrict__ recip, float* __restrict__ w_share, unsigned n_atoms) {
  __shared__ float2 d[FFT_TILE];
  __shared__ float2 stw[FFT_TW_MAX];
  if (partials && blockIdx.x == 0) {
    // the convolution's energy and virial partials are complete (written
    // by the a-axis pass before this launch): block 0 reduces them first,
    // in k_recip_reduce's order, with the tile's LDS as its scratch
    double* se = reinterpret_cast<double*>(d);
    recip_reduce_block(partials, np, recip, w_share, n_atoms, se, se + 256);
    __syncthreads();
  }
  unsigned h = nc >> 1, nch = h + 1;
  unsigned rows = FFT_TILE / h;
  unsigned r0 = blockIdx.x * rows;
  unsigned nr = min(rows, nrows - r0);
  fft_stage_twiddles(stw, twc, nc);
  __syncthreads();
  for (unsigned e = threadIdx.x; e < nr * h; e += blockDim.x) {
    unsigned r = e / h, k = e - r * h;
    const float2* row = cgrid + (size_t)(r0 + r) * nch;
    float2 xk = row[k], xc = row[h - k];
    xc.y = -xc.y;  // conj(X[h-k])
    float2 A = make_float2(xk.x + xc.x, xk.y + xc.y);
    float2 B = make_float2(xk.x - xc.x, xk.y - xc.y);
    float2 w = stw[k];
    w.y = -w.y;  // exp(+2 pi i k / nc)
    float2 wB = make_float2(w.x * B.x - w.y * B.y, w.x * B.y + w.y * B.x);
    // Z' = A + i * wB
    d[r * h + (MIXED ? k : bitrev(k, log2h))] = make_float2(A.x - wB.y, A.y + wB.x);
  }
  __syncthreads();
  if (MIXED)
    lds_fft_mixed(d, h, nr, h, +1, stw, nc);
  else
    lds_fft(d, h, log2h, nr, h, +1, stw, nc);
  for (unsigned e = threadIdx.x; e < nr * h; e += blockDim.x) {
    unsigned r = e / h, m = e - r * h;
    reinterpret_cast<float2*>(vgrid + (size_t)(r0 + r) * nc)[m] = d[r * h + m];
  }
}

// Strided axis pass over the complex grid: lines along an axis of length
// n with element stride `estride` (complex units); `nouter` groups of
// lines start at outer*ostride; within a group, CW consecutive columns.
#define FFT_CW 16
// LDS lines are padded to n+1 complex values to spread the column-wise
// accesses over the banks.  `rev_in` stores in bit-reversed order (for a
// DIT pass); `rev_out` reads a bit-reversed line (after a DIF pass).
__device__ __forceinline__ void strided_load(float2* d, const float2* __restrict__ g,
                                             size_t base, unsigned n, unsigned log2n,
                                             size_t estride, unsigned ncol, bool rev_in) {
  for (unsigned e = threadIdx.x; e < n * FFT_CW; e += blockDim.x) {
    unsigned k = e / FFT_CW, c = e - k * FFT_CW;
    float2 v = make_float2(0.f, 0.f);
    if (c < ncol) v = g[base + (size_t)k * estride + c];
    d[c * (n + 1) + (rev_in ? bitrev(k, log2n) : k)] = v;
  }
}
__device__ __forceinline__ void strided_store(const float2* d, float2* __restrict__ g,
                                              size_t base, unsigned n, unsigned log2n,
                                              size_t estride, unsigned ncol, bool rev_out) {
  for (unsigned e = threadIdx.x; e < n * FFT_CW; e += blockDim.x) {
    unsigned k = e / FFT_CW, c = e - k * FFT_CW;
    if (c < ncol) g[base + (size_t)k * estride + c] = d[c * (n + 1) + (rev_out ? bitrev(k, log2n) : k)];
  }
}

// b-axis pass (forward or inverse), in place.  grid: (na * nchunks).
template <bool MIXED>
__global__ void __launch_bounds__(FFT_THREADS) k_fft_b(float2* __restrict__ cgrid, unsigned na,
                                                       unsigned nb, unsigned nch,
                                                       unsigned log2b, int sign,
                                                       const float2* __restrict__ twb) {
  __shared__ float2 d[FFT_CW * 257];
  __shared__ float2 stw[FFT_TW_MAX];
  unsigned nchunk = (nch + FFT_CW - 1) / FFT_CW;
  unsigned a = blockIdx.x / nchunk, c0 = (blockIdx.x - a * nchunk) * FFT_CW;
  unsigned ncol = min(FFT_CW, nch - c0);
  size_t base = (size_t)a * nb * nch + c0;
  fft_stage_twiddles(stw, twb, nb);
  strided_load(d, cgrid, base, nb, log2b, nch, ncol, !MIXED);
  __syncthreads();
  if (MIXED)
    lds_fft_mixed(d, nb, FFT_CW, nb + 1, sign, stw, nb);
  else
    lds_fft(d, nb, log2b, FFT_CW, nb + 1, sign, stw, nb);
  strided_store(d, cgrid, base, nb, log2b, nch, ncol, false);
}

// Grids whose a-plane fits in LDS (nb * nc/2 <= FFT_TILE complex values
// and the plane's nc/2 + 1 columns of nb, padded, within FFT_PLANE_MAX):
// one workgroup per a-plane runs the c-axis and b-axis passes of the
// forward transform back to back (and of the inverse, b then c), with the
// plane staged in LDS between them instead of a round trip through the
// complex grid and a second launch.  Each line is transformed by the same
// LDS routines, on the same values, as in k_fft_c_fwd / k_fft_b /
// k_fft_c_inv; the compiler may round a few multiply-adds differently in
// the two kernels, so the results agree to f32 rounding.
#define FFT_PLANE_MAX 2176  // 33 columns x 65 (c <= 64, b <= 64)

__host__ __device__ inline bool fft_plane_fits(unsigned nb, unsigned nc) {
  return nb * (nc / 2) <= FFT_TILE && (nc / 2 + 1) * (nb + 1) <= FFT_PLANE_MAX;
}

template <bool MC, bool MB>
__global__ void __launch_bounds__(FFT_THREADS) k_fft_cb_fwd(
    const long long* __restrict__ rho, float2* __restrict__ cgrid, unsigned nb, unsigned nc,
    unsigned log2h, unsigned log2b, const float2* __restrict__ twc,
    const float2* __restrict__ twb) {
  __shared__ float2 d[FFT_TILE];
  __shared__ float2 col[FFT_PLANE_MAX];
  __shared__ float2 stw[FFT_TW_MAX], stwb[FFT_TW_MAX];
  const unsigned h = nc >> 1, nch = h + 1, nr = nb, ls = nb + 1;
  const unsigned r0 = blockIdx.x * nb;
  const float inv = 1.0f / 4294967296.0f;
  fft_stage_twiddles(stw, twc, nc);
  fft_stage_twiddles(stwb, twb, nb);
  for (unsigned e = threadIdx.x; e < nr * h; e += blockDim.x) {
    unsigned r = e / h, m = e - r * h;
    longlong2 v = reinterpret_cast<const longlong2*>(rho + (size_t)(r0 + r) * nc)[m];
    d[r * h + (MC ? m : bitrev(m, log2h))] = make_float2((float)v.x * inv, (float)v.y * inv);
  }
  __syncthreads();
  if (MC)
    lds_fft_mixed(d, h, nr, h, -1, stw, nc);
  else
    lds_fft(d, h, log2h, nr, h, -1, stw, nc);
  // k_fft_c_fwd's untangling, into the b-axis columns
  for (unsigned e = threadIdx.x; e < nr * nch; e += blockDim.x) {
    unsigned r = e / nch, k = e - r * nch;
    float2 zk = d[r * h + (k % h)];
    float2 zc = d[r * h + ((h - k) % h)];
    zc.y = -zc.y;
    float2 E = make_float2(0.5f * (zk.x + zc.x), 0.5f * (zk.y + zc.y));
    float2 O = make_float2(0.5f * (zk.y - zc.y), -0.5f * (zk.x - zc.x));
    float2 w = (k < h) ? stw[k] : make_float2(-1.f, 0.f);
    float2 wO = make_float2(w.x * O.x - w.y * O.y, w.x * O.y + w.y * O.x);
    col[k * ls + (MB ? r : bitrev(r, log2b))] = make_float2(E.x + wO.x, E.y + wO.y);
  }
  __syncthreads();
  if (MB)
    lds_fft_mixed(col, nb, nch, ls, -1, stwb, nb);
  else
    lds_fft(col, nb, log2b, nch, ls, -1, stwb, nb);
  for (unsigned e = threadIdx.x; e < nr * nch; e += blockDim.x) {
    unsigned r = e / nch, k = e - r * nch;
    cgrid[(size_t)(r0 + r) * nch + k] = col[k * ls + r];
  }
}

template <bool MB, bool MC>
__global__ void __launch_bounds__(FFT_THREADS) k_fft_bc_inv(
    const float2* __restrict__ cgrid, float* __restrict__ vgrid, unsigned nb, unsigned nc,
    unsigned log2h, unsigned log2b, const float2* __restrict__ twc,
    const float2* __restrict__ twb, const double2* __restrict__ partials, unsigned np,
    double* __restrict__ recip, float* __restrict__ w_share, unsigned n_atoms) {
  __shared__ float2 d[FFT_TILE];
  __shared__ float2 col[FFT_PLANE_MAX];
  __shared__ float2 stw[FFT_TW_MAX], stwb[FFT_TW_MAX];
  const unsigned h = nc >> 1, nch = h + 1, nr = nb, ls = nb + 1;
  const unsigned r0 = blockIdx.x * nb;
  if (partials && blockIdx.x == 0) {
    // as in k_fft_c_inv: block 0 reduces the energy and virial partials
    double* se = reinterpret_cast<double*>(d);
    recip_reduce_block(partials, np, recip, w_share, n_atoms, se, se + 256);
    __syncthreads();
  }
  fft_stage_twiddles(stw, twc, nc);
  fft_stage_twiddles(stwb, twb, nb);
  for (unsigned e = threadIdx.x; e < nr * nch; e += blockDim.x) {
    unsigned r = e / nch, k = e - r * nch;
    col[k * ls + (MB ? r : bitrev(r, log2b))] = cgrid[(size_t)(r0 + r) * nch + k];
  }
  __syncthreads();
  if (MB)
    lds_fft_mixed(col, nb, nch, ls, +1, stwb, nb);
  else
    lds_fft(col, nb, log2b, nch, ls, +1, stwb, nb);
  // k_fft_c_inv's packing of the row spectrum, from the b-axis columns
  for (unsigned e = threadIdx.x; e < nr * h; e += blockDim.x) {
    unsigned r = e / h, k = e - r * h;
    float2 xk = col[k * ls + r], xc = col[(h - k) * ls + r];
    xc.y = -xc.y;
    float2 A = make_float2(xk.x + xc.x, xk.y + xc.y);
    float2 B = make_float2(xk.x - xc.x, xk.y - xc.y);
    float2 w = stw[k];
    w.y = -w.y;
    float2 wB = make_float2(w.x * B.x - w.y * B.y, w.x * B.y + w.y * B.x);
    d[r * h + (MC ? k : bitrev(k, log2h))] = make_float2(A.x - wB.y, A.y + wB.x);
  }
  __syncthreads();
  if (MC)
    lds_fft_mixed(d, h, nr, h, +1, stw, nc);
  else
    lds_fft(d, h, log2h, nr, h, +1, stw, nc);
  for (unsigned e = threadIdx.x; e < nr * h; e += blockDim.x) {
    unsigned r = e / h, m = e - r * h;
    reinterpret_cast<float2*>(vgrid + (size_t)(r0 + r) * nc)[m] = d[r * h + m];
  }
}

// a-axis pass fused with the influence multiply:
//   forward FFT over a -> for every k: G(k), virial factor vf(k)
//   (spme_recip.cu:34-115 in f32 from the live lattice), energy and
//   virial partials hw*G*|rho^|^2 and hw*vf*|rho^|^2 (spme_recip.cu:
//   296-342) summed in FP64 by a fixed tree -> V^ = G rho^ -> inverse FFT
//   over a.  grid: (nb * nchunks); partials[blockIdx] = (E, W).
template <bool MIXED>
__global__ void __launch_bounds__(FFT_THREADS) k_fft_a_conv(
    float2* __restrict__ cgrid, unsigned na, unsigned nb, unsigned nc, unsigned nch,
    unsigned log2a, const float2* __restrict__ twa, const float* __restrict__ bfa,
    const float* __restrict__ bfb, const float* __restrict__ bfc,
    const float* __restrict__ lattice, float kc, float alpha, double2* __restrict__ partials) {
  __shared__ float2 d[FFT_CW * 257];
  __shared__ float2 stw[FFT_TW_MAX];
  __shared__ double red_e[FFT_THREADS], red_w[FFT_THREADS];
  unsigned nchunk = (nch + FFT_CW - 1) / FFT_CW;
  unsigned b = blockIdx.x / nchunk, c0 = (blockIdx.x - b * nchunk) * FFT_CW;
  unsigned ncol = min(FFT_CW, nch - c0);
  size_t base = (size_t)b * nch + c0;
  size_t estride = (size_t)nb * nch;
  unsigned ls = na + 1;
  fft_stage_twiddles(stw, twa, na);
  strided_load(d, cgrid, base, na, log2a, estride, ncol, !MIXED);
  __syncthreads();
  if (MIXED)
    lds_fft_mixed(d, na, FFT_CW, ls, -1, stw, na);
  else
    lds_fft(d, na, log2a, FFT_CW, ls, -1, stw, na);
  HdLattice L = hd_load_lattice(lattice);
  float v_box = L.lx * L.ly * L.lz;
  float four_alpha2 = 4.0f * alpha * alpha;
  const float pi_r = 3.14159265358979f;
  float four_pi = 4.0f * pi_r, two_pi = 2.0f * pi_r;
  float pref = kc / v_box;
  float ilx = 1.0f / L.lx, ily = 1.0f / L.ly, ilz = 1.0f / L.lz;
  float ra_x = ilx, ra_y = -L.xy * ilx * ily, ra_z = (L.xy * L.yz - L.xz * L.ly) * ilx * ily * ilz;
  float rb_y = ily, rb_z = -L.yz * ily * ilz, rc_z = ilz;
  float mb = (b <= nb / 2) ? (float)b : (float)b - (float)nb;
  double se = 0.0, sw = 0.0;
  for (unsigned e = threadIdx.x; e < na * FFT_CW; e += blockDim.x) {
    unsigned c = e / na, a = e - c * na;
    if (c >= ncol) continue;
    unsigned kcc = c0 + c;
    float ma = (a <= na / 2) ? (float)a : (float)a - (float)na;
    float mc = (kcc <= nc / 2) ? (float)kcc : (float)kcc - (float)nc;
    float kx = two_pi * (ma * ra_x);
    float ky = two_pi * (ma * ra_y + mb * rb_y);
    float kz = two_pi * (ma * ra_z + mb * rb_z + mc * rc_z);
    float k2 = kx * kx + ky * ky + kz * kz;
    float g = 0.f, vf = 0.f;
    if (k2 != 0.f) {
      g = pref * (four_pi / k2) * expf(-k2 / four_alpha2) * bfa[a] * bfb[b] * bfc[kcc];
      vf = g * (1.0f - k2 / (2.0f * alpha * alpha));
    }
    float2 v = d[c * ls + a];
    float rsq = v.x * v.x + v.y * v.y;
    double hw = (kcc == 0 || 2 * kcc == nc) ? 1.0 : 2.0;
    se += hw * (double)g * (double)rsq;
    sw += hw * (double)vf * (double)rsq;
    d[c * ls + a] = make_float2(g * v.x, g * v.y);
  }
  red_e[threadIdx.x] = se;
  red_w[threadIdx.x] = sw;
  __syncthreads();
  for (unsigned s = 1; s < FFT_THREADS; s <<= 1) {
    if ((threadIdx.x % (2 * s)) == 0) {
      red_e[threadIdx.x] += red_e[threadIdx.x + s];
      red_w[threadIdx.x] += red_w[threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) partials[blockIdx.x] = make_double2(red_e[0], red_w[0]);
  if (MIXED) {
    lds_fft_mixed(d, na, FFT_CW, ls, +1, stw, na);
    strided_store(d, cgrid, base, na, log2a, estride, ncol, false);
  } else {
    lds_fft_dif(d, na, log2a, FFT_CW, ls, +1, stw, na);
    strided_store(d, cgrid, base, na, log2a, estride, ncol, true);
  }
}

// Fixed-order FP64 reduction of the (E, W) partials; writes
//   recip[0] = E_recip (Ewald sum without self term), recip[1] = W_recip,
//   w_share[0] = (f32) W_recip / N  (the uniform per-atom share,
//   spme_recip.cu:376-403).
__global__ void __launch_bounds__(256) k_recip_reduce(const double2* __restrict__ partials,
                                                      unsigned np, double* __restrict__ recip,
                                                      float* __restrict__ w_share, unsigned n) {
  __shared__ double se[256], sw[256];
  recip_reduce_block(partials, np, recip, w_share, n, se, sw);
}

static unsigned ilog2u(unsigned v) {
  unsigned r = 0;
  while ((1u << r) < v) ++r;
  return r;
}

void hd_launch_spme_spread(hipStream_t st, const HdSpmeArgs& a) {
  unsigned brick[3];
  unsigned nbricks = hd_spread_bricks(a.na, a.nb, a.nc, brick);
  if (a.order == 5)
    hipLaunchKernelGGL(k_spread<5>, dim3(nbricks), dim3(SPREAD_THREADS), 0, st, a.spl, a.sg,
                       a.na, a.nb, a.nc, brick[0], brick[1], brick[2], a.voxel_rank, a.voxel_off,
                       a.nv[0], a.nv[1], a.nv[2], a.lattice, a.reach,
                       (unsigned long long*)a.rho_fixed);
  else
    hipLaunchKernelGGL(k_spread<4>, dim3(nbricks), dim3(SPREAD_THREADS), 0, st, a.spl, a.sg,
                       a.na, a.nb, a.nc, brick[0], brick[1], brick[2], a.voxel_rank, a.voxel_off,
                       a.nv[0], a.nv[1], a.nv[2], a.lattice, a.reach,
                       (unsigned long long*)a.rho_fixed);
}

void hd_launch_recip_reduce(hipStream_t st, const HdSpmeArgs& a, unsigned n_partials) {
  hipLaunchKernelGGL(k_recip_reduce, dim3(1), dim3(256), 0, st, a.partials, n_partials, a.recip,
                     a.w_share, a.n);
}

static bool pow2u(unsigned v) { return v && !(v & (v - 1)); }

template <bool MC, bool MB>
static void launch_plane_passes(hipStream_t st, const HdSpmeArgs& a, bool fwd, unsigned log2h,
                                unsigned log2b, unsigned np) {
  if (fwd)
    hipLaunchKernelGGL((k_fft_cb_fwd<MC, MB>), dim3(a.na), dim3(FFT_THREADS), 0, st,
                       a.rho_fixed, a.cgrid, a.nb, a.nc, log2h, log2b, a.tw_c, a.tw_b);
  else
    hipLaunchKernelGGL((k_fft_bc_inv<MB, MC>), dim3(a.na), dim3(FFT_THREADS), 0, st, a.cgrid,
                       a.vgrid, a.nb, a.nc, log2h, log2b, a.tw_c, a.tw_b, a.partials, np,
                       a.recip, a.w_share, a.n);
}

static void plane_passes(hipStream_t st, const HdSpmeArgs& a, bool fwd, bool mc, bool mb,
                         unsigned log2h, unsigned log2b, unsigned np) {
  if (mc && mb) launch_plane_passes<true, true>(st, a, fwd, log2h, log2b, np);
  else if (mc) launch_plane_passes<true, false>(st, a, fwd, log2h, log2b, np);
  else if (mb) launch_plane_passes<false, true>(st, a, fwd, log2h, log2b, np);
  else launch_plane_passes<false, false>(st, a, fwd, log2h, log2b, np);
}

void hd_launch_spme(hipStream_t st, const HdSpmeArgs& a) {
  unsigned nch = a.nc / 2 + 1;
  hd_launch_spme_spread(st, a);
  unsigned nrows = a.na * a.nb;
  unsigned h = a.nc / 2;
  unsigned rows = FFT_TILE / h;
  dim3 gc((nrows + rows - 1) / rows), tb(FFT_THREADS);
  bool mc = !pow2u(h), mb = !pow2u(a.nb), ma = !pow2u(a.na);
  if (!a.no_plane && fft_plane_fits(a.nb, a.nc)) {
    // c and b passes per a-plane in one launch each way
    unsigned nchunk = (nch + FFT_CW - 1) / FFT_CW;
    unsigned lh = mc ? 0u : ilog2u(h), lb = mb ? 0u : ilog2u(a.nb);
    plane_passes(st, a, true, mc, mb, lh, lb, 0);
    dim3 ga(a.nb * nchunk);
    if (ma)
      hipLaunchKernelGGL(k_fft_a_conv<true>, ga, tb, 0, st, a.cgrid, a.na, a.nb, a.nc, nch, 0u,
                         a.tw_a, a.bf_a, a.bf_b, a.bf_c, a.lattice, (float)a.kc, (float)a.alpha,
                         a.partials);
    else
      hipLaunchKernelGGL(k_fft_a_conv<false>, ga, tb, 0, st, a.cgrid, a.na, a.nb, a.nc, nch,
                         ilog2u(a.na), a.tw_a, a.bf_a, a.bf_b, a.bf_c, a.lattice, (float)a.kc,
                         (float)a.alpha, a.partials);
    plane_passes(st, a, false, mc, mb, lh, lb, a.nb * nchunk);
    return;
  }
  if (mc)
    hipLaunchKernelGGL(k_fft_c_fwd<true>, gc, tb, 0, st, a.rho_fixed, a.cgrid, nrows, a.nc, 0u,
                       a.tw_c);
  else
    hipLaunchKernelGGL(k_fft_c_fwd<false>, gc, tb, 0, st, a.rho_fixed, a.cgrid, nrows, a.nc,
                       ilog2u(h), a.tw_c);
  unsigned nchunk = (nch + FFT_CW - 1) / FFT_CW;
  dim3 gb(a.na * nchunk), ga(a.nb * nchunk);
  for (int sign = -1; sign <= 1; sign += 2) {
    if (sign > 0) {
      if (ma)
        hipLaunchKernelGGL(k_fft_a_conv<true>, ga, tb, 0, st, a.cgrid, a.na, a.nb, a.nc, nch, 0u,
                           a.tw_a, a.bf_a, a.bf_b, a.bf_c, a.lattice, (float)a.kc,
                           (float)a.alpha, a.partials);
      else
        hipLaunchKernelGGL(k_fft_a_conv<false>, ga, tb, 0, st, a.cgrid, a.na, a.nb, a.nc, nch,
                           ilog2u(a.na), a.tw_a, a.bf_a, a.bf_b, a.bf_c, a.lattice, (float)a.kc,
                           (float)a.alpha, a.partials);
    }
    if (mb)
      hipLaunchKernelGGL(k_fft_b<true>, gb, tb, 0, st, a.cgrid, a.na, a.nb, nch, 0u, sign,
                         a.tw_b);
    else
      hipLaunchKernelGGL(k_fft_b<false>, gb, tb, 0, st, a.cgrid, a.na, a.nb, nch, ilog2u(a.nb),
                         sign, a.tw_b);
  }
  // the inverse c pass also reduces the energy and virial partials
  if (mc)
    hipLaunchKernelGGL(k_fft_c_inv<true>, gc, tb, 0, st, a.cgrid, a.vgrid, nrows, a.nc, 0u,
                       a.tw_c, a.partials, a.nb * nchunk, a.recip, a.w_share, a.n);
  else
    hipLaunchKernelGGL(k_fft_c_inv<false>, gc, tb, 0, st, a.cgrid, a.vgrid, nrows, a.nc,
                       ilog2u(h), a.tw_c, a.partials, a.nb * nchunk, a.recip, a.w_share, a.n);
}

unsigned hd_spme_partials_count(unsigned nb, unsigned nc) {
  unsigned nch = nc / 2 + 1;
  return nb * ((nch + FFT_CW - 1) / FFT_CW);
}
