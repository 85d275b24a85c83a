/*
 * vw_kernels.h -- gfx950 kernels of the visibility / reconstruction path.
 *
 * Execution model (wave64, CDNA4):
 *  - Viss: a wave owns one chunk of sky tiles x RPW half rows.  Lanes hold
 *    pixels (4 per lane per 256-pixel sub-tile, coalesced SoA loads), rows
 *    are wave-uniform: row records, tile-cone classes and antenna frames
 *    arrive through scalar loads, so the all-hidden / all-visible / mixed
 *    decision is a scalar branch with no divergence.  Each lane keeps RPW
 *    complex partial sums in registers; one cross-lane tree per row per chunk
 *    writes a partial that a second kernel folds in chunk order
 *    (deterministic).  The plain form evaluates sin/cos from a 1024-entry
 *    LDS table (vw_shared.h).
 *  - Viss, antenna-factorized form (the mixed form's default): a wave owns
 *    one epoch and a chunk of tiles, lanes hold (antenna, pixel) pairs, and
 *    each step of 4 pixels feeds per-antenna exponentials to 16x16x4 matrix
 *    core products whose accumulators are the epoch's pair sums.
 *  - Recon: lanes hold output points (4 per lane, one output tile per wave),
 *    groups are wave-uniform and pass through a per-wave LDS ring; the group
 *    range of a segment is split into chunks whose partials a second kernel
 *    folds in order.
 * Workgroups are remapped so that consecutive logical blocks land on the same
 * XCD (hardware dispatches block b to XCD b % 8), keeping a chunk's pixel
 * data in one XCD's L2.
 */
#ifndef VW_KERNELS_H
#define VW_KERNELS_H

#include <hip/hip_runtime.h>
#include <float.h>
#include <stdint.h>
#include <type_traits>
#include "vw_shared.h"
#include "../../include/vissws.h"

struct RowRec {
  double u, v, w;
  int32_t ia, ib; /* antenna-frame indices g*A + a of the two endpoints */
};

/* chunk partials a fold kernel loads before adding them (in chunk order) */
#define VW_FOLD_BATCH 8

struct DevInfo {
  vw_segparams sp;
  int64_t nuniq;
  int64_t first_nz;
  int64_t wtotal;
  int32_t polar; /* the recon's polar terms may be used: bit 0 plain, bit 1 mixed (vw_polar_ok) */
  int32_t pad;
};

/* The segments that a launch of the one-sky step covers: one, or a run of short
 * ones.  Segment s has half rows [row0[s], row0[s + 1]) of the segment buffers
 * and its groups at positions base[s] + q, base a multiple of 64 with room for
 * one entry more than the segment has rows; its DevInfo is entry s. */
#define VW_MERGE_MAX 16
struct VwMerge {
  int n;
  int row0[VW_MERGE_MAX + 1], base[VW_MERGE_MAX + 1];
};

#define VW_FULLMASK 0xffffffffffffffffULL

__device__ __forceinline__ int vw_rfl(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ uint64_t vw_rfl64(uint64_t x) {
  return (uint64_t)(uint32_t)vw_rfl((int)(x >> 32)) << 32 | (uint32_t)vw_rfl((int)x);
}

/* Stage timing: the small kernels around a stage's large one write the device's
 * real-time counter to two words of host memory, ts[0] as the first workgroup
 * starts and ts[1] as the highest-numbered one ends (ts may be null).  The large
 * kernel's time runs from the latter of the kernel before it to the start of the
 * one after: all of the large kernel, and what the workgroups of the kernel before
 * it still do after its highest-numbered one.  (A stamp of the large kernel's own
 * start, a store before its loads, took the scalar loads of k_recon: 63 to 78
 * registers, 8 to 6 waves.)
 * Events recorded around every stage cost a barrier packet and a call each: a
 * whole run at Nside 32 went from 716 to 527 us, a one-segment predict with
 * adjoint at Nside 64 from 1000 to 845 us. */
__device__ __forceinline__ void vw_ts_begin(uint64_t* ts) {
  if (ts && blockIdx.x == 0 && threadIdx.x == 0) ts[0] = (uint64_t)wall_clock64();
}
__device__ __forceinline__ void vw_ts_end(uint64_t* ts) {
  if (ts && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) ts[1] = (uint64_t)wall_clock64();
}

/* logical block index with consecutive indices on one XCD */
__device__ __forceinline__ int64_t vw_xcd_block(int64_t b, int64_t nb) {
  int64_t q = nb / 8, r = nb % 8, x = b % 8, i = b / 8;
  return x * q + (x < r ? x : r) + i;
}

__device__ __forceinline__ double vw_wave_sum(double x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  return x;
}

__device__ __forceinline__ int64_t vw_wave_sum_i(int64_t x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  return x;
}

/* class byte of (tile, half row) from a [ntile][nh_pad] byte table, uniform */
__device__ __forceinline__ int vw_cls_lookup(const uint32_t* __restrict__ words, int64_t tile,
                                             int64_t nh_pad, int64_t h) {
  int64_t byte = tile * nh_pad + h;
  uint32_t w = words[byte >> 2];
  return vw_rfl((int)((w >> (8 * (byte & 3))) & 0xffu));
}

/* ------------------------------------------------------------------ */
/* resident geometry                                                    */
/* ------------------------------------------------------------------ */
__global__ void k_pix2lmn(int64_t nside, int64_t npix, double* __restrict__ l, double* __restrict__ m,
                          double* __restrict__ n, double* __restrict__ nm1) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npix) return;
  double a, b, c;
  vw_pix2lmn_nest(nside, p, &a, &b, &c);
  l[p] = a;
  m[p] = b;
  n[p] = c;
  nm1[p] = c - 1.0;
}

__global__ void k_grid_points(int64_t N, int64_t npts, const int64_t* __restrict__ gidx,
                              double* __restrict__ l, double* __restrict__ m, double* __restrict__ n) {
  int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= npts) return;
  int64_t id = gidx[k];
  double a, b, c;
  vw_grid_point(N, id / N, id % N, &a, &b, &c);
  l[k] = a;
  m[k] = b;
  n[k] = c;
}

/* Tile cone: stride-halving pairwise sum (a[i] += a[i+s], s = TP/2..1), centre,
 * minimum of c.s over the tile.  One workgroup of 256 per tile. */
template <int TP>
__global__ __launch_bounds__(256) void k_tile_cone(const double* __restrict__ l, const double* __restrict__ m,
                                                   const double* __restrict__ n, int64_t npts, int64_t ntile,
                                                   double* __restrict__ cone) {
  __shared__ double sx[TP / 2], sy[TP / 2], sz[TP / 2];
  __shared__ double smin[256];
  int64_t t = blockIdx.x;
  int64_t p0 = t * TP;
  int64_t cnt = npts - p0 < TP ? npts - p0 : TP;
  for (int i = threadIdx.x; i < TP / 2; i += 256) {
    int i2 = i + TP / 2;
    double x0 = i < cnt ? l[p0 + i] : 0.0, x1 = i2 < cnt ? l[p0 + i2] : 0.0;
    double y0 = i < cnt ? m[p0 + i] : 0.0, y1 = i2 < cnt ? m[p0 + i2] : 0.0;
    double z0 = i < cnt ? n[p0 + i] : 0.0, z1 = i2 < cnt ? n[p0 + i2] : 0.0;
    sx[i] = x0 + x1;
    sy[i] = y0 + y1;
    sz[i] = z0 + z1;
  }
  __syncthreads();
  for (int s = TP / 4; s > 0; s >>= 1) {
    for (int i = threadIdx.x; i < s; i += 256) {
      sx[i] = sx[i] + sx[i + s];
      sy[i] = sy[i] + sy[i + s];
      sz[i] = sz[i] + sz[i + s];
    }
    __syncthreads();
  }
  double cx, cy, cz;
  vw_cone_centre(sx[0], sy[0], sz[0], &cx, &cy, &cz);
  double mind = 1.0;
  for (int64_t i = threadIdx.x; i < cnt; i += 256)
    mind = fmin(mind, vw_dot3(cx, cy, cz, l[p0 + i], m[p0 + i], n[p0 + i]));
  smin[threadIdx.x] = mind;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) smin[threadIdx.x] = fmin(smin[threadIdx.x], smin[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    double ca, sa;
    vw_cone_radius(smin[0], &ca, &sa);
    cone[0 * ntile + t] = cx;
    cone[1 * ntile + t] = cy;
    cone[2 * ntile + t] = cz;
    cone[3 * ntile + t] = ca;
    cone[4 * ntile + t] = sa;
  }
}

/* ------------------------------------------------------------------ */
/* day geometry and segment rows                                        */
/* ------------------------------------------------------------------ */
struct DayArgs {
  int geometry;
  int T, A;
  int64_t orbit_res, seg_len, tw, day_offset;
  int day;
  const int64_t* t1s;
  const double* circ; /* 7*A: radius, phase, rate, sr, cr, si, ci */
  double dt;
};

__global__ void k_day_positions(DayArgs a, double* __restrict__ pos) {
  int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t TA = (int64_t)a.T * a.A;
  if (k >= TA) return;
  int64_t t = k / a.A;
  int s = (int)(k - t * a.A);
  double x, y, z;
  if (a.geometry == VW_GEOM_LUNAR8) {
    int64_t orb = t / a.seg_len, loc = t - orb * a.seg_len;
    int64_t row = a.t1s[orb] + loc;
    vw_lunar_sat(row, s, a.orbit_res, a.day, a.tw, a.day_offset, &x, &y, &z);
  } else {
    const double* c = a.circ;
    int A = a.A;
    vw_circ_orbit(c[s], c[A + s], c[2 * A + s], (double)t * a.dt, c[3 * A + s], c[4 * A + s],
                  c[5 * A + s], c[6 * A + s], &x, &y, &z);
  }
  pos[k] = x;
  pos[TA + k] = y;
  pos[2 * TA + k] = z;
}

/* A segment's geometry in one launch: per (epoch, antenna) the frame px, py, pz,
 * invn, ux, uy, uz, cosphi and, for the antenna-factorized Viss (aph not null),
 * the phase coefficients (x - x_0) * 1e3 / lambda with x_0 the epoch's antenna 0
 * and (aphl, may be null) the part that the roundings of the difference, the
 * product and the quotient left out; per (epoch, pair) the half row. */
__global__ void k_seg_gen(const double* __restrict__ pos, int T, int A, int P, int t0, int tlen, double occ_r,
                          double cosphi_glob, const int32_t* __restrict__ pa, const int32_t* __restrict__ pb,
                          double lambda, double* __restrict__ ant8, double4* __restrict__ aph,
                          double4* __restrict__ aphl, RowRec* __restrict__ rows, double4* __restrict__ rowt,
                          uint64_t* __restrict__ ts) {
  vw_ts_begin(ts);
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t TA = (int64_t)T * A;
  if (k < (int64_t)tlen * A) {
    const int64_t src = (int64_t)t0 * A + k;
    const double x[3] = {pos[src], pos[TA + src], pos[2 * TA + src]};
    double in, ux, uy, uz, cp;
    vw_antenna_frame(x[0], x[1], x[2], occ_r, cosphi_glob, &in, &ux, &uy, &uz, &cp);
    double* q = ant8 + k * 8;
    q[0] = x[0]; q[1] = x[1]; q[2] = x[2]; q[3] = in;
    q[4] = ux; q[5] = uy; q[6] = uz; q[7] = cp;
    if (aph) {
      const int64_t ref = (t0 + k / A) * A;
      double r[3], l[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double xr = pos[c * TA + ref];
        const double d = x[c] - xr, bb = d - x[c], de = (x[c] - (d - bb)) - (xr + bb); /* d + de = x - xr */
        const double p = d * 1e3, pe = fma(d, 1e3, -p) + de * 1e3;
        r[c] = p / lambda;
        l[c] = (fma(-r[c], lambda, p) + pe) / lambda;
      }
      aph[k] = make_double4(r[0], r[1], r[2], 0.0);
      if (aphl) aphl[k] = make_double4(l[0], l[1], l[2], 0.0);
    }
  }
  if (k < (int64_t)tlen * P) {
    const int64_t g = k / P;
    const int j = (int)(k - g * P);
    const int64_t ka = (t0 + g) * A + pa[j], kb = (t0 + g) * A + pb[j];
    RowRec r;
    r.u = vw_uvw_comp(pos[ka], pos[kb], lambda);
    r.v = vw_uvw_comp(pos[TA + ka], pos[TA + kb], lambda);
    r.w = vw_uvw_comp(pos[2 * TA + ka], pos[2 * TA + kb], lambda);
    r.ia = (int32_t)(g * A + pa[j]);
    r.ib = (int32_t)(g * A + pb[j]);
    rows[k] = r;
    /* the plain Viss phase in 1/1024 turns (exact power-of-two scaling) */
    rowt[k] = make_double4(r.u * VW_TAB_SCALE, r.v * VW_TAB_SCALE, r.w * VW_TAB_SCALE, 0.0);
  }
  vw_ts_end(ts);
}

/* reference full-row layout (orbit_online.cuh:186-231) into 9 SoA arrays */
__global__ void k_seg_full(const double* __restrict__ pos, int T, int A, int P, int t0, int64_t nh,
                           const int32_t* __restrict__ pa, const int32_t* __restrict__ pb,
                           const RowRec* __restrict__ rows, double* __restrict__ out) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t nf = 2 * nh;
  if (i >= nf) return;
  int64_t TA = (int64_t)T * A;
  int64_t g = i / (2 * P);
  int jj = (int)(i - g * 2 * P);
  bool neg = jj >= P;
  int j = neg ? jj - P : jj;
  int64_t h = g * P + j;
  int64_t ka = (t0 + g) * A + pa[j], kb = (t0 + g) * A + pb[j];
  int64_t k1 = neg ? kb : ka, k2 = neg ? ka : kb;
  RowRec r = rows[h];
  out[0 * nf + i] = neg ? -r.u : r.u;
  out[1 * nf + i] = neg ? -r.v : r.v;
  out[2 * nf + i] = neg ? -r.w : r.w;
  out[3 * nf + i] = pos[k1];
  out[4 * nf + i] = pos[TA + k1];
  out[5 * nf + i] = pos[2 * TA + k1];
  out[6 * nf + i] = pos[k2];
  out[7 * nf + i] = pos[TA + k2];
  out[8 * nf + i] = pos[2 * TA + k2];
}

/* cone bits of every antenna frame against tiles [tile0, tile0+nt) ->
 * bytes [nt][nfr_pad] (bit0 all visible, bit1 all hidden); cone arrays hold
 * all ntile tiles.  A row's class only combines the bits of its two frames,
 * so the cone tests run once per (tile, frame) instead of twice per
 * (tile, row): tlen*A frames against tlen*A(A-1)/2 rows. */
__global__ void k_ant_bits(const double* __restrict__ cone, int64_t ntile, int64_t tile0, int64_t nt,
                           const double* __restrict__ ant8, int64_t nfr, int64_t nfr_pad, uint8_t* __restrict__ bits,
                           uint64_t* __restrict__ ts) {
  vw_ts_begin(ts);
  int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < nt * nfr_pad) {
    int64_t tr = k / nfr_pad, f = k - tr * nfr_pad;
    int64_t t = tile0 + tr;
    const double* q = ant8 + (f < nfr ? f : 0) * 8;
    const int b = vw_cone_bits(q[4], q[5], q[6], cone[t], cone[ntile + t], cone[2 * ntile + t], cone[3 * ntile + t],
                               cone[4 * ntile + t], q[7]);
    bits[k] = (uint8_t)(f < nfr ? b : 0);
  }
  vw_ts_end(ts);
}

/* the cone bits of tile t's nfr frames (as k_ant_bits) into LDS */
__device__ __forceinline__ void vw_tile_bits_lds(uint8_t* sb, const double* __restrict__ cone, int64_t ntile,
                                                 int64_t t, const double* __restrict__ ant8, int64_t nfr) {
  const double cx = cone[t], cy = cone[ntile + t], cz = cone[2 * ntile + t];
  const double cA = cone[3 * ntile + t], sA = cone[4 * ntile + t];
  for (int64_t f = threadIdx.x; f < nfr; f += blockDim.x) {
    const double* q = ant8 + f * 8;
    sb[f] = (uint8_t)vw_cone_bits(q[4], q[5], q[6], cx, cy, cz, cA, sA, q[7]);
  }
}

/* pair class per (tile, half row) for the tiles of a pass -> bytes
 * [tiles][nh_pad] (rows past nh: hidden), from the frame bits.  A block
 * covers VW_GCLS_BLOCK rows of one tile, four a thread written as one class
 * word.  The rows' frame indices pass through LDS (loaded with consecutive
 * lanes on consecutive records, read back four rows a thread), beside the
 * tile's row of cone bits staged in LDS (STAGE; nfr_pad bytes of dynamic
 * LDS) or, for longer rows, gathered from global memory. */
#define VW_GCLS_BLOCK 1024
template <bool STAGE>
__global__ __launch_bounds__(256) void k_classify(const uint8_t* __restrict__ bits, int64_t nfr_pad, int nhb,
                                                  const RowRec* __restrict__ rows, int64_t nh, int64_t nh_pad,
                                                  uint32_t* __restrict__ cls, uint64_t* __restrict__ ts) {
  extern __shared__ uint4 sbits[];
  __shared__ int4 sab[VW_GCLS_BLOCK / 2]; /* (ia, ib) of rows 2 k and 2 k + 1 */
  static_assert(VW_GCLS_BLOCK == 4 * 256, "four entries a thread");
  const uint32_t tr = blockIdx.x / (uint32_t)nhb, hc = blockIdx.x - tr * (uint32_t)nhb;
  const int64_t hb = (int64_t)hc * VW_GCLS_BLOCK;
  const uint8_t* row = bits + (int64_t)tr * nfr_pad;
  /* rows past nh are not frames: frame 0 stands in (the row array holds at
   * least one record) */
  int2* sab2 = (int2*)sab;
  int2 ab[4];
  int keep[4]; /* all ones for a row, zero past nh (a mask, not a select, so
                * the four loads stay unconditional and in flight together) */
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int64_t h = hb + threadIdx.x + 256 * k;
    keep[k] = -(int)(h < nh);
    ab[k] = *(const int2*)&rows[h < nh ? h : 0].ia;
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) sab2[threadIdx.x + 256 * k] = make_int2(ab[k].x & keep[k], ab[k].y & keep[k]);
  if (STAGE) {
    /* nfr_pad is a multiple of 64 and the row starts 64-byte aligned */
    for (int64_t i = threadIdx.x; i < nfr_pad / 16; i += 256) sbits[i] = ((const uint4*)row)[i];
  }
  __syncthreads();
  const int64_t h0 = hb + 4 * threadIdx.x;
  if (h0 >= nh_pad) return; /* nh_pad is a multiple of 64: whole words only */
  const int4 p0 = sab[2 * threadIdx.x], p1 = sab[2 * threadIdx.x + 1];
  const int av[4] = {p0.x, p0.z, p1.x, p1.z}, bv[4] = {p0.y, p0.w, p1.y, p1.w};
  const uint8_t* b = STAGE ? (const uint8_t*)sbits : row;
  uint32_t w = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t c = (uint32_t)vw_pair_class(b[av[e]], b[bv[e]]);
    w |= (h0 + e < nh ? c : (uint32_t)VW_CLS_HIDDEN) << (8 * e);
  }
  cls[((int64_t)tr * nh_pad + h0) >> 2] = w;
  vw_ts_end(ts); /* thread 0 of a workgroup has rows */
}

/* k_classify with the cone bits made in place: one block per tile of the
 * pass computes the tile's frame bits into LDS (nfr bytes of dynamic LDS),
 * then walks the tile's rows VW_GCLS_BLOCK at a time as k_classify does, so
 * no bit table passes through global memory and each cone test runs once */
__global__ __launch_bounds__(256) void k_classify_tile(const double* __restrict__ cone, int64_t ntile,
                                                       int64_t tile0, const double* __restrict__ ant8, int64_t nfr,
                                                       const RowRec* __restrict__ rows, int64_t nh, int64_t nh_pad,
                                                       uint32_t* __restrict__ cls, uint64_t* __restrict__ ts) {
  vw_ts_begin(ts);
  extern __shared__ uint4 sbits[];
  __shared__ int4 sab[VW_GCLS_BLOCK / 2]; /* (ia, ib) of rows 2 k and 2 k + 1 */
  const int64_t tr = blockIdx.x;
  uint8_t* sb = (uint8_t*)sbits;
  vw_tile_bits_lds(sb, cone, ntile, tile0 + tr, ant8, nfr);
  int2* sab2 = (int2*)sab;
  for (int64_t hb = 0; hb < nh_pad; hb += VW_GCLS_BLOCK) {
    int2 ab[4];
    int keep[4]; /* a mask, not a select: the four loads stay in flight together */
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t h = hb + threadIdx.x + 256 * k;
      keep[k] = -(int)(h < nh);
      ab[k] = *(const int2*)&rows[h < nh ? h : 0].ia;
    }
    __syncthreads(); /* the bits are in; the last pass's reads of sab are done */
#pragma unroll
    for (int k = 0; k < 4; ++k) sab2[threadIdx.x + 256 * k] = make_int2(ab[k].x & keep[k], ab[k].y & keep[k]);
    __syncthreads();
    const int64_t h0 = hb + 4 * threadIdx.x;
    if (h0 < nh_pad) {
      const int4 p0 = sab[2 * threadIdx.x], p1 = sab[2 * threadIdx.x + 1];
      const int av[4] = {p0.x, p0.z, p1.x, p1.z}, bv[4] = {p0.y, p0.w, p1.y, p1.w};
      uint32_t w = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t c = (uint32_t)vw_pair_class(sb[av[e]], sb[bv[e]]);
        w |= (h0 + e < nh ? c : (uint32_t)VW_CLS_HIDDEN) << (8 * e);
      }
      cls[(tr * nh_pad + h0) >> 2] = w;
    }
  }
  vw_ts_end(ts);
}

/* effective mask of rows [row0, row0+nrows) x pixels (introspection) */
__global__ void k_masks(const double* __restrict__ l, const double* __restrict__ m, const double* __restrict__ n,
                        int64_t npix, int64_t TP, const uint8_t* __restrict__ cls, int64_t nh_pad,
                        const RowRec* __restrict__ rows, const double* __restrict__ ant8, int64_t row0,
                        int64_t nrows, uint8_t* __restrict__ mask) {
  int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nrows * npix) return;
  int64_t r = k / npix, p = k - r * npix;
  int64_t h = row0 + r;
  int c = cls[(p / TP) * nh_pad + h];
  uint8_t v;
  if (c == VW_CLS_VISIBLE) v = 1;
  else if (c == VW_CLS_HIDDEN) v = 0;
  else {
    RowRec rr = rows[h];
    const double* qa = ant8 + (int64_t)rr.ia * 8;
    const double* qb = ant8 + (int64_t)rr.ib * 8;
    v = (uint8_t)(vw_visible(l[p], m[p], n[p], qa[0], qa[1], qa[2], qa[3], qa[7]) &&
                  vw_visible(l[p], m[p], n[p], qb[0], qb[1], qb[2], qb[3], qb[7]));
  }
  mask[k] = v;
}

/* ------------------------------------------------------------------ */
/* Viss                                                                 */
/* ------------------------------------------------------------------ */
struct VissArgs {
  const double2* tab; /* the sine table (plain forms), built once per context */
  const double *l, *m, *n, *nm1, *B;
  const float* Bf;
  int64_t npix;
  int64_t tile0, ntile; /* tiles of this pass: [tile0, tile0 + ntile) */
  const RowRec* rows;
  const double4* rowt; /* (u, v, w) * 1024 per half row (plain form) */
  const double* ant8;
  const uint32_t* cls; /* [ntile][nh_pad] bytes (pass-relative) viewed as words */
  int64_t nh, nh_pad;
  int64_t tpc, nchunk, nrb, bpc;
  double2* part; /* [nchunk][nh_pad] */
  int64_t* cpart; /* [nchunk][nh_pad] (counting instance) */
};

/* the sine table: entry k = (cos, sin)(2 pi k / N), as vw_sincos_tab_build;
 * built once per context in device memory, copied into LDS by every
 * workgroup of the plain kernels (four 16-byte loads a thread) */
__global__ void k_tab_build(double2* __restrict__ tab) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= VW_TAB_N) return;
  double e[2]; /* (cos, sin) */
  vw_sincos_turn((double)i / (double)VW_TAB_N, &e[1], &e[0]);
  tab[i] = make_double2(e[0], e[1]);
}
__device__ __forceinline__ void vw_tab_fill(double2* tab, const double2* __restrict__ src) {
  for (int i = threadIdx.x; i < VW_TAB_N; i += blockDim.x) tab[i] = src[i];
}

__device__ __forceinline__ void vw_hw_sincos_turn(float r, float* s, float* c) {
  *s = __builtin_amdgcn_sinf(r);
  *c = __builtin_amdgcn_cosf(r);
}

/* occlusion of the PPL pixels of a lane against both endpoints of a row: the
 * plain kernels evaluate both tests without short circuit (straight-line
 * code, no exec-mask branches); the mixed kernels, at their tighter register
 * budget, keep the short-circuit form */
template <bool BRANCHFREE>
__device__ __forceinline__ bool vw_vis2(bool ok, double l, double m, double n, double ax, double ay, double az,
                                        double ai, double ac, double bx, double by, double bz, double bi, double bc) {
  if (BRANCHFREE)
    return ((int)ok & vw_visible(l, m, n, ax, ay, az, ai, ac) & vw_visible(l, m, n, bx, by, bz, bi, bc)) != 0;
  return ok && vw_visible(l, m, n, ax, ay, az, ai, ac) && vw_visible(l, m, n, bx, by, bz, bi, bc);
}

/* mixed form, one term: accumulate bf * exp(-j 2 pi x) in FP32 (the sign of
 * the imaginary part is applied when the partial is written) */
__device__ __forceinline__ void vw_viss_term_mixed(const RowRec& rec, double l, double m, double nm1, float bf,
                                                   float& fre, float& fim) {
  const double x = vw_viss_phase(rec.u, rec.v, rec.w, l, m, nm1);
  const float f = (float)__builtin_amdgcn_fract(x);
  float s, c;
  vw_hw_sincos_turn(f, &s, &c);
  fre = fmaf(bf, c, fre);
  fim = fmaf(bf, s, fim);
}

/* plain form, the PPL terms of one lane for one half row: phases (operands
 * pre-scaled by 1024), all table indices, the table reads, then polynomials
 * and rotations, so the LDS reads overlap the arithmetic */
/* The pixel weight bw is folded into the polynomial coefficients once per
 * sub-tile: w0 = bw, w1 = bw a, w2 = bw (-a^2/2), w3 = bw (-a^3/6) give
 *   bw cy = w0 + w2 z,  bw sy = f (w1 + w3 z),
 * and the rotation by the table entry (ec, es) is accumulated directly:
 *   dre += ec (bw cy) - es (bw sy),  dim += es (bw cy) + ec (bw sy),
 * four FMAs, two products fewer per term than rotating, then weighting.
 * MASK: a pixel with vis[k] false adds nothing (selects on bw cy, bw sy). */
template <int PPL, bool MASK>
__device__ __forceinline__ void vw_viss_terms_plain(const double4& rt, const double* pl, const double* pm,
                                                    const double* pz, const double* w0, const double* w1,
                                                    const double* w2, const double* w3, const bool* vis,
                                                    const double2* tab, double& dre, double& dim) {
  double f[PPL];
  int ix[PPL];
#pragma unroll
  for (int k = 0; k < PPL; ++k) f[k] = vw_tab_split(vw_viss_phase(rt.x, rt.y, rt.z, pl[k], pm[k], pz[k]), &ix[k]);
  double2 e[PPL];
#pragma unroll
  for (int k = 0; k < PPL; ++k) e[k] = tab[ix[k]];
#pragma unroll
  for (int k = 0; k < PPL; ++k) {
    const double z = f[k] * f[k];
    double cw = fma(z, w2[k], w0[k]);
    double sw = f[k] * fma(z, w3[k], w1[k]);
    if (MASK) {
      cw = vis[k] ? cw : 0.0;
      sw = vis[k] ? sw : 0.0;
    }
    dre = fma(-e[k].y, sw, fma(e[k].x, cw, dre));
    dim = fma(e[k].x, sw, fma(e[k].y, cw, dim));
  }
}

/* occupancy: the plain form keeps 8 FP64 row sums and 4 weight
 * coefficients per pixel per lane at 3 waves per SIMD; the mixed form (16
 * FP32 row sums) runs 5 (measured best) */
#ifndef VW_VISS_WAVES_PLAIN
#define VW_VISS_WAVES_PLAIN 3
#endif
#ifndef VW_VISS_WAVES_MIXED
#define VW_VISS_WAVES_MIXED 5
#endif
/* per-row Viss, mixed form (the plain form is k_viss_plain) */
template <int TP, int RPW, bool COUNT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(VW_VISS_WAVES_MIXED))) void k_viss(VissArgs a) {
  /* a tile is walked in sub-tiles of 256 pixels (4 per lane), so the
   * register footprint does not grow with the tile size */
  constexpr int PPL = 4;
  constexpr int NSUB = TP / 256;
  static_assert(RPW % 4 == 0, "class words hold 4 rows");
  const int64_t vb = vw_xcd_block(blockIdx.x, gridDim.x);
  const int64_t chunk = vb / a.bpc;
  const int wave = vw_rfl((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int64_t rb = (vb - chunk * a.bpc) * 4 + wave;
  if (chunk >= a.nchunk || rb >= a.nrb) return;
  const int64_t r0 = rb * RPW; /* r0 + RPW <= nh_pad: nh_pad is a multiple of 64 */
  const int64_t t0 = a.tile0 + chunk * a.tpc;
  const int64_t tend = a.tile0 + a.ntile;
  const int64_t t1 = (t0 + a.tpc < tend) ? t0 + a.tpc : tend;

  float fre[RPW], fim[RPW];
  int cnt[RPW];
#pragma unroll
  for (int r = 0; r < RPW; ++r) { fre[r] = 0.f; fim[r] = 0.f; cnt[r] = 0; }

  for (int64_t st = t0 * NSUB; st < t1 * NSUB; ++st) {
    const int64_t tile = st / NSUB;
    /* the class bytes of this wave's RPW rows for the tile: RPW/4 uniform words */
    uint32_t cw[RPW / 4];
    const uint32_t* cwp = a.cls + (((tile - a.tile0) * a.nh_pad + r0) >> 2);
#pragma unroll
    for (int j = 0; j < RPW / 4; ++j) cw[j] = (uint32_t)vw_rfl((int)cwp[j]);
    double pl[PPL], pm[PPL], pn[PPL], pz[PPL];
    float pbf[PPL];
    bool ok[PPL];
#pragma unroll
    for (int k = 0; k < PPL; ++k) {
      int64_t p = st * 256 + lane + 64 * k;
      ok[k] = p < a.npix;
      int64_t pp = ok[k] ? p : 0;
      pl[k] = a.l[pp];
      pm[k] = a.m[pp];
      pn[k] = a.n[pp];
      pz[k] = a.nm1[pp];
      /* weights are zero outside the sky, so the visible path needs no mask */
      pbf[k] = ok[k] ? a.Bf[pp] : 0.0f;
    }
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
      const int64_t h = r0 + r;
      /* rows past nh carry the hidden class */
      const int cls = (int)((cw[r >> 2] >> (8 * (r & 3))) & 0xffu);
      if (cls == VW_CLS_VISIBLE) {
        const RowRec rec = a.rows[h];
#pragma unroll
        for (int k = 0; k < PPL; ++k) vw_viss_term_mixed(rec, pl[k], pm[k], pz[k], pbf[k], fre[r], fim[r]);
        if (COUNT) {
#pragma unroll
          for (int k = 0; k < PPL; ++k) cnt[r] += ok[k] ? 1 : 0;
        }
      } else if (cls == VW_CLS_MIXED) {
        const RowRec rec = a.rows[h];
        const double* qa = a.ant8 + (int64_t)rec.ia * 8;
        const double* qb = a.ant8 + (int64_t)rec.ib * 8;
        const double ax = qa[0], ay = qa[1], az = qa[2], ai = qa[3], ac = qa[7];
        const double bx = qb[0], by = qb[1], bz = qb[2], bi = qb[3], bc = qb[7];
        bool vis[PPL];
#pragma unroll
        for (int k = 0; k < PPL; ++k)
          vis[k] = vw_vis2<true>(ok[k], pl[k], pm[k], pn[k], ax, ay, az, ai, ac, bx, by, bz, bi, bc);
#pragma unroll
        for (int k = 0; k < PPL; ++k)
          vw_viss_term_mixed(rec, pl[k], pm[k], pz[k], vis[k] ? pbf[k] : 0.f, fre[r], fim[r]);
        if (COUNT) {
#pragma unroll
          for (int k = 0; k < PPL; ++k) cnt[r] += vis[k] ? 1 : 0;
        }
      }
    }
  }
  /* one cross-lane tree per row; FP64 above the per-lane FP32 blocks */
#pragma unroll
  for (int r = 0; r < RPW; ++r) {
    const int64_t h = r0 + r;
    double re = vw_wave_sum((double)fre[r]);
    double im = vw_wave_sum((double)fim[r]);
    int64_t cc = 0;
    if (COUNT) cc = vw_wave_sum_i((int64_t)cnt[r]);
    if (lane == 0 && h < a.nh) {
      a.part[chunk * a.nh_pad + h] = make_double2(re, -im);
      if (COUNT) a.cpart[chunk * a.nh_pad + h] = cc;
    }
  }
}

/* Plain per-row Viss with the pixel data prefetched into LDS.  Each wave
 * keeps its own LDS copy of the next sub-tile's l, m, n and weights, written
 * by direct global-to-LDS loads (16 bytes a lane: two neighbouring pixels)
 * while the current sub-tile is summed, together with the next class words;
 * a sub-tile then starts with LDS reads, and no registers hold the data in
 * flight.  Nothing else in the sub-tile loop reads global memory, so the
 * loop never waits on the prefetch: the wave's rows are read once up front
 * ((u, v, w) into scalar registers, the antenna data of the occlusion
 * predicates into LDS).  Lane i owns pixels 128 j + 2 i + e (j, e in {0, 1})
 * of a 256-pixel sub-tile; pixel counts are even, so a pair is in the sky or
 * out of it whole, and pairs outside it read pixels 0 and 1 under a zero
 * weight.  n - 1 is formed as in k_pix2lmn.  Terms, masks and partials as
 * k_viss. */
template <int TP, int RPW, bool COUNT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(VW_VISS_WAVES_PLAIN))) void k_viss_plain(
    VissArgs a) {
  constexpr int PPL = 4;
  constexpr int SUB = 64 * PPL;
  constexpr int NSUB = TP / SUB;
  constexpr int NCW = RPW / 4; /* class words per sub-tile */
  static_assert(RPW % 4 == 0 && NCW <= 64, "class words hold 4 rows");
  static_assert(TP % SUB == 0, "tiles hold whole sub-tiles");
  __shared__ double2 tab[VW_TAB_N];
  __shared__ double2 pre[4][4][2][64]; /* [wave][l, m, n, B][half][lane] */
  __shared__ double rant[4][RPW][10];  /* [wave][row][antenna a (x y z i c), b (...)] */
  vw_tab_fill(tab, a.tab);
  __syncthreads();
  const int64_t vb = vw_xcd_block(blockIdx.x, gridDim.x);
  const int64_t chunk = vb / a.bpc;
  const int wave = vw_rfl((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int64_t rb = (vb - chunk * a.bpc) * 4 + wave;
  if (chunk >= a.nchunk || rb >= a.nrb) return;
  const int64_t r0 = rb * RPW; /* r0 + RPW <= nh_pad: nh_pad is a multiple of 64 */
  const int64_t t0 = a.tile0 + chunk * a.tpc;
  const int64_t tend = a.tile0 + a.ntile;
  const int64_t t1 = (t0 + a.tpc < tend) ? t0 + a.tpc : tend;
  const int64_t s0 = t0 * NSUB, s1 = t1 * NSUB;

  /* the wave's rows; rows past nh are hidden and never summed */
  double4 rt[RPW];
#pragma unroll
  for (int r = 0; r < RPW; ++r) rt[r] = (r0 + r < a.nh) ? a.rowt[r0 + r] : make_double4(0.0, 0.0, 0.0, 0.0);
  if (lane < RPW && r0 + lane < a.nh) {
    const RowRec rec = a.rows[r0 + lane];
    const double* qa = a.ant8 + (int64_t)rec.ia * 8;
    const double* qb = a.ant8 + (int64_t)rec.ib * 8;
    double* d = rant[wave][lane];
    d[0] = qa[0]; d[1] = qa[1]; d[2] = qa[2]; d[3] = qa[3]; d[4] = qa[7];
    d[5] = qb[0]; d[6] = qb[1]; d[7] = qb[2]; d[8] = qb[3]; d[9] = qb[7];
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

  typedef __attribute__((address_space(3))) void* lds_ptr;
  uint32_t cwn = 0; /* lane j < NCW: class word j of the prefetched sub-tile */
  auto prefetch = [&](int64_t s) {
    const double* src[4] = {a.l, a.m, a.n, a.B};
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int64_t p = s * SUB + 128 * j + 2 * lane;
      const int64_t pp = p < a.npix ? p : 0;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        __builtin_amdgcn_global_load_lds((const void*)(src[q] + pp), (lds_ptr)&pre[wave][q][j][0], 16, 0, 0);
    }
    const uint32_t* cwp = a.cls + ((((s / NSUB) - a.tile0) * a.nh_pad + r0) >> 2);
    cwn = cwp[lane < NCW ? lane : 0];
  };

  double dre[RPW], dim[RPW];
  int cnt[RPW];
#pragma unroll
  for (int r = 0; r < RPW; ++r) { dre[r] = 0.0; dim[r] = 0.0; cnt[r] = 0; }

  prefetch(s0);
  for (int64_t st = s0; st < s1; ++st) {
    /* this sub-tile's prefetch has landed */
    __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
    uint32_t cw[NCW];
#pragma unroll
    for (int j = 0; j < NCW; ++j) cw[j] = (uint32_t)__builtin_amdgcn_readlane((int)cwn, j);
    double pl[PPL], pm[PPL], pn[PPL], pz[PPL], w0[PPL], w1[PPL], w2[PPL], w3[PPL];
    bool ok[PPL];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const double2 L = pre[wave][0][j][lane], M = pre[wave][1][j][lane];
      const double2 N = pre[wave][2][j][lane], W = pre[wave][3][j][lane];
      pl[2 * j] = L.x;
      pl[2 * j + 1] = L.y;
      pm[2 * j] = M.x;
      pm[2 * j + 1] = M.y;
      pn[2 * j] = N.x;
      pn[2 * j + 1] = N.y;
      const bool okj = st * SUB + 128 * j + 2 * lane < a.npix;
      ok[2 * j] = okj;
      ok[2 * j + 1] = okj;
      w0[2 * j] = okj ? W.x : 0.0;
      w0[2 * j + 1] = okj ? W.y : 0.0;
    }
    /* the reads are done before the buffer is refilled */
    __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (st + 1 < s1) prefetch(st + 1);
#pragma unroll
    for (int k = 0; k < PPL; ++k) {
      pz[k] = pn[k] - 1.0;
      w1[k] = w0[k] * VW_SHORT_S1;
      w2[k] = w0[k] * VW_SHORT_C2;
      w3[k] = w0[k] * VW_SHORT_S3;
    }
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
      /* rows past nh carry the hidden class */
      const int cls = (int)((cw[r >> 2] >> (8 * (r & 3))) & 0xffu);
      if (cls == VW_CLS_VISIBLE) {
        vw_viss_terms_plain<PPL, false>(rt[r], pl, pm, pz, w0, w1, w2, w3, ok, tab, dre[r], dim[r]);
        if (COUNT) {
#pragma unroll
          for (int k = 0; k < PPL; ++k) cnt[r] += ok[k] ? 1 : 0;
        }
      } else if (cls == VW_CLS_MIXED) {
        const double* d = rant[wave][r];
        const double ax = d[0], ay = d[1], az = d[2], ai = d[3], ac = d[4];
        const double bx = d[5], by = d[6], bz = d[7], bi = d[8], bc = d[9];
        bool vis[PPL];
#pragma unroll
        for (int k = 0; k < PPL; ++k)
          vis[k] = vw_vis2<true>(ok[k], pl[k], pm[k], pn[k], ax, ay, az, ai, ac, bx, by, bz, bi, bc);
        vw_viss_terms_plain<PPL, true>(rt[r], pl, pm, pz, w0, w1, w2, w3, vis, tab, dre[r], dim[r]);
        if (COUNT) {
#pragma unroll
          for (int k = 0; k < PPL; ++k) cnt[r] += vis[k] ? 1 : 0;
        }
      }
    }
  }
  /* one cross-lane tree per row */
#pragma unroll
  for (int r = 0; r < RPW; ++r) {
    const int64_t h = r0 + r;
    const double re = vw_wave_sum(dre[r]);
    const double im = vw_wave_sum(dim[r]);
    int64_t cc = 0;
    if (COUNT) cc = vw_wave_sum_i((int64_t)cnt[r]);
    if (lane == 0 && h < a.nh) {
      a.part[chunk * a.nh_pad + h] = make_double2(re, -im);
      if (COUNT) a.cpart[chunk * a.nh_pad + h] = cc;
    }
  }
}

/* adjoint of the plain Viss sum (a real-linear map from pixel weights to
 * raw half visibilities): for one tile pass and one chunk of half rows,
 * g_p = sum_h M_hp Re(r_h exp(+j 2 pi (u l + v m + w (n-1)))) per pixel,
 * with the effective mask M of the Viss (tile class, then the per-pixel
 * predicate on partly visible tiles) and its table sincos.  A wave owns one
 * 256-pixel sub-tile (4 pixels per lane) and a chunk of rows; rows are
 * wave-uniform, their class one byte of a uniform class word.  Partials
 * [chunk][pixel of the pass]; the fold applies the pixel area. */
struct VissAdjArgs {
  const double2* tab; /* the sine table (plain forms), built once per context */
  const double *l, *m, *n, *nm1;
  int64_t npix;
  int64_t tile0, ntile; /* tiles of this pass: [tile0, tile0 + ntile) */
  const RowRec* rows;
  const double4* rowt; /* (u, v, w) * 1024 per half row */
  const double* ant8;
  const uint32_t* cls; /* [ntile][nh_pad] bytes (pass-relative) viewed as words */
  int64_t nh, nh_pad;
  const double2* res;  /* [nh] residual half visibilities (raw convention) */
  int64_t rpc, nchunk; /* rows per chunk (a multiple of 4), chunks */
  int64_t nsub;        /* 256-pixel sub-tiles of the pass */
  double* part;        /* [nchunk][nsub * 256] */
};

template <int TP>
__global__ __launch_bounds__(256) void k_viss_adj(VissAdjArgs a) {
  constexpr int PPL = 4;
  __shared__ double2 tab[VW_TAB_N];
  vw_tab_fill(tab, a.tab);
  __syncthreads();
  const int wave = vw_rfl((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int64_t wv = (int64_t)blockIdx.x * 4 + wave;
  const int64_t chunk = wv / a.nsub, sub = wv - chunk * a.nsub;
  if (chunk >= a.nchunk) return;
  const int64_t p0 = a.tile0 * TP + sub * 256; /* first pixel of the sub-tile */
  const int64_t tile = p0 / TP;
  const int64_t h0 = chunk * a.rpc;
  const int64_t h1 = h0 + a.rpc < a.nh ? h0 + a.rpc : a.nh;
  double pl[PPL], pm[PPL], pn[PPL], pz[PPL], acc[PPL];
  bool ok[PPL];
#pragma unroll
  for (int k = 0; k < PPL; ++k) {
    const int64_t p = p0 + lane + 64 * k;
    ok[k] = p < a.npix;
    const int64_t pp = ok[k] ? p : 0;
    pl[k] = a.l[pp];
    pm[k] = a.m[pp];
    pn[k] = a.n[pp];
    pz[k] = a.nm1[pp];
    acc[k] = 0.0;
  }
  const uint32_t* cwp = a.cls + (((tile - a.tile0) * a.nh_pad) >> 2);
  for (int64_t h4 = h0; h4 < h1; h4 += 4) {
    const uint32_t cw = (uint32_t)vw_rfl((int)cwp[h4 >> 2]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t h = h4 + j;
      const int cls = (int)((cw >> (8 * j)) & 0xffu);
      if (h >= h1 || cls == VW_CLS_HIDDEN) continue;
      const double2 r = a.res[h];
      bool mk[PPL];
      if (cls == VW_CLS_VISIBLE) {
#pragma unroll
        for (int k = 0; k < PPL; ++k) mk[k] = ok[k];
      } else {
        const RowRec rec = a.rows[h];
        const double* qa = a.ant8 + (int64_t)rec.ia * 8;
        const double* qb = a.ant8 + (int64_t)rec.ib * 8;
#pragma unroll
        for (int k = 0; k < PPL; ++k)
          mk[k] = vw_vis2<true>(ok[k], pl[k], pm[k], pn[k], qa[0], qa[1], qa[2], qa[3], qa[7], qb[0], qb[1], qb[2],
                                qb[3], qb[7]);
      }
      const double4 rt = a.rowt[h];
      double f[PPL];
      int ix[PPL];
#pragma unroll
      for (int k = 0; k < PPL; ++k) f[k] = vw_tab_split(vw_viss_phase(rt.x, rt.y, rt.z, pl[k], pm[k], pz[k]), &ix[k]);
      double2 e[PPL];
#pragma unroll
      for (int k = 0; k < PPL; ++k) e[k] = tab[ix[k]];
#pragma unroll
      for (int k = 0; k < PPL; ++k) {
        double sy, cy, sn, cs;
        vw_tab_poly_short(f[k], &sy, &cy);
        vw_tab_rotate(e[k].x, e[k].y, sy, cy, &sn, &cs);
        /* Re(r exp(+j x)) = r.x cos x - r.y sin x */
        const double t = fma(r.x, cs, fma(-r.y, sn, acc[k]));
        acc[k] = mk[k] ? t : acc[k];
      }
    }
  }
  const int64_t stride = a.nsub * 256;
#pragma unroll
  for (int k = 0; k < PPL; ++k) a.part[chunk * stride + sub * 256 + lane + 64 * k] = acc[k];
}

/* adjoint partials of a pass -> g[p] = area * sum over chunks (ascending) */
__global__ void k_viss_adj_fold(const double* __restrict__ part, int64_t nchunk, int64_t stride, int64_t p0,
                                int64_t np, double area, double* __restrict__ g) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np) return;
  double s = 0.0;
  for (int64_t k = 0; k < nchunk; ++k) s = s + part[k * stride + i];
  g[p0 + i] = area * s;
}

/* a raw half sum, phase-corrected (vh not null: whole steps, where the
 * correction is no stage of its own) */
__device__ __forceinline__ void vw_store_half(double2* __restrict__ vraw, double2* __restrict__ vh,
                                              const RowRec* __restrict__ rows, int64_t h, double re, double im) {
  vraw[h] = make_double2(re, im);
  if (vh) {
    double cr, ci;
    vw_phase_correct(re, im, rows[h].w, &cr, &ci);
    vh[h] = make_double2(cr, ci);
  }
}

/* partials -> raw half sums, chunks folded in ascending order; passes after
 * the first add to the running sums */
__global__ void k_viss_reduce(const double2* __restrict__ part, int64_t nchunk, int64_t nh, int64_t nh_pad,
                              int accumulate, double2* __restrict__ vraw, const int64_t* __restrict__ cpart,
                              int64_t* __restrict__ counts, const RowRec* __restrict__ rows,
                              double2* __restrict__ vh, uint64_t* __restrict__ ts) {
  vw_ts_begin(ts);
  int64_t h = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (h >= nh) return;
  double re = 0.0, im = 0.0;
  int64_t c = 0;
  /* VW_FOLD_BATCH chunks' loads in flight at a time; the sums keep chunk order */
  int64_t k = 0;
  for (; k + VW_FOLD_BATCH <= nchunk; k += VW_FOLD_BATCH) {
    double2 v[VW_FOLD_BATCH];
#pragma unroll
    for (int e = 0; e < VW_FOLD_BATCH; ++e) v[e] = part[(k + e) * nh_pad + h];
#pragma unroll
    for (int e = 0; e < VW_FOLD_BATCH; ++e) {
      re += v[e].x;
      im += v[e].y;
    }
    if (counts) {
#pragma unroll
      for (int e = 0; e < VW_FOLD_BATCH; ++e) c += cpart[(k + e) * nh_pad + h];
    }
  }
  for (; k < nchunk; ++k) {
    double2 v = part[k * nh_pad + h];
    re += v.x;
    im += v.y;
    if (counts) c += cpart[k * nh_pad + h];
  }
  if (accumulate) {
    double2 o = vraw[h];
    re = o.x + re;
    im = o.y + im;
    if (counts) c += counts[h];
  }
  vw_store_half(vraw, vh, rows, h, re, im);
  if (counts) counts[h] = c;
  vw_ts_end(ts); /* thread 0 of a workgroup has a row */
}

/* ------------------------------------------------------------------ */
/* Viss, antenna-factorized form on the matrix cores                    */
/* ------------------------------------------------------------------ */
/* The phase of half row (a, b) is a difference of antenna phases,
 *   u l + v m + w (n-1) = psi_b - psi_a,  psi_x = (x - x_0).(l, m, n-1) 1e3/lambda
 * (x_0: the epoch's antenna 0, which cancels), and its mask is a product of
 * per-antenna masks (below).  With e_x = exp(+2 pi j psi_x) = c_x + j s_x one
 * epoch's half visibilities are entries of
 *   V[a][b] = sum_p I_p m_a m_b e_a conj(e_b):
 *   Re V = Y11[a][b] + Y22[a][b],  Im V = Y21[a][b] - Y21[b][a],
 *   Y11 = sum I c c^T,  Y22 = sum I s s^T,  Y21 = sum I s c^T,
 * three real (16 x 4) x (4 x 16) products per 4 pixels and 16 antennas on
 * the FP64 matrix cores (FP32 in the mixed form), where the row form
 * evaluates 120 phase / sin / cos terms per pixel one by one.  Lane l
 * computes the exponential of antenna 16 gi + l % 16 at pixel l / 16 of the
 * step, which is at once its A operand (row, k) and its B operand (k, column)
 * element.  Accumulator layout (measured on gfx950): FP64 lane l register r
 * holds D[l/16 + 4r][l%16]; FP32 D[4(l/16) + r][l%16].
 *
 * Masks.  The mask of row (a, b) on a pixel is 1 when both endpoint cones
 * hold the tile (class visible), 0 when either cone misses it (hidden), else
 * the product of the two per-pixel predicates.  In a tile where no antenna
 * is partly visible the per-antenna mask m = hidden ? 0 : 1 gives exactly
 * that; otherwise m = hidden ? 0 : predicate does, unless the predicate of an
 * all-visible antenna fails on a pixel of the tile (the cone bound is
 * conservative, so only rounding at the horizon can do that), which would
 * drop terms of pairs of two all-visible antennas.  The summing pass flags
 * that case; the tile then gets a correction pass adding, for those pairs,
 *   Y += sum_p I_p (o_a o_b - o_a p_a o_b p_b) (...)   (o: all-visible),
 * two more products per block on the same accumulators. */
typedef double vw_d4 __attribute__((ext_vector_type(4)));
typedef float vw_f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ vw_d4 vw_mfma(double a, double b, vw_d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ vw_f4 vw_mfma(float a, float b, vw_f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

struct VissFArgs {
  const double2* tab; /* the sine table (plain forms), built once per context */
  const double *l, *m, *n, *nm1, *B;
  const float* Bf;
  int64_t npix;
  int64_t tile0, ntile;   /* tiles of this pass: [tile0, tile0 + ntile) */
  const double4* aph;     /* [tlen*A] (x - x_0) * 1e3 / lambda per antenna frame */
  const double4* aphl;    /* what its roundings left out (plain form)           */
  const double* ant8;     /* [tlen*A][8] antenna frames */
  const uint8_t* bits;    /* [ntile][nfr_pad] cone bits, pass-relative tiles */
  int64_t nfr_pad;
  int32_t A, tlen;
  int64_t tpc, nchunk, nquad;
  int32_t check;          /* 1: every tile with a partly visible antenna takes the two-mask sum */
  double* part;           /* [tlen][nchunk][NB][256] */
};

/* blocks of one wave's accumulators for G groups of 16 antennas: Y11 and Y22
 * for gi >= gj (symmetric), Y21 for all (gi, gj) */
template <int G> struct VfShape {
  static constexpr int NS = G * (G + 1) / 2;
  static constexpr int NB = NS + G * G; /* partial blocks: Re = Y11 + Y22 (NS), Y21 (G*G) */
};

/* one tile's pixel data staged in LDS for the four waves of a workgroup
 * (weights zero past the end of the sky) */
template <int TP> struct VfTileLds {
  double l[TP], m[TP], n[TP], nm1[TP], w[TP];
};

template <int G> struct VfLane {
  double kx[G], ky[G], kz[G];                 /* phase coefficients, turns        */
  double jx[G], jy[G], jz[G];                 /* their low parts (plain form)     */
  double px[G], py[G], pz[G], pinv[G], pcos[G]; /* predicate frame */
};

/* An antenna's phase in turns, up to whole turns: the fractions of the three
 * products, each exact before its one rounding (a multiply-add from the
 * product's nearest integer), with the low parts of the coefficients.  A row is
 * the difference of two such phases, so plain products would double the variance
 * of the row form's phase rounding; these 14 operations leave 2^-52 turns, and
 * most of them run under the products on the matrix cores (Nside 256, 16
 * epochs: 0.525 -> 0.583 ms with 16 antennas, 1.31 -> 1.41 ms with 32). */
__device__ __forceinline__ double vw_ant_phase_frac(double kx, double ky, double kz, double jx, double jy, double jz,
                                                    double l, double m, double nm1) {
  const double f1 = fma(kx, l, -rint(kx * l)), f2 = fma(ky, m, -rint(ky * m)), f3 = fma(kz, nm1, -rint(kz * nm1));
  return (fma(jx, l, f1) + fma(jy, m, f2)) + fma(jz, nm1, f3);
}

/* the product-mask sum of one tile.  PRED false (no partly visible
 * antenna in the tile): m = hidden ? 0 : 1.  PRED: m = hidden ? 0 :
 * predicate, and the return value is nonzero when the predicate of an
 * all-visible antenna failed on some pixel of the tile.  CORR:
 * the correction pass instead, for pairs of two all-visible antennas
 * (o = all-visible): Y += sum w (o_a o_b - o_a p_a o_b p_b) (...). */
template <int TP, int G, bool MIXED, bool PRED, bool CORR>
__device__ __forceinline__ uint64_t vf_tile(const VfTileLds<TP>& px, const VfLane<G>& L, const int (&bt)[G],
                                            const double2* tab,
                                            typename std::conditional<MIXED, vw_f4, vw_d4>::type (&y11)[VfShape<G>::NS],
                                            typename std::conditional<MIXED, vw_f4, vw_d4>::type (&y22)[VfShape<G>::NS],
                                            typename std::conditional<MIXED, vw_f4, vw_d4>::type (&y21)[G * G]) {
  using T = typename std::conditional<MIXED, float, double>::type;
  constexpr bool NEED_N = PRED || CORR;
  const int q = (threadIdx.x & 63) >> 4;
  bool vis[G], allv[G];
  uint64_t allm[G]; /* lanes whose antenna of group gi is all-visible */
#pragma unroll
  for (int gi = 0; gi < G; ++gi) {
    vis[gi] = (bt[gi] & 2) == 0;
    allv[gi] = (bt[gi] & 1) != 0;
    allm[gi] = __ballot(allv[gi]);
  }
  uint64_t failed = 0;
  /* not unrolled: the mixed form then fits 5 waves per SIMD (measured 4 %
   * faster than the compiler's two-step unroll at 4 waves) */
#pragma unroll 1
  for (int st = 0; st < TP / 4; ++st) {
    const int e = 4 * st + q;
    const double l = px.l[e], m = px.m[e], nm1 = px.nm1[e];
    const double n = NEED_N ? px.n[e] : 0.0;
    const T w = (T)px.w[e];
    T cm[G], sm[G], co[G], so[G];
#pragma unroll
    for (int gi = 0; gi < G; ++gi) {
      bool msk, omk = false;
      if (PRED || CORR) {
        const bool pv = vw_visible(l, m, n, L.px[gi], L.py[gi], L.pz[gi], L.pinv[gi], L.pcos[gi]);
        if (CORR) {
          omk = allv[gi];
          msk = allv[gi] & pv;
        } else {
          msk = vis[gi] & pv;
          failed |= ~__ballot(pv) & allm[gi];
        }
      } else {
        msk = vis[gi];
      }
      T c, s;
      if (MIXED) {
        /* the fraction in [0, 1) */
        const double x = vw_viss_phase(L.kx[gi], L.ky[gi], L.kz[gi], l, m, nm1);
        float sf, cf;
        vw_hw_sincos_turn((float)__builtin_amdgcn_fract(x), &sf, &cf);
        c = cf;
        s = sf;
      } else {
        int ix;
        const double x =
            vw_ant_phase_frac(L.kx[gi], L.ky[gi], L.kz[gi], L.jx[gi], L.jy[gi], L.jz[gi], l, m, nm1);
        const double f = vw_tab_split(x * VW_TAB_SCALE, &ix);
        const double2 te = tab[ix];
        double sy, cy, sd, cd;
        vw_tab_poly_short(f, &sy, &cy);
        vw_tab_rotate(te.x, te.y, sy, cy, &sd, &cd);
        c = (T)cd;
        s = (T)sd;
      }
      cm[gi] = msk ? c : (T)0;
      sm[gi] = msk ? s : (T)0;
      co[gi] = omk ? c : (T)0;
      so[gi] = omk ? s : (T)0;
    }
#pragma unroll
    for (int gi = 0; gi < G; ++gi) {
      /* CORR: the second product of each block carries the minus sign */
      const T wm = CORR ? -w : w;
      const T wc = wm * cm[gi], ws = wm * sm[gi];
      const T wco = w * co[gi], wso = w * so[gi];
#pragma unroll
      for (int gj = 0; gj <= gi; ++gj) {
        const int b = gi * (gi + 1) / 2 + gj;
        if (CORR) {
          y11[b] = vw_mfma(wc, cm[gj], vw_mfma(wco, co[gj], y11[b]));
          y22[b] = vw_mfma(ws, sm[gj], vw_mfma(wso, so[gj], y22[b]));
        } else {
          y11[b] = vw_mfma(wc, cm[gj], y11[b]);
          y22[b] = vw_mfma(ws, sm[gj], y22[b]);
        }
      }
#pragma unroll
      for (int gj = 0; gj < G; ++gj) {
        if (CORR) y21[gi * G + gj] = vw_mfma(ws, cm[gj], vw_mfma(wso, co[gj], y21[gi * G + gj]));
        else y21[gi * G + gj] = vw_mfma(ws, cm[gj], y21[gi * G + gj]);
      }
    }
  }
  return failed;
}

#ifndef VW_VISSF_WAVES_G2
#define VW_VISSF_WAVES_G2 2
#endif
template <int TP, int G, bool MIXED>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(G == 1 ? 4 : VW_VISSF_WAVES_G2))) void k_vissf(
    VissFArgs a) {
  using Acc = typename std::conditional<MIXED, vw_f4, vw_d4>::type;
  constexpr int NS = VfShape<G>::NS, NB = VfShape<G>::NB;
  constexpr int EPT = TP / 256; /* pixels staged per thread */
  __shared__ double2 tab[MIXED ? 1 : VW_TAB_N];
  __shared__ VfTileLds<TP> px;
  if (!MIXED) vw_tab_fill(tab, a.tab);
  const int64_t vb = vw_xcd_block(blockIdx.x, gridDim.x);
  const int64_t chunk = vb / a.nquad;
  if (chunk >= a.nchunk) return; /* whole workgroup */
  const int wave = vw_rfl((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int64_t g = (vb - chunk * a.nquad) * 4 + wave; /* epoch of this wave */
  /* waves past the last epoch stage pixels and meet the barriers, nothing else */
  const bool active = g < a.tlen;
  const int64_t t0 = a.tile0 + chunk * a.tpc;
  const int64_t tend = a.tile0 + a.ntile;
  const int64_t t1 = (t0 + a.tpc < tend) ? t0 + a.tpc : tend;

  VfLane<G> L;
  int64_t fr[G];
  bool have[G];
#pragma unroll
  for (int gi = 0; gi < G; ++gi) {
    const int ant = gi * 16 + (lane & 15);
    have[gi] = active && ant < a.A;
    fr[gi] = have[gi] ? g * a.A + ant : 0;
    const double4 k = a.aph[fr[gi]];
    const double* q8 = a.ant8 + fr[gi] * 8;
    L.kx[gi] = have[gi] ? k.x : 0.0;
    L.ky[gi] = have[gi] ? k.y : 0.0;
    L.kz[gi] = have[gi] ? k.z : 0.0;
    if (!MIXED) {
      const double4 j = a.aphl[fr[gi]];
      L.jx[gi] = have[gi] ? j.x : 0.0;
      L.jy[gi] = have[gi] ? j.y : 0.0;
      L.jz[gi] = have[gi] ? j.z : 0.0;
    }
    L.px[gi] = q8[0]; L.py[gi] = q8[1]; L.pz[gi] = q8[2]; L.pinv[gi] = q8[3]; L.pcos[gi] = q8[7];
  }
  /* the plain form sums in the FP64 accumulators of the matrix cores; the
   * mixed form sums each tile in FP32 and adds it to FP64 totals */
  Acc y11[NS], y22[NS], y21[G * G];
  vw_d4 s11[NS], s22[NS], s21[G * G];
#pragma unroll
  for (int i = 0; i < NS; ++i) { y11[i] = Acc{0, 0, 0, 0}; y22[i] = Acc{0, 0, 0, 0}; s11[i] = vw_d4{0, 0, 0, 0}; s22[i] = vw_d4{0, 0, 0, 0}; }
#pragma unroll
  for (int i = 0; i < G * G; ++i) { y21[i] = Acc{0, 0, 0, 0}; s21[i] = vw_d4{0, 0, 0, 0}; }

  /* pixel data of the next tile, loaded one tile ahead */
  double nl[EPT], nm[EPT], nn[EPT], nz[EPT], nw[EPT];
  auto fetch = [&](int64_t tile) {
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
      const int64_t p = tile * TP + threadIdx.x + 256 * k;
      const bool ok = p < a.npix;
      /* past the end of the sky: the tile's first pixel with weight zero, so
       * the predicate test sees only the tile's own directions */
      const int64_t pp = ok ? p : tile * TP;
      nl[k] = a.l[pp]; nm[k] = a.m[pp]; nn[k] = a.n[pp]; nz[k] = a.nm1[pp];
      nw[k] = ok ? (MIXED ? (double)a.Bf[pp] : a.B[pp]) : 0.0;
    }
  };
  fetch(t0);
  for (int64_t tile = t0; tile < t1; ++tile) {
    __syncthreads(); /* the previous tile's readers are done (and the table is built) */
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
      const int e = threadIdx.x + 256 * k;
      px.l[e] = nl[k]; px.m[e] = nm[k]; px.n[e] = nn[k]; px.nm1[e] = nz[k]; px.w[e] = nw[k];
    }
    __syncthreads();
    if (tile + 1 < t1) fetch(tile + 1);
    if (!active) continue;
    const uint8_t* brow = a.bits + (tile - a.tile0) * a.nfr_pad;
    int bt[G];
    int nvis = 0;
    bool any_mixed = false;
#pragma unroll
    for (int gi = 0; gi < G; ++gi) {
      bt[gi] = have[gi] ? (int)brow[fr[gi]] : 2;
      nvis += __popcll(__ballot((bt[gi] & 2) == 0) & 0xffffull);
      any_mixed |= (__ballot((bt[gi] & 3) == 0) & 0xffffull) != 0;
    }
    /* fewer than two antennas see any of the tile: every pair is hidden */
    if (nvis < 2) continue;
    if (!any_mixed) {
      vf_tile<TP, G, MIXED, false, false>(px, L, bt, tab, y11, y22, y21);
    } else {
      const uint64_t failed = vf_tile<TP, G, MIXED, true, false>(px, L, bt, tab, y11, y22, y21);
      if (a.check || failed != 0) vf_tile<TP, G, MIXED, true, true>(px, L, bt, tab, y11, y22, y21);
    }
    if (MIXED) {
#pragma unroll
      for (int i = 0; i < NS; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s11[i][r] += (double)y11[i][r];
          s22[i][r] += (double)y22[i][r];
          y11[i][r] = 0;
          y22[i][r] = 0;
        }
#pragma unroll
      for (int i = 0; i < G * G; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s21[i][r] += (double)y21[i][r];
          y21[i][r] = 0;
        }
    }
  }
  if (!active) return;
  /* partial blocks: Re = Y11 + Y22 for gi >= gj, then Y21; row-major 16 x 16 */
  double* out = a.part + (g * a.nchunk + chunk) * (int64_t)NB * 256;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = MIXED ? 4 * (lane >> 4) + r : (lane >> 4) + 4 * r, j = lane & 15;
#pragma unroll
    for (int s = 0; s < NS; ++s)
      out[s * 256 + i * 16 + j] = MIXED ? s11[s][r] + s22[s][r] : (double)y11[s][r] + (double)y22[s][r];
#pragma unroll
    for (int s = 0; s < G * G; ++s) out[(NS + s) * 256 + i * 16 + j] = MIXED ? s21[s][r] : (double)y21[s][r];
  }
}

/* partial blocks -> per-epoch block sums.  Workgroup (epoch, slice of 32
 * entries); its eight 32-lane groups take every eighth chunk (256-byte
 * reads), then the eight sums are added in a fixed order (deterministic). */
__global__ __launch_bounds__(256) void k_vissf_fold(const double* __restrict__ part, int64_t nchunk, int64_t nent,
                                                    double* __restrict__ esum, uint64_t* __restrict__ ts) {
  vw_ts_begin(ts);
  __shared__ double red[8][32];
  const int64_t nslice = nent / 32;
  const int64_t g = blockIdx.x / nslice, sl = blockIdx.x - g * nslice;
  const int t = threadIdx.x & 31, c0 = threadIdx.x >> 5;
  const int64_t e = sl * 32 + t;
  double s = 0.0;
  for (int64_t k = c0; k < nchunk; k += 8) s += part[(g * nchunk + k) * nent + e];
  red[c0][t] = s;
  __syncthreads();
  if (c0 == 0) {
    double r = red[0][t];
#pragma unroll
    for (int i = 1; i < 8; ++i) r += red[i][t];
    esum[g * nent + e] = r;
  }
}

/* per-epoch block sums -> raw half sums of the epoch's pairs (pa[j], pb[j]);
 * passes after the first add to the running sums */
__global__ void k_vissf_rows(const double* __restrict__ esum, int64_t nh, int P, int G,
                             const int32_t* __restrict__ pa, const int32_t* __restrict__ pb, int accumulate,
                             double2* __restrict__ vraw, const RowRec* __restrict__ rows, double2* __restrict__ vh,
                             uint64_t* __restrict__ ts) {
  int64_t h = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (h >= nh) return;
  const int64_t g = h / P;
  const int j = (int)(h - g * P);
  const int ea = pa[j], eb = pb[j];
  const int hi = ea > eb ? ea : eb, lo = ea > eb ? eb : ea;
  const int NS = G * (G + 1) / 2, NB = NS + G * G;
  const int64_t ire = (int64_t)((hi >> 4) * ((hi >> 4) + 1) / 2 + (lo >> 4)) * 256 + (hi & 15) * 16 + (lo & 15);
  const int64_t iab = (int64_t)(NS + (ea >> 4) * G + (eb >> 4)) * 256 + (ea & 15) * 16 + (eb & 15);
  const int64_t iba = (int64_t)(NS + (eb >> 4) * G + (ea >> 4)) * 256 + (eb & 15) * 16 + (ea & 15);
  const double* b = esum + g * (int64_t)NB * 256;
  double re = b[ire], im = b[iab] - b[iba];
  if (accumulate) {
    double2 o = vraw[h];
    re = o.x + re;
    im = o.y + im;
  }
  vw_store_half(vraw, vh, rows, h, re, im);
  vw_ts_end(ts);
}

/* phase correction + conjugate completion (common.hpp:255-277) */
__global__ void k_conj_fill(const double2* __restrict__ vraw, const RowRec* __restrict__ rows, int64_t nh, int P,
                            double2* __restrict__ vh, double2* __restrict__ vfull, uint64_t* __restrict__ ts) {
  vw_ts_begin(ts);
  int64_t h = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (h >= nh) return;
  double2 z = vraw[h];
  double re, im;
  vw_phase_correct(z.x, z.y, rows[h].w, &re, &im);
  vh[h] = make_double2(re, im);
  int64_t g = h / P, j = h - g * P;
  vfull[2 * P * g + j] = make_double2(re, im);
  vfull[2 * P * g + P + j] = make_double2(re, -im);
  vw_ts_end(ts);
}

/* ------------------------------------------------------------------ */
/* segment parameters, keys, stable grouping                            */
/* ------------------------------------------------------------------ */
/* The polar terms round the phase after adding the visibility's argument, the
 * (re, im) terms without it: they differ by the rounding of phases of up to
 * umax (2 + |fa| + |fb|) turns.  Below 2^22 turns that is under 1e-9 of the
 * maps; it stays below for baselines of 14,000 km at 30 MHz.  Beyond it, and for
 * the unbounded slopes of rows that span no plane, the plain recon keeps the
 * (re, im) terms and their rounding.  So does the mixed recon beyond 2^25 turns,
 * up to where the difference, 2^-28 turns, stays an eighth of the rounding of
 * its FP32 fraction (one row at 1 MHz, phases of 2^39 turns: polar terms 3.3e-4
 * of the map off, the others below 5e-6). */
__device__ __forceinline__ int vw_polar_ok(const vw_segparams& sp) {
  const double turns = (double)sp.half * sp.du * (2.0 + fabs(sp.fa) + fabs(sp.fb));
  return (turns <= 4194304.0 ? 1 : 0) | (turns <= 33554432.0 ? 2 : 0);
}

/* The five sums of the w-plane fit over the full rows, in 256 strided partial
 * sums (partial t: full rows t, t + 256, ... in order) that a pairwise tree
 * folds: the order every build of this path and its oracle use.  A full row's
 * products are its half row's (the signs cancel).  One wave per 64 partials on
 * four CUs, VW_SEG_BATCH rows' loads in flight before they are added in order;
 * one workgroup with a 64-bit division and a load waited for per row took 86 us
 * for 31,744 half rows. */
#define VW_SEG_BATCH 16
__device__ __forceinline__ void vw_segsum_partial(const RowRec* __restrict__ rows, int64_t nh, int P, int t,
                                                  double* __restrict__ sums) {
  const int64_t n = 2 * nh;
  double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0, a4 = 0.0;
  const int64_t gstep = (int64_t)(256 / (2 * P)) * P; /* full row i -> i + 256: epochs (as half rows) and pairs */
  const int jstep = 256 % (2 * P);
  int64_t gP = (int64_t)(t / (2 * P)) * P; /* first half row of the epoch of full row i */
  int jj = t % (2 * P);
  for (int64_t i = t; i < n; i += 256 * VW_SEG_BATCH) {
    double u[VW_SEG_BATCH], v[VW_SEG_BATCH], w[VW_SEG_BATCH];
#pragma unroll
    for (int e = 0; e < VW_SEG_BATCH; ++e) {
      const RowRec& r = rows[i + 256 * e < n ? gP + (jj >= P ? jj - P : jj) : 0];
      u[e] = r.u; v[e] = r.v; w[e] = r.w;
      jj += jstep;
      gP += gstep;
      if (jj >= 2 * P) { jj -= 2 * P; gP += P; }
    }
#pragma unroll
    for (int e = 0; e < VW_SEG_BATCH; ++e)
      if (i + 256 * e < n) {
        a0 = a0 + u[e] * u[e];
        a1 = a1 + v[e] * v[e];
        a2 = a2 + u[e] * v[e];
        a3 = a3 + u[e] * w[e];
        a4 = a4 + v[e] * w[e];
      }
  }
  sums[t] = a0; sums[256 + t] = a1; sums[512 + t] = a2; sums[768 + t] = a3; sums[1024 + t] = a4;
}
__global__ __launch_bounds__(64) void k_segsums(const RowRec* __restrict__ rows, int64_t nh, int P,
                                                double* __restrict__ sums, uint64_t* __restrict__ ts) {
  vw_ts_begin(ts);
  vw_segsum_partial(rows, nh, P, blockIdx.x * 64 + threadIdx.x, sums);
}

/* mode row -> (half row, conjugate flag) */
__device__ __forceinline__ int64_t vw_row_half(int64_t r, int P, bool full, bool* neg) {
  if (!full) { *neg = false; return r; }
  int64_t g = r / (2 * P);
  int jj = (int)(r - g * 2 * P);
  *neg = jj >= P;
  return g * P + (jj >= P ? jj - P : jj);
}

/* segment parameters from the partial sums (every workgroup folds them, the
 * first writes them), then the uv-grid key of each row and, in idx, its index
 * (iota, for the radix sort) or zero (for k_rank_count) */
__global__ __launch_bounds__(256) void k_keys(const double* __restrict__ sums, const RowRec* __restrict__ rows,
                                              int64_t nr, int P, int full, double bl_max, double lambda,
                                              DevInfo* __restrict__ info, int64_t* __restrict__ keys,
                                              int32_t* __restrict__ idx, int iota) {
  __shared__ double s[5][256];
  __shared__ vw_segparams ssp;
  const int t = threadIdx.x;
#pragma unroll
  for (int k = 0; k < 5; ++k) s[k][t] = sums[256 * k + t];
  const int64_t r = (int64_t)blockIdx.x * 256 + t;
  bool neg;
  const int64_t h = vw_row_half(r < nr ? r : 0, P, full != 0, &neg);
  const RowRec rec = rows[h];
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if (t < st)
      for (int k = 0; k < 5; ++k) s[k][t] = s[k][t] + s[k][t + st];
    __syncthreads();
  }
  if (t == 0) {
    vw_segparams_from_sums(s[0][0], s[1][0], s[2][0], s[3][0], s[4][0], bl_max, lambda, &ssp);
    if (blockIdx.x == 0) {
      info->sp = ssp;
      info->polar = vw_polar_ok(ssp);
    }
  }
  __syncthreads();
  if (r >= nr) return;
  const vw_segparams sp = ssp;
  const double sg = neg ? -1.0 : 1.0;
  keys[r] = vw_grid_key(sg * rec.u, sg * rec.v, &sp, full ? 0 : 1);
  idx[r] = iota ? (int32_t)r : 0;
}

/* Stable order by (key, row index): all-pairs rank counted over a 2-D grid
 * of (256-row block, jblk-row block) compare tiles with integer atomics
 * (exact, order-independent), then a scatter.  The grid is sized for about
 * 2,048 workgroups, so a segment of a few thousand rows costs a few
 * microseconds instead of a one-workgroup sort. */
__global__ __launch_bounds__(256) void k_rank_count(const int64_t* __restrict__ keys, int64_t nr, int64_t jblk,
                                                    int32_t* __restrict__ rank) {
  __shared__ int64_t sk[256];
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t j0 = (int64_t)blockIdx.y * jblk;
  const int64_t j1 = j0 + jblk < nr ? j0 + jblk : nr;
  const int64_t ki = i < nr ? keys[i] : 0;
  int32_t cnt = 0;
  for (int64_t base = j0; base < j1; base += 256) {
    int64_t j = base + threadIdx.x;
    sk[threadIdx.x] = j < j1 ? keys[j] : INT64_MAX;
    __syncthreads();
    int64_t lim = j1 - base < 256 ? j1 - base : 256;
    for (int64_t q = 0; q < lim; ++q) {
      int64_t kj = sk[q];
      cnt += (kj < ki) || (kj == ki && base + q < i);
    }
    __syncthreads();
  }
  if (i < nr && cnt) atomicAdd(&rank[i], cnt);
}

/* segments longer than this many rows are ordered by a radix sort */
#define VW_RANK_MAX 8192

__global__ void k_rank_scatter(const int64_t* __restrict__ keys, const int32_t* __restrict__ rank, int64_t nr,
                               int32_t* __restrict__ idx_sorted, int64_t* __restrict__ keys_sorted) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nr) return;
  idx_sorted[rank[i]] = (int32_t)i;
  keys_sorted[rank[i]] = keys[i];
}

/* run boundaries -> keys, offsets, nuniq (single workgroup): 4,096 sorted keys
 * at a time, four consecutive ones a thread, the next ones loaded while these
 * are counted; boundary counts are scanned in the waves, then over the 16 waves.
 * (A run of nr / 1024 keys a thread, walked twice from global memory, took 82 us
 * for 31,744 rows.) */
__global__ __launch_bounds__(1024) void k_groups(const int64_t* __restrict__ ks, int64_t nr, int blockage,
                                                 int64_t* __restrict__ gkeys, int32_t* __restrict__ goff,
                                                 DevInfo* __restrict__ info, uint64_t* __restrict__ ts) {
  __shared__ int32_t wtot[2][16];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  int64_t k[4], prev;
  auto load = [&](int64_t i0) {
#pragma unroll
    for (int e = 0; e < 4; ++e) k[e] = i0 + e < nr ? ks[i0 + e] : 0;
    prev = i0 > 0 && i0 <= nr ? ks[i0 - 1] : 0;
  };
  int64_t i = 4 * t;
  load(i);
  int32_t base = 0; /* groups before this block of 4,096 keys */
  int buf = 0;
  for (int64_t b0 = 0; b0 < nr; b0 += 4096, i += 4096, buf ^= 1) {
    int64_t c[4];
    int f[4], cnt = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      c[e] = k[e];
      f[e] = i + e < nr && (i + e == 0 || k[e] != (e ? k[e > 0 ? e - 1 : 0] : prev)) ? 1 : 0;
      cnt += f[e];
    }
    if (b0 + 4096 < nr) load(i + 4096);
    int inc = cnt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(inc, o, 64);
      if (lane >= o) inc += v;
    }
    if (lane == 63) wtot[buf][wave] = inc;
    __syncthreads();
    int32_t before = 0, all = 0;
#pragma unroll
    for (int wv = 0; wv < 16; ++wv) {
      const int32_t x = wtot[buf][wv];
      before += wv < wave ? x : 0;
      all += x;
    }
    int32_t g = base + before + inc - cnt;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (f[e]) {
        gkeys[g] = c[e];
        goff[g] = (int32_t)(i + e);
        ++g;
      }
    base += all;
  }
  if (t == 0) {
    goff[base] = (int32_t)nr;
    info->nuniq = base;
    info->first_nz = (base > 0 && ks[0] == 0) ? 1 : 0;
    if (!blockage) info->wtotal += base;
  }
  vw_ts_end(ts);
}

/* The whole grouping of short segments, one workgroup each: the w-plane sums and
 * parameters as k_segsums and k_keys compute them, the rows' keys, their stable
 * order (a bitonic sort of the distinct (key, row) pairs, one a thread, strides
 * below 64 by lane exchange, the rest through LDS) and the runs.  For up to
 * 1,024 rows; with four rows a thread, for 3,840, the one workgroup waited so
 * long for a CU beside the recon kernel that a 16-segment run at Nside 128 took
 * 9.3 instead of 9.0 ms. */
#define VW_GROUP_ONE_MAX 1024
__global__ __launch_bounds__(1024) void k_group_one(VwMerge mg, const RowRec* __restrict__ rows, int P, int full,
                                                    double bl_max, double lambda, int blockage,
                                                    int32_t* __restrict__ idx_sorted, int64_t* __restrict__ gkeys,
                                                    int32_t* __restrict__ goff, DevInfo* __restrict__ info,
                                                    uint64_t* __restrict__ ts) {
  vw_ts_begin(ts);
  constexpr int N = 1024;
  __shared__ double sums[5 * 256];
  __shared__ vw_segparams ssp;
  __shared__ int64_t sk[N];
  __shared__ int32_t si[N];
  __shared__ int32_t wtot[16];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, sg = blockIdx.x;
  const int nh = mg.row0[sg + 1] - mg.row0[sg], nr = full ? 2 * nh : nh; /* <= VW_GROUP_ONE_MAX */
  rows += mg.row0[sg];
  idx_sorted += mg.base[sg];
  gkeys += mg.base[sg];
  goff += mg.base[sg];
  info += sg;
  if (t < 256) vw_segsum_partial(rows, nh, P, t, sums);
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    /* the five sums' trees side by side */
    const int k = t >> 8, j = t & 255;
    if (j < st) {
      sums[256 * k + j] = sums[256 * k + j] + sums[256 * k + j + st];
      if (k == 0) sums[1024 + j] = sums[1024 + j] + sums[1024 + j + st];
    }
    __syncthreads();
  }
  if (t == 0) {
    vw_segparams_from_sums(sums[0], sums[256], sums[512], sums[768], sums[1024], bl_max, lambda, &ssp);
    info->sp = ssp;
    info->polar = vw_polar_ok(ssp);
  }
  __syncthreads();
  const vw_segparams sp = ssp;
  bool neg;
  const int64_t h = vw_row_half(t < nr ? t : 0, P, full != 0, &neg);
  const double sgn = neg ? -1.0 : 1.0;
  const int64_t k0 = vw_grid_key(sgn * rows[h].u, sgn * rows[h].v, &sp, full ? 0 : 1);
  int64_t key = t < nr ? k0 : INT64_MAX; /* keys are non-negative and below it */
  int32_t idx = t;
  for (int k = 2; k <= N; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      int64_t kb;
      int32_t ib;
      if (j >= 64) {
        __syncthreads();
        sk[t] = key;
        si[t] = idx;
        __syncthreads();
        kb = sk[t ^ j];
        ib = si[t ^ j];
      } else {
        kb = __shfl_xor(key, j, 64);
        ib = __shfl_xor(idx, j, 64);
      }
      const bool less = kb < key || (kb == key && ib < idx);
      if (less == (((t & k) == 0) == ((t & j) == 0))) {
        key = kb;
        idx = ib;
      }
    }
  __syncthreads();
  sk[t] = key;
  if (t < nr) idx_sorted[t] = idx;
  __syncthreads();
  const bool f = t < nr && (t == 0 || key != sk[t > 0 ? t - 1 : 0]);
  const uint64_t b = __ballot(f);
  if (lane == 0) wtot[wave] = __popcll(b);
  __syncthreads();
  int32_t before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    const int32_t x = wtot[w];
    before += w < wave ? x : 0;
    all += x;
  }
  if (f) {
    const int32_t g = before + __popcll(b & ((1ull << lane) - 1));
    gkeys[g] = key;
    goff[g] = t;
  }
  if (t == 0) {
    goff[all] = nr;
    info->nuniq = all;
    info->first_nz = (all > 0 && key == 0) ? 1 : 0;
    if (!blockage) info->wtotal += all; /* blockage 0 takes one segment a launch */
  }
  vw_ts_end(ts);
}

/* Occlusion in FP32, exact where it decides.  d = s . u - cosphi with every
 * operand rounded to FP32 is within 4e-7 of the FP64 test's difference
 * (operands 2^-24 relative each, |s| = |u| = 1, three roundings of sums below
 * 2, the threshold), so outside +-VW_VIS_EPS its sign is the FP64 test's
 * result; closer in, the caller evaluates the FP64 test.  A frame that is not
 * finite (an antenna at the origin) fails the FP64 test everywhere: threshold
 * 2 here. */
#define VW_VIS_EPS 1e-6f
__device__ __forceinline__ void vw_frame32(const double* __restrict__ q8, float* __restrict__ f) {
  const bool ok = isfinite(q8[4]) && isfinite(q8[5]) && isfinite(q8[6]) && isfinite(q8[7]);
  f[0] = ok ? (float)q8[4] : 0.f;
  f[1] = ok ? (float)q8[5] : 0.f;
  f[2] = ok ? (float)q8[6] : 0.f;
  f[3] = ok ? (float)q8[7] : 2.f;
}
/* the smaller of the two endpoints' differences: above VW_VIS_EPS both see
 * the direction, below -VW_VIS_EPS one does not */
__device__ __forceinline__ float vw_vis32(float l, float m, float n, const float* f) {
  const float a = fmaf(n, f[2], fmaf(m, f[1], fmaf(l, f[0], -f[3])));
  const float b = fmaf(n, f[6], fmaf(m, f[5], fmaf(l, f[4], -f[7])));
  return fminf(a, b);
}

/* Per-group records as SoA (uniform loads of four groups per array in one
 * scalar load): cell centre, visibility (representative or group mean) in
 * polar form, the representative's antenna frames and member range.  The
 * one-sky recon adds Re(V exp(2 pi j x)) = |V| cos(2 pi (x + arg)), arg in
 * turns: the argument rides in the phase's first multiply-add, so a term
 * needs one cosine and one product instead of sine, cosine and two. */
struct GRec {
  double ugu, vgu; /* wavelengths; x1024 for the plain generic kind  */
  double arg, amp; /* visibility: argument in turns, magnitude        */
};
struct GroupSoA {
  GRec* rec;    /* 32 B */
  double2* v;   /* the visibility as (re, im), for segments without polar terms */
  double* ant;  /* [q][10]: representative's antenna frames a and b (plain form; */
  float* ant32; /* [q][8]: in FP32, vw_frame32; null in the mixed form)        */
  int32_t *gia, *gib; /* the representative's frames' indices */
};

__global__ void k_group_data(VwMerge mg, const int64_t* __restrict__ gkeys, const int32_t* __restrict__ goff,
                             const int32_t* __restrict__ idx_sorted, const double2* __restrict__ vh,
                             const RowRec* __restrict__ rows, const double* __restrict__ ant8, int P, int full,
                             int blockage, int occ_mode, double uv_scale,
                             DevInfo* __restrict__ info, GroupSoA g, uint64_t* __restrict__ ts) {
  vw_ts_begin(ts);
  int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int base = 0, row0 = 0;
  for (int k = 1; k < mg.n; ++k)
    if (q >= mg.base[k]) {
      base = mg.base[k];
      row0 = mg.row0[k];
      ++info;
    }
  if (q - base >= info->nuniq) {
    vw_ts_end(ts); /* the grid covers the rows: the last workgroup often holds no group */
    return;
  }
  vw_segparams sp = info->sp;
  int64_t key = gkeys[q];
  int32_t s0 = goff[q], s1 = goff[q + 1];
  double ugu = 0.0, vgu = 0.0;
  if (key != 0) vw_key_uv(key, &sp, &ugu, &vgu);
  idx_sorted += base;
  rows += row0;
  vh += row0;
  bool neg;
  /* the one member a single-representative rule reads: occ_mode 1 the
   * first of the sorted run, occ_mode 2 the median (viss_recon_kernel.cuh:
   * 603-614; mirror_tile_recon_group .cuh:782-792) */
  int64_t hr = vw_row_half(idx_sorted[occ_mode == 1 ? s0 : s0 + (s1 - s0) / 2], P, full != 0, &neg);
  double vr, vi;
  if (blockage) {
    /* representative value (signed for rows of the conjugate half) */
    double2 v = vh[hr];
    vr = v.x;
    vi = neg ? -v.y : v.y;
  } else {
    /* group mean over members in sorted order (compute_avg, viss_recon_kernel.cuh:327-333) */
    double sr = 0.0, si = 0.0;
    for (int32_t k = s0; k < s1; ++k) {
      bool ng;
      int64_t h = vw_row_half(idx_sorted[k], P, full != 0, &ng);
      double2 v = vh[h];
      sr = sr + v.x;
      si = si + (ng ? -v.y : v.y);
    }
    vr = sr / (double)(s1 - s0);
    vi = si / (double)(s1 - s0);
  }
  GRec gr;
  gr.ugu = ugu * uv_scale; /* 1024 for the plain generic kind's table sincos, else 1 (exact) */
  gr.vgu = vgu * uv_scale;
  /* finite parts give a finite magnitude, others none: the finite-value filter
   * reads it.  A magnitude past what the polar terms hold (2 |V| from each of 32
   * groups before a fold in FP64, |V| in FP32), or infinite parts, leave the
   * segment to the (re, im) terms, which overflow where the sum of the parts does;
   * a NaN is NaN in both */
  const double mag = hypot(vr, vi);
  gr.amp = isfinite(vr) && isfinite(vi) ? fmin(mag, DBL_MAX) : NAN;
  if (!isnan(vr) && !isnan(vi) && !(mag <= FLT_MAX)) atomicAnd(&info->polar, mag < 0x1p1000 ? 1 : 0);
  gr.arg = atan2(vi, vr) * VW_INV_TWOPI;
  g.rec[q] = gr;
  g.v[q] = make_double2(vr, vi);
  RowRec r = rows[hr];
  g.gia[q] = r.ia;
  g.gib[q] = r.ib;
  if (g.ant) {
    const double* qa = ant8 + (int64_t)r.ia * 8;
    const double* qb = ant8 + (int64_t)r.ib * 8;
    double* d = g.ant + q * 10;
    d[0] = qa[0]; d[1] = qa[1]; d[2] = qa[2]; d[3] = qa[3]; d[4] = qa[7];
    d[5] = qb[0]; d[6] = qb[1]; d[7] = qb[2]; d[8] = qb[3]; d[9] = qb[7];
    vw_frame32(qa, g.ant32 + q * 8);
    vw_frame32(qb, g.ant32 + q * 8 + 4);
  }
  vw_ts_end(ts);
}

/* The output sets of one recon launch (HEALPix map, lm image, one tile pass of
 * each): each kernel of the recon stage takes both, the blocks of the second
 * after those of the first. */
struct ReconSet {
  const double *l, *m, *n;
  const double* cone; /* [5][ntile] */
  int64_t ntile;      /* tiles of the whole set                                  */
  int64_t tile0, nt;  /* tiles of this pass                                      */
  int64_t pt0, npts;  /* its points [pt0, pt0 + npts), pt0 = tile0 * TP          */
  uint64_t* cls;      /* [nt][nq_pad / 16] mask words of 16 groups (representative
                       * kinds), [nt][nh_pad] row class bytes (generic kind)     */
  const uint8_t* bits; /* [nt][nfr_pad] cone bits (long frame rows)               */
  uint64_t* fvis;     /* [nt][nfr_pad][TP / 64] points seen (representative kinds) */
  int64_t nchunk;     /* group ranges per point block                            */
  int cst[VW_MERGE_MAX + 1]; /* of them, segment s has [cst[s], cst[s + 1])      */
  int64_t pwaves;     /* point blocks (waves) per group range                    */
  int64_t nblk;       /* workgroups of the recon kernel                          */
  double* part;       /* [nchunk][npts]                                          */
  uint32_t* wpart;    /* [nchunk][npts]                                          */
  double* acc;        /* accumulators of the whole set                           */
  uint32_t* wacc;
};
struct ReconSets {
  ReconSet s[2]; /* a set without tiles or blocks is absent */
};

/* Which of a wave's 64 points (lane: pl, pm, pn; ok) each of 64 antenna frames
 * sees: lane f returns frame f0 + f's word, bit j = point j.  cb: the frame's
 * cone bits on the points' tile, which decide it where they can; the partly
 * visible frames are broadcast one by one for the FP64 test of every point. */
__device__ __forceinline__ uint64_t vw_frame_words(const double* __restrict__ ant8, int64_t f, int64_t nfr, int cb,
                                                   double pl, double pm, double pn, bool ok) {
  const uint64_t all = ~0ull;
  uint64_t word = !(cb & 2) && (cb & 1) ? all : 0ull;
  uint64_t some = __ballot(f < nfr && !(cb & 3));
  if (!some) return word;
  const double* q = ant8 + (f < nfr ? f : nfr - 1) * 8;
  const double x = q[0], y = q[1], z = q[2], in = q[3], cp = q[7];
  const int lane = threadIdx.x & 63;
  while (some) {
    const int j = __builtin_ctzll(some);
    some &= some - 1;
    auto at = [j](double v) {
      const uint64_t w = __builtin_bit_cast(uint64_t, v);
      const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)w, j);
      const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(w >> 32), j);
      return __builtin_bit_cast(double, (uint64_t)c << 32 | a);
    };
    const uint64_t v = __ballot(ok && vw_visible(pl, pm, pn, at(x), at(y), at(z), at(in), at(cp)));
    word = lane == j ? v : word;
  }
  return word;
}

/* Occlusion bits of the frames that a tile's cone leaves open, neither hidden nor
 * visible by more than rounding (b: the tile's cone bits), for one block of 64
 * points, by one wave: fo[f * stride], bit j = point j is seen from frame f.  The
 * wave gathers open frames in LDS and takes 64 at a time, a lane a frame, against
 * the points in turn (LDS broadcasts).  Broadcasting the frames one by one and
 * writing the decided frames' words too took twice the time; points as scalar
 * loads or lane by lane, a queue shared by the workgroup, and further workgroups
 * for 256 frames each, which test the cones again, were no faster where the tiles
 * fill the chip (337 us for 6,289 tiles x 2,048 frames).  Frames [f0, f1). */
__device__ __forceinline__ void vw_open_frames(const uint8_t* b, int64_t f0, int64_t f1, const double* __restrict__ ant8,
                                               double pl, double pm, double pn, bool ok, double* pts /* [3][64] */,
                                               int32_t* queue /* [128] */, uint64_t* __restrict__ fo, int stride) {
  const int lane = threadIdx.x & 63;
  const uint64_t okm = __ballot(ok);
  auto settle = [] { /* the wave's LDS writes are seen by its reads, and its reads done before its writes */
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  settle();
  pts[lane] = pl;
  pts[64 + lane] = pm;
  pts[128 + lane] = pn;
  auto take = [&](int n) { /* the queue's first n <= 64 frames */
    settle();
    const int f = lane < n ? queue[lane] : -1;
    const double* q = ant8 + (int64_t)(f < 0 ? 0 : f) * 8;
    const double x = q[0], y = q[1], z = q[2], in = q[3], cp = q[7];
    uint32_t w[2];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      uint32_t v = 0;
#pragma unroll 8
      for (int j = 0; j < 32; ++j) {
        const int p = 32 * hf + j;
        v |= (uint32_t)vw_visible(pts[p], pts[64 + p], pts[128 + p], x, y, z, in, cp) << j;
      }
      w[hf] = v;
    }
    if (f >= 0) fo[(int64_t)f * stride] = ((uint64_t)w[1] << 32 | w[0]) & okm;
    settle();
  };
  int cnt = 0;
  for (; f0 < f1; f0 += 64) {
    const int64_t f = f0 + lane;
    const bool open = f < f1 && !(b[f] & 6);
    const uint64_t m = __ballot(open);
    if (open) queue[cnt + __popcll(m & ((1ull << lane) - 1))] = (int32_t)f;
    cnt += __popcll(m);
    if (cnt >= 64) {
      take(64);
      cnt -= 64;
      const int32_t r = queue[64 + lane];
      settle();
      if (lane < cnt) queue[lane] = r;
    }
  }
  if (cnt) take(cnt);
}

/* The one-sky recon's form of the same classes: per (tile, 16 groups) one
 * 64-bit word, bit j = group j is visible from the whole tile, bits 16 + j and
 * 32 + j = it is partly, with its first, its second antenna's frame left open
 * by the tile's cone (not visible by more than rounding); hidden groups, groups
 * below first_nz (the key-0 group) and past nuniq have none of them, so the recon
 * walks set bits and needs no range test.  TILE: one block per tile
 * makes the tile's cone bits in LDS (frame rows up to VW_GCLS_LDS_MAX bytes);
 * else they come from the bit table of the pass.  A wave takes 4 x 64 groups
 * at a time, a lane one group of each 64 (coalesced index loads, all issued
 * before the gathers), and writes the masks of ballots.  Words of entries
 * below nuniq rounded up to 64 are written: the recon reads no others.
 * BITS (mixed form): the block also writes the open frames' occlusion bits
 * (vw_open_frames), whose AND over a partly visible group's open frames is its
 * mask, the same as the two tests of each point; the recon loads the words as scalars.  Testing both antennas of every
 * (point, group) in FP32, with an FP64 fallback, as the plain form does, cost it
 * as much as two terms and 26 registers (5 instead of 8 waves a SIMD): two Nside
 * 256 segments 24.3 -> 22.5 ms, the Nside 128 day 8.98 -> 8.56.  The plain form is
 * bound by its FP64 terms and gained nothing (Nside 256 -2%, short segments and
 * the lunar formation, with few groups a frame, +2 to 4%).
 * A tile's frames and groups are shared by gridDim.x / tiles workgroups
 * (group_mask_parts). */
template <bool TILE, bool BITS>
__global__ __launch_bounds__(256) void k_group_mask(VwMerge mg, ReconSets sets, const double* __restrict__ ant8, int64_t nfr,
                                                    int64_t nfr_pad, int64_t TP, const int32_t* __restrict__ ia,
                                                    const int32_t* __restrict__ ib, const DevInfo* __restrict__ info,
                                                    int64_t nq_pad, uint64_t* __restrict__ ts) {
  vw_ts_begin(ts);
  extern __shared__ uint4 sbits[];
  const uint32_t ntot = (uint32_t)(sets.s[0].nt + sets.s[1].nt);
  const uint32_t parts = gridDim.x / ntot, part = blockIdx.x / ntot, blk_t = blockIdx.x - part * ntot;
  const int si = (int)blk_t >= (int)sets.s[0].nt;
  const ReconSet& S = sets.s[si];
  const int64_t tr = blk_t - (si ? sets.s[0].nt : 0);
  const uint8_t* b = TILE ? (const uint8_t*)sbits : S.bits + tr * nfr_pad;
  if (TILE) {
    vw_tile_bits_lds((uint8_t*)sbits, S.cone, S.ntile, S.tile0 + tr, ant8, nfr);
    __syncthreads();
  }
  const int wave = vw_rfl((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  if (BITS) {
    __shared__ double spt[4][192];
    __shared__ int32_t squeue[4][128];
    const int nblk = (int)(TP / 64);
    const int64_t per = ((nfr + parts - 1) / parts + 63) / 64 * 64, f0 = part * per;
    for (int blk = wave; blk < nblk; blk += 4) {
      const int64_t p = tr * TP + 64 * blk + lane; /* pass-relative */
      const bool ok = p < S.npts;
      const int64_t pp = S.pt0 + (ok ? p : 0);
      vw_open_frames(b, f0, f0 + per < nfr ? f0 + per : nfr, ant8, S.l[pp], S.m[pp], S.n[pp], ok, spt[wave], squeue[wave],
                     S.fvis + tr * nfr_pad * nblk + blk, nblk);
    }
  }
  uint64_t* out = S.cls + tr * (nq_pad >> 4);
  for (int sg = 0; sg < mg.n; ++sg) {
    const int base = mg.base[sg], nu = base + vw_rfl((int)info[sg].nuniq), q0 = base + vw_rfl((int)info[sg].first_nz);
    const int qend = (nu + 63) / 64 * 64; /* <= nq_pad, a multiple of 64 */
    for (int j0 = base + 256 * (wave + 4 * (int)part); j0 < qend; j0 += 1024 * (int)parts) {
      int av[4], bv[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int q = j0 + 64 * e + lane;
        /* indices past nuniq are not frames: frame 0 stands in for them */
        av[e] = q < nu ? ia[q] : 0;
        bv[e] = q < nu ? ib[q] : 0;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int q = j0 + 64 * e + lane;
        const bool in = q >= q0 && q < nu;
        const int ba = b[av[e]], bb = b[bv[e]], c = vw_pair_class(ba, bb);
        const uint64_t v = __ballot(in && c == VW_CLS_VISIBLE);
        const uint64_t ma = __ballot(in && c == VW_CLS_MIXED && !(ba & 4));
        const uint64_t mb = __ballot(in && c == VW_CLS_MIXED && !(bb & 4));
        if (lane < 4 && j0 + 64 * e < qend) {
          const int sh = 16 * lane;
          out[((j0 + 64 * e) >> 4) + lane] =
              ((v >> sh) & 0xffffu) | ((ma >> sh) & 0xffffu) << 16 | ((mb >> sh) & 0xffffu) << 32;
        }
      }
    }
  }
  vw_ts_end(ts);
}

/* ------------------------------------------------------------------ */
/* reconstruction                                                       */
/* ------------------------------------------------------------------ */
struct ReconArgs {
  VwMerge mg;
  const double2* tab;  /* the sine table (plain), built once per context */
  ReconSets sets;
  int64_t TP, nq_pad, nh_pad, nfr_pad;
  GroupSoA g;
  const int32_t* goff;
  const int32_t* idx_sorted;
  const double2* vh;
  const RowRec* rows;
  const double* ant8;
  const DevInfo* info;
  int P, full, occ_mode;
};

#define VW_KIND_REP 0
#define VW_KIND_GENERIC 1
#define VW_KIND_AVG 2
#define VW_KIND_REP_FINITE 3 /* representatives, groups with a non-finite value skipped */
#define VW_KIND_IS_REP(k) ((k) == VW_KIND_REP || (k) == VW_KIND_REP_FINITE)

/* visibility of one row for the PPL points of a lane given the class */
template <int PPL, bool BRANCHFREE>
__device__ __forceinline__ void vw_ant_vis(const double* __restrict__ ant8, int ia, int ib, const double* pl,
                                           const double* pm, const double* pn, const bool* ok, bool* vis) {
  const double* qa = ant8 + (int64_t)ia * 8;
  const double* qb = ant8 + (int64_t)ib * 8;
  const double ax = qa[0], ay = qa[1], az = qa[2], ai = qa[3], ac = qa[7];
  const double bx = qb[0], by = qb[1], bz = qb[2], bi = qb[3], bc = qb[7];
#pragma unroll
  for (int k = 0; k < PPL; ++k)
    vis[k] = vw_vis2<BRANCHFREE>(ok[k], pl[k], pm[k], pn[k], ax, ay, az, ai, ac, bx, by, bz,
             bi, bc);
}

/* FP64 phase and turn reduction, hardware FP32 sin/cos, FP32 sums over blocks
 * of at most 32 groups, added up in FP64 (mixed form, one point) */
struct ReconAccF32 {
  float b = 0.f;
  double s = 0.0;
  /* b + amp cos(2 pi (ugu lp + vgu mp + arg)) */
  __device__ float term(double ugu, double vgu, double arg, float amp, double lp, double mp) const {
    /* the fraction in [0, 1) turns: one v_fract_f64 */
    const double x = fma(vgu, mp, fma(ugu, lp, arg));
    const float f = (float)__builtin_amdgcn_fract(x);
    return fmaf(amp, __builtin_amdgcn_cosf(f), b);
  }
  /* the (re, im) form of a term, kept only where use holds: a select, not a branch */
  __device__ void term_ri(bool use, double ugu, double vgu, float vrf, float vif, double lp, double mp) {
    const double x = vw_recon_phase(ugu, vgu, lp, mp);
    const float f = (float)__builtin_amdgcn_fract(x);
    const float sn = __builtin_amdgcn_sinf(f), cs = __builtin_amdgcn_cosf(f);
    const float nb = fmaf(vrf, cs, fmaf(-vif, sn, b));
    b = use ? nb : b;
  }
  __device__ void fold() {
    s += (double)b;
    b = 0.f;
  }
  __device__ double value() const { return s + (double)b; }
};

/* cos(2 pi x) without a table.  q = fract(x) and r = q - 1/2 give cos(2 pi x) =
 * -cos(2 pi r) = -T4(c), c = cos(pi r / 2), T4(c) = 8 (u^2 - u) + 1 with u = c^2.
 * c is even in r, and r^2 = w + 1/4 with w = q^2 - q, one multiply-add, so c is a
 * polynomial in w on [-1/4, 0]: degree 5, the minimax fit to |T4'(c)| times the
 * error, which leaves 1.9e-13 of the cosine.  Seven operations to v = u^2 - u,
 * with cos(2 pi x) = -8 v - 1; the -1 is summed per group, not per point
 * (ReconLane::fold). */
__device__ __forceinline__ double vw_cos_v(double x) {
  const double q = __builtin_amdgcn_fract(x);
  const double w = fma(q, q, -q);
  double c = fma(w, -0x1.a1f326935c708p-16, 0x1.d198ac4ebf5c1p-11);
  c = fma(w, c, -0x1.4705ad44bdfc1p-6);
  c = fma(w, c, 0x1.e82ab50a06c0cp-3);
  c = fma(w, c, -0x1.1c5831ae32c64p+0);
  c = fma(w, c, 0x1.6a09e667f13cap-1);
  const double u = c * c;
  return fma(u, u, -u);
}

/* the PPL points of one lane and one group; a point with use[k] false keeps
 * its sum.  A plain term is 12 FP64 instructions (phase 2, cosine 9, sum 1)
 * and nothing else: sine and cosine from the 1024-entry LDS table took 15 and
 * a 16-byte read at a random entry, whose bank conflicts (8 lanes a phase on 8
 * bank groups, 20 cycles of the CU's one LDS pipe a read) had become the bound.
 * A mixed term saves the sine and a product of the (re, im) form, 16.2 -> 11.5
 * issue slots of an FP32 FMA.  Both are bound by VALU issue. */
template <int PPL, bool MIXED>
struct ReconLane {
  double d[PPL];
  double ones = 0.0; /* minus the magnitudes of the groups that every point sees (plain polar terms) */
  ReconAccF32 f[PPL];
  __device__ ReconLane() {
#pragma unroll
    for (int k = 0; k < PPL; ++k) d[k] = 0.0;
  }
  template <bool MASK>
  __device__ __forceinline__ void add(const GRec& g, const bool* use, const double* lp, const double* mp) {
    if (MIXED) {
      const float amp = (float)g.amp;
#pragma unroll
      for (int k = 0; k < PPL; ++k) {
        const float t = f[k].term(g.ugu, g.vgu, g.arg, amp, lp[k], mp[k]);
        f[k].b = !MASK || use[k] ? t : f[k].b;
      }
    } else {
      const double a8 = -8.0 * g.amp;
      if (!MASK) ones -= g.amp;
#pragma unroll
      for (int k = 0; k < PPL; ++k) {
        const double v = vw_cos_v(fma(g.vgu, mp[k], fma(g.ugu, lp[k], g.arg)));
        const double t = fma(a8, v, MASK ? d[k] - g.amp : d[k]);
        d[k] = !MASK || use[k] ? t : d[k];
      }
    }
  }
  /* the (re, im) form, a value per point: averages over the members that
   * each point sees */
  __device__ __forceinline__ void add_ri(double ugu, double vgu, const double* vr, const double* vi, const bool* use,
                                         const double* lp, const double* mp, const double2* tab) {
    if (MIXED) {
#pragma unroll
      for (int k = 0; k < PPL; ++k) f[k].term_ri(use[k], ugu, vgu, (float)vr[k], (float)vi[k], lp[k], mp[k]);
    } else {
      double fr[PPL];
      int ix[PPL];
#pragma unroll
      for (int k = 0; k < PPL; ++k) fr[k] = vw_tab_split(vw_recon_phase(ugu, vgu, lp[k], mp[k]), &ix[k]);
      double2 e[PPL];
#pragma unroll
      for (int k = 0; k < PPL; ++k) e[k] = tab[ix[k]];
#pragma unroll
      for (int k = 0; k < PPL; ++k) {
        double sy, cy, sn, cs;
        vw_tab_poly_short(fr[k], &sy, &cy);
        vw_tab_rotate(e[k].x, e[k].y, sy, cy, &sn, &cs);
        const double t = vw_recon_add(d[k], vr[k], vi[k], sn, cs);
        d[k] = use[k] ? t : d[k];
      }
    }
  }
  /* the (re, im) form of a group's terms, point after point (segments without
   * polar terms), in the plain form with the sine table in global memory; use ==
   * nullptr: every point */
  __device__ __forceinline__ void add_one(const GRec& g, const double2& v, const bool* use, const double* lp,
                                          const double* mp, const double2* __restrict__ gtab) {
#pragma unroll
    for (int k = 0; k < PPL; ++k) {
      if (MIXED) {
        f[k].term_ri(use == nullptr || use[k], g.ugu, g.vgu, (float)v.x, (float)v.y, lp[k], mp[k]);
        continue;
      }
      int ix;
      const double fr = vw_tab_split(vw_recon_phase(g.ugu, g.vgu, lp[k], mp[k]) * VW_TAB_SCALE, &ix);
      const double2 e = gtab[ix];
      double sy, cy, sn, cs;
      vw_tab_poly_short(fr, &sy, &cy);
      vw_tab_rotate(e.x, e.y, sy, cy, &sn, &cs);
      const double t = vw_recon_add(d[k], v.x, v.y, sn, cs);
      d[k] = use == nullptr || use[k] ? t : d[k];
    }
  }
  /* every 32 groups.  Plain: the terms -8 v |V| are positive and grow with the
   * groups, the sum with |V| as their root, so the magnitudes come off while both
   * are small: left to the end of a range of 77,658 groups, the sums were 7.6e-10
   * |V| off, with the folds 9.3e-11 (rms). */
  __device__ void fold() {
#pragma unroll
    for (int k = 0; k < PPL; ++k) {
      if (MIXED) f[k].fold();
      else d[k] += ones;
    }
    ones = 0.0;
  }
  __device__ double value(int k) const { return MIXED ? f[k].value() : d[k] + ones; }
};

#ifndef VW_RECON_WAVES_PLAIN
#define VW_RECON_WAVES_PLAIN 5
#endif
#ifndef VW_RECON_WAVES_MIXED
#define VW_RECON_WAVES_MIXED 5
#endif
#ifndef VW_RECON_WAVES_GENERIC
#define VW_RECON_WAVES_GENERIC 4
#endif
template <int PPL, bool MIXED, int KIND>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(
    KIND == VW_KIND_GENERIC ? VW_RECON_WAVES_GENERIC : MIXED ? VW_RECON_WAVES_MIXED : VW_RECON_WAVES_PLAIN))) void k_recon(ReconArgs a) {
  constexpr bool TABLE = !MIXED && KIND == VW_KIND_GENERIC;
  constexpr bool BITS = MIXED && VW_KIND_IS_REP(KIND); /* occlusion bits, see k_group_mask */
  __shared__ double2 tab[TABLE ? VW_TAB_N : 1];
  __shared__ double gring[4][2 * 64]; /* per wave: two blocks of 16 group records */
  if (TABLE) {
    vw_tab_fill(tab, a.tab);
    __syncthreads();
  }
  const int lane = threadIdx.x & 63;
  const int si = (int)blockIdx.x >= (int)a.sets.s[0].nblk;
  const ReconSet& S = a.sets.s[si];
  const int64_t wid =
      (int64_t)(blockIdx.x - (si ? (uint32_t)a.sets.s[0].nblk : 0u)) * 4 + vw_rfl((int)(threadIdx.x >> 6));
  const int64_t chunk = wid / S.pwaves;
  const int64_t pw = wid - chunk * S.pwaves;
  if (chunk >= S.nchunk) return;
  const int64_t pbase = pw * 64 * PPL; /* pass-relative */
  const int64_t tile = pbase / a.TP;   /* pass-relative tile (class tables are per pass) */
  int sg = 0; /* the chunk's segment */
  while (sg + 1 < a.mg.n && (int)chunk >= S.cst[sg + 1]) ++sg;
  const DevInfo* info = a.info + sg;
  const vw_segparams sp = info->sp;
  /* group positions fit 32 bits; uniform values keep the range tests scalar */
  const int64_t nu = a.mg.base[sg] + vw_rfl((int)info->nuniq);
  const int64_t q0 = a.mg.base[sg] + vw_rfl((int)info->first_nz);
  const bool polar = (vw_rfl(info->polar) & (MIXED ? 2 : 1)) != 0;
  /* group range of this chunk, aligned to 16 groups */
  const int64_t base = q0 & ~(int64_t)15;
  const int64_t nch = S.cst[sg + 1] - S.cst[sg];
  const int64_t span = ((nu - base) + nch - 1) / nch;
  const int64_t spanA = (span + 15) & ~(int64_t)15;
  const int64_t qa_ = vw_rfl((int)(base + (chunk - S.cst[sg]) * spanA));
  const int64_t qb_ = vw_rfl((int)(qa_ + spanA < nu ? qa_ + spanA : nu));

  double pl[PPL], pm[PPL], pn[PPL], lp[PPL], mp[PPL];
  float fl[PPL], fm[PPL], fn[PPL]; /* FP32 directions (partly visible groups, plain form) */
  bool ok[PPL];
#pragma unroll
  for (int k = 0; k < PPL; ++k) {
    int64_t p = pbase + lane + 64 * k;
    ok[k] = p < S.npts;
    int64_t pp = S.pt0 + (ok[k] ? p : 0);
    pl[k] = S.l[pp];
    pm[k] = S.m[pp];
    pn[k] = S.n[pp];
    lp[k] = fma(sp.fa, pn[k], pl[k]);
    mp[k] = fma(sp.fb, pn[k], pm[k]);
    if (!BITS) {
      fl[k] = (float)pl[k];
      fm[k] = (float)pm[k];
      fn[k] = (float)pn[k];
    }
  }
  ReconLane<PPL, MIXED> acc;
  uint32_t wl[PPL];
#pragma unroll
  for (int k = 0; k < PPL; ++k) wl[k] = 0;
  uint32_t wu = 0;
  int nblk = 0;

  if (VW_KIND_IS_REP(KIND) || KIND == VW_KIND_AVG) {
    /* records pass through a per-wave LDS ring in blocks of 16 (512 B: one
     * double per lane, loaded one block ahead); each group is then read with
     * a uniform LDS address.  The mask words of 16 groups are scalar loads
     * fetched one block ahead; the set bits are walked, the groups visible
     * from the whole tile first, so that a hidden group costs nothing and
     * each kind of term has one place in the code (the sums stay in their
     * registers): a class byte per group tested in turn, with a fourfold
     * unrolled site per class, cost a dozen scalar instructions a group and
     * eight moves a term.  Nside 256, 32 antennas, 1024^2 image, one 64-epoch
     * segment: 30.6 -> 29.6 ms plain, 15.0 -> 12.7 ms mixed; Nside 128 mixed
     * day 10.8 -> 10.0 ms.  Blocks start at multiples of 16 and nq_pad is a multiple of
     * 64, so every block lies inside the records and the masks. */
    double* ring = gring[vw_rfl((int)(threadIdx.x >> 6))];
    const double* recd = (const double*)a.g.rec;
    const uint64_t* mrow = VW_KIND_IS_REP(KIND) ? S.cls + tile * (a.nq_pad >> 4) : nullptr;
    double stage = (qa_ < qb_) ? recd[qa_ * 4 + lane] : 0.0;
    uint64_t nmw = 0;
    if (VW_KIND_IS_REP(KIND) && qa_ < qb_) nmw = vw_rfl64(mrow[qa_ >> 4]);
    /* lane j < 16: the frames of the block's group j; the words of the wave's
     * points, 64 k points on for point k of a lane */
    const int fw = (int)(a.TP / 64);
    const uint64_t* fv = BITS ? S.fvis + tile * a.nfr_pad * fw + (pbase - tile * a.TP) / 64 : nullptr;
    int32_t nia = 0, nib = 0;
    if (BITS && qa_ < qb_) {
      nia = a.g.gia[qa_ + (lane & 15)];
      nib = a.g.gib[qa_ + (lane & 15)];
    }
    /* the walk, built with and without the polar terms: a choice per term cost
     * the mixed form 3% (Nside 256, 32 antennas, 64 epochs: 7.28 -> 7.51 ms) */
    auto walk = [&](auto polar_) {
      constexpr bool POLAR = decltype(polar_)::value;
      int buf = 0;
      for (int q16 = (int)qa_; q16 < (int)qb_; q16 += 16, buf ^= 1) {
        ring[buf * 64 + lane] = stage;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        uint64_t mw = nmw;
        const int32_t cia = nia, cib = nib;
        if (q16 + 16 < (int)qb_) {
          stage = recd[(int64_t)(q16 + 16) * 4 + lane];
          if (VW_KIND_IS_REP(KIND)) {
            nmw = vw_rfl64(mrow[(q16 + 16) >> 4]);
            if (BITS) {
              nia = a.g.gia[q16 + 16 + (lane & 15)];
              nib = a.g.gib[q16 + 16 + (lane & 15)];
            }
          }
        }
        if (KIND == VW_KIND_AVG) { /* every group of nonzero key, no classes */
          const int lo = (int)q0 > q16 ? (int)q0 - q16 : 0, hi = (int)qb_ - q16 < 16 ? (int)qb_ - q16 : 16;
          mw = ((1u << hi) - 1u) & ~((1u << lo) - 1u);
        }
        const GRec* blk = (const GRec*)(ring + buf * 64);
        uint32_t vis = (uint32_t)mw & 0xffffu;
        const uint32_t opa = (uint32_t)(mw >> 16) & 0xffffu, opb = (uint32_t)(mw >> 32);
        uint32_t part = opa | opb;
        if (KIND != VW_KIND_REP_FINITE) wu += (uint32_t)__builtin_popcount(vis);
        while (vis) {
          const int j = __builtin_ctz(vis);
          vis &= vis - 1;
          const GRec g = blk[j];
          if (KIND == VW_KIND_REP_FINITE) {
            if (!isfinite(g.amp)) continue;
            wu += 1;
          }
          if (POLAR) acc.template add<false>(g, nullptr, lp, mp);
          else acc.add_one(g, a.g.v[q16 + j], nullptr, lp, mp, a.tab);
        }
        if (VW_KIND_IS_REP(KIND)) {
          while (part) {
            const int j = __builtin_ctz(part);
            part &= part - 1;
            const GRec g = blk[j];
            if (KIND == VW_KIND_REP_FINITE && !isfinite(g.amp)) continue;
            bool use[PPL];
            if constexpr (BITS) {
              /* both frames' words, the one's twice where only it is open */
              const int32_t fa = __builtin_amdgcn_readlane(cia, j), fb = __builtin_amdgcn_readlane(cib, j);
              const uint64_t* va = fv + (int64_t)(opa >> j & 1 ? fa : fb) * fw;
              const uint64_t* vb = fv + (int64_t)(opb >> j & 1 ? fb : fa) * fw;
#pragma unroll
              for (int k = 0; k < PPL; ++k) use[k] = __builtin_amdgcn_inverse_ballot_w64(va[k] & vb[k]);
            } else {
              float fr[8];
#pragma unroll
              for (int e = 0; e < 8; ++e) fr[e] = a.g.ant32[(int64_t)(q16 + j) * 8 + e];
              float vd[PPL], near_ = 4.f;
#pragma unroll
              for (int k = 0; k < PPL; ++k) {
                vd[k] = vw_vis32(fl[k], fm[k], fn[k], fr);
                near_ = fminf(near_, fabsf(vd[k]));
                use[k] = vd[k] > 0.f;
              }
              if (__ballot(near_ <= VW_VIS_EPS)) { /* a point on the horizon: the FP64 test */
                const double* d = a.g.ant + (int64_t)(q16 + j) * 10;
#pragma unroll
                for (int k = 0; k < PPL; ++k) {
                  int ln = lane; /* opaque: the addresses are formed here, not kept in registers across the loop */
                  __asm__ volatile("" : "+v"(ln));
                  const int64_t pp = S.pt0 + (ok[k] ? pbase + ln + 64 * k : 0);
                  use[k] = vw_vis2<true>(ok[k], S.l[pp], S.m[pp], S.n[pp], d[0], d[1], d[2], d[3], d[4], d[5], d[6],
                                         d[7], d[8], d[9]);
                }
              }
            }
#pragma unroll
            for (int k = 0; k < PPL; ++k) wl[k] += use[k] ? 1 : 0;
            if (POLAR) acc.template add<true>(g, use, lp, mp);
            else acc.add_one(g, a.g.v[q16 + j], use, lp, mp, a.tab);
          }
        }
        if (buf) acc.fold();
      }
    };
    if (polar) walk(std::true_type{});
    else walk(std::false_type{});
  } else {
    /* generic representative sets (viss_recon_kernel.cuh:603-614, isfinite filter) */
    for (int64_t q = (qa_ > q0 ? qa_ : q0); q < qb_; ++q) {
      const int32_t s0 = a.goff[q], s1 = a.goff[q + 1], L = s1 - s0;
      int32_t posv[4];
      int np;
      if (a.occ_mode == 0) np = -1;
      else if (a.occ_mode == 1) { posv[0] = s0; np = 1; }
      else if (a.occ_mode == 2) { posv[0] = s0 + (L >> 1); np = 1; }
      else { posv[0] = s0; posv[1] = s0 + L / 3; posv[2] = s0 + (2 * L) / 3; posv[3] = s1 - 1; np = 4; }
      double sr[PPL], si[PPL];
      int cn[PPL];
#pragma unroll
      for (int k = 0; k < PPL; ++k) { sr[k] = 0.0; si[k] = 0.0; cn[k] = 0; }
      const int32_t kend = (np < 0) ? s1 : np;
      for (int32_t kk = (np < 0 ? s0 : 0); kk < kend; ++kk) {
        const int32_t pos = (np < 0) ? kk : posv[kk];
        bool ng;
        const int64_t h = vw_row_half(a.idx_sorted[pos], a.P, a.full != 0, &ng);
        const int cls = vw_cls_lookup((const uint32_t*)S.cls, tile, a.nh_pad, h);
        if (cls == VW_CLS_HIDDEN) continue;
        bool mv[PPL];
        if (cls == VW_CLS_VISIBLE) {
#pragma unroll
          for (int k = 0; k < PPL; ++k) mv[k] = ok[k];
        } else {
          const RowRec rec = a.rows[h];
          vw_ant_vis<PPL, !MIXED>(a.ant8, rec.ia, rec.ib, pl, pm, pn, ok, mv);
        }
        const double2 v = a.vh[h];
        const double wr = v.x, wi = ng ? -v.y : v.y;
        const bool fin = isfinite(wr) && isfinite(wi);
#pragma unroll
        for (int k = 0; k < PPL; ++k)
          if (mv[k] && fin) { sr[k] = sr[k] + wr; si[k] = si[k] + wi; cn[k] += 1; }
      }
      const double ugu = a.g.rec[q].ugu, vgu = a.g.rec[q].vgu;
      double ar[PPL], ai[PPL];
      bool use[PPL];
#pragma unroll
      for (int k = 0; k < PPL; ++k) {
        use[k] = cn[k] > 0;
        const double invc = 1.0 / (double)(use[k] ? cn[k] : 1);
        ar[k] = sr[k] * invc;
        ai[k] = si[k] * invc;
        wl[k] += use[k] ? 1 : 0;
      }
      acc.add_ri(ugu, vgu, ar, ai, use, lp, mp, tab);
      if (MIXED && ++nblk == 32) {
        nblk = 0;
        acc.fold();
      }
    }
  }
#pragma unroll
  for (int k = 0; k < PPL; ++k) {
    if (!ok[k]) continue;
    const int64_t p = pbase + lane + 64 * k;
    S.part[chunk * S.npts + p] = acc.value(k);
    S.wpart[chunk * S.npts + p] = wu + wl[k];
  }
}

/* fold group-range partials in order into the accumulators (add_inplace) for
 * the points of a pass, both output sets */
__global__ void k_recon_reduce(ReconSets sets, int weights, uint64_t* __restrict__ ts) {
  vw_ts_begin(ts);
  const int64_t nb0 = (sets.s[0].npts + blockDim.x - 1) / blockDim.x;
  const int si = (int64_t)blockIdx.x >= nb0;
  const ReconSet& S = sets.s[si];
  const int64_t p = ((int64_t)blockIdx.x - (si ? nb0 : 0)) * blockDim.x + threadIdx.x;
  if (p >= S.npts) return;
  const double* __restrict__ part = S.part;
  const uint32_t* __restrict__ wpart = S.wpart;
  const int64_t nchunk = S.nchunk, pstride = S.npts;
  double s = part[p];
  uint32_t w = wpart[p];
  /* VW_FOLD_BATCH chunks' loads in flight at a time; the sum keeps chunk order */
  int64_t k = 1;
  for (; k + VW_FOLD_BATCH <= nchunk; k += VW_FOLD_BATCH) {
    double x[VW_FOLD_BATCH];
    uint32_t y[VW_FOLD_BATCH];
#pragma unroll
    for (int e = 0; e < VW_FOLD_BATCH; ++e) {
      x[e] = part[(k + e) * pstride + p];
      y[e] = wpart[(k + e) * pstride + p];
    }
#pragma unroll
    for (int e = 0; e < VW_FOLD_BATCH; ++e) {
      s = s + x[e];
      w += y[e];
    }
  }
  for (; k < nchunk; ++k) {
    s = s + part[k * pstride + p];
    w += wpart[k * pstride + p];
  }
  S.acc[S.pt0 + p] = S.acc[S.pt0 + p] + s;
  if (weights) S.wacc[S.pt0 + p] += w;
  vw_ts_end(ts); /* thread 0 of a workgroup has a point */
}

/* Final maps of every sky of both output sets: C = acc / W (blockage 1) or
 * acc * (1/W_total) (blockage 0), one thread per output value; inv (lm image)
 * gives an output pixel's point, -1 outside the unit disk, which gets zeros.
 * Weight maps: one for all skies (wstride 0, written with sky 0) or one a sky. */
struct FinalSet {
  const double* acc;      /* [nsky][nin]               */
  const uint32_t* w;      /* [nin] or [nsky][nin]      */
  const int32_t* inv;     /* [nout] or null            */
  int64_t nin, nout;
  int64_t wstride;        /* 0 or nin                  */
  double* out;            /* [nsky][nout]              */
  uint32_t* wout;         /* [nout] or [nsky][nout]; null: not wanted */
};
struct FinalArgs {
  FinalSet s[2]; /* nout 0: absent */
  int64_t nsky;
  int blockage;
  const DevInfo* info;
};
__global__ __launch_bounds__(256) void k_finalize(FinalArgs a, uint64_t* __restrict__ ts) {
  vw_ts_begin(ts);
  const int64_t nb0 = (a.nsky * a.s[0].nout + 255) / 256;
  const int si = (int64_t)blockIdx.x >= nb0;
  const FinalSet& S = a.s[si];
  const int64_t k = ((int64_t)blockIdx.x - (si ? nb0 : 0)) * 256 + threadIdx.x;
  if (k >= a.nsky * S.nout) return;
  const int64_t sk = k / S.nout, o = k - sk * S.nout;
  const int64_t i = S.inv ? S.inv[o] : o;
  double v = 0.0;
  uint32_t wi = 0;
  if (i >= 0) {
    wi = S.w[sk * S.wstride + i];
    const double x = S.acc[sk * S.nin + i];
    if (a.blockage) v = wi > 0 ? x / (double)wi : 0.0;
    else {
      const int64_t wt = a.info->wtotal;
      const double r = wt > 0 ? 1.0 / (double)wt : 0.0;
      v = x * r;
    }
  }
  S.out[k] = v;
  if (S.wout && (S.wstride || sk == 0)) S.wout[k] = wi;
  vw_ts_end(ts);
}

/* point index of each image pixel (inv filled with -1 before) */
__global__ void k_grid_inv(int64_t npts, const int64_t* __restrict__ gidx, int32_t* __restrict__ inv) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < npts) inv[gidx[k]] = (int32_t)k;
}

/* zeroes up to eight arrays of 32-bit words in one launch (kernels, not memset
 * nodes: a captured step holds it).  Arrays start 16-byte aligned. */
struct ClearArgs {
  uint32_t* p[8];
  int64_t n[8];
  int cnt;
};
__global__ __launch_bounds__(256) void k_clear(ClearArgs a) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x, nt = (int64_t)gridDim.x * 256;
  for (int j = 0; j < a.cnt; ++j) {
    const int64_t n4 = a.n[j] / 4;
    for (int64_t i = t; i < n4; i += nt) ((uint4*)a.p[j])[i] = make_uint4(0, 0, 0, 0);
    if (t < a.n[j] - 4 * n4) a.p[j][4 * n4 + t] = 0;
  }
}

#endif
