/*
 * vw_batch.h -- sky batches: many sky realisations through one geometry.
 *
 * The skies of a batch share antennas, epochs, the segment schedule and so
 * the rows, tile classes, w-plane fit, uv cells and groups of every segment.
 * Both sums then become products of a phasor matrix that depends only on
 * the geometry with a matrix that holds one column per sky:
 *
 *   Viss   V[h][s] = sum_p  M[h][p] exp(-j 2 pi x_hp) I[p][s]
 *          (rows x pixels) x (pixels x skies)
 *   recon  C[q][s] = sum_g  M[q][g] Re(exp(+j 2 pi y_qg) V_g[s])
 *          (points x groups) x (groups x skies)
 *
 * The phasor tiles are made on the fly (FP64 phase and its reduction mod 1
 * turn, hardware FP32 sin/cos, the occlusion mask as zeros) and never stored;
 * the products run on the BF16 matrix cores (v_mfma_f32_16x16x32_bf16) with
 * both operands split x = hi + lo into two BF16 values and three products
 * hi*hi + hi*lo + lo*hi per real multiply-add (about 2^-16 relative per
 * term), FP32 accumulation over one 256-pixel sub-tile or 256-group block,
 * then FP64 sums across blocks, chunks and passes.
 *
 * Operand layout of v_mfma_f32_16x16x32_bf16 (wave64), as used here:
 *   A (16 x 32, rows x k):  lane l holds row l % 16, k = 8 (l / 16) + i, i < 8
 *   B (32 x 16, k x cols):  lane l holds column l % 16, the same k
 *   D (16 x 16, f32):       lane l holds D[4 (l / 16) + i][l % 16], i < 4
 * A and B use the same k assignment, so any permutation of k inside the
 * instruction leaves the product unchanged.
 *
 * Packed operand matrices (sky, group visibilities) are stored as
 * [k / 32][nsky_pad][32] BF16, so a lane's 8 values are one 16-byte load.
 */
#ifndef VW_BATCH_H
#define VW_BATCH_H

#include "vw_kernels.h"

typedef __bf16 vw_bf16x8 __attribute__((ext_vector_type(8)));
typedef float vw_f32x4b __attribute__((ext_vector_type(4)));

typedef float vw_f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 vw_bf16x2 __attribute__((ext_vector_type(2)));

/* x = hi + lo with hi = bf16(x) and lo = bf16(x - hi), both rounded to
 * nearest even: x - hi is exact in FP32 and |x - hi| <= 2^-9 |x|, so
 * |x - hi - lo| <= 2^-18 |x| and the omitted lo*lo product of a split
 * multiply is below 2^-18 of the term.  Per pair of values: one packed
 * conversion, a shift and a mask back to FP32, two subtractions, one packed
 * conversion of the remainders. */
__device__ __forceinline__ void vw_split8(const float (&x)[8], vw_bf16x8& hi, vw_bf16x8& lo) {
  uint32_t h[4], l[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const vw_f32x2 v = {x[2 * j], x[2 * j + 1]};
    const uint32_t hp = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, vw_bf16x2));
    const float h0 = __builtin_bit_cast(float, hp << 16), h1 = __builtin_bit_cast(float, hp & 0xffff0000u);
    const vw_f32x2 rr = {x[2 * j] - h0, x[2 * j + 1] - h1};
    h[j] = hp;
    l[j] = __builtin_bit_cast(uint32_t, __builtin_convertvector(rr, vw_bf16x2));
  }
  hi = __builtin_bit_cast(vw_bf16x8, h);
  lo = __builtin_bit_cast(vw_bf16x8, l);
}

__device__ __forceinline__ vw_bf16x8 vw_ld_bf16x8(const uint4* p) {
  return __builtin_bit_cast(vw_bf16x8, *p);
}

__device__ __forceinline__ vw_f32x4b vw_mfma_bf16(vw_bf16x8 a, vw_bf16x8 b, vw_f32x4b c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

/* three-product split multiply-accumulate: (ah + al)(bh + bl) without al*bl */
__device__ __forceinline__ vw_f32x4b vw_mac3(vw_bf16x8 ah, vw_bf16x8 al, vw_bf16x8 bh, vw_bf16x8 bl,
                                             vw_f32x4b c) {
  c = vw_mfma_bf16(al, bh, c);
  c = vw_mfma_bf16(ah, bl, c);
  return vw_mfma_bf16(ah, bh, c);
}

/* ------------------------------------------------------------------ */
/* packing                                                              */
/* ------------------------------------------------------------------ */

/* sky batch [nsky][npix] FP32 (already scaled by the pixel area) ->
 * hi / lo [npix_pad / 32][nsky_pad][32]; zero for padding pixels and skies */
__global__ void k_sky_pack(const float* __restrict__ sky, int64_t nsky, int64_t npix, int64_t npix_pad,
                           int64_t nsky_pad, __bf16* __restrict__ hi, __bf16* __restrict__ lo) {
  int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= npix_pad * nsky_pad) return;
  const int64_t kb = k / (nsky_pad * 32);
  const int64_t r = k - kb * nsky_pad * 32;
  const int64_t s = r / 32, j = r - s * 32;
  const int64_t p = kb * 32 + j;
  const float x = (s < nsky && p < npix) ? sky[s * npix + p] : 0.0f;
  const __bf16 h = (__bf16)x;
  hi[k] = h;
  lo[k] = (__bf16)(x - (float)h);
}

/* ------------------------------------------------------------------ */
/* work order                                                           */
/* ------------------------------------------------------------------ */

/* The batched kernels walk rows (Viss) and groups (recon) in an order that
 * keeps rows with similar occlusion together, so that more 16-row blocks are
 * hidden on a whole tile and skipped: the sort key of a row is the unordered
 * pair of the coarse direction cells of its two antennas (each unit vector
 * quantised to 4 levels per axis and Morton-interleaved: 64 cells).  At
 * Nside 128 / 16 antennas this takes the share of skipped (tile, 16-row)
 * blocks from 4% to 35% (the per-tile bound is 43%).  Entries past the count
 * get key 4096 and sort last; the sort is stable, so ties keep index order. */
#define VW_ORDER_BITS 13
__device__ __forceinline__ int vw_dir_cell(double x, double y, double z) {
  const double v[3] = {x, y, z};
  int c = 0;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    int q = (int)((v[d] + 1.0) * 2.0);
    q = q < 0 ? 0 : (q > 3 ? 3 : q);
    c |= ((q >> 1) & 1) << (3 + d);
    c |= (q & 1) << d;
  }
  return c;
}
__device__ __forceinline__ int32_t vw_pair_key(const double* __restrict__ ant8, int ia, int ib) {
  const double* qa = ant8 + (int64_t)ia * 8;
  const double* qb = ant8 + (int64_t)ib * 8;
  const int ca = vw_dir_cell(qa[4], qa[5], qa[6]), cb = vw_dir_cell(qb[4], qb[5], qb[6]);
  return (ca < cb) ? (ca << 6) | cb : (cb << 6) | ca;
}
__global__ void k_row_keys(const RowRec* __restrict__ rows, const double* __restrict__ ant8, int64_t nh, int64_t n,
                           int32_t* __restrict__ keys, int32_t* __restrict__ idx) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  keys[i] = i < nh ? vw_pair_key(ant8, rows[i].ia, rows[i].ib) : 4096;
  idx[i] = (int32_t)i;
}
/* cell centres and the representatives' antenna-frame indices in the recon's
 * work order */
__global__ void k_group_order_recs(const int32_t* __restrict__ order, const GRec* __restrict__ rec,
                                   const int32_t* __restrict__ gia, const int32_t* __restrict__ gib, int64_t n,
                                   double2* __restrict__ orec, int32_t* __restrict__ oia, int32_t* __restrict__ oib) {
  int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const int64_t q = order[j];
  const GRec g = rec[q];
  orec[j] = make_double2(g.ugu, g.vgu);
  oia[j] = gia[q];
  oib[j] = gib[q];
}
__global__ void k_group_keys(const int32_t* __restrict__ gia, const int32_t* __restrict__ gib,
                             const double* __restrict__ ant8, const DevInfo* __restrict__ info, int64_t n,
                             int32_t* __restrict__ keys, int32_t* __restrict__ idx) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  keys[i] = i < info->nuniq ? vw_pair_key(ant8, gia[i], gib[i]) : 4096;
  idx[i] = (int32_t)i;
}

/* ------------------------------------------------------------------ */
/* occlusion bits                                                       */
/* ------------------------------------------------------------------ */

/* Which points each antenna frame sees, one word per (32-point block of the
 * pass, frame): out[block][nfr_pad], bit j = point 32 block + j.  A row's or a
 * group's mask over 32 points is the AND of its two frames' words, so the
 * occlusion test runs once per (point, frame) instead of twice per masked term
 * (an epoch's A frames serve A (A - 1) / 2 rows), and the term loops of the
 * products hold no test.  A frame that the tile's cone finds all visible or
 * all hidden needs none at all; bits are the per-point FP64 test's otherwise.  A
 * mask so equals the pair class with its per-point tests, but for a point at the
 * far end of a cone whose rounded bound passes the frame by less than the point
 * fails it (1e-15; bit 2 of vw_cone_bits): the class tests it for a pair whose
 * other frame is partly visible, and passes it for one whose other frame is all
 * visible; a frame has one word for both, and passes it here.
 * A wave owns 64 points and 64 frames (vw_frame_words); 50 us for 196,608
 * points x 2,080 frames.  64 skies at Nside 128, 16 antennas, 205 epochs and a
 * 256^2 image, against class bytes with the FP64 test in the term loops (a
 * divergent branch per masked term in the recon): k_reconb 22.3 -> 16.3 ms and
 * k_vissb 7.4 -> 6.5 ms of overlapped kernel time, the call 36.8 -> 33.8 ms,
 * results equal bit for bit.
 * A one-dimensional grid, point blocks fastest: a second dimension ends at 65,536
 * workgroups, 4.2 million frames. */
__global__ __launch_bounds__(256) void k_frame_vis(const double* __restrict__ l, const double* __restrict__ m,
                                                   const double* __restrict__ n, int64_t npts,
                                                   const double* __restrict__ cone, int64_t ntile, int64_t tile0,
                                                   int64_t nblk, int64_t TP, const double* __restrict__ ant8,
                                                   int64_t nfr, int64_t nfr_pad, uint32_t* __restrict__ out) {
  const int lane = threadIdx.x & 63;
  const uint32_t npb = (uint32_t)((nblk + 3) / 4), fb = blockIdx.x / npb;
  const int64_t b = (int64_t)(blockIdx.x - fb * npb) * 4 + vw_rfl((int)(threadIdx.x >> 6));
  if (b >= nblk) return;
  const int64_t t = tile0 + b * 64 / TP;
  const int64_t p = tile0 * TP + b * 64 + lane;
  const bool ok = p < npts;
  const int64_t pp = ok ? p : npts - 1;
  const double pl = l[pp], pm = m[pp], pn = n[pp];
  const int64_t f = (int64_t)fb * 64 + lane;
  const double* q = ant8 + (f < nfr ? f : nfr - 1) * 8;
  const int cb = vw_cone_bits(q[4], q[5], q[6], cone[t], cone[ntile + t], cone[2 * ntile + t], cone[3 * ntile + t],
                              cone[4 * ntile + t], q[7]);
  const uint64_t w = vw_frame_words(ant8, f, nfr, cb, pl, pm, pn, ok);
  out[2 * b * nfr_pad + f] = (uint32_t)w;
  out[(2 * b + 1) * nfr_pad + f] = (uint32_t)(w >> 32);
}

/* all ones where bit `bit` of x is set, else zero */
__device__ __forceinline__ int vw_bit_mask(uint32_t x, int bit) { return __builtin_amdgcn_sbfe((int)x, bit, 1); }
__device__ __forceinline__ float vw_and_f32(float x, int mask) {
  return __builtin_bit_cast(float, __builtin_bit_cast(int, x) & mask);
}

/* ------------------------------------------------------------------ */
/* Viss                                                                 */
/* ------------------------------------------------------------------ */
struct VissBArgs {
  const double *l, *m, *nm1;
  const uint4 *skyh, *skyl; /* packed sky, 16-byte units                        */
  int64_t npix, nsky_pad;
  int64_t tile0, ntile, TP;  /* tiles of this pass                              */
  const RowRec* rows;
  const uint32_t* fvis;      /* [32-pixel block of the pass][nfr_pad] occlusion bits */
  int64_t nfr_pad;
  const int32_t* perm;       /* work order: block row j is half row perm[j]       */
  int64_t nh, nh_pad;
  int64_t tpc, nchunk, nrb, nrbw; /* tiles per chunk, chunks, 16-row blocks, blocks of 4 */
  double2* part;             /* [nchunk][nsky_pad][nh_pad]                        */
};

/* LDS staging of one k-step of a packed operand: NARR arrays x (16 NB)
 * rows of 32 BF16, each row padded to 40 BF16 (80 B) so that the 16 rows a
 * 16-lane phase reads fall on disjoint banks.  A workgroup loads step k + 1
 * into registers (16 B per thread and array) while it computes step k, then
 * stores them into the other buffer. */
#define VW_LROW 40
typedef unsigned int vw_u32x4 __attribute__((ext_vector_type(4)));
template <int NARR, int NB>
struct VwStage {
  static constexpr int ROWS = NARR * 16 * NB; /* LDS rows per k-step */
  vw_u32x4 r0, r1, r2, r3;
  /* thread t < 64 NB holds the 16-byte unit t of every array's block kb:
   * row row0 + t / 4 of the sky group, quarter t % 4 of its 32 values */
  __device__ __forceinline__ void load(const uint4* p0, const uint4* p1, const uint4* p2, const uint4* p3, int64_t kb,
                                       int64_t nsky_pad, int64_t row0) {
    const int t = (int)threadIdx.x;
    if (t < 64 * NB) {
      const int64_t off = (kb * nsky_pad + row0 + (t >> 2)) * 4 + (t & 3);
      r0 = *(const vw_u32x4*)(p0 + off);
      if (NARR > 1) r1 = *(const vw_u32x4*)(p1 + off);
      if (NARR > 2) r2 = *(const vw_u32x4*)(p2 + off);
      if (NARR > 3) r3 = *(const vw_u32x4*)(p3 + off);
    }
  }
  __device__ __forceinline__ void store(__bf16* buf) const {
    const int t = (int)threadIdx.x;
    if (t < 64 * NB) {
      __bf16* d = buf + (t >> 2) * VW_LROW + (t & 3) * 8;
      *(vw_u32x4*)d = r0;
      if (NARR > 1) *(vw_u32x4*)(d + 16 * NB * VW_LROW) = r1;
      if (NARR > 2) *(vw_u32x4*)(d + 32 * NB * VW_LROW) = r2;
      if (NARR > 3) *(vw_u32x4*)(d + 48 * NB * VW_LROW) = r3;
    }
  }
};

__device__ __forceinline__ vw_bf16x8 vw_lds_bf16x8(const __bf16* buf, int row, int g) {
  return *(const vw_bf16x8*)(buf + row * VW_LROW + g * 8);
}

/* one wave: 16 half rows x (16 NB) skies over the tiles of one chunk; a
 * workgroup is four waves (64 consecutive rows) on the same pixels.  Per
 * k-step of 32 pixels the workgroup stages the sky operand and the pixels' l,
 * m, n - 1 through double-buffered LDS; a lane's row takes its mask over the
 * step's pixels from its two frames' words of the occlusion bits.  Every step
 * issues the same global loads, for the next step, unconditionally (indices
 * clamped in range), and waits for them only before their LDS stores at its
 * end: a load waited for right after it is issued would also wait for the
 * loads in flight before it (the vector memory counter is in order), exposing
 * their latency. */
#ifndef VW_VISSB_WAVES
#define VW_VISSB_WAVES 3
#endif
template <int NB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(VW_VISSB_WAVES))) void k_vissb(VissBArgs a) {
  using Stage = VwStage<2, NB>;
  __shared__ __attribute__((aligned(16))) __bf16 bsh[2][Stage::ROWS * VW_LROW];
  __shared__ double px[2][3][32]; /* l, m, n - 1 of a k-step's pixels */
  const int64_t vb = vw_xcd_block(blockIdx.x, gridDim.x);
  const int64_t rbw = vb % a.nrbw;
  const int64_t rest = vb / a.nrbw;
  const int64_t chunk = rest % a.nchunk;
  const int64_t sg = rest / a.nchunk;
  const int wave = vw_rfl((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  const int64_t rb = rbw * 4 + wave;
  const bool wave_on = rb < a.nrb; /* uniform; every wave still joins the barriers */
  const int64_t jr = rb * 16 + r;  /* block row */
  /* the sorted order puts the padding rows (index >= nh) last */
  const bool row_on = jr < a.nh;
  const RowRec rec = a.rows[a.perm[row_on ? jr : 0]];
  const uint32_t rmask = row_on ? 0xffffffffu : 0u;
  const int64_t t0 = a.tile0 + chunk * a.tpc;
  const int64_t tend = a.tile0 + a.ntile;
  const int64_t t1 = (t0 + a.tpc < tend) ? t0 + a.tpc : tend;
  const int ksh = a.TP == 512 ? 4 : 3; /* k-steps per tile: 1 << ksh */
  const int64_t kb0 = t0 << ksh;       /* first k-step block of the chunk */
  const int64_t K = (t1 - t0) << ksh;  /* k-steps of 32 pixels (> 0) */
  const int64_t row0 = sg * 16 * NB;

  Stage stg;
  /* thread t < 96: coordinate t / 32 of pixel t % 32 of a step (the others
   * repeat a load, unstored) */
  const int xc_ = (int)(threadIdx.x >> 5);
  const double* xsrc = xc_ == 0 ? a.l : (xc_ == 1 ? a.m : a.nm1);
  const uint32_t* fv = a.fvis + (kb0 - (a.tile0 << ksh)) * a.nfr_pad;
  double xp;
  uint32_t xa, xb; /* the next step's words of the row's two frames */
#define VW_X_LOAD(k_)                                             \
  do {                                                            \
    const int64_t p_ = ((kb0 + (k_)) << 5) + (threadIdx.x & 31);  \
    const double v_ = xsrc[p_ < a.npix ? p_ : a.npix - 1];        \
    xp = p_ < a.npix ? v_ : 0.0;                                  \
    xa = fv[(k_) * a.nfr_pad + rec.ia];                           \
    xb = fv[(k_) * a.nfr_pad + rec.ib];                           \
  } while (0)
#define VW_X_STORE(b_)                                          \
  do {                                                          \
    if (threadIdx.x < 96) px[b_][xc_][threadIdx.x & 31] = xp;   \
  } while (0)

  vw_f32x4b accR[NB], accI[NB], sumR[NB], sumI[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    accR[nb] = vw_f32x4b{0.f, 0.f, 0.f, 0.f};
    accI[nb] = vw_f32x4b{0.f, 0.f, 0.f, 0.f};
    sumR[nb] = vw_f32x4b{0.f, 0.f, 0.f, 0.f};
    sumI[nb] = vw_f32x4b{0.f, 0.f, 0.f, 0.f};
  }

  /* prologue: step 0 */
  VW_X_LOAD(0);
  stg.load(a.skyh, a.skyl, nullptr, nullptr, kb0, a.nsky_pad, row0);
  VW_X_STORE(0);
  stg.store(bsh[0]);
  __syncthreads();

  bool dirty = false; /* uniform: the block's accumulators hold products */
  for (int64_t k = 0; k < K; ++k) {
    const int buf = (int)(k & 1);
    const int64_t kn = k + 1 < K ? k + 1 : k; /* the last step reloads itself */
    const uint32_t mw = xa & xb & rmask;      /* bit kk: pixel kk of the step is seen */
    stg.load(a.skyh, a.skyl, nullptr, nullptr, kb0 + kn, a.nsky_pad, row0);
    VW_X_LOAD(kn);
    if (wave_on && __ballot(mw != 0) != 0) {
      const double* pl_ = px[buf][0];
      const double* pm_ = px[buf][1];
      const double* pz_ = px[buf][2];
      float cv[8], sv[8];
      /* two forms of the step, chosen per wave: with and without masks */
#define VW_PHASOR(MASKED_)                                                  \
  do {                                                                      \
    _Pragma("unroll") for (int i = 0; i < 8; ++i) {                         \
      const int kk = g * 8 + i;                                             \
      const double x = vw_viss_phase(rec.u, rec.v, rec.w, pl_[kk], pm_[kk], pz_[kk]); \
      const float f = (float)__builtin_amdgcn_fract(x);                     \
      const float sn = __builtin_amdgcn_sinf(f), cs = __builtin_amdgcn_cosf(f); \
      const int on = MASKED_ ? vw_bit_mask(m8, i) : -1;                     \
      cv[i] = MASKED_ ? vw_and_f32(cs, on) : cs;                            \
      sv[i] = MASKED_ ? vw_and_f32(sn, on) : sn;                            \
    }                                                                       \
  } while (0)
      const uint32_t m8 = mw >> (8 * g);
      if (__ballot(mw != 0xffffffffu)) VW_PHASOR(true);
      else VW_PHASOR(false);
#undef VW_PHASOR
      vw_bf16x8 ach, acl, ash, asl;
      vw_split8(cv, ach, acl);
      vw_split8(sv, ash, asl);
      const __bf16* bb = bsh[buf];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const vw_bf16x8 bh = vw_lds_bf16x8(bb, nb * 16 + r, g);
        const vw_bf16x8 bl = vw_lds_bf16x8(bb, 16 * NB + nb * 16 + r, g);
        accR[nb] = vw_mac3(ach, acl, bh, bl, accR[nb]);
        accI[nb] = vw_mac3(ash, asl, bh, bl, accI[nb]);
      }
      dirty = true;
    }
    if ((k & 7) == 7 && dirty) {
      /* blocked sums: the products of 256 pixels accumulate in the matrix
       * core's FP32 accumulators, which are then added to FP32 block sums
       * (folded across chunks in FP64): error ~ (256 + K / 256) ulp
       * rather than K ulp */
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        sumR[nb] += accR[nb];
        sumI[nb] += accI[nb];
        accR[nb] = vw_f32x4b{0.f, 0.f, 0.f, 0.f};
        accI[nb] = vw_f32x4b{0.f, 0.f, 0.f, 0.f};
      }
      dirty = false;
    }
    /* buffers of step k - 1: every wave passed the barrier after reading
     * them (the last step writes its own reload there, unread) */
    stg.store(bsh[buf ^ 1]);
    VW_X_STORE(buf ^ 1);
    __syncthreads();
  }
#undef VW_X_LOAD
#undef VW_X_STORE
  if (!wave_on) return;
  /* D[4 g + i][r]: block row rb * 16 + 4 g + i, sky column r */
  int64_t hw[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t jj = rb * 16 + 4 * g + i;
    hw[i] = jj < a.nh ? a.perm[jj] : -1;
  }
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int64_t sky = (sg * NB + nb) * 16 + r;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (hw[i] >= 0) a.part[(chunk * a.nsky_pad + sky) * a.nh_pad + hw[i]] = make_double2((double)sumR[nb][i], -(double)sumI[nb][i]);
  }
}

/* chunk partials -> raw half sums [nsky][nh], chunks in ascending order;
 * passes after the first add to the running sums */
__global__ void k_vissb_fold(const double2* __restrict__ part, int64_t nchunk, int64_t nsky, int64_t nsky_pad,
                             int64_t nh, int64_t nh_pad, int accumulate, double2* __restrict__ vraw) {
  int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nsky * nh) return;
  const int64_t s = k / nh, h = k - s * nh;
  double re = 0.0, im = 0.0;
  for (int64_t c = 0; c < nchunk; ++c) {
    const double2 v = part[(c * nsky_pad + s) * nh_pad + h];
    re += v.x;
    im += v.y;
  }
  if (accumulate) {
    re += vraw[k].x;
    im += vraw[k].y;
  }
  vraw[k] = make_double2(re, im);
}

/* phase correction and conjugate completion of every sky [nsky][nh] ->
 * [nsky][nh] and [nsky][2 nh] (common.hpp:255-277) */
__global__ void k_conj_fill_b(const double2* __restrict__ vraw, const RowRec* __restrict__ rows, int64_t nh, int P,
                              int64_t nsky, double2* __restrict__ vh, double2* __restrict__ vfull) {
  int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nsky * nh) return;
  const int64_t s = k / nh, h = k - s * nh;
  double re, im;
  vw_phase_correct(vraw[k].x, vraw[k].y, rows[h].w, &re, &im);
  vh[k] = make_double2(re, im);
  const int64_t g = h / P, j = h - g * P;
  double2* vf = vfull + s * 2 * nh;
  vf[2 * P * g + j] = make_double2(re, im);
  vf[2 * P * g + P + j] = make_double2(re, -im);
}

/* ------------------------------------------------------------------ */
/* reconstruction                                                       */
/* ------------------------------------------------------------------ */

/* group visibilities of every sky -> packed real and imaginary parts in the
 * recon's work order, [nq_pad / 32][nsky_pad][32] hi / lo; zero outside
 * [first_nz, nuniq) and for padding skies.  blockage 1: the representative's value (occ_mode 1
 * first member, else the median member, signed for rows of the conjugate
 * half); blockage 0: the group mean over members in sorted order. */
__global__ void k_group_pack(const int32_t* __restrict__ goff, const int32_t* __restrict__ idx_sorted,
                             const double2* __restrict__ vh, int64_t nh, int P, int full, int blockage, int occ_mode,
                             const DevInfo* __restrict__ info, const int32_t* __restrict__ gperm, int64_t nq_pad,
                             int64_t nsky, int64_t nsky_pad, __bf16* __restrict__ rh, __bf16* __restrict__ rl,
                             __bf16* __restrict__ ih, __bf16* __restrict__ il) {
  int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nq_pad * nsky_pad) return;
  const int64_t qb = k / (nsky_pad * 32);
  const int64_t rr = k - qb * nsky_pad * 32;
  const int64_t s = rr / 32, j = rr - s * 32;
  const int64_t q = gperm[qb * 32 + j]; /* position j of the work order holds group gperm[j] */
  float vr = 0.f, vi = 0.f;
  if (s < nsky && q >= info->first_nz && q < info->nuniq) {
    const int32_t s0 = goff[q], s1 = goff[q + 1];
    const double2* v = vh + s * nh;
    if (blockage) {
      bool neg;
      const int64_t hr = vw_row_half(idx_sorted[occ_mode == 1 ? s0 : s0 + (s1 - s0) / 2], P, full != 0, &neg);
      vr = (float)v[hr].x;
      vi = (float)(neg ? -v[hr].y : v[hr].y);
    } else {
      double sr = 0.0, si = 0.0;
      for (int32_t t = s0; t < s1; ++t) {
        bool ng;
        const int64_t hh = vw_row_half(idx_sorted[t], P, full != 0, &ng);
        sr = sr + v[hh].x;
        si = si + (ng ? -v[hh].y : v[hh].y);
      }
      vr = (float)(sr / (double)(s1 - s0));
      vi = (float)(si / (double)(s1 - s0));
    }
  }
  const __bf16 a = (__bf16)vr, b = (__bf16)vi;
  rh[k] = a;
  rl[k] = (__bf16)(vr - (float)a);
  ih[k] = b;
  il[k] = (__bf16)(vi - (float)b);
}

struct ReconBArgs {
  const double *l, *m, *n;
  int64_t pt0, npts;          /* points [pt0, pt0 + npts) of this pass            */
  const uint32_t* fvis;       /* [32-point block of the pass][nfr_pad] occlusion bits */
  int64_t nfr_pad;
  const int32_t* gperm;       /* work order: position j is group gperm[j]          */
  const double2* orec;        /* (ugu, vgu) in work order                          */
  const int32_t *oia, *oib;   /* the representative's antenna frames, work order   */
  const DevInfo* info;
  const uint4 *vrh, *vrl, *vih, *vil; /* packed group visibilities, 16-byte units */
  int64_t nsky_pad;
  int rep;                    /* 1: the representative's mask; 0: every group counts */
  int64_t nchunk, pblk, pbw;  /* group ranges, 16-point blocks, blocks of 4        */
  double* part;               /* [nchunk][nsky_pad][pstride]                       */
  uint32_t* wpart;            /* [nchunk][pstride]                                 */
  int64_t pstride;
};

/* one wave: 16 output points x (16 NB) skies over one range of groups; a
 * workgroup is four waves (64 consecutive points of one output tile).  Per
 * k-step of 32 groups the workgroup stages the packed group visibilities, the
 * groups' cell centres and, per wave, the groups' masks over its 16 points
 * through double-buffered LDS.  A mask is the AND of two words of the
 * occlusion bits; the words are gathered one step ahead, their frame indices
 * two.  Masks are zero for positions out of range and for the key-0 group, so
 * they are all the term loop asks. */
#ifndef VW_RECONB_WAVES
#define VW_RECONB_WAVES 3
#endif
template <int NB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(VW_RECONB_WAVES))) void k_reconb(ReconBArgs a) {
  using Stage = VwStage<4, NB>;
  __shared__ __attribute__((aligned(16))) __bf16 bsh[2][Stage::ROWS * VW_LROW];
  __shared__ double2 grec[2][32]; /* (ugu, vgu) */
  __shared__ __attribute__((aligned(16))) uint16_t gm[2][4][32]; /* masks: bit r = point r of the wave */
  const int64_t vb = vw_xcd_block(blockIdx.x, gridDim.x);
  const int64_t pbw = vb % a.pbw;
  const int64_t rest = vb / a.pbw;
  const int64_t chunk = rest % a.nchunk;
  const int64_t sg = rest / a.nchunk;
  const int wave = vw_rfl((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  const int64_t pb = pbw * 4 + wave;
  const bool wave_on = pb < a.pblk;
  const int64_t pbase = pb * 16;          /* pass-relative */
  const int64_t p = pbase + r;
  const bool okp = wave_on && p < a.npts;
  const int64_t pp = a.pt0 + (okp ? p : 0);
  const vw_segparams sp = a.info->sp;
  const double pl = a.l[pp], pm = a.m[pp], pn = a.n[pp];
  const double lp = fma(sp.fa, pn, pl), mp = fma(sp.fb, pn, pm);
  const int64_t nu = a.info->nuniq, q0 = a.info->first_nz;
  /* this chunk's positions [qa, qe) of the work order (positions below nuniq
   * hold the segment's groups), aligned to 256 */
  const int64_t span = (nu + a.nchunk - 1) / a.nchunk;
  const int64_t spanA = (span + 255) & ~(int64_t)255;
  const int64_t qa = chunk * spanA;
  const int64_t qe = qa + spanA < nu ? qa + spanA : nu;
  const int64_t K = qe > qa ? (qe - qa + 31) >> 5 : 0; /* uniform over the workgroup */
  const int64_t row0 = sg * 16 * NB;

  Stage stg;
  /* wave 0, threads 0-31: the cell centre (ugu, vgu) of one position of the
   * k-step; wave 1: lane (b, j) the mask of position j over the workgroup's
   * 32-point block b */
  const int xj = lane & 31, xb = lane >> 5;
  const uint32_t* fv = a.fvis + (pbw * 2 + xb) * a.nfr_pad;
  double2 xr = make_double2(0.0, 0.0);
  int32_t xia = 0, xib = 0; /* frames of the step after the staged one; < 0: no group */
  uint32_t xm0 = 0, xm1 = 0;
#define VW_X_INDEX(k_)                                         \
  do {                                                         \
    if (wave == 1) {                                           \
      const int64_t j_ = qa + 32 * (k_) + xj;                  \
      const int64_t jc_ = j_ < qe ? j_ : qa;                   \
      const bool in_ = j_ < qe && a.gperm[jc_] >= q0;          \
      const int32_t ia_ = a.oia[jc_], ib_ = a.oib[jc_];        \
      xia = in_ ? ia_ : -1;                                    \
      xib = ib_;                                               \
    }                                                          \
  } while (0)
#define VW_X_LOAD(k_)                                                       \
  do {                                                                      \
    if (wave == 0) {                                                        \
      /* qa + 32 k + 32 <= nq_pad: both are multiples of 32 */              \
      if (lane < 32) xr = a.orec[qa + 32 * (k_) + lane];                    \
    } else if (wave == 1) {                                                 \
      xm0 = xm1 = xia >= 0 ? 0xffffffffu : 0u;                              \
      if (a.rep && xia >= 0) {                                              \
        xm0 = fv[xia];                                                      \
        xm1 = fv[xib];                                                      \
      }                                                                     \
    }                                                                       \
  } while (0)
#define VW_X_STORE(b_)                                        \
  do {                                                        \
    if (wave == 0) {                                          \
      if (lane < 32) grec[b_][lane] = xr;                     \
    } else if (wave == 1) {                                   \
      const uint32_t m_ = xm0 & xm1;                          \
      gm[b_][2 * xb][xj] = (uint16_t)m_;                      \
      gm[b_][2 * xb + 1][xj] = (uint16_t)(m_ >> 16);          \
    }                                                         \
  } while (0)
  vw_f32x4b acc[NB];
  double sum[NB][4];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    acc[nb] = vw_f32x4b{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i) sum[nb][i] = 0.0;
  }
  uint32_t cnt = 0;

  if (K > 0) {
    VW_X_INDEX(0);
    stg.load(a.vrh, a.vrl, a.vih, a.vil, qa >> 5, a.nsky_pad, row0);
    VW_X_LOAD(0);
    VW_X_INDEX(1);
    stg.store(bsh[0]);
    VW_X_STORE(0);
  }
  __syncthreads();
  for (int64_t k = 0; k < K; ++k) {
    const int buf = (int)(k & 1);
    const bool more = k + 1 < K;
    if (more) {
      stg.load(a.vrh, a.vrl, a.vih, a.vil, (qa >> 5) + k + 1, a.nsky_pad, row0);
      VW_X_LOAD(k + 1);
      VW_X_INDEX(k + 2);
    }
    /* masks of the lane's positions 8 g .. 8 g + 7; a k-step that no point of
     * the wave sees adds nothing, one that all see needs no masks */
    const vw_u32x4 mw = *(const vw_u32x4*)(&gm[buf][wave][g * 8]);
    const uint32_t ml = gm[buf][wave][lane & 31];
    if (wave_on && __ballot(ml != 0) != 0) {
      float cv[8], sv[8];
      if (__ballot(ml != 0xffffu) == 0) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const double2 u = grec[buf][g * 8 + i];
          const double x = vw_recon_phase(u.x, u.y, lp, mp);
          const float f = (float)__builtin_amdgcn_fract(x);
          cv[i] = __builtin_amdgcn_cosf(f);
          sv[i] = -__builtin_amdgcn_sinf(f);
        }
        cnt += 8u;
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int on = vw_bit_mask(mw[i >> 1] >> r, 16 * (i & 1));
          const double2 u = grec[buf][g * 8 + i];
          const double x = vw_recon_phase(u.x, u.y, lp, mp);
          const float f = (float)__builtin_amdgcn_fract(x);
          cv[i] = vw_and_f32(__builtin_amdgcn_cosf(f), on);
          sv[i] = vw_and_f32(-__builtin_amdgcn_sinf(f), on);
          cnt -= (uint32_t)on;
        }
      }
      vw_bf16x8 ach, acl, ash, asl;
      vw_split8(cv, ach, acl);
      vw_split8(sv, ash, asl);
      const __bf16* bb = bsh[buf];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        acc[nb] = vw_mac3(ach, acl, vw_lds_bf16x8(bb, nb * 16 + r, g),
                          vw_lds_bf16x8(bb, 16 * NB + nb * 16 + r, g), acc[nb]);
        acc[nb] = vw_mac3(ash, asl, vw_lds_bf16x8(bb, 32 * NB + nb * 16 + r, g),
                          vw_lds_bf16x8(bb, 48 * NB + nb * 16 + r, g), acc[nb]);
      }
    }
    if (wave_on && ((k & 7) == 7 || !more)) {
      /* FP64 sums across blocks of 256 groups (also after skipped steps) */
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[nb][i] += (double)acc[nb][i];
        acc[nb] = vw_f32x4b{0.f, 0.f, 0.f, 0.f};
      }
    }
    if (more) {
      stg.store(bsh[buf ^ 1]);
      VW_X_STORE(buf ^ 1);
    }
    __syncthreads();
  }
#undef VW_X_INDEX
#undef VW_X_LOAD
#undef VW_X_STORE
  if (!wave_on) return;
  /* the four lanes of a point (r, r + 16, r + 32, r + 48) hold its counts */
  cnt += (uint32_t)__shfl_xor((int)cnt, 16, 64);
  cnt += (uint32_t)__shfl_xor((int)cnt, 32, 64);
  if (sg == 0 && g == 0 && p < a.npts) a.wpart[chunk * a.pstride + p] = cnt;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int64_t sky = (sg * NB + nb) * 16 + r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t pt = pbase + 4 * g + i;
      if (pt < a.npts) a.part[(chunk * a.nsky_pad + sky) * a.pstride + pt] = sum[nb][i];
    }
  }
}

/* group-range partials -> accumulators [nsky][npts_all] (add_inplace); the
 * sky-0 threads also fold the weights */
__global__ void k_reconb_fold(const double* __restrict__ part, const uint32_t* __restrict__ wpart, int64_t nchunk,
                              int64_t nsky, int64_t nsky_pad, int64_t pstride, int64_t pt0, int64_t npts,
                              int64_t npts_all, int weights, double* __restrict__ acc, uint32_t* __restrict__ wacc) {
  int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nsky * npts) return;
  const int64_t s = k / npts, p = k - s * npts;
  double v = part[s * pstride + p];
  /* VW_FOLD_BATCH chunks' loads in flight at a time; the sum keeps chunk order */
  int64_t c = 1;
  for (; c + VW_FOLD_BATCH <= nchunk; c += VW_FOLD_BATCH) {
    double x[VW_FOLD_BATCH];
#pragma unroll
    for (int e = 0; e < VW_FOLD_BATCH; ++e) x[e] = part[((c + e) * nsky_pad + s) * pstride + p];
#pragma unroll
    for (int e = 0; e < VW_FOLD_BATCH; ++e) v = v + x[e];
  }
  for (; c < nchunk; ++c) v = v + part[(c * nsky_pad + s) * pstride + p];
  acc[s * npts_all + pt0 + p] += v;
  if (weights && s == 0) {
    uint32_t w = wpart[p];
    for (int64_t c2 = 1; c2 < nchunk; ++c2) w += wpart[c2 * pstride + p];
    wacc[pt0 + p] += w;
  }
}

/* every sky's phase-corrected half visibilities of the current segment
 * [nsky][nh] into the day buffer [nsky][day_rows] at row offset row0 */
__global__ void k_vday_store(const double2* __restrict__ vh, int64_t nsky, int64_t nh, int64_t row0, int64_t day_rows,
                             double2* __restrict__ vday) {
  int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nsky * nh) return;
  const int64_t s = k / nh, h = k - s * nh;
  vday[s * day_rows + row0 + h] = vh[k];
}

/* ------------------------------------------------------------------ */
/* stable LSD radix sort without memsets (graph-capturable)             */
/* ------------------------------------------------------------------ */
/* One pass sorts by the 8-bit digit (key >> shift) & 255 of blocks of
 * VW_RS_BLOCK elements: k_rs_hist counts each block's digits (LDS counters),
 * k_rs_scan turns the digit-major table [256][nblk] into exclusive offsets
 * within each digit plus the digit totals, k_rs_scatter places each block's
 * elements at the digit's base (the scan of the totals) plus the block's
 * offset plus the element's place among the block's equal digits, in input
 * order (stable). */
#define VW_RS_BLOCK 128
template <typename K>
__global__ __launch_bounds__(256) void k_rs_hist(const K* __restrict__ keys, int64_t n, int shift,
                                                 int32_t* __restrict__ hist, int64_t nblk) {
  __shared__ int32_t h[256];
  const int64_t b = blockIdx.x;
  h[threadIdx.x] = 0;
  __syncthreads();
  const int64_t i0 = b * VW_RS_BLOCK, i1 = i0 + VW_RS_BLOCK < n ? i0 + VW_RS_BLOCK : n;
  for (int64_t i = i0 + threadIdx.x; i < i1; i += 256) atomicAdd(&h[(int)((keys[i] >> shift) & 255)], 1);
  __syncthreads();
  hist[(int64_t)threadIdx.x * nblk + b] = h[threadIdx.x];
}
/* exclusive scan of each digit's row of the digit-major table [256][nblk]
 * in place, one workgroup per digit (a lane takes a contiguous run of the
 * row, the run totals are scanned in LDS); the digit's total goes to
 * tot[digit] */
__global__ __launch_bounds__(256) void k_rs_scan(int32_t* __restrict__ a, int64_t nblk, int32_t* __restrict__ tot) {
  __shared__ int32_t t[256];
  int32_t* row = a + (int64_t)blockIdx.x * nblk;
  const int64_t per = (nblk + 255) / 256;
  const int64_t i0 = threadIdx.x * per, i1 = i0 + per < nblk ? i0 + per : nblk;
  int32_t s = 0;
  for (int64_t i = i0; i < i1; ++i) s += row[i];
  t[threadIdx.x] = s;
  __syncthreads();
  for (int o = 1; o < 256; o <<= 1) {
    const int32_t v = threadIdx.x >= (unsigned)o ? t[threadIdx.x - o] : 0;
    __syncthreads();
    t[threadIdx.x] += v;
    __syncthreads();
  }
  int32_t run = threadIdx.x ? t[threadIdx.x - 1] : 0;
  for (int64_t i = i0; i < i1; ++i) {
    const int32_t c = row[i];
    row[i] = run;
    run += c;
  }
  if (threadIdx.x == 255) tot[blockIdx.x] = t[255];
}
/* Each of the first two waves holds 64 elements, one a lane; the lanes of equal
 * digit find each other by eight ballots, so an element's place among its
 * wave's equals is a population count and the second wave starts after the
 * first one's count.  (One lane per digit walking the block's 128 digits took
 * 13-15 us a pass.) */
template <typename K, typename V>
__global__ __launch_bounds__(256) void k_rs_scatter(const K* __restrict__ kin, const V* __restrict__ vin, int64_t n,
                                                    int shift, const int32_t* __restrict__ offs, int64_t nblk,
                                                    const int32_t* __restrict__ tot, K* __restrict__ kout,
                                                    V* __restrict__ vout) {
  static_assert(VW_RS_BLOCK == 128, "two waves of elements");
  __shared__ int32_t pos0[256]; /* where the block's elements of a digit start   */
  __shared__ int32_t cnt0[256]; /* elements of a digit in the block's first wave */
  __shared__ int32_t wsum[4];
  const int64_t b = blockIdx.x;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int64_t i = b * VW_RS_BLOCK + t;
  const bool mine = t < VW_RS_BLOCK && i < n;
  K key = 0;
  V val = 0;
  if (mine) { key = kin[i]; val = vin[i]; }
  const int32_t off = offs[(int64_t)t * nblk + b]; /* digit t's elements in earlier blocks */
  /* digit bases: exclusive scan of the digit totals, one digit a thread */
  const int32_t tt = tot[t];
  int32_t inc = tt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int32_t v = __shfl_up(inc, o, 64);
    if (lane >= o) inc += v;
  }
  if (lane == 63) wsum[wave] = inc;
  cnt0[t] = 0;
  __syncthreads();
  int32_t before = 0;
#pragma unroll
  for (int wv = 0; wv < 3; ++wv) before += wv < wave ? wsum[wv] : 0;
  pos0[t] = before + inc - tt + off;
  /* the lanes with this lane's digit (lanes without an element: none) */
  const int d = (int)((key >> shift) & 255);
  uint64_t same = __ballot(mine);
#pragma unroll
  for (int bit = 0; bit < 8; ++bit) {
    const uint64_t m = __ballot((d >> bit) & 1);
    same &= ((d >> bit) & 1) ? m : ~m;
  }
  const uint64_t lower = same & ((1ull << lane) - 1);
  if (wave == 0 && mine && lower == 0) cnt0[d] = __popcll(same);
  __syncthreads();
  if (mine) {
    const int32_t p = pos0[d] + (wave == 1 ? cnt0[d] : 0) + __popcll(lower);
    kout[p] = key;
    vout[p] = val;
  }
}

#endif
