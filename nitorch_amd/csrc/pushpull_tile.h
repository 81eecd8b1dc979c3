// LDS-tiled push / count for 3-D float fields (isotropic order ORD), and the
// dispatch of every mode over the tiles, gathers and bins.
//
// One work-group owns a TX x TY x TZ tile of samples (grid points); each
// thread owns R of them.  The work-group reduces the bounding box of the
// first taps of its in-bound samples, and when the box (extended by the
// ORD + 1 taps) fits in LDS, it accumulates the tile's splats into an LDS
// box of FP64 values with FP64 LDS atomics (gfx950 runs ds_add_f64 at ~80%
// of the rate of its 64-bit integer atomics, and ~40x faster than
// ds_add_f32), then adds the box to the output once, folded and signed, with
// one FP32 global atomic per non-zero box element.  At orders >= 1 a
// thread's z-consecutive samples whose taps are z-consecutive too first sum
// their splats along z in registers (at most R = 4 or 2 FP32 terms a box
// element) and add one FP64 atomic a position.  Every box element is a
// double sum of its splats (FP64 products at order 0; above, FP32 sums of at
// most R FP32 products), so each output element keeps float's relative
// accuracy against the sum of its splats' magnitudes however small it is
// next to the tile's other values, and NaN / Inf values propagate as in the
// reference's float sums.
// The box has fixed dimensions per order (every tap offset is then an
// immediate of the LDS instruction); channels are accumulated one at a time.
// A tile whose box does not fit is listed for a second pass: in calls of at
// least BIN_MIN_SAMPLES samples scatter_kernel (pushpull_scatter.h) takes those
// that fit one or two larger boxes, and the others' samples are sorted by
// first-tap bin, every bin with a box of its own (pushpull_bin.h); in smaller
// calls, and in the entry point that allocates nothing, tile_dyn cuts each
// listed tile into sub-tiles with boxes sized to their own spread and runs the
// direct per-sample routine pp_sample for a sub-tile that still does not fit.
// Every sample is handled exactly once; the result never depends on the
// route, only the speed does.
//
// Weights, the out-of-bound rule and the splat order of each sample are
// those of pp_sample (nitorch/_C/src/impl/pushpull_common.cpp: OOB :926-974,
// splat3d :1235-1290, linear :1653-1858, nearest :2314-2341); folding and
// signs follow bounds_common.h:28-219.
#pragma once
#include <algorithm>
#include <climits>
#include <type_traits>

#include "pushpull_impl.h"

namespace ni_amd {

#define TL_SLACK 2     // extra box extent per axis for the spread of a tile's coordinates
#define BIN_MIN_SAMPLES (int64_t(1) << 20)   // smallest call whose listed tiles take the binned pass
// Tiles whose bounding box holds at most ST_MAX_VOL elements (one or two boxes
// of scatter_kernel) go to it, unless more than 1 / ST_FAR as many tiles are
// wider: then all are binned -- a bin costs the same with few samples in it.
// 181 x 217 x 181, order 3, one channel, all binned against this rule: rotation
// by 15 degrees and zoom 1.1 543 and 342 us; smooth warps of 2 / 4 / 6 / 8
// voxels RMS 688 / 716 / 716 / 721 and 461 / 624 / 701 / 713.  Order 1, 8
// channels: 963 and 876; 1111 / 1230 / 1263 / 1261 and 974 / 1140 / 1262 / 1256.
// No call measured at orders 1 to 7 with 1 to 8 channels on these grids is
// slower by more than 1 %; the one shape that is (2000 x 30 x 30 under a noise
// of 0.3 voxels, order 3, 8 channels: 896 and 1034) leaves most work-groups
// with one tile.
#define ST_MAX_VOL 14000
#define ST_FAR 8

// Tile and box geometry of the scatter of order ORD, fixed at compile time.
//  * Up to order 5: 512 threads, 8 x 16 x 16 tiles, four z-consecutive samples
//    per thread -- every box element is one global atomic in the flush and a
//    box exceeds its tile by the ORD + 1 taps plus TL_SLACK voxels per axis,
//    so the atomics per sample fall with the tile size, and the register
//    window of the splat spans four samples.  Above order 5 (the window's
//    weights of four samples would not fit the registers, a box of 94 KB one
//    CU's LDS twice): 256 threads, 4 x 8 x 16, two samples per thread.
//  * Lanes: ZL = TZ / R threads per z-row, then R y-rows, then x-rows.
//  * The box is [x][y][z] with x stride DYZ padded to 48 (mod 64) words and
//    DZ = 1 (mod R): neighbouring lanes adding one tap fall on distinct LDS
//    banks (R y-rows in the R residue classes mod R, lanes R banks apart in a
//    row).
template <int ORD>
struct TileBox {
  static constexpr bool BIG = ORD <= 5;                // the 512-thread scatter
  static constexpr int NTH = BIG ? 512 : 256;          // threads per work-group
  static constexpr int NW = NTH / 64;                  // waves
  static constexpr int R = BIG ? 4 : 2;                // samples per thread
  static constexpr int TX = BIG ? 8 : 4;
  static constexpr int TY = BIG ? 16 : 8;
  static constexpr int TZ = 16;
  static constexpr int ZL = TZ / R;                    // threads per z-row of the tile
  static constexpr int RY = R;                         // y-rows per wave
  static constexpr int RX = 64 / ZL / RY;              // x-rows per wave
  static constexpr int WX = TX / RX;                   // waves along x
  static constexpr int DX = TX + ORD + TL_SLACK;
  static constexpr int DY = TY + ORD + TL_SLACK;
  static constexpr int DZ0 = TZ + ORD + TL_SLACK;
  static constexpr int DZ = DZ0 + ((1 - DZ0) % R + R) % R;
  static constexpr int DYZ0 = DY * DZ;
  static constexpr int DYZ = DYZ0 + ((48 - DYZ0) % 64 + 64) % 64;
  static constexpr int VOL = DX * DYZ;
  static constexpr int NPP = (DYZ0 + NTH - 1) / NTH;   // y-z plane positions per thread
  // waves per SIMD asked of the register allocator for the 512-thread
  // scatter: the window (orders 1-5) holds its samples' weights and needs 97
  // (order 3) to 128 (order 5) VGPRs, two work-groups a CU
  static constexpr int MINW = BIG ? (ORD >= 1 ? 4 : 6) : 1;
  static_assert(TX * TY * TZ == NTH * R, "R samples per thread");
  static_assert(WX * RX == TX && (NW / WX) * RY == TY, "waves tile the rows");
};

// First sample of this thread within its tile (sample i adds i to z).
template <class B>
__device__ __forceinline__ void tl_thread(int &sx, int &sy, int &sz0) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, row = lane / B::ZL;
  sx = row / B::RY + B::RX * (w % B::WX);
  sy = row % B::RY + B::RY * (w / B::WX);
  sz0 = (lane % B::ZL) * B::R;
}

// The y-z plane of a box's ext[1] x ext[2] corner, split over the threads:
// position j of a thread is (by, bz), with folded source offset and sign
// from the axis tables and the LDS offset by * DZ + bz.
template <class B>
struct TilePlane {
  int yz_ofs[B::NPP];   // folded y + z offset in the tensor, elements
  int yz_lds[B::NPP];   // by * DZ + bz, or -1 when the position is outside the plane
  float yz_sg[B::NPP];  // product of the y and z signs
  __device__ __forceinline__ void init(int E1, int E2, const int *fofs, const float *fsg) {
    const float r2 = 1.f / (float)E2;
#pragma unroll
    for (int j = 0; j < B::NPP; ++j) {
      const int p = threadIdx.x + j * B::NTH;
      int by = (int)((float)p * r2);   // floor(p / E2): exact after the fix-ups (p < 2^22)
      by -= by * E2 > p;
      by += (by + 1) * E2 <= p;
      const int bz = p - by * E2;
      const bool in = by < E1;
      yz_lds[j] = in ? by * B::DZ + bz : -1;
      yz_ofs[j] = in ? fofs[B::DX + by] + fofs[B::DX + B::DY + bz] : 0;
      yz_sg[j] = in ? fsg[B::DX + by] * fsg[B::DX + B::DY + bz] : 0.f;
    }
  }
};

// Gather modes stage the source box; scatter modes accumulate one.
//   TM_PULL  : out[c]      = sum_t w(t) src(t, c)                   (F_PULL)
//   TM_SGRAD : out[c][d]   = sum_t dw_d(t) src(t, c)                (F_SGRAD)
//   TM_GGRAD : gout[d]     = sum_t dw_d(t) sum_c src(t, c) trgt(c)  (F_GRAD | F_TRGT,
//              or F_GRAD with a single channel and no target: trgt = 1)
//   TM_PUSH  : out(t, c)  += w(t) trgt(c)                           (F_PUSH | F_TRGT)
//   TM_COUNT : out(t)     += w(t)                                   (F_COUNT)
enum TileMode { TM_PULL = 0, TM_PUSH = 1, TM_COUNT = 2, TM_SGRAD = 3, TM_GGRAD = 4, TM_GGRAD1 = 5 };

template <int MODE>
struct TileMeta {
  static constexpr bool gather = MODE == TM_PULL || MODE == TM_SGRAD || MODE == TM_GGRAD || MODE == TM_GGRAD1;
  static constexpr bool deriv = MODE == TM_SGRAD || MODE == TM_GGRAD || MODE == TM_GGRAD1;
};

// Samples of a tile (work-group): 4 x 8 x 16 for the gathers (larger tiles
// re-read less halo but cost occupancy), TileBox's for the scatters.
template <int ORD, int MODE>
struct TileDims {
  static constexpr int TX = TileMeta<MODE>::gather ? 4 : TileBox<ORD>::TX;
  static constexpr int TY = TileMeta<MODE>::gather ? 8 : TileBox<ORD>::TY;
  static constexpr int TZ = 16;
};

// Spline weight / derivative of tap T at signed distance d: the
// evaluation of spl_w / spl_g (common.h), with the piece and its Horner
// coefficients fixed at compile time (immediates, never table loads).
template <int O, int P, int I>
__device__ __forceinline__ float tl_horner_w(float u) {
  constexpr float c = (float)SplTab<O>::W[P][I];
  if constexpr (I == SplTab<O>::NDW - 1) return c;
  else return tl_horner_w<O, P, I + 1>(u) * u + c;
}
template <int O, int P, int I>
__device__ __forceinline__ float tl_horner_g(float u) {
  constexpr float c = (float)SplTab<O>::G[P][I];
  if constexpr (I == SplTab<O>::NDG - 1) return c;
  else return tl_horner_g<O, P, I + 1>(u) * u + c;
}
template <int ORD, bool DERIV, int T>
__device__ __forceinline__ void tl_weight(float x, int lo, float (&w)[ORD + 1], float (&g)[ORD + 1]) {
  if constexpr (T <= ORD) {
    if constexpr (T == 0 || T == ORD) {   // last piece, from x itself (spl_outer_s)
      float h;
      spl_outer<float, ORD>(T == 0, spl_outer_s<float, int>(ORD, T, x, lo), w[T], g[T], h);
    } else {
      constexpr int P = tap_piece<ORD>(T);
      constexpr float centre = (float)piece_centre<ORD>(P);
      const float d = x - (float)(lo + T);
      const float a = d < 0.f ? -d : d;
      w[T] = tl_horner_w<ORD, P, 0>(a - centre);
      if constexpr (DERIV) {
        const float gg = tl_horner_g<ORD, P, 0>(a - centre);
        g[T] = d < 0.f ? -gg : gg;
      }
    }
    tl_weight<ORD, DERIV, T + 1>(x, lo, w, g);
  }
}

// First tap index and the ORD + 1 weights (and, when DERIV, first
// derivatives) of coordinate x, as pp_sample computes them.
template <int ORD, bool DERIV = false>
__device__ __forceinline__ int tl_taps(float x, float (&w)[ORD + 1], float (&g)[ORD + 1]) {
  if constexpr (ORD == 0) {
    w[0] = 1.f;
    g[0] = 0.f;
    return (int)roundf(x);
  } else if constexpr (ORD == 1) {
    // weights as distances to the far tap: exact when small
    const int j0 = (int)floorf(x);
    w[0] = (float)(j0 + 1) - x;
    w[1] = x - (float)j0;
    g[0] = -1.f;
    g[1] = 1.f;
    return j0;
  } else {
    const int lo = (int)floorf(x - first_tap_offset<float>(ORD));
    tl_weight<ORD, DERIV, 0>(x, lo, w, g);
    return lo;
  }
}

// First tap index of coordinate x (as tl_taps).
template <int ORD>
__device__ __forceinline__ int tl_first(float x) {
  if constexpr (ORD == 0) return (int)roundf(x);
  else if constexpr (ORD == 1) return (int)floorf(x);
  else return (int)floorf(x - first_tap_offset<float>(ORD));
}

__device__ __forceinline__ int wave_min(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ int wave_max(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
  return v;
}

// p / d for 0 <= p, d < 2^22 from the float reciprocal rinv = 1 / d: the
// float quotient is within 1 of the exact one, one correction each way
// (a runtime integer division costs ~30 VALU operations)
__device__ __forceinline__ int tl_div(int p, int d, float rinv) {
  int q = (int)((float)p * rinv);
  q -= q * d > p;
  q += (q + 1) * d <= p;
  return q;
}

// Rotate a small register array left by one: a rolled tap loop reads
// element 0 and rotates, so that no array is indexed by the loop counter
// (which would put it in scratch memory); NT rotations restore the order.
template <typename T, int N>
__device__ __forceinline__ void tl_rot(T (&v)[N]) {
  const T t = v[0];
#pragma unroll
  for (int j = 0; j + 1 < N; ++j) v[j] = v[j + 1];
  v[N - 1] = t;
}

// Hide a register array's values from the optimiser for one loop
// iteration, so that products of it are not hoisted out of the loop (where
// they would all be live at once).
template <int N>
__device__ __forceinline__ void tl_opaque(float (&v)[N]) {
#pragma unroll
  for (int j = 0; j < N; ++j) asm volatile("" : "+v"(v[j]));
}

template <int MODE>
struct TileFlags {
  static constexpr int value = MODE == TM_PULL ? F_PULL : MODE == TM_PUSH ? (F_PUSH | F_TRGT)
                               : MODE == TM_COUNT ? F_COUNT : MODE == TM_SGRAD ? F_SGRAD
                               : MODE == TM_GGRAD ? (F_GRAD | F_TRGT) : F_GRAD;
};

// Tiles whose box fits the static one; the others are listed: in mid, when
// given (two counts, then tile ids), those that scatter_kernel can take in few
// boxes, else in fb (a count, then tile ids).
template <int ORD, int MODE>
__global__ __launch_bounds__((TileBox<ORD>::NTH),
                             (TileBox<ORD>::MINW)) void tile_kernel(PPArgs<float> a, int ntx, int nty, int ntz,
                                                                    int64_t nblocks, int *fb, int *mid) {
  constexpr int NT = ORD + 1;
  using B = TileBox<ORD>;
  constexpr int R = B::R, NTH = B::NTH;
  constexpr int DY = B::DY, DZ = B::DZ, DYZ = B::DYZ, VOL = B::VOL;
  __shared__ __align__(16) double box[VOL];
  __shared__ int red[B::NW][6];

  const int64_t tile = xcd_block(nblocks);
  int64_t r = tile;
  const int tz = (int)(r % ntz); r /= ntz;
  const int ty = (int)(r % nty); r /= nty;
  const int tx = (int)(r % ntx);
  const int n = (int)(r / ntx);
  const int X = (int)a.tX, Y = (int)a.tY, Z = (int)a.tZ;
  const int sz[3] = {(int)a.sX, (int)a.sY, (int)a.sZ};

  // ---- samples of this thread: in-bound flags, taps ----
  // sample i is (px, py, pz0 + i)
  int sx, sy, sz0;
  tl_thread<B>(sx, sy, sz0);
  const int px = tx * B::TX + sx, py = ty * B::TY + sy, pz0 = tz * B::TZ + sz0;
  bool valid[R], inb[R];
  // orders >= 1 keep every sample's weights
  constexpr bool WIN = ORD >= 1;
  constexpr int NW = WIN ? R : 1;
  int lo[R][3];
  float w[NW][3][NT];
  if constexpr (WIN) {   // the window multiplies the weights of samples outside a group by 0: keep them finite
#pragma unroll
    for (int i = 0; i < NW; ++i)
#pragma unroll
      for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int t = 0; t < NT; ++t) w[i][d][t] = 0.f;
  }
  int mn[3] = {INT_MAX, INT_MAX, INT_MAX}, mx[3] = {INT_MIN, INT_MIN, INT_MIN};
  const float tol = (a.extrap & 2) ? 0.55f : 0.05f;
  const int gD = (int)a.grid_s[4];
  const int gS = (int)a.grid_s[3];
  const float *gp0 = a.grid + (int)(n * a.grid_s[0] + px * a.grid_s[1] + py * a.grid_s[2] + pz0 * a.grid_s[3]);
#pragma unroll
  for (int i = 0; i < R; ++i) {
    valid[i] = px < X && py < Y && pz0 + i < Z;
    inb[i] = false;
    if (valid[i]) {
      const float *gp = gp0 + i * gS;
      const float xs[3] = {gp[0], gp[gD], gp[2 * gD]};
      bool ok = true;
      if (!(a.extrap & 1))
#pragma unroll
        for (int d = 0; d < 3; ++d) ok = ok && (xs[d] >= -tol && xs[d] < (float)(sz[d] - 1) + tol);
      inb[i] = ok;
      if (ok) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          float wtmp[NT], gtmp[NT];
          lo[i][d] = tl_taps<ORD>(xs[d], wtmp, gtmp);
          if constexpr (NW == R) {
#pragma unroll
            for (int t = 0; t < NT; ++t) w[i][d][t] = wtmp[t];
          }
          mn[d] = min(mn[d], lo[i][d]);
          mx[d] = max(mx[d], lo[i][d]);
        }
      }
    }
  }

  // ---- bounding box of the work-group's first taps ----
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    mn[d] = wave_min(mn[d]);
    mx[d] = wave_max(mx[d]);
  }
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      red[threadIdx.x >> 6][d] = mn[d];
      red[threadIdx.x >> 6][3 + d] = mx[d];
    }
  }
  __syncthreads();
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    mn[d] = red[0][d];
    mx[d] = red[0][3 + d];
#pragma unroll
    for (int wv = 1; wv < B::NW; ++wv) {
      mn[d] = min(mn[d], red[wv][d]);
      mx[d] = max(mx[d], red[wv][3 + d]);
    }
  }

  const int oC = (int)a.out_s[1];
  if (mn[0] > mx[0]) return;   // no in-bound sample in this tile
  int ext[3];
  bool fits = true;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const int64_t e = (int64_t)mx[d] - (int64_t)mn[d] + NT;
    fits = fits && e <= (d == 0 ? B::DX : d == 1 ? DY : DZ);
    ext[d] = (int)(e < 0x7fffffff ? e : 0x7fffffff);
  }
  if (!fits) {   // scattered tile
    if (threadIdx.x == 0) {
      if (mid && (double)ext[0] * (double)ext[1] * (double)ext[2] <= (double)ST_MAX_VOL) {
        mid[2 + atomicAdd(mid, 1)] = (int)tile;
      } else if (fb) {
        fb[1 + atomicAdd(fb, 1)] = (int)tile;
        if (mid) atomicAdd(mid + 1, 1);
      }
    }
    return;
  }
  int off[R];
#pragma unroll
  for (int i = 0; i < R; ++i)
    off[i] = inb[i] ? (lo[i][0] - mn[0]) * DYZ + (lo[i][1] - mn[1]) * DZ + (lo[i][2] - mn[2]) : 0;

  const int C = MODE == TM_COUNT ? 1 : (int)a.C;

  // folded offsets (in elements of the staged / scattered tensor) and signs
  // of the box positions along each axis: fold() runs once per position
  constexpr int NF = B::DX + DY + DZ;
  __shared__ int fofs[NF];
  __shared__ float fsg[NF];
  {
    const int64_t *st = a.out_s;
    const int st0 = (int)st[2], st1 = (int)st[3], st2 = (int)st[4];
    for (int i = threadIdx.x; i < NF; i += NTH) {
      const int d = i < B::DX ? 0 : i < B::DX + DY ? 1 : 2;
      const int b = i - (d == 0 ? 0 : d == 1 ? B::DX : B::DX + DY);
      const int e = d == 0 ? ext[0] : d == 1 ? ext[1] : ext[2];
      const int m = d == 0 ? mn[0] : d == 1 ? mn[1] : mn[2];
      const int nn = d == 0 ? sz[0] : d == 1 ? sz[1] : sz[2];
      const int bd = d == 0 ? a.bound[0] : d == 1 ? a.bound[1] : a.bound[2];
      int sg = 0, j = 0;
      if (b < e) j = fold<int>(bd, tap_at(m, b), nn, sg);
      fofs[i] = j * (d == 0 ? st0 : d == 1 ? st1 : st2);
      fsg[i] = (float)sg;
    }
  }
  __syncthreads();
  TilePlane<B> pl;
  pl.init(ext[1], ext[2], fofs, fsg);
  // cleared once; each flush clears what it read
  for (int i = threadIdx.x; i < VOL; i += NTH) box[i] = 0.0;
  __syncthreads();

  for (int c = 0; c < C; ++c) {
    if (c) __syncthreads();   // previous channel fully consumed
    // keep the per-tap weight products inside the channel loop (hoisting
    // them would hold (ORD + 1)^3 products per sample in registers)
#pragma unroll
    for (int i = 0; i < NW; ++i)
#pragma unroll
      for (int d = 0; d < 3; ++d) tl_opaque(w[i][d]);
    float tv[R];
    const float *tp0 = MODE == TM_PUSH ? a.trgt + (int)(n * a.trgt_s[0] + (int64_t)c * a.trgt_s[1] + px * a.trgt_s[2] +
                                                        py * a.trgt_s[3] + pz0 * a.trgt_s[4])
                                       : nullptr;
#pragma unroll
    for (int i = 0; i < R; ++i) tv[i] = !inb[i] ? 0.f : (MODE == TM_PUSH ? tp0[i * (int)a.trgt_s[4]] : 1.f);
    __syncthreads();
    if constexpr (WIN) {
      // push / count, orders >= 1: a thread's R z-consecutive samples whose
      // first taps share x and y and advance by one along z with the sample
      // share a window of R + NT - 1 z positions per (x, y) tap row.  Their
      // splats are summed in registers (FP32, at most R terms a position:
      // sample i reaches positions i .. i + NT - 1 of the window) and each
      // position is added to the box by one FP64 atomic: R + NT - 1 atomics
      // a row instead of R * NT.  Sample i's taps start at box element
      // off[i], so samples with equal off[i] - i are exactly those one
      // window at base off[i] - i serves.  A thread's samples split into
      // such groups (anchored at its first sample left); the lanes of a wave
      // loop until every group is done, so any grid is handled, a smooth
      // one in one pass.  A non-finite value reaches only its own taps.
      constexpr int WS = R + NT - 1;
      unsigned rem = 0;
#pragma unroll
      for (int i = 0; i < R; ++i) rem |= inb[i] ? 1u << i : 0u;
      while (rem) {
        const int an = __builtin_ctz(rem);
        int base = off[0];
#pragma unroll
        for (int i = 1; i < R; ++i)
          if (an == i) base = off[i] - i;
        unsigned gm = 0;
#pragma unroll
        for (int i = 0; i < R; ++i)
          if (((rem >> i) & 1u) && off[i] - i == base) gm |= 1u << i;
        rem &= ~gm;
        const int hi = 31 - __builtin_clz(gm) + NT - 1;   // last window position reached
        // window position s is box element base + s (an <= s <= hi)
        double *bp = box + base;
#pragma unroll 1
        for (int kx = 0; kx < NT; ++kx, bp += DYZ) {
          float xv[R];
#pragma unroll
          for (int i = 0; i < R; ++i) xv[i] = ((gm >> i) & 1u) ? w[i][0][0] * tv[i] : 0.f;
#pragma unroll
          for (int ky = 0; ky < NT; ++ky) {
            float acc[WS];
#pragma unroll
            for (int s = 0; s < WS; ++s) acc[s] = 0.f;
#pragma unroll
            for (int i = 0; i < R; ++i) {
              const float cw = xv[i] * w[i][1][ky];
#pragma unroll
              for (int kz = 0; kz < NT; ++kz) acc[i + kz] = fmaf(cw, w[i][2][kz], acc[i + kz]);
            }
#pragma unroll
            for (int s = 0; s < WS; ++s)
              if (s >= an && s <= hi) atomicAdd(bp + ky * DZ + s, (double)acc[s]);
          }
#pragma unroll
          for (int i = 0; i < R; ++i) tl_rot(w[i][0]);
        }
      }
    } else {
      // order 0: one tap a sample
#pragma unroll
      for (int i = 0; i < R; ++i)
        if (inb[i]) atomicAdd(box + off[i], (double)tv[i]);
    }
    // ---- add the box to the output, folded and signed; clear it for
    // the next channel (the splats never leave the ext corner) ----
    __syncthreads();
    float *out = a.out + (int)(n * a.out_s[0] + (int64_t)c * oC);
    const int e0 = ext[0] - 1;
#pragma unroll
    for (int j = 0; j < B::NPP; ++j) {
      if (pl.yz_lds[j] < 0) continue;
      // a whole x row of the box read (and cleared) at once, then its
      // atomics issued back to back
      double *bq = box + pl.yz_lds[j];
      float fv[B::DX];   // the row, rounded to float (0 where the box is empty)
#pragma unroll
      for (int bx = 0; bx < B::DX; ++bx) fv[bx] = (float)bq[bx * DYZ];
#pragma unroll
      for (int bx = 0; bx < B::DX; ++bx) bq[bx * DYZ] = 0.0;
      float *op = out + pl.yz_ofs[j];
#pragma unroll
      for (int bx = 0; bx < B::DX; ++bx) {
        const float sg = fsg[bx] * pl.yz_sg[j];
        if (bx <= e0 && fv[bx] != 0.f && sg != 0.f) atomic_add(op + fofs[bx], fv[bx] * sg);
        if ((bx & 3) == 3) __builtin_amdgcn_sched_barrier(0);   // bound the addresses held at once
      }
    }
  }
}

// Tiles whose box does not fit, by the direct per-sample routine, where no list
// can be had: every tile repeats tile_kernel's bounding-box test (bit-identical,
// so every tile is handled by exactly one of the two kernels).  Kept apart from
// tile_kernel so that its register demand does not lower that kernel's
// occupancy.
template <int ORD, int MODE>
__global__ __launch_bounds__((TileBox<ORD>::NTH)) void tile_fallback(PPArgs<float> a, int ntx, int nty, int ntz,
                                                                     int64_t nblocks) {
  constexpr int NT = ORD + 1;
  constexpr int FL = TileFlags<MODE>::value;
  using B = TileBox<ORD>;
  constexpr int R = B::R;
  const int X = (int)a.tX, Y = (int)a.tY, Z = (int)a.tZ;
  int sx, sy, sz0;
  tl_thread<B>(sx, sy, sz0);
  __shared__ int red[B::NW][6];
  int64_t r = xcd_block(nblocks);
  const int tz = (int)(r % ntz); r /= ntz;
  const int ty = (int)(r % nty); r /= nty;
  const int tx = (int)(r % ntx);
  const int n = (int)(r / ntx);
  const int sz[3] = {(int)a.sX, (int)a.sY, (int)a.sZ};
  const int px = tx * B::TX + sx, py = ty * B::TY + sy, pz0 = tz * B::TZ + sz0;
  bool valid[R], inb[R];
  int mn[3] = {INT_MAX, INT_MAX, INT_MAX}, mx[3] = {INT_MIN, INT_MIN, INT_MIN};
  const float tol = (a.extrap & 2) ? 0.55f : 0.05f;
  const int gD = (int)a.grid_s[4];
  const int gS = (int)a.grid_s[3];
  const float *gp0 = a.grid + (int)(n * a.grid_s[0] + px * a.grid_s[1] + py * a.grid_s[2] + pz0 * a.grid_s[3]);
#pragma unroll
  for (int i = 0; i < R; ++i) {
    valid[i] = px < X && py < Y && pz0 + i < Z;
    inb[i] = false;
    if (valid[i]) {
      const float *gp = gp0 + i * gS;
      const float xs[3] = {gp[0], gp[gD], gp[2 * gD]};
      bool ok = true;
      if (!(a.extrap & 1))
#pragma unroll
        for (int d = 0; d < 3; ++d) ok = ok && (xs[d] >= -tol && xs[d] < (float)(sz[d] - 1) + tol);
      inb[i] = ok;
      if (ok) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          float wd[NT], gd[NT];
          const int l = tl_taps<ORD>(xs[d], wd, gd);
          mn[d] = min(mn[d], l);
          mx[d] = max(mx[d], l);
        }
      }
    }
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    mn[d] = wave_min(mn[d]);
    mx[d] = wave_max(mx[d]);
  }
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      red[threadIdx.x >> 6][d] = mn[d];
      red[threadIdx.x >> 6][3 + d] = mx[d];
    }
  }
  __syncthreads();
  bool fits = true;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    int m0 = red[0][d], m1 = red[0][3 + d];
#pragma unroll
    for (int wv = 1; wv < B::NW; ++wv) {
      m0 = min(m0, red[wv][d]);
      m1 = max(m1, red[wv][3 + d]);
    }
    if (m0 > m1) return;   // no in-bound sample: handled by tile_kernel
    const int64_t e = (int64_t)m1 - (int64_t)m0 + NT;
    fits = fits && e <= (d == 0 ? B::DX : d == 1 ? B::DY : B::DZ);
  }
  if (fits) return;
#pragma unroll 1
  for (int i = 0; i < R; ++i)
    if (valid[i]) pp_sample<float, int32_t, ORD, FL, true>(a, n, px, py, pz0 + i);
}

// Tiles that tile_kernel listed (taps too spread for the static box): each
// listed tile is cut into sub-tiles of
// 4 x 8 x 8 samples (one per thread of a 256-thread work-group), and each
// sub-tile accumulates an LDS box sized from its own first-tap
// spread (runtime strides, up to DYN_MAXE elements per channel).  Strongly
// deformed grids (large rotations, zooms, displacements with a large
// Jacobian) keep most of the tile path's reuse this way: a sub-tile's box is
// a few times its sample count instead of the per-sample kernel's 64 taps
// x channels of scattered global traffic.  A sub-tile whose box is still
// too large runs the per-sample routine.  Same weights, out-of-bound rule,
// FP64 accumulation as tile_kernel.
#define DYN_TX 4
#define DYN_TY 8
#define DYN_TZ 8
#define DYN_NTH 256
#define DYN_MAXE 8192        // box elements (64 KB of doubles)
#define DYN_MAXAX 128        // box extent per axis

template <int ORD, int MODE>
__global__ __launch_bounds__(DYN_NTH) void tile_dyn(PPArgs<float> a, int ntx, int nty, int ntz, const int *fb) {
  constexpr int NT = ORD + 1;
  constexpr int FL = TileFlags<MODE>::value;
  using B = TileBox<ORD>;
  constexpr int NW = DYN_NTH / 64;
  static_assert(DYN_TX * DYN_TY * DYN_TZ == DYN_NTH, "one sample per thread");
  static_assert(B::TX % DYN_TX == 0 && B::TY % DYN_TY == 0 && B::TZ % DYN_TZ == 0, "sub-tiles tile the tile");
  constexpr int NSX = B::TX / DYN_TX, NSY = B::TY / DYN_TY, NSZ = B::TZ / DYN_TZ;
  __shared__ double box[DYN_MAXE];
  __shared__ int fofs[3 * DYN_MAXAX];
  __shared__ float fsg[3 * DYN_MAXAX];
  __shared__ int red[NW][6];

  const int X = (int)a.tX, Y = (int)a.tY, Z = (int)a.tZ;
  const int sz[3] = {(int)a.sX, (int)a.sY, (int)a.sZ};
  const float tol = (a.extrap & 2) ? 0.55f : 0.05f;
  const int lx = threadIdx.x / (DYN_TY * DYN_TZ), ly = (threadIdx.x / DYN_TZ) % DYN_TY, lz = threadIdx.x % DYN_TZ;
  const int cnt = fb[0];
  for (int64_t j = blockIdx.x; j < (int64_t)cnt * NSX * NSY * NSZ; j += gridDim.x) {
    const int sub = (int)(j % (NSX * NSY * NSZ));
    int64_t r = fb[1 + j / (NSX * NSY * NSZ)];
    const int tz = (int)(r % ntz); r /= ntz;
    const int ty = (int)(r % nty); r /= nty;
    const int tx = (int)(r % ntx);
    const int n = (int)(r / ntx);
    const int px = tx * B::TX + (sub / (NSY * NSZ)) * DYN_TX + lx;
    const int py = ty * B::TY + ((sub / NSZ) % NSY) * DYN_TY + ly;
    const int pz = tz * B::TZ + (sub % NSZ) * DYN_TZ + lz;
    const bool valid = px < X && py < Y && pz < Z;
    bool inb = false;
    float xq[3] = {0.f, 0.f, 0.f};
    int lo[3] = {0, 0, 0};
    int mn[3] = {INT_MAX, INT_MAX, INT_MAX}, mx[3] = {INT_MIN, INT_MIN, INT_MIN};
    if (valid) {
      const float *gp = a.grid + (int64_t)n * a.grid_s[0] + (int64_t)px * a.grid_s[1] + (int64_t)py * a.grid_s[2] +
                        (int64_t)pz * a.grid_s[3];
      const int gD = (int)a.grid_s[4];
      xq[0] = gp[0]; xq[1] = gp[gD]; xq[2] = gp[2 * gD];
      bool ok = true;
      if (!(a.extrap & 1))
#pragma unroll
        for (int d = 0; d < 3; ++d) ok = ok && (xq[d] >= -tol && xq[d] < (float)(sz[d] - 1) + tol);
      inb = ok;
      if (ok) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          float wt[NT], gt[NT];
          lo[d] = tl_taps<ORD>(xq[d], wt, gt);
          mn[d] = lo[d];
          mx[d] = lo[d];
        }
      }
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      mn[d] = wave_min(mn[d]);
      mx[d] = wave_max(mx[d]);
    }
    __syncthreads();   // previous sub-tile done with red / box / tables
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        red[threadIdx.x >> 6][d] = mn[d];
        red[threadIdx.x >> 6][3 + d] = mx[d];
      }
    }
    __syncthreads();
    int ext[3];
    bool none = false, fits = true;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      int m0 = red[0][d], m1 = red[0][3 + d];
#pragma unroll
      for (int wv = 1; wv < NW; ++wv) {
        m0 = min(m0, red[wv][d]);
        m1 = max(m1, red[wv][3 + d]);
      }
      mn[d] = m0;
      none = none || m0 > m1;
      const int64_t e = (int64_t)m1 - (int64_t)m0 + NT;
      fits = fits && e <= DYN_MAXAX;
      ext[d] = fits && !none ? (int)e : 1;
    }
    if (none) continue;   // no in-bound sample
    const int DZ = ext[2], DYZ = ext[1] * ext[2];
    fits = fits && (int64_t)ext[0] * DYZ <= DYN_MAXE;
    if (!fits) {   // per-sample routine for this sub-tile
      if (valid) pp_sample<float, int32_t, ORD, FL, true>(a, n, px, py, pz);
      continue;
    }
    const int VOL = ext[0] * DYZ;
    const float rz = 1.f / (float)DZ, ry = 1.f / (float)ext[1];
    // folded offsets and signs of the box positions along each axis
    {
      const int64_t *st = a.out_s;
      for (int i = threadIdx.x; i < ext[0] + ext[1] + ext[2]; i += DYN_NTH) {
        const int d = i < ext[0] ? 0 : (i < ext[0] + ext[1] ? 1 : 2);
        const int b = i - (d == 0 ? 0 : (d == 1 ? ext[0] : ext[0] + ext[1]));
        int sg = 0;
        const int jj = fold<int>(a.bound[d], tap_at(mn[d], b), sz[d], sg);
        fofs[i] = jj * (int)st[2 + d];
        fsg[i] = (float)sg;
      }
    }
    // this sample's box offset and weights
    float w[3][NT], g[3][NT];
    int off = 0;
    if (inb) {
#pragma unroll
      for (int d = 0; d < 3; ++d) tl_taps<ORD>(xq[d], w[d], g[d]);
      off = (lo[0] - mn[0]) * DYZ + (lo[1] - mn[1]) * DZ + (lo[2] - mn[2]);
    }
    __syncthreads();
    for (int q = threadIdx.x; q < VOL; q += DYN_NTH) box[q] = 0.0;
    const float *tq = MODE == TM_PUSH ? a.trgt + (int64_t)n * a.trgt_s[0] + (int64_t)px * a.trgt_s[2] +
                                            (int64_t)py * a.trgt_s[3] + (int64_t)pz * a.trgt_s[4]
                                      : nullptr;
    float *out = a.out + (int64_t)n * a.out_s[0];
    const int C = MODE == TM_COUNT ? 1 : (int)a.C;
    for (int c = 0; c < C; ++c) {
      const float v = !inb ? 0.f : (MODE == TM_PUSH ? tq[(int64_t)c * a.trgt_s[1]] : 1.f);
      __syncthreads();   // box cleared (first channel) / flushed (later ones)
      if (inb && v != 0.f) {
        const double vd = (double)v;
        double *bp = box + off;
#pragma unroll 1
        for (int kx = 0; kx < NT; ++kx, bp += DYZ) {
#pragma unroll
          for (int ky = 0; ky < NT; ++ky) {
            const double t = (double)w[0][kx] * (double)w[1][ky] * vd;
            double *bq = bp + ky * DZ;
#pragma unroll
            for (int kz = 0; kz < NT; ++kz) atomicAdd(bq + kz, t * (double)w[2][kz]);
          }
        }
      }
      __syncthreads();
      // flush: one FP32 global atomic per non-zero box element; clear it
      float *oc = out + (int64_t)c * a.out_s[1];
      for (int q = threadIdx.x; q < VOL; q += DYN_NTH) {
        const double dv = box[q];
        box[q] = 0.0;
        if (dv == 0.0) continue;
        const int row = tl_div(q, DZ, rz), bz = q - row * DZ;
        const int bx = tl_div(row, ext[1], ry), by = row - bx * ext[1];
        const float sg = fsg[bx] * fsg[ext[0] + by] * fsg[ext[0] + ext[1] + bz];
        if (sg != 0.f)
          atomic_add(oc + fofs[bx] + fofs[ext[0] + by] + fofs[ext[0] + ext[1] + bz], (float)dv * sg);
      }
    }
  }
}

}  // namespace ni_amd

#include "pushpull_bin.h"   // the binned second pass (uses the helpers above)
#include "pushpull_scatter.h"
#include "pushpull_gather.h"
#include "pushpull_gtile.h"

namespace ni_amd {

// Channels from which the tiles of a large pull or grid_grad that are too
// spread are sorted into bins instead of staging one or two channels at a
// time: with fewer, or in small calls, the sort costs more than it saves (order
// 3, 181 x 217 x 181, a warp of 8 voxels RMS: 8 channels 1.2 ms binned, 2.6
// not; one channel 0.58 and 0.38).
#define BIN_MIN_CHANNELS 3

// Such a tile's box holds more than 1 / bin_parts of the LDS.  Two channels at
// a time beat the bins up to order 4 (181 x 217 x 181, 4 channels, order 3, warp
// of 4 voxels RMS: 0.50 against 0.57 ms), not where a sample has 216 taps or
// more and the box most of a tile's time (order 5, warp of 8: 1.40 against 1.21;
// of 2: 0.67 and 0.75, few tiles; order 4, 8 channels, warp of 8: 1.92 and 1.60),
// but again at order 7, whose bins of 15^3 voxels are slow (rotation by 30
// degrees: 1.57 and 1.96), nor where each stage re-reads the source's cache
// lines (16 channels last, order 3, rotation by 30 degrees: 2.68 and 1.56).
template <int ORD, int MODE>
static int bin_parts(const PPArgs<float> &a) {
  const bool taps = MODE == TM_PULL && (ORD == 5 || ORD == 6 || (ORD == 4 && a.C > 4));
  return taps || wide_strided(a) ? 4 : 2;
}

// A gather's samples are independent, and its blocks long along z: lattices of
// few z are relabelled (points in a row and single slices to the last axes; two
// or three slices trade z and y), so that their blocks are not mostly idle.
// Pull, order 3: 10^6 points 0.90 -> 0.25 ms, 2048 x 2048 x 1 0.76 -> 0.23,
// 1024 x 1024 x 2 0.21 -> 0.09.
static PPArgs<float> gather_lattice(PPArgs<float> a) {
  int64_t *t[3] = {&a.tX, &a.tY, &a.tZ};
  auto swap = [&](int i, int j) {
    std::swap(*t[i], *t[j]);
    std::swap(a.grid_s[1 + i], a.grid_s[1 + j]);
    std::swap(a.trgt_s[2 + i], a.trgt_s[2 + j]);
    std::swap(a.out_s[2 + i], a.out_s[2 + j]);
    std::swap(a.gout_s[1 + i], a.gout_s[1 + j]);
  };
  if (a.tZ == 1 && a.tY == 1) {
    swap(0, 2);
  } else if (a.tZ == 1) {   // (X, Y, 1) -> (1, X, Y)
    swap(1, 2);
    swap(0, 1);
  } else if (a.tZ <= 3 && a.tY >= 16) {
    swap(1, 2);
  }
  return a;
}

template <int ORD, int MODE>
static void launch_gather_mode(const PPArgs<float> &a, hipStream_t st) {
  if (a.C <= gather_channels<ORD, MODE>(a)) {
    launch_gather<ORD, MODE>(a, st);
    return;
  }
  if constexpr (ORD >= 1 && (MODE == TM_PULL || MODE == TM_SGRAD)) {
    using B = TileDims<ORD, MODE>;
    const int ntx = (int)((a.tX + B::TX - 1) / B::TX);
    const int nty = (int)((a.tY + B::TY - 1) / B::TY);
    const int ntz = (int)((a.tZ + B::TZ - 1) / B::TZ);
    BinPlan p;
    if ((ORD > 1 || wide_strided(a)) && a.C >= BIN_MIN_CHANNELS && a.N * a.tX * a.tY * a.tZ >= BIN_MIN_SAMPLES &&
        bin_plan(a, a.N * (int64_t)ntx * nty * ntz, B::TX * B::TY * B::TZ, p, st)) {
      launch_gtile<ORD, MODE>(a, p.fb, bin_parts<ORD, MODE>(a), st);
      launch_binned<ORD, MODE>(a, ntx, nty, ntz, p, st);
      return;
    }
  }
  if constexpr (ORD > 0) launch_gtile<ORD, MODE>(a, nullptr, 0, st);
}

// Whether the mode's first kernel can cover the samples in one launch (thin or
// very many lattices leave most of a block idle, up to 255 of 256 threads).
template <int ORD, int MODE>
static bool tile_fits(const PPArgs<float> &call) {
  const PPArgs<float> a = TileMeta<MODE>::gather ? gather_lattice(call) : call;
  using B = TileDims<ORD, MODE>;
  const bool cache = TileMeta<MODE>::gather && a.C <= gather_channels<ORD, MODE>(a);
  const int64_t bx = cache ? GA_TX : B::TX, by = cache ? GA_TY : B::TY, bz = cache ? GA_TZ : B::TZ;
  return launch_fits(a.N * ((a.tX + bx - 1) / bx) * ((a.tY + by - 1) / by) * ((a.tZ + bz - 1) / bz),
                     TileMeta<MODE>::gather ? GA_NTH : TileBox<ORD>::NTH);
}

// Push / count: tile_kernel, then the tiles it listed as too scattered.  In
// calls of at least BIN_MIN_SAMPLES samples that may allocate: scatter_kernel
// on those that fit a few larger boxes, the binned pass on the others.
// Below, where these launches cost more than they save, tile_dyn (list in
// stream-ordered scratch or the caller's; without either, tile_fallback
// repeats the bounding-box test on every tile).
template <int ORD, int MODE>
static void launch_tile(const PPArgs<float> &a, hipStream_t st) {
  if constexpr (TileMeta<MODE>::gather) {
    launch_gather_mode<ORD, MODE>(gather_lattice(a), st);
  } else {
    using B = TileBox<ORD>;
    const int ntx = (int)((a.tX + B::TX - 1) / B::TX);
    const int nty = (int)((a.tY + B::TY - 1) / B::TY);
    const int ntz = (int)((a.tZ + B::TZ - 1) / B::TZ);
    const int64_t nb = a.N * (int64_t)ntx * nty * ntz;
    const dim3 g((unsigned)nb), b(B::NTH);
    const bool own = a.scratch == nullptr;
    BinPlan p;
    if (own && a.N * a.tX * a.tY * a.tZ >= BIN_MIN_SAMPLES && bin_plan(a, nb, B::TX * B::TY * B::TZ, p, st)) {
      hipLaunchKernelGGL((tile_kernel<ORD, MODE>), g, b, 0, st, a, ntx, nty, ntz, nb, p.fb, p.tiles);
      const dim3 gs((unsigned)(nb < 1024 ? nb : 1024));
      hipLaunchKernelGGL((scatter_kernel<ORD, MODE == TM_COUNT>), gs, b, 0, st, a, ntx, nty, ntz, (const int *)p.tiles,
                         p.fb);
      launch_binned<ORD, MODE>(a, ntx, nty, ntz, p, st);
      return;
    }
    int *fb = nullptr;
    if (!own) {
      fb = a.scratch;   // the caller checked nb + 1 <= a.scratch_cap
    } else if (scratch_alloc((void **)&fb, sizeof(int) * (size_t)(nb + 1), st) != hipSuccess) {
      (void)hipGetLastError();
      fb = nullptr;
    }
    if (fb) hipLaunchKernelGGL(fill_zero<int>, dim3(1), dim3(NI_BLOCK), 0, st, fb, (int64_t)1);
    hipLaunchKernelGGL((tile_kernel<ORD, MODE>), g, b, 0, st, a, ntx, nty, ntz, nb, fb, (int *)nullptr);
    if (fb) {
      constexpr int nsub = (B::TX / DYN_TX) * (B::TY / DYN_TY) * (B::TZ / DYN_TZ);
      const int64_t want = nb * nsub;
      const unsigned gd = (unsigned)(want < 4096 ? want : 4096);
      hipLaunchKernelGGL((tile_dyn<ORD, MODE>), dim3(gd), dim3(DYN_NTH), 0, st, a, ntx, nty, ntz, (const int *)fb);
      if (own) (void)hipFreeAsync(fb, st);
    } else {
      hipLaunchKernelGGL((tile_fallback<ORD, MODE>), g, b, 0, st, a, ntx, nty, ntz, nb);
    }
  }
}

// Every mode of a call, or false (nothing launched) if one does not fit.
template <int ORD, int... MODES>
static bool launch_tiles(const PPArgs<float> &a, hipStream_t st) {
  if (!(tile_fits<ORD, MODES>(a) && ...)) return false;
  (launch_tile<ORD, MODES>(a, st), ...);
  return true;
}

}  // namespace ni_amd
