// Row-gather pull / gradients of 3-D float fields (isotropic order ORD):
// one thread per sample, taps read straight from the caches.
//
// A work-group covers a 4 x 4 x 16 block of samples (a wave: 4 y-rows of 16
// z-consecutive samples), so that neighbouring lanes read neighbouring
// source voxels on any smooth grid and the CU's vector cache serves the
// re-reads that an LDS box would.  The ORD + 1 z-taps of a sample are
// consecutive in memory when the source's z stride is 1 and none of them
// folds: one load of up to 16 bytes a tap row.  No box means no limit on
// how far a block's samples spread: rotated, zoomed and strongly warped
// grids take the same single launch as near-identity ones, with no list of
// scattered tiles, no sort and no scratch.
//
// Taps, weights, the out-of-bound rule and folding are pp_sample's; a tap
// row is summed along z first (weights and derivatives), then weighted
// along y and x, which differs from pp_sample's order only by rounding.
#pragma once
#include <type_traits>

namespace ni_amd {

#ifndef GA_TX
#define GA_TX 4
#define GA_TY 4
#define GA_TZ 16
#endif
#define GA_NTH 256

// Folded offsets and signed weights of one axis's taps.  Bit t of `ok` is
// set when tap t lies inside (sign != 0): a tap that reads as zero must not
// let its voxel's value through (it may be a NaN), nor its weight (infinite
// or NaN at an infinite coordinate).
template <int ORD, bool DERIV>
__device__ __forceinline__ unsigned ga_fold(int bound, int lo, int n, int stride, float (&w)[ORD + 1],
                                            float (&g)[ORD + 1], int (&of)[ORD + 1]) {
  unsigned ok = 0;
  // rolled: taps shift through the last element, NT shifts restore the order
#pragma unroll 1
  for (int t = 0; t <= ORD; ++t) {
    int s;
    const int j = fold<int>(bound, tap_at(lo, t), n, s) * stride;
    ok |= s != 0 ? 1u << t : 0u;
    tl_rot(of);
    tl_rot(w);
    of[ORD] = j;
    w[ORD] = s != 0 ? w[ORD] * (float)s : 0.f;
    if constexpr (DERIV) {
      tl_rot(g);
      g[ORD] = s != 0 ? g[ORD] * (float)s : 0.f;
    }
  }
  return ok;
}

// Taps of one sample: first-tap offset and strides when every tap of the
// wave lies inside the source (INNER), folded offsets and `ok` bits per axis
// otherwise.
template <int ORD, bool INNER, bool ZU, bool ROLL>
struct GaTaps {
  int base, s0, s1, s2;
  // of[0] (and, with ROLL, of[1]) is rotated by the tap loop: element 0 is the
  // current plane (row)
  int of[3][ORD + 1];
  unsigned ok[3];
  __device__ __forceinline__ void row(const float *sp, int kx, int ky, float (&v)[ORD + 1]) const {
    if constexpr (INNER) {
      const float *rp = sp + (base + kx * s0 + ky * s1);
#pragma unroll
      for (int kz = 0; kz <= ORD; ++kz) v[kz] = rp[ZU ? kz : kz * s2];
    } else {
      const float *rp = sp + (of[0][0] + of[1][ROLL ? 0 : ky]);
      const bool in = (ok[0] >> kx) & (ok[1] >> ky) & 1u;
#pragma unroll
      for (int kz = 0; kz <= ORD; ++kz) {
        const float t = rp[of[2][kz]];
        v[kz] = in && ((ok[2] >> kz) & 1u) ? t : 0.f;
      }
    }
  }
  __device__ __forceinline__ void next(int axis) {
    if constexpr (!INNER) tl_rot(of[axis]);
  }
};

// Value (ax) or spatial gradient (ax, ay, az) of the channel at `sp`.  ROLL:
// the rows are looped over instead of unrolled with every load in flight
// (the tile kernel's rare samples, whose registers would lower its occupancy).
template <int ORD, bool DERIV, bool ROLL, class TAPS>
__device__ __forceinline__ void ga_sum(TAPS &tp, const float *sp, float (&w)[3][ORD + 1], float (&g)[3][ORD + 1],
                                       float &ax, float &ay, float &az) {
  constexpr int NT = ORD + 1;
  ax = ay = az = 0.f;
  float sw, sg, sv;   // plane sums: w_y w_z, g_y w_z, w_y g_z
  auto row = [&](int kx, int ky) {
    float v[NT];
    tp.row(sp, kx, ky, v);
    float rw = v[0] * w[2][0], rg = 0.f;
    if constexpr (DERIV) rg = v[0] * g[2][0];
#pragma unroll
    for (int kz = 1; kz < NT; ++kz) {
      rw += v[kz] * w[2][kz];
      if constexpr (DERIV) rg += v[kz] * g[2][kz];
    }
    const int j = ROLL ? 0 : ky;
    sw += w[1][j] * rw;
    if constexpr (DERIV) {
      sg += g[1][j] * rw;
      sv += w[1][j] * rg;
    }
    if constexpr (ROLL) {   // NT rotations restore the order
      tl_rot(w[1]);
      if constexpr (DERIV) tl_rot(g[1]);
      tp.next(1);
    }
  };
  auto plane = [&](int kx) {
    sw = sg = sv = 0.f;
    if constexpr (ROLL) {
#pragma unroll 1
      for (int ky = 0; ky < NT; ++ky) row(kx, ky);
    } else {
#pragma unroll
      for (int ky = 0; ky < NT; ++ky) row(kx, ky);
    }
    ax += (DERIV ? g[0][0] : w[0][0]) * sw;
    if constexpr (DERIV) {
      ay += w[0][0] * sg;
      az += w[0][0] * sv;
    }
    tl_rot(w[0]);
    if constexpr (DERIV) tl_rot(g[0]);
    tp.next(0);
  };
  if constexpr (ROLL) {
#pragma unroll 1
    for (int kx = 0; kx < NT; ++kx) plane(kx);
  } else {
#pragma unroll
    for (int kx = 0; kx < NT; ++kx) plane(kx);
  }
}

// Where a sample's results go (and, for the grid gradient, its target).
struct GaOut {
  float *op;
  int oC, oK;
  const float *tp;
  int tC;
};

// Taps of NC channels at once, each multiplied by its target: their grid
// gradients share the weights.
template <int ORD, int NC, class TAPS>
struct GaDot {
  TAPS &t;
  int sC;
  float tv[NC];
  __device__ __forceinline__ void row(const float *sp, int kx, int ky, float (&v)[ORD + 1]) const {
    float u[NC][ORD + 1];
#pragma unroll
    for (int c = 0; c < NC; ++c) t.row(sp + c * sC, kx, ky, u[c]);
#pragma unroll
    for (int k = 0; k <= ORD; ++k) {
      v[k] = u[0][k] * tv[0];
#pragma unroll
      for (int c = 1; c < NC; ++c) v[k] += u[c][k] * tv[c];
    }
  }
  __device__ __forceinline__ void next(int axis) { t.next(axis); }
};

// DOT: grid gradients take four channels at a time (sources whose channels
// lie side by side: a cache line is read by few loads, not by one a channel).
template <int ORD, int MODE, bool ROLL, bool DOT, class TAPS>
__device__ __forceinline__ void ga_run(TAPS &taps, const float *src, int sC, int C, bool inb, bool valid,
                                       float (&w)[3][ORD + 1], float (&g)[3][ORD + 1], const GaOut &o,
                                       float (&og)[3]) {
  constexpr bool DERIV = TileMeta<MODE>::deriv;
  int first = 0;
  if constexpr (MODE == TM_GGRAD && DOT) {
#pragma unroll 1
    for (; first + 4 <= C; first += 4) {
      if (!inb) continue;
      GaDot<ORD, 4, TAPS> q{taps, sC, {}};
#pragma unroll
      for (int c = 0; c < 4; ++c) q.tv[c] = o.tp[(first + c) * o.tC];
      float ax, ay, az;
      ga_sum<ORD, DERIV, ROLL>(q, src + first * sC, w, g, ax, ay, az);
      og[0] += ax;
      og[1] += ay;
      og[2] += az;
    }
  }
#pragma unroll 1
  for (int c = first; c < C; ++c) {
    float ax = 0.f, ay = 0.f, az = 0.f;
    if (inb) ga_sum<ORD, DERIV, ROLL>(taps, src + c * sC, w, g, ax, ay, az);
    if (!valid) continue;
    if constexpr (MODE == TM_PULL) {
      o.op[c * o.oC] = ax;
    } else if constexpr (MODE == TM_SGRAD) {
      float *op = o.op + c * o.oC;
      op[0] = ax;
      op[o.oK] = ay;
      op[2 * o.oK] = az;
    } else if (inb) {
      const float t = MODE == TM_GGRAD ? o.tp[c * o.tC] : 1.f;
      og[0] += t * ax;
      og[1] += t * ay;
      og[2] += t * az;
    }
  }
}

template <int ORD, int MODE, bool ZU, bool ROLL, bool DOT = false>
__device__ __forceinline__ void ga_sample(const PPArgs<float> &a, int n, int px, int py, int pz, bool valid) {
  constexpr int NT = ORD + 1;
  constexpr bool DERIV = TileMeta<MODE>::deriv;
  const int sz[3] = {(int)a.sX, (int)a.sY, (int)a.sZ};
  const float tol = (a.extrap & 2) ? 0.55f : 0.05f;
  float w[3][NT], g[3][NT];
  int lo[3] = {0, 0, 0};
  bool inb = false, inner[3] = {true, true, true};
  if (valid) {
    const float *gp = a.grid + (int)(n * a.grid_s[0] + px * a.grid_s[1] + py * a.grid_s[2] + pz * a.grid_s[3]);
    const int gD = (int)a.grid_s[4];
    const float xs[3] = {gp[0], gp[gD], gp[2 * gD]};
    inb = true;
    if (!(a.extrap & 1))
#pragma unroll
      for (int d = 0; d < 3; ++d) inb = inb && (xs[d] >= -tol && xs[d] < (float)(sz[d] - 1) + tol);
    if (inb)
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        lo[d] = tl_taps<ORD, DERIV>(xs[d], w[d], g[d]);
        inner[d] = lo[d] >= 0 && lo[d] <= sz[d] - NT;
      }
  }
  const int st[3] = {(int)a.src_s[2], (int)a.src_s[3], (int)a.src_s[4]};
  const int C = (int)a.C, sC = (int)a.src_s[1];
  const float *src = a.src + (int)(n * a.src_s[0]);
  GaOut o{nullptr, (int)a.out_s[1], (int)a.out_s[5], nullptr, (int)a.trgt_s[1]};
  if constexpr (MODE == TM_PULL || MODE == TM_SGRAD)
    o.op = a.out + (int)(n * a.out_s[0] + px * a.out_s[2] + py * a.out_s[3] + pz * a.out_s[4]);
  if constexpr (MODE == TM_GGRAD)
    o.tp = a.trgt + (int)(n * a.trgt_s[0] + px * a.trgt_s[2] + py * a.trgt_s[3] + pz * a.trgt_s[4]);
  float og[3] = {0.f, 0.f, 0.f};
  if constexpr (ORD == 0 && (MODE == TM_GGRAD || MODE == TM_GGRAD1)) {
    // zero everywhere: nothing to read
  } else if (!ROLL && __all(inner[0] && inner[1] && inner[2])) {
    GaTaps<ORD, true, ZU, ROLL> t;
    t.base = lo[0] * st[0] + lo[1] * st[1] + lo[2] * st[2];
    t.s0 = st[0];
    t.s1 = st[1];
    t.s2 = st[2];
    ga_run<ORD, MODE, ROLL, DOT>(t, src, sC, C, inb, valid, w, g, o, og);
  } else {
    GaTaps<ORD, false, ZU, ROLL> t;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      if (!ROLL && __all(inner[d])) {   // no lane folds along this axis
        t.ok[d] = ~0u;
#pragma unroll
        for (int k = 0; k < NT; ++k) t.of[d][k] = (lo[d] + k) * st[d];
      } else if (inb) {
        t.ok[d] = ga_fold<ORD, DERIV>(a.bound[d], lo[d], sz[d], st[d], w[d], g[d], t.of[d]);
      }
    }
    ga_run<ORD, MODE, ROLL, DOT>(t, src, sC, C, inb, valid, w, g, o, og);
  }
  if constexpr (MODE == TM_GGRAD || MODE == TM_GGRAD1) {
    if (valid) {
      float *gq = a.gout + (int)(n * a.gout_s[0] + px * a.gout_s[1] + py * a.gout_s[2] + pz * a.gout_s[3]);
      const int gDo = (int)a.gout_s[4];
      gq[0] = og[0];
      gq[gDo] = og[1];
      gq[2 * gDo] = og[2];
    }
  }
}

template <int ORD, int MODE, bool ZU>
__global__ __launch_bounds__(GA_NTH) void gather_kernel(PPArgs<float> a, int ntx, int nty, int ntz, int64_t nblocks) {
  int64_t r = xcd_block(nblocks);
  const int tz = (int)(r % ntz); r /= ntz;
  const int ty = (int)(r % nty); r /= nty;
  const int tx = (int)(r % ntx);
  const int n = (int)(r / ntx);
  const int px = tx * GA_TX + (int)(threadIdx.x / (GA_TY * GA_TZ));
  const int py = ty * GA_TY + (int)(threadIdx.x / GA_TZ) % GA_TY;
  const int pz = tz * GA_TZ + (int)(threadIdx.x % GA_TZ);
  ga_sample<ORD, MODE, ZU, false>(a, n, px, py, pz, px < a.tX && py < a.tY && pz < a.tZ);
}

template <int ORD, int MODE>
static void launch_gather(const PPArgs<float> &a, hipStream_t st) {
  const int ntx = (int)((a.tX + GA_TX - 1) / GA_TX);
  const int nty = (int)((a.tY + GA_TY - 1) / GA_TY);
  const int ntz = (int)((a.tZ + GA_TZ - 1) / GA_TZ);
  const int64_t nb = a.N * (int64_t)ntx * nty * ntz;
  if (a.src_s[4] == 1)
    hipLaunchKernelGGL((gather_kernel<ORD, MODE, true>), dim3((unsigned)nb), dim3(GA_NTH), 0, st, a, ntx, nty, ntz, nb);
  else
    hipLaunchKernelGGL((gather_kernel<ORD, MODE, false>), dim3((unsigned)nb), dim3(GA_NTH), 0, st, a, ntx, nty, ntz, nb);
}

}  // namespace ni_amd
