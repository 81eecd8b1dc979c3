// Scaling and squaring of a stationary velocity field and its analytic
// backward (nitorch/spatial/_svf.py).
//
// One linear squaring is one launch (svf_step): the velocity at id + v, the
// composed Jacobian (_svf.py:449-478) and the pushed-forward gradient
// (:271-279) all read the same small neighbourhood of each voxel, so the
// sampling grid, the central-difference Jacobian field and the pulled fields
// are never written to memory.  svf_rotate is the backward's start (:255-269).
//
// The rest handles fields of 3 x 3 matrices at other interpolation orders
// (:271-284 and :480): the product of two Jacobian fields, and the
// push-forward of a gradient through one squaring, g0 + det(J) J^T p, fused
// into one pass.  There every field is addressed by element strides: a vector field by (per
// voxel, per component), a matrix field by (per voxel, per row, per
// column), so transposed and channel-first views are read in place.  The
// voxel index runs over the N x D x H x W voxels of a view whose leading
// dims collapse to one stride (the caller checks).  Outputs are dense,
// [V, 3, 3] or [V, 3].  Each lane handles one voxel; the bound is HBM.
#include <cstdint>

#include "common.h"
#include "nitorch_amd.h"

namespace ni_amd {

#define SV3_BLOCK 256
// voxels of a work-group of the linear squaring (SV3_BLOCK of them); the
// forward and backward of 160 x 192 x 160, 8 squarings, take 3.47 ms with
// 4 x 2 x 32, 3.70 with 4 x 4 x 16, 3.92 with 2 x 2 x 64, 4.28 with 8 x 4 x 8
#define SVF_TX 4
#define SVF_TY 2
#define SVF_TZ 32

struct Mat3 {
  int64_t v, r, c;
};

template <typename T>
__device__ __forceinline__ void load3x3(const T *p, const Mat3 &s, int64_t i, T m[3][3]) {
  const T *q = p + i * s.v;
#pragma unroll
  for (int r = 0; r < 3; ++r)
#pragma unroll
    for (int c = 0; c < 3; ++c) m[r][c] = q[r * s.r + c * s.c];
}

// O[i] = A[i] B[i]
template <typename T>
__global__ __launch_bounds__(SV3_BLOCK) void mat3_mul(int64_t V, const T *__restrict__ A, Mat3 sa,
                                                      const T *__restrict__ B, Mat3 sb, T *__restrict__ O) {
  const int64_t i = (int64_t)blockIdx.x * SV3_BLOCK + threadIdx.x;
  if (i >= V) return;
  T a[3][3], b[3][3];
  load3x3(A, sa, i, a);
  load3x3(B, sb, i, b);
  T *o = O + i * 9;
#pragma unroll
  for (int r = 0; r < 3; ++r)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      // summed in k order, as the rank-one accumulation it replaces
      T s = a[r][0] * b[0][c];
      s = s + a[r][1] * b[1][c];
      s = s + a[r][2] * b[2][c];
      o[r * 3 + c] = s;
    }
}

// O[i] = G0[i] + det(J[i]) * J[i]^T P[i]
template <typename T>
__global__ __launch_bounds__(SV3_BLOCK) void grad_step(int64_t V, const T *__restrict__ J, Mat3 sj,
                                                       const T *__restrict__ P, int64_t pv, int64_t pc,
                                                       const T *__restrict__ G0, int64_t gv, int64_t gc,
                                                       T *__restrict__ O) {
  const int64_t i = (int64_t)blockIdx.x * SV3_BLOCK + threadIdx.x;
  if (i >= V) return;
  T m[3][3];
  load3x3(J, sj, i, m);
  const T det = m[0][0] * (m[1][1] * m[2][2] - m[1][2] * m[2][1]) -
                m[0][1] * (m[1][0] * m[2][2] - m[1][2] * m[2][0]) +
                m[0][2] * (m[1][0] * m[2][1] - m[1][1] * m[2][0]);
  const T p0 = P[i * pv], p1 = P[i * pv + pc], p2 = P[i * pv + 2 * pc];
  T *o = O + i * 3;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    T s = m[0][c] * p0;
    s = s + m[1][c] * p1;
    s = s + m[2][c] * p2;
    o[c] = G0[i * gv + c * gc] + s * det;
  }
}

// ---------------------------------------------------------------------------
// One linear squaring of channel-last fields [N, X, Y, Z, 3].
// ---------------------------------------------------------------------------
struct SvfGeo {
  int n[3];          // X, Y, Z (each >= 2)
  int bound[3];      // of the pulls of v and g (the Jacobian's is dft)
  int ntx, nty, ntz; // blocks of SVF_TX x SVF_TY x SVF_TZ voxels
};

// This thread's voxel (batch b, coordinates p); false outside the lattice.
// Lanes run along z first, so that neighbouring lanes read neighbouring
// voxels; blocks of one XCD are contiguous.
__device__ __forceinline__ bool svf_voxel(const SvfGeo &G, int &b, int (&p)[3]) {
  const int64_t nb = gridDim.x, q = nb / 8, rem = nb % 8;
  const int64_t xcd = blockIdx.x % 8, local = blockIdx.x / 8;
  int64_t r = xcd * q + (xcd < rem ? xcd : rem) + local;
  const int tz = (int)(r % G.ntz); r /= G.ntz;
  const int ty = (int)(r % G.nty); r /= G.nty;
  const int tx = (int)(r % G.ntx);
  b = (int)(r / G.ntx);
  p[0] = tx * SVF_TX + (int)(threadIdx.x / (SVF_TY * SVF_TZ));
  p[1] = ty * SVF_TY + (int)(threadIdx.x / SVF_TZ) % SVF_TY;
  p[2] = tz * SVF_TZ + (int)(threadIdx.x % SVF_TZ);
  return p[0] < G.n[0] && p[1] < G.n[1] && p[2] < G.n[2];
}

template <typename T> __device__ __forceinline__ int svf_floor(T x);
template <> __device__ __forceinline__ int svf_floor<float>(float x) { return (int)floorf(x); }
template <> __device__ __forceinline__ int svf_floor<double>(double x) { return (int)floor(x); }

template <typename T>
__device__ __forceinline__ T det3(const T (&m)[3][3]) {
  return m[0][0] * (m[1][1] * m[2][2] - m[1][2] * m[2][1]) - m[0][1] * (m[1][0] * m[2][2] - m[1][2] * m[2][0]) +
         m[0][2] * (m[1][0] * m[2][1] - m[1][1] * m[2][0]);
}

// Linear pull of the 3-channel field f at taps (lo, lo + 1) with weights w,
// folded by the bounds.
template <typename T>
__device__ __forceinline__ void svf_pull(const T *f, const SvfGeo &G, const int (&lo)[3], const T (&w)[3][2],
                                         T (&out)[3]) {
  int of[3][2];
  T ws[3][2];
  bool on[3][2];
  const int st[3] = {G.n[1] * G.n[2] * 3, G.n[2] * 3, 3};
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      int s;
      of[d][t] = fold<int>(G.bound[d], tap_at(lo[d], t), G.n[d], s) * st[d];
      on[d][t] = s != 0;
      ws[d][t] = s < 0 ? -w[d][t] : w[d][t];
    }
  out[0] = out[1] = out[2] = T(0);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const T wxy = ws[0][i] * ws[1][j];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        if (!(on[0][i] && on[1][j] && on[2][k])) continue;   // reads as zero
        const T *q = f + (of[0][i] + of[1][j] + of[2][k]);
        const T ww = wxy * ws[2][k];
#pragma unroll
        for (int c = 0; c < 3; ++c) out[c] += q[c] * ww;
      }
    }
}

// Matrix fields: [N, X, Y, Z, 3, 3] (PLANAR false) or one plane of voxels an
// entry, [9, N, X, Y, Z], whose accesses are contiguous across lanes.
template <bool PLANAR, typename T>
__device__ __forceinline__ T *svf_mat(T *m, int64_t vox, int64_t nvox, int e) {
  return PLANAR ? m + e * nvox + vox : m + vox * 9 + e;
}

// With u = scale v (scale: +-2^-steps on the first squaring, else 1):
// v_out = u + u o (id + u) (+ id if add_id), unless null;
// JAC:  jac_out = ((I + D u) o (id + u)) jac, with D periodic central
//       differences (jac null: the identity);
// GRAD: g_out = gscale (g + det(jac) jac^T (g o (id + u))).
// The pulled I + D u is summed from the 32 voxels its 8 taps' differences
// touch (12 rows along z): at 160 x 192 x 160 the step with all three moves
// 120 B a voxel (0.12 ms at the rate of a large copy) and takes 0.24 ms, where
// the separate grid, difference, pull and product passes took 1.34.
template <typename T, bool JAC, bool GRAD, bool PLANAR>
__global__ __launch_bounds__(SV3_BLOCK) void svf_step(SvfGeo G, int64_t nvox, const T *__restrict__ v, T scale,
                                                      const T *jac, const T *__restrict__ g, T gscale,
                                                      T *__restrict__ v_out, T *jac_out, T *__restrict__ g_out,
                                                      int add_id) {
  int b, p[3];
  if (!svf_voxel(G, b, p)) return;
  const int64_t V = (int64_t)G.n[0] * G.n[1] * G.n[2];
  const int64_t vox = b * V + ((int64_t)p[0] * G.n[1] + p[1]) * G.n[2] + p[2];
  const T *vb = v + b * V * 3;
  T own[3], w[3][2];
  int lo[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    own[d] = v[vox * 3 + d] * scale;
    const T x = (T)p[d] + own[d];
    lo[d] = svf_floor<T>(x);
    // weights as distances to the far tap: exact when small
    w[d][0] = (T)(lo[d] + 1) - x;
    w[d][1] = x - (T)lo[d];
  }
  T m[3][3];
  if constexpr (JAC || GRAD) {
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c)
        m[r][c] = jac ? *svf_mat<PLANAR>(jac, vox, nvox, r * 3 + c) : (r == c ? T(1) : T(0));
  }
  if constexpr (GRAD) {
    T pg[3];
    svf_pull<T>(g + b * V * 3, G, lo, w, pg);
    const T det = det3(m);
#pragma unroll
    for (int c = 0; c < 3; ++c)
      g_out[vox * 3 + c] = (g[vox * 3 + c] + (m[0][c] * pg[0] + m[1][c] * pg[1] + m[2][c] * pg[2]) * det) * gscale;
    __builtin_amdgcn_sched_barrier(0);   // the pulled gradient's registers are free below
  }
  T pv[3];
  if constexpr (JAC) {
    // position a of an axis is voxel lo - 1 + a (a = 0..3), periodic
    int ix[4], iy[4], iz[4];
    const int sx = G.n[1] * G.n[2] * 3, sy = G.n[2] * 3;
    bool inner = true;
#pragma unroll
    for (int d = 0; d < 3; ++d) inner = inner && lo[d] >= 1 && lo[d] <= G.n[d] - 3;
    int s;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      ix[a] = (inner ? lo[0] - 1 + a : fold<int>(B_DFT, tap_at(lo[0], a - 1), G.n[0], s)) * sx;
      iy[a] = (inner ? lo[1] - 1 + a : fold<int>(B_DFT, tap_at(lo[1], a - 1), G.n[1], s)) * sy;
      iz[a] = (inner ? lo[2] - 1 + a : fold<int>(B_DFT, tap_at(lo[2], a - 1), G.n[2], s)) * 3;
    }
    T J[3][3];   // [component][axis], pulled central differences
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      pv[c] = T(0);
      J[c][0] = J[c][1] = J[c][2] = T(0);
    }
    // coefficients of the 4 positions in the sum of (v[a + 1] - v[a - 1]) over
    // the taps a = 1, 2 (halved below)
    const T dx[4] = {-w[0][0], -w[0][1], w[0][0], w[0][1]};
    const T dy[4] = {-w[1][0], -w[1][1], w[1][0], w[1][1]};
    // Their sums are zero: everything is summed of what exceeds the first tap's
    // velocity, so that the differences round as those of neighbours do and not
    // as the velocities, whose constant part may be large (30 voxels: 3e-6 of
    // rounding in the Jacobian against 3e-7).  In time it is even: 3.11 -> 3.08
    // ms the backward of 160 x 192 x 160.
    T first[3];
    {
      const T *q = vb + (ix[1] + iy[1] + iz[1]);
#pragma unroll
      for (int c = 0; c < 3; ++c) first[c] = q[c];
    }
#pragma unroll
    for (int ax = 0; ax < 4; ++ax)
#pragma unroll
      for (int ay = 0; ay < 4; ++ay) {
        const bool cx = ax == 1 || ax == 2, cy = ay == 1 || ay == 2;
        if (!cx && !cy) continue;
        const T *q = vb + (ix[ax] + iy[ay]);
        T zs[3], zd[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const T v1 = q[iz[1] + c], v2 = q[iz[2] + c];
          zs[c] = (v1 - first[c]) + w[2][1] * (v2 - v1);
          if (cx && cy) zd[c] = w[2][0] * (v2 - q[iz[0] + c]) + w[2][1] * (q[iz[3] + c] - v1);
        }
        const T wx = cx ? w[0][ax == 2] : T(0), wy = cy ? w[1][ay == 2] : T(0);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          if (cy) J[c][0] += dx[ax] * wy * zs[c];
          if (cx) J[c][1] += wx * dy[ay] * zs[c];
          if (cx && cy) {
            J[c][2] += wx * wy * zd[c];
            pv[c] += wx * wy * zs[c];
          }
        }
        if (ay & 1) __builtin_amdgcn_sched_barrier(0);   // bound the rows in flight (registers)
      }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      pv[c] = (pv[c] + first[c]) * scale;
#pragma unroll
      for (int d = 0; d < 3; ++d) J[c][d] = J[c][d] * (scale * T(0.5)) + (c == d ? T(1) : T(0));
    }
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c)
        *svf_mat<PLANAR>(jac_out, vox, nvox, r * 3 + c) = J[r][0] * m[0][c] + J[r][1] * m[1][c] + J[r][2] * m[2][c];
    // (the pull's own bound, where it is not the Jacobian's)
    const bool per = G.bound[0] == B_DFT && G.bound[1] == B_DFT && G.bound[2] == B_DFT;
    if (!per && !inner && v_out) {
      svf_pull<T>(vb, G, lo, w, pv);
#pragma unroll
      for (int c = 0; c < 3; ++c) pv[c] *= scale;
    }
  } else if (v_out) {
    svf_pull<T>(vb, G, lo, w, pv);
#pragma unroll
    for (int c = 0; c < 3; ++c) pv[c] *= scale;
  }
  if (!v_out) return;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    T o = own[c] + pv[c];
    if (add_id) o += (T)p[c];
    v_out[vox * 3 + c] = o;
  }
}

// jac_out = I + D (scale v) (central differences under the bounds), and
// g_out = (2 I - jac_out)^-T rot^T g (rot null: the identity): the gradient
// that the first squaring of the backward pushes forward.  Matrix fields are
// planar; jac_out may be rot.
template <typename T>
__global__ __launch_bounds__(SV3_BLOCK) void svf_rotate(SvfGeo G, int64_t nvox, const T *__restrict__ v, T scale,
                                                        const T *rot, const T *__restrict__ g, T *jac_out,
                                                        T *__restrict__ g_out) {
  int b, p[3];
  if (!svf_voxel(G, b, p)) return;
  const int64_t V = (int64_t)G.n[0] * G.n[1] * G.n[2];
  const int64_t vox = b * V + ((int64_t)p[0] * G.n[1] + p[1]) * G.n[2] + p[2];
  const int64_t st[3] = {(int64_t)G.n[1] * G.n[2] * 3, (int64_t)G.n[2] * 3, 3};
  T m[3][3];
  if (rot)
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c) m[r][c] = *svf_mat<true>(rot, vox, nvox, r * 3 + c);
  T a[3][3];   // J, then 2 I - J
  const T *q = v + vox * 3;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    int sp, sm;
    const int jp = fold<int>(G.bound[d], p[d] + 1, G.n[d], sp), jm = fold<int>(G.bound[d], p[d] - 1, G.n[d], sm);
    const T fp = (T)sp * scale, fm = (T)sm * scale;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const T vp = sp ? q[(jp - p[d]) * st[d] + c] * fp : T(0);
      const T vm = sm ? q[(jm - p[d]) * st[d] + c] * fm : T(0);
      a[c][d] = (vp - vm) * T(0.5) + (c == d ? T(1) : T(0));
    }
  }
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      *svf_mat<true>(jac_out, vox, nvox, c * 3 + d) = a[c][d];
      a[c][d] = (c == d ? T(2) : T(0)) - a[c][d];
    }
  T u[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) u[c] = g[vox * 3 + c];
  if (rot) {
    T t[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) t[c] = m[0][c] * u[0] + m[1][c] * u[1] + m[2][c] * u[2];
#pragma unroll
    for (int c = 0; c < 3; ++c) u[c] = t[c];
  }
  // a^T x = u by cofactors: x_i = sum_j cof(a)[i][j] u_j / det
  const T det = det3(a);
  const T c00 = a[1][1] * a[2][2] - a[1][2] * a[2][1], c01 = a[1][2] * a[2][0] - a[1][0] * a[2][2],
          c02 = a[1][0] * a[2][1] - a[1][1] * a[2][0];
  const T c10 = a[0][2] * a[2][1] - a[0][1] * a[2][2], c11 = a[0][0] * a[2][2] - a[0][2] * a[2][0],
          c12 = a[0][1] * a[2][0] - a[0][0] * a[2][1];
  const T c20 = a[0][1] * a[1][2] - a[0][2] * a[1][1], c21 = a[0][2] * a[1][0] - a[0][0] * a[1][2],
          c22 = a[0][0] * a[1][1] - a[0][1] * a[1][0];
  g_out[vox * 3 + 0] = (c00 * u[0] + c01 * u[1] + c02 * u[2]) / det;
  g_out[vox * 3 + 1] = (c10 * u[0] + c11 * u[1] + c12 * u[2]) / det;
  g_out[vox * 3 + 2] = (c20 * u[0] + c21 * u[1] + c22 * u[2]) / det;
}

static int svf_geo(int32_t dtype, int64_t N, const int64_t *shape, const int32_t *bound, SvfGeo &G, int64_t &nb) {
  NI_CHECK(dtype == NI_FLOAT32 || dtype == NI_FLOAT64, "svf: unsupported dtype %d", dtype);
  NI_CHECK(shape && bound && N >= 0, "svf: missing argument");
  int64_t vox = 1;
  for (int d = 0; d < 3; ++d) {
    NI_CHECK(shape[d] >= 2 && shape[d] < (1 << 30), "svf: each axis needs at least 2 voxels (got %lld)",
             (long long)shape[d]);
    NI_CHECK(bound[d] >= 0 && bound[d] <= 8, "svf: unknown bound code %d", bound[d]);
    vox *= shape[d];
    NI_CHECK(vox * 3 < (int64_t(1) << 31) - 1, "svf: volume too large");
    G.n[d] = (int)shape[d];
    G.bound[d] = bound[d];
  }
  G.ntx = (G.n[0] + SVF_TX - 1) / SVF_TX;
  G.nty = (G.n[1] + SVF_TY - 1) / SVF_TY;
  G.ntz = (G.n[2] + SVF_TZ - 1) / SVF_TZ;
  nb = N * (int64_t)G.ntx * G.nty * G.ntz;
  NI_CHECK(launch_fits(nb, SV3_BLOCK), "svf: too many voxels");
  return 0;
}

template <typename T>
static void svf_launch(const SvfGeo &G, int64_t N, int64_t nb, const void *v, double scale, const void *jac,
                       const void *g, double gscale, void *v_out, void *jac_out, void *g_out, bool planar, int add_id,
                       hipStream_t st) {
  const dim3 grid((unsigned)nb), block(SV3_BLOCK);
  const int64_t nvox = N * G.n[0] * G.n[1] * G.n[2];
#define SVF_LAUNCH(J, D, P)                                                                                     \
  hipLaunchKernelGGL((svf_step<T, J, D, P>), grid, block, 0, st, G, nvox, (const T *)v, (T)scale, (const T *)jac, \
                     (const T *)g, (T)gscale, (T *)v_out, (T *)jac_out, (T *)g_out, add_id)
  if (g_out && jac_out) {
    if (planar) SVF_LAUNCH(true, true, true);
    else SVF_LAUNCH(true, true, false);
  } else if (g_out) {
    if (planar) SVF_LAUNCH(false, true, true);
    else SVF_LAUNCH(false, true, false);
  } else if (jac_out) {
    if (planar) SVF_LAUNCH(true, false, true);
    else SVF_LAUNCH(true, false, false);
  } else {
    SVF_LAUNCH(false, false, false);
  }
#undef SVF_LAUNCH
}

static inline Mat3 mat3(const int64_t *s) { return Mat3{s[0], s[1], s[2]}; }

}  // namespace ni_amd

using namespace ni_amd;

extern "C" {

int ni_svf_mat3_mul(int32_t dtype, int64_t nvox, const void *a, const int64_t *a_stride, const void *b,
                    const int64_t *b_stride, void *out, void *stream) {
  set_error("");
  NI_CHECK(dtype == NI_FLOAT32 || dtype == NI_FLOAT64, "svf_mat3_mul: unsupported dtype %d", dtype);
  NI_CHECK(nvox >= 0, "svf_mat3_mul: negative voxel count");
  if (nvox == 0) return 0;
  NI_CHECK(a && b && out && a_stride && b_stride, "svf_mat3_mul: missing argument");
  hipStream_t st = (hipStream_t)stream;
  const unsigned nb = (unsigned)((nvox + SV3_BLOCK - 1) / SV3_BLOCK);
  NI_CHECK((nvox + SV3_BLOCK - 1) / SV3_BLOCK < (int64_t(1) << 31), "svf_mat3_mul: too many voxels");
  if (dtype == NI_FLOAT32)
    hipLaunchKernelGGL(mat3_mul<float>, dim3(nb), dim3(SV3_BLOCK), 0, st, nvox, (const float *)a,
                       mat3(a_stride), (const float *)b, mat3(b_stride), (float *)out);
  else
    hipLaunchKernelGGL(mat3_mul<double>, dim3(nb), dim3(SV3_BLOCK), 0, st, nvox, (const double *)a,
                       mat3(a_stride), (const double *)b, mat3(b_stride), (double *)out);
  NI_HIP_CHECK(hipGetLastError());
  return 0;
}

int ni_svf_grad_step(int32_t dtype, int64_t nvox, const void *jac, const int64_t *jac_stride, const void *p,
                     const int64_t *p_stride, const void *g0, const int64_t *g0_stride, void *out, void *stream) {
  set_error("");
  NI_CHECK(dtype == NI_FLOAT32 || dtype == NI_FLOAT64, "svf_grad_step: unsupported dtype %d", dtype);
  NI_CHECK(nvox >= 0, "svf_grad_step: negative voxel count");
  if (nvox == 0) return 0;
  NI_CHECK(jac && p && g0 && out && jac_stride && p_stride && g0_stride, "svf_grad_step: missing argument");
  NI_CHECK((nvox + SV3_BLOCK - 1) / SV3_BLOCK < (int64_t(1) << 31), "svf_grad_step: too many voxels");
  hipStream_t st = (hipStream_t)stream;
  const unsigned nb = (unsigned)((nvox + SV3_BLOCK - 1) / SV3_BLOCK);
  if (dtype == NI_FLOAT32)
    hipLaunchKernelGGL(grad_step<float>, dim3(nb), dim3(SV3_BLOCK), 0, st, nvox, (const float *)jac,
                       mat3(jac_stride), (const float *)p, p_stride[0], p_stride[1], (const float *)g0,
                       g0_stride[0], g0_stride[1], (float *)out);
  else
    hipLaunchKernelGGL(grad_step<double>, dim3(nb), dim3(SV3_BLOCK), 0, st, nvox, (const double *)jac,
                       mat3(jac_stride), (const double *)p, p_stride[0], p_stride[1], (const double *)g0,
                       g0_stride[0], g0_stride[1], (double *)out);
  NI_HIP_CHECK(hipGetLastError());
  return 0;
}

int ni_svf_step(int32_t dtype, int64_t N, const int64_t *shape, const int32_t *bound, const void *v, double scale,
                const void *jac, const void *g, double gscale, void *v_out, void *jac_out, void *g_out, int32_t planar,
                int32_t add_identity, void *stream) {
  set_error("");
  SvfGeo G;
  int64_t nb = 0;
  if (int rc = svf_geo(dtype, N, shape, bound, G, nb)) return rc;
  if (nb == 0) return 0;
  NI_CHECK(v && v != v_out, "svf_step: the velocity needs an output of its own");
  NI_CHECK(v_out || jac_out || g_out, "svf_step: no output");
  NI_CHECK(!g_out || (g && g != g_out), "svf_step: the gradient needs an output of its own");
  if (dtype == NI_FLOAT32)
    svf_launch<float>(G, N, nb, v, scale, jac, g, gscale, v_out, jac_out, g_out, planar != 0, add_identity,
                      (hipStream_t)stream);
  else
    svf_launch<double>(G, N, nb, v, scale, jac, g, gscale, v_out, jac_out, g_out, planar != 0, add_identity,
                       (hipStream_t)stream);
  NI_HIP_CHECK(hipGetLastError());
  return 0;
}

int ni_svf_rotate(int32_t dtype, int64_t N, const int64_t *shape, const int32_t *bound, const void *v, double scale,
                  const void *rot, const void *g, void *jac_out, void *g_out, void *stream) {
  set_error("");
  SvfGeo G;
  int64_t nb = 0;
  if (int rc = svf_geo(dtype, N, shape, bound, G, nb)) return rc;
  if (nb == 0) return 0;
  NI_CHECK(v && g && jac_out && g_out && g != g_out, "svf_rotate: missing argument");
  const dim3 grid((unsigned)nb), block(SV3_BLOCK);
  const int64_t nvox = N * G.n[0] * G.n[1] * G.n[2];
  if (dtype == NI_FLOAT32)
    hipLaunchKernelGGL(svf_rotate<float>, grid, block, 0, (hipStream_t)stream, G, nvox, (const float *)v, (float)scale,
                       (const float *)rot, (const float *)g, (float *)jac_out, (float *)g_out);
  else
    hipLaunchKernelGGL(svf_rotate<double>, grid, block, 0, (hipStream_t)stream, G, nvox, (const double *)v, scale,
                       (const double *)rot, (const double *)g, (double *)jac_out, (double *)g_out);
  NI_HIP_CHECK(hipGetLastError());
  return 0;
}

}  // extern "C"
