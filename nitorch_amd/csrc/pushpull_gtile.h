// LDS-tiled gathers (pull, spatial gradients, grid gradients) of 3-D float
// fields (isotropic order ORD).
//
// One 256-thread work-group owns a 4 x 8 x 16 tile of samples, two a thread
// (4 y-rows apart; a wave covers 4 x-rows of 16 z-consecutive samples).  It
// reduces the bounding box of its in-bound samples' taps and stages that
// box of the source -- folded by the boundary condition and signed, so the
// taps need no folding -- in LDS, NCC channels interleaved per voxel, so
// that a tap of 4 channels is one 16-byte LDS read (gfx950's LDS serves
// 128-bit reads at ~1.5x the bytes per clock of 32-bit ones).  The box has
// the extents the tile needs: a rotation, a zoom or a displacement with a
// moderate Jacobian widens it, and the tile stages fewer channels at a time
// (4, 2, 1) until it fits.  A tile whose box does not fit with one channel
// (scattered or far-extrapolated coordinates) reads its taps straight from
// the caches (ga_sample): the result never depends on the data's
// smoothness, only the speed does, and a call is one launch without scratch.
//
// A tap row is summed along z first (weights and derivatives), then
// weighted along y and x; weights, the out-of-bound rule and folding are
// those of pp_sample.
#pragma once

namespace ni_amd {

#define FAR_TAP (1 << 30)   // first taps beyond are a saturated conversion's

// ONE: single-channel calls, whose kernels need fewer registers.
template <int ORD, bool DERIV, bool ONE>
struct GTile {
  static constexpr int NTH = 256, NW = NTH / 64, R = 2;
  static constexpr int TX = 4, TY = 8, TZ = 16;
  static constexpr int MAXE = 64;   // box extent per axis
  // work-groups that share a CU's 160 KB of LDS: what the kernel's registers
  // let run, except above order 3 with several channels, where a third
  // work-group leaves too small a box for rotated grids (order 5, 8 channels,
  // 181 x 217 x 181: 0.93 / 1.02 ms near the identity / rotated by 15 degrees
  // with 2, 0.74 / 1.46 with 3)
  static constexpr int WGS = ORD <= 2 ? 5 : ORD == 3 ? (ONE && !DERIV ? 5 : 4) : ONE ? 3 : 2;
  static constexpr int CAP = WGS == 5 ? 7592 : WGS == 4 ? 9824 : WGS == 3 ? 13024 : 20064;   // box, floats
};

// Voxels between the x planes of a box of E1 x E2 planes with ncc channels
// a voxel: padded so that the x-rows read in one LDS cycle fall on different
// banks (two rows of 16 z-samples half the banks apart), when that fits.
template <int CAP>
__device__ __forceinline__ int gt_plane(int E0, int E1, int E2, int ncc) {
  const int v = E1 * E2;
  const int m = ncc == 4 ? 31 : 63, r = ncc == 4 ? 16 : ncc == 2 ? 32 : 16;
  const int p = v + ((r - v) & m);
  return E0 * p * ncc <= CAP ? p : v;
}

// What a tile's samples need from its box, uniform over the work-group.
struct GBoxDims {
  int e[3];    // extents
  int DYZ;     // voxels between x planes (z rows are e[2] apart)
  bool inner;  // no position folds: box (x, y, z) is source element base + strides . (x, y, z)
  int base;
};

template <int NCC> struct GVec;
template <> struct GVec<1> { using T = float; };
template <> struct GVec<2> { using T = float2; };
template <> struct GVec<4> { using T = float4; };
__device__ __forceinline__ void g_unpack(const float &v, float (&o)[1]) { o[0] = v; }
__device__ __forceinline__ void g_unpack(const float2 &v, float (&o)[2]) { o[0] = v.x; o[1] = v.y; }
__device__ __forceinline__ void g_unpack(const float4 &v, float (&o)[4]) { o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w; }
__device__ __forceinline__ void g_pack(const float (&o)[1], float &v) { v = o[0]; }
__device__ __forceinline__ void g_pack(const float (&o)[2], float2 &v) { v = make_float2(o[0], o[1]); }
__device__ __forceinline__ void g_pack(const float (&o)[4], float4 &v) { v = make_float4(o[0], o[1], o[2], o[3]); }

// Stage channels src + c * sC (c < nc; zeros past nc) of the box: each thread
// owns y-z positions of the plane and walks x, XB positions of every channel
// in flight.  INNER: no position of the box folds, so that addresses are a
// uniform base plus one 32-bit offset a thread, and nothing is signed.
template <int NCC, bool INNER>
__device__ __forceinline__ void gt_fill(float *box, const float *src, int sC, int nc, const GBoxDims &d,
                                        const int (&st)[3], const int *fofs, const float *fsg) {
  constexpr int NTH = 256, MAXE = 64;
  using V = typename GVec<NCC>::T;
  constexpr int XB = NCC == 4 ? 4 : 8;
  const int plane = d.e[1] * d.e[2];
  const float r2 = 1.f / (float)d.e[2];
  V *vbox = (V *)box;
  for (int p = threadIdx.x; p < plane; p += NTH) {
    const int by = tl_div(p, d.e[2], r2), bz = p - by * d.e[2];
    unsigned yzb = 0;
    const float *sp = nullptr;
    float yz = 0.f;
    if constexpr (INNER) {
      yzb = (unsigned)(by * st[1] + bz * st[2]) * 4u;
    } else {
      sp = src + (fofs[MAXE + by] + fofs[2 * MAXE + bz]);
      yz = fsg[MAXE + by] * fsg[2 * MAXE + bz];
    }
    V *bp = vbox + p;
    auto rows = [&](auto xb, int x0) {
      constexpr int N = decltype(xb)::value;
      float v[N][NCC];
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int c = 0; c < NCC; ++c) {
          if constexpr (INNER)
            v[i][c] = c < nc ? *(const float *)((const char *)(src + (c * sC + (x0 + i) * st[0])) + yzb) : 0.f;
          else
            v[i][c] = c < nc ? sp[c * sC + fofs[x0 + i]] : 0.f;
        }
#pragma unroll
      for (int i = 0; i < N; ++i) {
        if constexpr (!INNER) {
          const float sg = fsg[x0 + i] * yz;
#pragma unroll
          for (int c = 0; c < NCC; ++c) v[i][c] = sg != 0.f ? v[i][c] * sg : 0.f;
        }
        g_pack(v[i], bp[(x0 + i) * d.DYZ]);
      }
    };
    int x0 = 0;
#pragma unroll 1
    for (; x0 + XB <= d.e[0]; x0 += XB) rows(std::integral_constant<int, XB>{}, x0);
    if (XB > 4 && x0 + 4 <= d.e[0]) {
      rows(std::integral_constant<int, 4>{}, x0);
      x0 += 4;
    }
    if (x0 + 2 <= d.e[0]) {
      rows(std::integral_constant<int, 2>{}, x0);
      x0 += 2;
    }
    if (x0 < d.e[0]) rows(std::integral_constant<int, 1>{}, x0);
  }
}

// Sums of one sample over its taps in the box: values (ax), or derivatives
// along x, y, z (ax, ay, az), of NCC channels; with DOT, of their dot product
// with tv (ax[0], ay[0], az[0]).
template <int ORD, bool DERIV, bool DOT, int NCC>
__device__ __forceinline__ void gt_sum(const typename GVec<NCC>::T *bp, const GBoxDims &d, float (&w)[3][ORD + 1],
                                       float (&g)[3][ORD + 1], const float (&tv)[NCC],
                                       float (&ax)[DOT ? 1 : NCC], float (&ay)[DOT ? 1 : NCC],
                                       float (&az)[DOT ? 1 : NCC]) {
  constexpr int NT = ORD + 1, NA = DOT ? 1 : NCC;
#pragma unroll
  for (int c = 0; c < NA; ++c) ax[c] = ay[c] = az[c] = 0.f;
#pragma unroll 1
  for (int kx = 0; kx < NT; ++kx, bp += d.DYZ) {
    float sw[NA], sg[NA], sv[NA];   // plane sums: w_y w_z, g_y w_z, w_y g_z
#pragma unroll
    for (int c = 0; c < NA; ++c) sw[c] = sg[c] = sv[c] = 0.f;
    const typename GVec<NCC>::T *bq = bp;
#pragma unroll
    for (int ky = 0; ky < NT; ++ky, bq += d.e[2]) {
      float rw[NA], rg[NA];
#pragma unroll
      for (int kz = 0; kz < NT; ++kz) {
        float v[NCC], u[NA];
        g_unpack(bq[kz], v);
        if constexpr (DOT) {
          u[0] = v[0] * tv[0];
#pragma unroll
          for (int c = 1; c < NCC; ++c) u[0] += v[c] * tv[c];
        } else {
#pragma unroll
          for (int c = 0; c < NCC; ++c) u[c] = v[c];
        }
#pragma unroll
        for (int c = 0; c < NA; ++c) {
          rw[c] = kz ? rw[c] + u[c] * w[2][kz] : u[c] * w[2][kz];
          if constexpr (DERIV) rg[c] = kz ? rg[c] + u[c] * g[2][kz] : u[c] * g[2][kz];
        }
      }
#pragma unroll
      for (int c = 0; c < NA; ++c) {
        sw[c] += w[1][ky] * rw[c];
        if constexpr (DERIV) {
          sg[c] += g[1][ky] * rw[c];
          sv[c] += w[1][ky] * rg[c];
        }
      }
      // bound the rows in flight (registers; at order 2 the three rows of a plane
      // fit, and the fence costs 2 to 5 %)
      if constexpr (ORD != 2) __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int c = 0; c < NA; ++c) {
      ax[c] += (DERIV ? g[0][0] : w[0][0]) * sw[c];
      if constexpr (DERIV) {
        ay[c] += w[0][0] * sg[c];
        az[c] += w[0][0] * sv[c];
      }
    }
    tl_rot(w[0]);   // NT rotations restore the order
    if constexpr (DERIV) tl_rot(g[0]);
  }
}

// State of a thread's samples.
template <int ORD>
struct GSamples {
  bool valid[2], inb[2];
  int off[2];          // voxel offset of the first tap in the box
  float xq[2][3];
  int px, py, pz, n;
};

template <int ORD, int MODE, int NCC>
__device__ __forceinline__ void gt_run(const PPArgs<float> &a, float *box, const GBoxDims &d, const int *fofs,
                                       const float *fsg, GSamples<ORD> &s) {
  constexpr int NT = ORD + 1;
  constexpr bool DERIV = TileMeta<MODE>::deriv, GG = MODE == TM_GGRAD || MODE == TM_GGRAD1;
  constexpr int STEP = GTile<ORD, false, false>::NW;   // y-rows between a thread's samples
  const int C = (int)a.C, sC = (int)a.src_s[1];
  const int st[3] = {(int)a.src_s[2], (int)a.src_s[3], (int)a.src_s[4]};
  const float *src = a.src + (int)(s.n * a.src_s[0]);
  float og[2][3] = {{0.f, 0.f, 0.f}, {0.f, 0.f, 0.f}};
#pragma unroll 1
  for (int c0 = 0; c0 < C; c0 += NCC) {
    const int nc = C - c0 < NCC ? C - c0 : NCC;
    if (c0) __syncthreads();   // previous chunk fully read
    if (d.inner) gt_fill<NCC, true>(box, src + (c0 * sC + d.base), sC, nc, d, st, fofs, fsg);
    else gt_fill<NCC, false>(box, src + c0 * sC, sC, nc, d, st, fofs, fsg);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (!s.valid[i]) continue;
      float ax[GG ? 1 : NCC], ay[GG ? 1 : NCC], az[GG ? 1 : NCC], tv[NCC];
#pragma unroll
      for (int c = 0; c < (GG ? 1 : NCC); ++c) ax[c] = ay[c] = az[c] = 0.f;
      if (s.inb[i]) {
        float w[3][NT], g[3][NT];
#pragma unroll
        for (int k = 0; k < 3; ++k) (void)tl_taps<ORD, DERIV>(s.xq[i][k], w[k], g[k]);
        if constexpr (MODE == TM_GGRAD) {
          const float *tp = a.trgt + (int)(s.n * a.trgt_s[0] + c0 * a.trgt_s[1] + s.px * a.trgt_s[2] +
                                           (s.py + i * STEP) * a.trgt_s[3] + s.pz * a.trgt_s[4]);
          const int tC = (int)a.trgt_s[1];
#pragma unroll
          for (int c = 0; c < NCC; ++c) tv[c] = c < nc ? tp[c * tC] : 0.f;
        } else {
#pragma unroll
          for (int c = 0; c < NCC; ++c) tv[c] = c < nc ? 1.f : 0.f;
        }
        gt_sum<ORD, DERIV, GG, NCC>((const typename GVec<NCC>::T *)box + s.off[i], d, w, g, tv, ax, ay, az);
      }
      if constexpr (GG) {
        og[i][0] += ax[0];
        og[i][1] += ay[0];
        og[i][2] += az[0];
      } else {
        const int oC = (int)a.out_s[1], oK = (int)a.out_s[5];
        float *op = a.out + (int)(s.n * a.out_s[0] + (int64_t)c0 * oC + s.px * a.out_s[2] +
                                  (s.py + i * STEP) * a.out_s[3] + s.pz * a.out_s[4]);
#pragma unroll
        for (int c = 0; c < NCC; ++c) {
          if (c >= nc) break;
          op[c * oC] = ax[c];
          if constexpr (MODE == TM_SGRAD) {
            op[c * oC + oK] = ay[c];
            op[c * oC + 2 * oK] = az[c];
          }
        }
      }
    }
  }
  if constexpr (GG) {
    const int gD = (int)a.gout_s[4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
      if (s.valid[i]) {
        float *gq = a.gout + (int)(s.n * a.gout_s[0] + s.px * a.gout_s[1] + (s.py + i * STEP) * a.gout_s[2] +
                                   s.pz * a.gout_s[3]);
        gq[0] = og[i][0];
        gq[gD] = og[i][1];
        gq[2 * gD] = og[i][2];
      }
  }
}

// fb: list of the tiles left to the binned pass, or null: those whose box holds
// more than 1 / parts of the LDS.  DIRECT (wide strided sources at order 1):
// tiles that would stage one channel at a time (grid gradients: two) are read
// from the caches instead.
template <int ORD, int MODE, bool ONE, bool DIRECT>
__global__ __launch_bounds__(256) void gtile_kernel(PPArgs<float> a, int ntx, int nty, int ntz,
                                                    int64_t nblocks, int *fb, int parts) {
  using B = GTile<ORD, TileMeta<MODE>::deriv, ONE>;
  constexpr int NT = ORD + 1, R = B::R, STEP = B::NW;
  __shared__ __align__(16) float box[B::CAP];
  __shared__ int fofs[3 * B::MAXE];
  __shared__ float fsg[3 * B::MAXE];
  __shared__ int red[B::NW][6];

  const int64_t tile = xcd_block(nblocks);
  int64_t r = tile;
  const int tz = (int)(r % ntz); r /= ntz;
  const int ty = (int)(r % nty); r /= nty;
  const int tx = (int)(r % ntx);
  const int sz[3] = {(int)a.sX, (int)a.sY, (int)a.sZ};
  const int lane = threadIdx.x & 63;
  GSamples<ORD> s;
  s.n = (int)(r / ntx);
  s.px = tx * B::TX + lane / B::TZ;
  s.py = ty * B::TY + (int)(threadIdx.x >> 6);
  s.pz = tz * B::TZ + lane % B::TZ;

  int lo[R][3];
  int mn[3] = {INT_MAX, INT_MAX, INT_MAX}, mx[3] = {INT_MIN, INT_MIN, INT_MIN};
  const float tol = (a.extrap & 2) ? 0.55f : 0.05f;
  const int gD = (int)a.grid_s[4];
  const float *gp0 = a.grid + (int)(s.n * a.grid_s[0] + s.px * a.grid_s[1] + s.py * a.grid_s[2] + s.pz * a.grid_s[3]);
#pragma unroll
  for (int i = 0; i < R; ++i) {
    s.valid[i] = s.px < a.tX && s.py + i * STEP < a.tY && s.pz < a.tZ;
    s.inb[i] = false;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      s.xq[i][d] = 0.f;
      lo[i][d] = 0;
    }
    if (s.valid[i]) {
      const float *gp = gp0 + i * STEP * (int)a.grid_s[2];
      bool ok = true;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        s.xq[i][d] = gp[d * gD];
        if (!(a.extrap & 1)) ok = ok && (s.xq[i][d] >= -tol && s.xq[i][d] < (float)(sz[d] - 1) + tol);
      }
      s.inb[i] = ok;
      if (ok)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          lo[i][d] = tl_first<ORD>(s.xq[i][d]);
          mn[d] = min(mn[d], lo[i][d]);
          mx[d] = max(mx[d], lo[i][d]);
        }
    }
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    mn[d] = wave_min(mn[d]);
    mx[d] = wave_max(mx[d]);
  }
  if (lane == 0)
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      red[threadIdx.x >> 6][d] = mn[d];
      red[threadIdx.x >> 6][3 + d] = mx[d];
    }
  __syncthreads();
  GBoxDims d;
  bool fits = true, none = false;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    mn[k] = red[0][k];
    mx[k] = red[0][3 + k];
#pragma unroll
    for (int v = 1; v < B::NW; ++v) {
      mn[k] = min(mn[k], red[v][k]);
      mx[k] = max(mx[k], red[v][3 + k]);
    }
    mn[k] = __builtin_amdgcn_readfirstlane(mn[k]);
    mx[k] = __builtin_amdgcn_readfirstlane(mx[k]);
    none = none || mn[k] > mx[k];
    const int64_t e = (int64_t)mx[k] - (int64_t)mn[k] + NT;
    // (coordinates beyond the integer range have weights that a staged zero
    // would not cancel: ga_sample drops them)
    fits = fits && e <= B::MAXE && mn[k] > -FAR_TAP && mx[k] < FAR_TAP;
    d.e[k] = (int)(e <= B::MAXE ? e : B::MAXE);
  }
  // no in-bound sample: one channel of an (unread) unit box, so that the
  // outputs' zeros are written by the same code
  if (none) d.e[0] = d.e[1] = d.e[2] = 1;
  fits = fits || none;
  int ncc = ONE ? 1 : a.C >= 3 ? 4 : (int)a.C;
  const int vol = d.e[0] * d.e[1] * d.e[2];
  if (fb && (!fits || vol * parts > B::CAP)) {   // listed for the binned pass
    if (threadIdx.x == 0) fb[1 + atomicAdd(fb, 1)] = (int)tile;
    return;
  }
  while (ncc > 1 && vol * ncc > B::CAP) ncc >>= 1;
  constexpr int DIRECT_NCC = !DIRECT ? 0 : MODE == TM_GGRAD ? 2 : 1;
  if (!fits || vol > B::CAP || ncc <= DIRECT_NCC) {   // taps from the caches
#pragma unroll 1
    for (int py = s.py; py < s.py + R * STEP; py += STEP)
      ga_sample<ORD, MODE, false, !DIRECT, DIRECT>(a, s.n, s.px, py, s.pz, s.px < a.tX && py < a.tY && s.pz < a.tZ);
    return;
  }
  d.DYZ = gt_plane<B::CAP>(d.e[0], d.e[1], d.e[2], ncc);
  // (unsigned 32-bit byte offsets of a plane position: 2 * 64 strides below
  // 2^31, and none that steps back, as a flipped view's do)
  d.inner = !none && (uint64_t)a.src_s[3] < (1u << 22) && (uint64_t)a.src_s[4] < (1u << 22);
#pragma unroll
  for (int k = 0; k < 3; ++k) d.inner = d.inner && axis_inside(mn[k], d.e[k], sz[k]);
  d.base = mn[0] * (int)a.src_s[2] + mn[1] * (int)a.src_s[3] + mn[2] * (int)a.src_s[4];
  if (!d.inner)
    // folded offsets and signs of the box positions along each axis
    for (int i = threadIdx.x; i < 3 * B::MAXE; i += B::NTH) {
      const int k = i / B::MAXE, b = i % B::MAXE;
      const int e = k == 0 ? d.e[0] : k == 1 ? d.e[1] : d.e[2];
      if (b < e && !none) {
        const int m = k == 0 ? mn[0] : k == 1 ? mn[1] : mn[2];
        const int nn = k == 0 ? sz[0] : k == 1 ? sz[1] : sz[2];
        const int bd = k == 0 ? a.bound[0] : k == 1 ? a.bound[1] : a.bound[2];
        const int st = (int)(k == 0 ? a.src_s[2] : k == 1 ? a.src_s[3] : a.src_s[4]);
        int sg;
        const int j = fold<int>(bd, tap_at(m, b), nn, sg);
        fofs[i] = j * st;
        fsg[i] = (float)sg;
      } else if (b == 0) {
        fofs[i] = 0;
        fsg[i] = 0.f;
      }
    }
#pragma unroll
  for (int i = 0; i < R; ++i)
    s.off[i] = s.inb[i] ? (lo[i][0] - mn[0]) * d.DYZ + (lo[i][1] - mn[1]) * d.e[2] + (lo[i][2] - mn[2]) : 0;
  __syncthreads();
  if constexpr (!ONE) {
    if (ncc == 4) return gt_run<ORD, MODE, 4>(a, box, d, fofs, fsg, s);
    if (ncc == 2) return gt_run<ORD, MODE, 2>(a, box, d, fofs, fsg, s);
  }
  gt_run<ORD, MODE, 1>(a, box, d, fofs, fsg, s);
}

// Sources of many channels whose z neighbours are apart (channels-last views):
// staging fewer than four channels at a time reads every cache line once for
// each stage.
static inline bool wide_strided(const PPArgs<float> &a) { return a.src_s[4] != 1 && a.C >= 8; }

// fb: list of tiles left to the binned pass (a count, then tile ids), or null.
template <int ORD, int MODE>
static void launch_gtile(const PPArgs<float> &a, int *fb, int parts, hipStream_t st) {
  using B = GTile<ORD, false, false>;
  const int ntx = (int)((a.tX + B::TX - 1) / B::TX);
  const int nty = (int)((a.tY + B::TY - 1) / B::TY);
  const int ntz = (int)((a.tZ + B::TZ - 1) / B::TZ);
  const int64_t nb = a.N * (int64_t)ntx * nty * ntz;
  const dim3 g((unsigned)nb), b(B::NTH);
  if (ORD == 1 && wide_strided(a))
    hipLaunchKernelGGL((gtile_kernel<ORD, MODE, false, ORD == 1>), g, b, 0, st, a, ntx, nty, ntz, nb, fb, parts);
  else if (a.C == 1)
    hipLaunchKernelGGL((gtile_kernel<ORD, MODE, true, false>), g, b, 0, st, a, ntx, nty, ntz, nb, fb, parts);
  else
    hipLaunchKernelGGL((gtile_kernel<ORD, MODE, false, false>), g, b, 0, st, a, ntx, nty, ntz, nb, fb, parts);
}

// Channels up to which a call's taps are read straight from the caches
// (gather_kernel) rather than staged in LDS.  Order 0 has one tap, nothing to
// stage (8 channels, 181 x 217 x 181: 0.15 ms against the tiles' 0.19, 0.35
// against 0.73 on a warped grid).  At order 1 each channel re-reads 8 taps
// from the caches, where a tile stages 4 channels at once: pull of 3 channels
// 0.074 against 0.090 ms and 0.165 against 0.22 warped, of 8 channels 0.25
// against 0.20; the spatial gradient, whose stores weigh more, changes over
// earlier.  Above, the (ORD + 1)^2 rows of a tap box cost the caches more
// than the tile (order 3, one channel, rotated: 0.22 against 0.13 ms).  Where
// z neighbours are apart (channels-last views), neighbouring lanes and the taps
// of a row share cache lines less, and one channel is the limit at order 1
// (pull of 3: 0.12 against 0.09 ms near the identity, 0.21 and 0.10 rotated).
template <int ORD, int MODE>
static int gather_channels(const PPArgs<float> &a) {
  if (ORD != 1) return ORD == 0 ? INT_MAX : 0;
  return a.src_s[4] != 1 ? 1 : MODE == TM_SGRAD ? 2 : 3;
}

}  // namespace ni_amd
