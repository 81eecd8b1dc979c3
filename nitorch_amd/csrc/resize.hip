// Generic resize of [N, C, *spatial] tensors (1-3 spatial dims) for gfx950.
//
// Replaces ni::resize (nitorch/_C/src/resize.cpp:25-59, implementation
// nitorch/_C/src/impl/resize_common.cpp): every target voxel w samples the
// source at the separable affine coordinate x = scale * w + shift (per axis,
// computed in double and rounded to the data type as the reference does)
// with the order-`order` B-spline and the boundary folding of the pull --
// with no out-of-bound masking (the reference's resize always interpolates).
// `do_adjoint` swaps the roles (source = output, target = input) and splats
// instead (the transpose), into a zeroed source.  shift / scale per axis
// follow prepare_affine (resize_common.cpp:1548-1567):
//   edge:   shift = (Ds/Dt - 1) / 2,            scale = Ds / Dt
//   center: shift = 0,                          scale = (Ds - 1) / (Dt - 1)
//   first:  shift = 0,                          scale = 1 / f
//   last:   shift = f (Ds - 1) / (Dt - 1),      scale = 1 / f
// with f the factor (inverted when do_adjoint), and `normalize` multiplies
// the result by the scales with the reference's fall-through switch
// (resize_common.cpp:1640-1646): 1-D by s0 * (s0 s1) * (s0 s1 s2), 2-D by
// (s0 s1) * (s0 s1 s2), 3-D by s0 s1 s2.
//
// MI355X layout: one lane per target voxel, z fastest, so the lanes of a
// wave read neighbouring source voxels and write (or, adjoint, scatter
// into) one contiguous run; per-axis taps, weights, signs and folded
// offsets are computed once per lane and reused over the channels.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>

#include "common.h"
#include "nitorch_amd.h"

namespace ni_amd {

#define RS_BLOCK 256
#define RS_MAXT 8

struct RsArgs {
  int N, C;
  int ns[3], nt[3];   // source / target sizes (1 for unused axes)
  int bound[3], order[3];
  double shift[3], scale[3];
  int accumulate;     // pull: add into the target instead of overwriting it
  int nearest_dbl;    // isotropic nearest: round scale * w + shift in double
};

template <typename T> __device__ inline T rs_floor(T x);
template <> __device__ inline float rs_floor<float>(float x) { return floorf(x); }
template <> __device__ inline double rs_floor<double>(double x) { return floor(x); }
template <typename T> __device__ inline T rs_round(T x);
template <> __device__ inline float rs_round<float>(float x) { return roundf(x); }
template <> __device__ inline double rs_round<double>(double x) { return round(x); }

// Taps of target index w along one axis: count, weights, signed source offsets.
template <typename T>
__device__ inline int rs_taps(const RsArgs &a, int d, int w, long long stride, T (&wt)[RS_MAXT],
                              long long (&off)[RS_MAXT], int (&sg)[RS_MAXT]) {
#pragma clang fp contract(off)
  const int o = a.order[d];
  // product and sum rounded separately, as the reference computes them (a
  // fused multiply-add moves coordinates such as 4.499999999999999 onto 4.5)
  const double xd = a.scale[d] * (double)w + a.shift[d];
  const T x = (T)xd;
  const int lo = o == 0 ? (a.nearest_dbl ? (int)round(xd) : (int)rs_round<T>(x))
                        : (int)rs_floor<T>(x - first_tap_offset<T>(o));
#pragma unroll
  for (int t = 0; t < RS_MAXT; ++t) {
    if (t > o) break;
    const int b = tap_at(lo, t);
    T g, h;
    spl_eval<T>(o, t, x - T(b), wt[t], g, h);
    int s;
    const int j = fold<int>(a.bound[d], b, a.ns[d], s);
    sg[t] = s;
    off[t] = (long long)j * stride;
  }
  return o + 1;
}

// ADJ == false: out (target) [+]= sum_taps w * s * in(source)
// ADJ == true : out (source) += w * s * in(target), by atomics
template <typename T, bool ADJ>
__global__ __launch_bounds__(RS_BLOCK) void resize_kernel(const T *__restrict__ in, T *__restrict__ out,
                                                          RsArgs a) {
  const long long Vt = (long long)a.nt[0] * a.nt[1] * a.nt[2];
  const long long Vs = (long long)a.ns[0] * a.ns[1] * a.ns[2];
  const long long gid = (long long)blockIdx.x * RS_BLOCK + threadIdx.x;
  if (gid >= (long long)a.N * Vt) return;
  const int n = (int)(gid / Vt);
  const long long v = gid - (long long)n * Vt;
  const int wz = (int)(v % a.nt[2]);
  const int wy = (int)((v / a.nt[2]) % a.nt[1]);
  const int wx = (int)(v / ((long long)a.nt[2] * a.nt[1]));
  T w0[RS_MAXT], w1[RS_MAXT], w2[RS_MAXT];
  long long o0[RS_MAXT], o1[RS_MAXT], o2[RS_MAXT];
  int s0[RS_MAXT], s1[RS_MAXT], s2[RS_MAXT];
  const int t0 = rs_taps<T>(a, 0, wx, (long long)a.ns[1] * a.ns[2], w0, o0, s0);
  const int t1 = rs_taps<T>(a, 1, wy, (long long)a.ns[2], w1, o1, s1);
  const int t2 = rs_taps<T>(a, 2, wz, 1, w2, o2, s2);
  const long long C = a.C;
  if constexpr (!ADJ) {
    const T *src = in + (long long)n * C * Vs;
    T *tgt = out + (long long)n * C * Vt + v;
    for (long long c = 0; c < C; ++c) {
      const T *sc = src + c * Vs;
      T acc = a.accumulate ? tgt[c * Vt] : T(0);
      // same order as the reference: z taps outer, x taps inner,
      // weight (wz * wy) * wx
      for (int k = 0; k < t2; ++k)
        for (int j = 0; j < t1; ++j) {
          const int syz = s2[k] * s1[j];
          const T wyz = w2[k] * w1[j];
          const long long oyz = o2[k] + o1[j];
          for (int i = 0; i < t0; ++i) {
            const int s = syz * s0[i];
            if (s) {
              const T val = sc[oyz + o0[i]];
              acc += (s < 0 ? -val : val) * (wyz * w0[i]);
            }
          }
        }
      tgt[c * Vt] = acc;
    }
  } else {
    const T *tg = in + (long long)n * C * Vt + v;
    T *src = out + (long long)n * C * Vs;
    for (int k = 0; k < t2; ++k)
      for (int j = 0; j < t1; ++j) {
        const int syz = s2[k] * s1[j];
        const T wyz = w2[k] * w1[j];
        const long long oyz = o2[k] + o1[j];
        for (int i = 0; i < t0; ++i) {
          const int s = syz * s0[i];
          if (!s) continue;
          const T wxyz = wyz * w0[i];
          for (long long c = 0; c < C; ++c) {
            const T val = tg[c * Vt] * wxyz;
            unsafeAtomicAdd(src + c * Vs + oyz + o0[i], s < 0 ? -val : val);
          }
        }
      }
  }
}

// One axis of the separable forward resize: in [A, nin, B] -> out [A, nout, B],
// out[a, j, b] = (accumulate ? out : 0) + sum_t w_t(j) s_t in[a, fold(lo_j + t), b].
// Lanes run along b (contiguous), so every tap is a coalesced row read.
template <typename T>
__global__ __launch_bounds__(RS_BLOCK) void resize_axis(const T *__restrict__ in, T *__restrict__ out,
                                                        long long A, long long B, RsArgs a, int d,
                                                        int accumulate) {
  const int nout = a.nt[d], nin = a.ns[d];
  const long long gid = (long long)blockIdx.x * RS_BLOCK + threadIdx.x;
  if (gid >= A * nout * B) return;
  const long long b = gid % B;
  const int j = (int)((gid / B) % nout);
  const long long o = gid / (B * nout);
  T w[RS_MAXT];
  long long off[RS_MAXT];
  int sg[RS_MAXT];
  const int nt = rs_taps<T>(a, d, j, B, w, off, sg);
  const T *src = in + o * nin * B + b;
  T acc = accumulate ? out[gid] : T(0);
  for (int t = 0; t < nt; ++t) {
    if (sg[t]) {
      const T v = src[off[t]];
      acc += (sg[t] < 0 ? -v : v) * w[t];
    }
  }
  out[gid] = acc;
}

// Logical block id with the blocks of each XCD contiguous: the hardware
// deals consecutive block ids round-robin over the 8 XCDs, so output rows
// that share input rows would otherwise fetch them through different L2s.
__device__ __forceinline__ unsigned rs_xcd_block() {
  const unsigned b = blockIdx.x, n = gridDim.x;
  const unsigned xcd = b % 8u, local = b / 8u, q = n / 8u, r = n % 8u;
  return xcd * q + (xcd < r ? xcd : r) + local;
}

// Tap table of one axis: for each target index j, RS_MAXT entries of folded
// source index (-1: no tap or sign 0, which the reference never reads) and
// weight times sign.
template <typename T>
__global__ __launch_bounds__(RS_BLOCK) void rs_table(RsArgs a, int d, T *__restrict__ tw, int *__restrict__ ti) {
  const int j = blockIdx.x * RS_BLOCK + threadIdx.x;
  if (j >= a.nt[d]) return;
  T w[RS_MAXT];
  long long off[RS_MAXT];
  int sg[RS_MAXT];
  const int nt = rs_taps<T>(a, d, j, 1, w, off, sg);
#pragma unroll
  for (int t = 0; t < RS_MAXT; ++t) {
    const bool on = t < nt && sg[t] != 0;
    tw[j * RS_MAXT + t] = on ? (sg[t] < 0 ? -w[t] : w[t]) : T(0);
    ti[j * RS_MAXT + t] = on ? (int)off[t] : -1;
  }
}

// The same pass for long rows (B >= 64): work-group row r = (a, j) is uniform,
// so its taps are read once from the table (scalar loads); lanes cover b.
template <typename T>
__global__ __launch_bounds__(RS_BLOCK) void resize_rows(const T *__restrict__ in, T *__restrict__ out, int nbx,
                                                        long long B, int nin, int nout, int ntap,
                                                        const T *__restrict__ tw, const int *__restrict__ ti,
                                                        int accumulate) {
  const unsigned blk = rs_xcd_block();
  const int row = (int)(blk / (unsigned)nbx);
  const long long b = (long long)(blk - (unsigned)row * (unsigned)nbx) * RS_BLOCK + threadIdx.x;
  if (b >= B) return;
  const int j = row % nout;
  const long long o = row / nout;
  const T *src = in + o * nin * B + b;
  T *dst = out + (long long)row * B + b;
  T acc = accumulate ? *dst : T(0);
  for (int t = 0; t < ntap; ++t) {
    const int i = ti[j * RS_MAXT + t];
    if (i >= 0) acc += src[(long long)i * B] * tw[j * RS_MAXT + t];
  }
  *dst = acc;
}

// Long rows with B % 4 == 0: four consecutive values per lane (16-byte
// loads and stores for float).
template <typename T>
__global__ __launch_bounds__(RS_BLOCK) void resize_rows4(const T *__restrict__ in, T *__restrict__ out, int nbx,
                                                         long long B, int nin, int nout, int ntap,
                                                         const T *__restrict__ tw, const int *__restrict__ ti,
                                                         int accumulate) {
  using V = HIP_vector_type<T, 4>;
  const unsigned blk = rs_xcd_block();
  const int row = (int)(blk / (unsigned)nbx);
  const long long b = ((long long)(blk - (unsigned)row * (unsigned)nbx) * RS_BLOCK + threadIdx.x) * 4;
  if (b >= B) return;
  const int j = row % nout;
  const long long o = row / nout;
  const T *src = in + o * nin * B + b;
  V *dst = (V *)(out + (long long)row * B + b);
  V acc = accumulate ? *dst : V(T(0));
  for (int t = 0; t < ntap; ++t) {
    const int i = ti[j * RS_MAXT + t];
    if (i >= 0) {
      const V v = *(const V *)(src + (long long)i * B);
      const T w = tw[j * RS_MAXT + t];
      acc.x += v.x * w; acc.y += v.y * w; acc.z += v.z * w; acc.w += v.w * w;
    }
  }
  *dst = acc;
}

// The contiguous axis (B == 1): a work-group stages `rows` whole input rows
// (one contiguous chunk) and the axis's tap table in LDS, then writes its
// rows x nout outputs as one contiguous chunk.
template <typename T>
__global__ __launch_bounds__(RS_BLOCK) void resize_contig(const T *__restrict__ in, T *__restrict__ out,
                                                          long long A, int rows, int nin, int nout, int ntap,
                                                          const T *__restrict__ tw, const int *__restrict__ ti,
                                                          int accumulate) {
  extern __shared__ char rs_smem[];
  T *lw = (T *)rs_smem;                                  // nout * RS_MAXT weights
  int *li = (int *)(lw + (size_t)nout * RS_MAXT);        // nout * RS_MAXT indices
  T *lx = (T *)(li + (size_t)nout * RS_MAXT + ((sizeof(T) == 8) ? ((nout * RS_MAXT) & 1) : 0));
  const long long r0 = (long long)blockIdx.x * rows;
  const int nr = (int)(A - r0 < rows ? A - r0 : rows);
  for (int k = threadIdx.x; k < nout * RS_MAXT; k += RS_BLOCK) { lw[k] = tw[k]; li[k] = ti[k]; }
  const T *src = in + r0 * nin;
  for (int k = threadIdx.x; k < nr * nin; k += RS_BLOCK) lx[k] = src[k];
  __syncthreads();
  T *dst = out + r0 * nout;
  for (int k = threadIdx.x; k < nr * nout; k += RS_BLOCK) {
    const int r = k / nout, j = k - r * nout;
    const T *x = lx + r * nin;
    T acc = accumulate ? dst[k] : T(0);
    for (int t = 0; t < ntap; ++t) {
      const int i = li[j * RS_MAXT + t];
      if (i >= 0) acc += x[i] * lw[j * RS_MAXT + t];
    }
    dst[k] = acc;
  }
}

// Short rows (B < 64) with fewer than 2^31 outputs: 32-bit index math.
template <typename T>
__global__ __launch_bounds__(RS_BLOCK) void resize_short(const T *__restrict__ in, T *__restrict__ out, int total,
                                                         int B, int nin, int nout, int ntap,
                                                         const T *__restrict__ tw, const int *__restrict__ ti,
                                                         int accumulate) {
  const int gid = blockIdx.x * RS_BLOCK + threadIdx.x;
  if (gid >= total) return;
  int b = 0, r = gid;
  if (B > 1) { b = gid % B; r = gid / B; }
  const int j = r % nout, o = r / nout;
  const T *src = in + ((long long)o * nin) * B + b;
  T acc = accumulate ? out[gid] : T(0);
  for (int t = 0; t < ntap; ++t) {
    const int i = ti[j * RS_MAXT + t];
    if (i >= 0) acc += src[(long long)i * B] * tw[j * RS_MAXT + t];
  }
  out[gid] = acc;
}

template <typename T>
__global__ __launch_bounds__(RS_BLOCK) void rs_fill(T *__restrict__ p, long long n, T v) {
  const long long i = (long long)blockIdx.x * RS_BLOCK + threadIdx.x;
  if (i < n) p[i] = v;
}

template <typename T>
__global__ __launch_bounds__(RS_BLOCK) void rs_scale(T *__restrict__ p, long long n, T f) {
  const long long i = (long long)blockIdx.x * RS_BLOCK + threadIdx.x;
  if (i < n) p[i] *= f;
}

static unsigned rs_blocks(long long n) { return (unsigned)((n + RS_BLOCK - 1) / RS_BLOCK); }

// shift and scale of one axis (resize_common.cpp:1548-1567); GridAlignType
// edge = 0, center = 1, first = 2, last = 3
static void rs_affine(double f, double Ds, double Dt, int mode, double &shift, double &scale) {
  shift = 0.;
  scale = 1. / f;
  switch (mode) {
    case 0: shift = 0.5 * (Ds / Dt - 1); scale = Ds / Dt; break;
    case 1: shift = 0.; scale = (Ds - 1) / (Dt - 1); break;
    case 3: shift = f * (Ds - 1) / (Dt - 1); break;
    default: break;
  }
}

// Forward resize as separable passes x -> y -> z (axes of size 1 on both
// sides are skipped): each pass streams its input once with coalesced tap
// rows, instead of one lane gathering (O+1)^3 taps per channel from three
// strided axes.  Intermediates come from a stream-ordered allocation; false
// if it fails (the caller then uses the direct kernel).
template <typename T>
static bool rs_separable(const T *input, T *output, const RsArgs &a, hipStream_t st) {
  int axes[3], np = 0;
  for (int d = 0; d < 3; ++d)
    if (!(a.ns[d] == 1 && a.nt[d] == 1)) axes[np++] = d;
  if (np == 0) return false;
  const long long NC = (long long)a.N * a.C;
  long long cur[3] = {a.ns[0], a.ns[1], a.ns[2]};
  // sizes of the intermediates (after each pass but the last)
  long long tmp_elems[2] = {0, 0};
  {
    long long c[3] = {a.ns[0], a.ns[1], a.ns[2]};
    for (int p = 0; p + 1 < np; ++p) {
      c[axes[p]] = a.nt[axes[p]];
      tmp_elems[p % 2] = std::max(tmp_elems[p % 2], NC * c[0] * c[1] * c[2]);
    }
  }
  // buffer: the two intermediates, then per pass a tap table of nt[d] x
  // RS_MAXT weights and as many int indices
  long long tab_w[3], tab_i[3], tot = tmp_elems[0] + tmp_elems[1];
  for (int p = 0; p < np; ++p) {
    tab_w[p] = tot;
    tot += (long long)a.nt[axes[p]] * RS_MAXT;
    tab_i[p] = tot;
    tot += ((long long)a.nt[axes[p]] * RS_MAXT * sizeof(int) + sizeof(T) - 1) / sizeof(T);
  }
  T *buf = nullptr;
  if (scratch_alloc((void **)&buf, (size_t)tot * sizeof(T), st) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  T *tmp[2] = {buf, buf + tmp_elems[0]};
  for (int p = 0; p < np; ++p)
    hipLaunchKernelGGL(rs_table<T>, dim3(rs_blocks(a.nt[axes[p]])), dim3(RS_BLOCK), 0, st, a, axes[p],
                       buf + tab_w[p], (int *)(buf + tab_i[p]));
  const T *src = input;
  for (int p = 0; p < np; ++p) {
    const int d = axes[p];
    long long A = NC, B = 1;
    for (int e = 0; e < d; ++e) A *= cur[e];
    for (int e = d + 1; e < 3; ++e) B *= cur[e];
    const bool last = p + 1 == np;
    T *dst = last ? output : tmp[p % 2];
    const long long n = A * a.nt[d] * B;
    const int acc = last ? a.accumulate : 0;
    const long long nbx = (B + RS_BLOCK - 1) / RS_BLOCK;
    const T *tw = buf + tab_w[p];
    const int *ti = (const int *)(buf + tab_i[p]);
    const int ntap = a.order[d] + 1;
    const long long nbx4 = (B / 4 + RS_BLOCK - 1) / RS_BLOCK;
    // contiguous axis: rows of nin inputs staged in LDS (about 16 KB of them)
    const int crows = (int)std::max<long long>(1, std::min<long long>(A, 16384 / ((long long)a.ns[d] * sizeof(T))));
    const size_t clds = (size_t)a.nt[d] * RS_MAXT * (sizeof(T) + sizeof(int)) + sizeof(T) +
                        (size_t)crows * a.ns[d] * sizeof(T);
    // 4-wide accesses need both base pointers aligned to the vector (a
    // caller's view may start at any element)
    const bool al4 = ((uintptr_t)src % (4 * sizeof(T))) == 0 && ((uintptr_t)dst % (4 * sizeof(T))) == 0;
    if (B >= 64 && B % 4 == 0 && al4 && A * a.nt[d] * nbx4 < (1LL << 31))
      hipLaunchKernelGGL(resize_rows4<T>, dim3((unsigned)(A * a.nt[d] * nbx4)), dim3(RS_BLOCK), 0, st, src, dst,
                         (int)nbx4, B, a.ns[d], a.nt[d], ntap, tw, ti, acc);
    else if (B >= 64 && A * a.nt[d] * nbx < (1LL << 31))
      hipLaunchKernelGGL(resize_rows<T>, dim3((unsigned)(A * a.nt[d] * nbx)), dim3(RS_BLOCK), 0, st, src, dst,
                         (int)nbx, B, a.ns[d], a.nt[d], ntap, tw, ti, acc);
    else if (B == 1 && clds <= 32768 && (A + crows - 1) / crows < (1LL << 31) &&
             (long long)crows * std::max(a.ns[d], a.nt[d]) < (1LL << 30))
      hipLaunchKernelGGL(resize_contig<T>, dim3((unsigned)((A + crows - 1) / crows)), dim3(RS_BLOCK), clds, st,
                         src, dst, A, crows, a.ns[d], a.nt[d], ntap, tw, ti, acc);
    else if (n < (1LL << 31) - RS_BLOCK)
      hipLaunchKernelGGL(resize_short<T>, dim3(rs_blocks(n)), dim3(RS_BLOCK), 0, st, src, dst, (int)n, (int)B,
                         a.ns[d], a.nt[d], ntap, tw, ti, acc);
    else
      hipLaunchKernelGGL(resize_axis<T>, dim3(rs_blocks(n)), dim3(RS_BLOCK), 0, st, src, dst, A, B, a, d, acc);
    cur[d] = a.nt[d];
    src = dst;
  }
  (void)hipFreeAsync(buf, st);
  return true;
}

// Voxel coordinates A [x y z] + t of a lattice: out[b, x, y, z, :], mat[b] =
// [A | t] (3 x 4).  Products and sums in double, rounded once; bound by the
// store of 3 values a voxel (181 x 217 x 181: 0.03 ms, where the same grid
// from elementwise and reduction passes took 0.36).
template <typename T>
__global__ __launch_bounds__(RS_BLOCK) void affine_lattice(const T *__restrict__ mat, T *__restrict__ out, int nx,
                                                           int ny, int nz, long long nvox) {
  const long long v = (long long)blockIdx.x * RS_BLOCK + threadIdx.x;
  if (v >= nvox) return;
  const unsigned V = (unsigned)nx * (unsigned)ny * (unsigned)nz;   // < 2^31 (checked by the caller)
  const long long b = v / V;
  const unsigned w = (unsigned)(v - b * V);
  const unsigned z = w % (unsigned)nz, r = w / (unsigned)nz;
  const double p[3] = {(double)(r / (unsigned)ny), (double)(r % (unsigned)ny), (double)z};
  const T *m = mat + b * 12;
  T *o = out + v * 3;
#pragma unroll
  for (int d = 0; d < 3; ++d)
    o[d] = (T)((double)m[4 * d] * p[0] + (double)m[4 * d + 1] * p[1] + (double)m[4 * d + 2] * p[2] +
               (double)m[4 * d + 3]);
}

// ---------------------------------------------------------------------------
// Forward resize of a 3-D volume in one pass.
//
// A work-group owns TXO x 8 x 32 outputs of one channel, one (y, z) position a
// thread.  It walks the source planes that its outputs' x taps use: stages the
// rows and columns of the plane that the y and z taps use (the next plane's
// loads in flight meanwhile), sums along z into LDS, along y into one value a
// thread, and adds that to the accumulators of the outputs that use the plane.
// The source is read once (plus the tiles' halos, mostly from L2) and the
// result written once: 1.02 GB for the half-size cubic resize of 4 x 8 x 192^3
// (0.21 ms at the rate of a large copy), where a pass an axis moves 2.4 GB:
// 0.27 against 0.65 ms.
//
// Which planes, rows and columns the taps use (folding and wrapping included)
// is a bitmap a axis; a set bit's rank is its place in the staged lists.
// ---------------------------------------------------------------------------
#define RF_OY 8
#define RF_OZ 32
#define RF_STAGE 2048   // staged values of a plane
#define RF_WORDS 64     // bitmap words an axis: source axes up to 2048

// Lattice positions that `cnt` consecutive outputs' taps can use.
static int rf_extent(const RsArgs &a, int d, int cnt) {
  const int nt = a.order[d] + 1;
  cnt = std::min(cnt, a.nt[d]);
  const double span = (cnt - 1) * std::fabs(a.scale[d]) + 2 + nt;
  return (int)std::min<double>(std::min<double>(span, (double)cnt * nt), a.ns[d]);
}

template <typename T, int TXO, int MT>
__global__ __launch_bounds__(RS_BLOCK) void resize_fused(const T *__restrict__ in, T *__restrict__ out, RsArgs a,
                                                         int ntx, int nty, int ntz) {
  __shared__ T stage[RF_STAGE];
  __shared__ T tz[RF_OY * MT * RF_OZ];
  __shared__ T wx[TXO * MT * TXO];
  __shared__ unsigned xmask[TXO * MT];
  __shared__ int list[3][RF_OZ * MT];
  __shared__ unsigned bits[3][RF_WORDS];
  __shared__ int base[3][RF_WORDS + 1];
  unsigned r = rs_xcd_block();
  const int bz = (int)(r % (unsigned)ntz); r /= (unsigned)ntz;
  const int by = (int)(r % (unsigned)nty); r /= (unsigned)nty;
  const int bx = (int)(r % (unsigned)ntx);
  const long long nc = r / (unsigned)ntx;
  const int t = threadIdx.x, lz = t % RF_OZ, ly = t / RF_OZ;
  const int oz = bz * RF_OZ + lz, oy = by * RF_OY + ly, ox0 = bx * TXO;
  const bool vz = oz < a.nt[2], vy = oy < a.nt[1];

  // ---- taps: this thread's along z and y, and of output plane t along x ----
  T wz[MT], wy[MT], wxt[MT];
  int iz[MT], iy[MT], ix[MT];
  auto taps = [&](int d, int w, bool on, T (&wt)[MT], int (&it)[MT]) {
    T w8[RS_MAXT];
    long long o8[RS_MAXT];
    int s8[RS_MAXT];
    const int n = on ? rs_taps<T>(a, d, w, 1, w8, o8, s8) : 0;
#pragma unroll
    for (int k = 0; k < MT; ++k) {
      const bool use = k < n && s8[k] != 0;   // (a tap of sign 0 is never read)
      it[k] = use ? (int)o8[k] : -1;
      wt[k] = use ? (s8[k] < 0 ? -w8[k] : w8[k]) : T(0);
    }
  };
  taps(2, oz, vz, wz, iz);
  taps(1, oy, vy, wy, iy);
  const bool isx = t < TXO && ox0 + t < a.nt[0];
  taps(0, ox0 + t, isx, wxt, ix);

  // ---- lists of used planes, rows and columns ----
  for (int k = t; k < 3 * RF_WORDS; k += RS_BLOCK) ((unsigned *)bits)[k] = 0u;
  for (int k = t; k < TXO * MT * TXO; k += RS_BLOCK) wx[k] = T(0);
  for (int k = t; k < TXO * MT; k += RS_BLOCK) xmask[k] = 0u;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < MT; ++k) {
    if (ly == 0 && iz[k] >= 0) atomicOr(&bits[2][iz[k] >> 5], 1u << (iz[k] & 31));
    if (lz == 0 && iy[k] >= 0) atomicOr(&bits[1][iy[k] >> 5], 1u << (iy[k] & 31));
    if (ix[k] >= 0) atomicOr(&bits[0][ix[k] >> 5], 1u << (ix[k] & 31));
  }
  __syncthreads();
  if (t < 3 * 64) {   // one wave an axis: ranks of the words, then the lists
    const int d = t >> 6, l = t & 63;
    unsigned b = bits[d][l];
    int inc = __popc(b);
    const int own = inc;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int u = __shfl_up(inc, o, 64);
      if (l >= o) inc += u;
    }
    base[d][l] = inc - own;
    if (l == 63) base[d][64] = inc;
    for (int at = inc - own; b; ++at) {
      const int j = __ffs((int)b) - 1;
      list[d][at] = l * 32 + j;
      b &= b - 1u;
    }
  }
  __syncthreads();
  auto rank = [&](int d, int i) { return base[d][i >> 5] + __popc(bits[d][i >> 5] & ((1u << (i & 31)) - 1u)); };
#pragma unroll
  for (int k = 0; k < MT; ++k) {
    if (iz[k] >= 0) iz[k] = rank(2, iz[k]);
    if (iy[k] >= 0) iy[k] = rank(1, iy[k]);
    if (ix[k] >= 0) {   // (one thread an output: no two write one weight)
      const int at = rank(0, ix[k]);
      wx[at * TXO + t] += wxt[k];
      atomicOr(&xmask[at], 1u << t);
    }
  }
  const int np = base[0][64], ny = base[1][64], nz = base[2][64];
  __syncthreads();

  // ---- staged elements of this thread: offsets within a source plane ----
  constexpr int NL = RF_STAGE / RS_BLOCK;
  const int cnt = ny * nz;
  const float rz = 1.f / (float)nz;
  int off[NL];
#pragma unroll
  for (int k = 0; k < NL; ++k) {
    const int e = t + k * RS_BLOCK;
    int row = (int)((float)e * rz);   // floor(e / nz): within 1, fixed up
    row -= row * nz > e;
    row += (row + 1) * nz <= e;
    off[k] = e < cnt ? list[1][row] * a.ns[2] + list[2][e - row * nz] : -1;
  }
  const long long plane = (long long)a.ns[1] * a.ns[2];
  const T *src = in + nc * a.ns[0] * plane;
  T pre[NL], acc[TXO];
#pragma unroll
  for (int j = 0; j < TXO; ++j) acc[j] = T(0);
  auto fetch = [&](int pi) {
    const T *sp = src + list[0][pi] * plane;
#pragma unroll
    for (int k = 0; k < NL; ++k) pre[k] = off[k] >= 0 ? sp[off[k]] : T(0);
  };
  if (np > 0) fetch(0);
  for (int pi = 0; pi < np; ++pi) {
#pragma unroll
    for (int k = 0; k < NL; ++k)
      if (off[k] >= 0) stage[t + k * RS_BLOCK] = pre[k];
    __syncthreads();
    if (pi + 1 < np) fetch(pi + 1);
    for (int row = ly; row < ny; row += RF_OY) {
      T v = T(0);
#pragma unroll
      for (int k = 0; k < MT; ++k)
        if (iz[k] >= 0) v += stage[row * nz + iz[k]] * wz[k];
      tz[row * RF_OZ + lz] = v;
    }
    __syncthreads();
    T v = T(0);
#pragma unroll
    for (int k = 0; k < MT; ++k)
      if (iy[k] >= 0) v += tz[iy[k] * RF_OZ + lz] * wy[k];
    const unsigned m = xmask[pi];
    // (an output that does not use the plane must not see it: it may hold a NaN)
#pragma unroll
    for (int j = 0; j < TXO; ++j)
      if ((m >> j) & 1u) acc[j] += v * wx[pi * TXO + j];
  }
  if (!vz || !vy) return;
  T *dst = out + ((nc * a.nt[0] + ox0) * a.nt[1] + oy) * (long long)a.nt[2] + oz;
  const long long oplane = (long long)a.nt[1] * a.nt[2];
#pragma unroll
  for (int j = 0; j < TXO; ++j)
    if (ox0 + j < a.nt[0]) dst[j * oplane] = a.accumulate ? dst[j * oplane] + acc[j] : acc[j];
}

// Estimated time of a pass an axis, in us: elements written and taps, by the
// kernel that the length and alignment of the rows select (16-byte rows, rows,
// the contiguous axis, short rows), and never less than its six launches.
template <typename T>
static double rs_passes_time(const RsArgs &a, bool aligned) {
  static const double f32[4][2] = {{1.8, 0.19}, {2.4, 0.61}, {1.6, 1.1}, {0, 0.37}};
  static const double f64[4][2] = {{2.2, 0.44}, {2.8, 0.66}, {3.1, 1.5}, {0, 0.19}};
  const bool f = sizeof(T) == 4;
  double us = f ? 35 : 30, n = 1e-6 * a.N * a.C * (double)a.ns[0] * a.ns[1] * a.ns[2];
  for (int d = 0; d < 3; ++d) {
    long long B = 1;
    for (int e = d + 1; e < 3; ++e) B *= a.ns[e];
    n = n / a.ns[d] * a.nt[d];
    const int kind = B >= 64 ? (B % 4 == 0 && aligned ? 0 : 1) : B == 1 ? 2 : 3;
    const double(&c)[2] = (f ? f32 : f64)[kind];
    us += n * (c[0] + c[1] * (a.order[d] + 1));
  }
  return std::max(us, 57.);
}

// Estimated time of resize_fused: per work-group, per plane that it walks, and
// per plane for the rows summed along z, the values staged and the outputs
// accumulated.
template <typename T>
static double rf_time(const RsArgs &a, bool wide, int txo, long long nb) {
  // us per million: work-groups, planes, z rows / 8, values / 256, outputs, tap weights; us a launch
  static const double cost[2][2][7] = {{{0, 270, 180, 16, 5, 12, 15}, {4000, 220, 200, 52, 23, 21, 25}},
                                       {{520, 750, 230, 21, 0, 18, 8}, {4300, 0, 150, 45, 140, 68, 27}}};
  const double(&c)[7] = cost[sizeof(T) == 8][wide];
  const double b = 1e-6 * nb, np = rf_extent(a, 0, txo), ny = rf_extent(a, 1, RF_OY), nz = rf_extent(a, 2, RF_OZ);
  return b * (c[0] + c[5] * txo * txo + np * (c[1] + c[2] * std::ceil(ny / RF_OY) + c[3] * ny * nz / RS_BLOCK +
                                              c[4] * txo)) + c[6];
}

// One launch when the taps of a tile fit what the kernel stages: 3-D volumes
// resized by a factor of about a third or more (2048 staged values: 8 x 32
// outputs of a cubic half-size resize use 19 x 67), axes up to 2048, a sane
// affine map -- and the tiles are not mostly idle: a block has 8 x 32 rows of
// outputs whatever the volume, so that very many small or flat volumes take a
// pass an axis sooner (16384 x 2 volumes of 4^3 to 2^3, order 3: 0.23 ms fused,
// 0.06 not), and so do double volumes above order 3, where a plane's 16
// outputs a thread cost most (512 x 512 x 24 by 1.5: 0.69 and 0.36).  The
// choice compares the two estimates, which were fitted to 1335 resizes (14
// lattices, 13 factors, orders 0 to 7, both types), four in five within 15 %.
// Of the 203 that the kernel would slow down by more than 5 % it leaves 13; of
// 1068 on other lattices, 8 (at worst 0.27 -> 0.38 ms, 20000 volumes of 6^3
// doubled, order 3).
// False otherwise (the caller then runs a pass an axis).
template <typename T>
static bool rs_fused(const T *input, T *output, const RsArgs &a, hipStream_t st) {
  for (int d = 0; d < 3; ++d)
    if (a.ns[d] > 32 * RF_WORDS || a.nt[d] < 2 || !(std::fabs(a.scale[d]) < 1e3) || !(std::fabs(a.shift[d]) < 1e6))
      return false;
  if ((long long)rf_extent(a, 1, RF_OY) * rf_extent(a, 2, RF_OZ) > RF_STAGE) return false;
  const int nty = (a.nt[1] + RF_OY - 1) / RF_OY, ntz = (a.nt[2] + RF_OZ - 1) / RF_OZ;
  const bool wide = a.order[0] > 3 || a.order[1] > 3 || a.order[2] > 3;
  // 16 output planes a work-group re-read the fewest source planes; small
  // volumes take 4, for more work-groups (each walks its planes in turn)
  const long long per = (long long)a.N * a.C * nty * ntz;
  const bool tall = per * ((a.nt[0] + 15) / 16) >= 1024;
  const int txo = tall ? 16 : 4;
  const int ntx = (a.nt[0] + txo - 1) / txo;
  const long long nb = per * ntx;
  const bool aligned = ((uintptr_t)input | (uintptr_t)output) % (4 * sizeof(T)) == 0;
  if (!launch_fits(nb, RS_BLOCK) || rf_time<T>(a, wide, txo, nb) >= rs_passes_time<T>(a, aligned)) return false;
  const dim3 g((unsigned)nb), b(RS_BLOCK);
#define RF_LAUNCH(TX, M) \
  hipLaunchKernelGGL((resize_fused<T, TX, M>), g, b, 0, st, input, output, a, ntx, nty, ntz)
  if (tall) {
    if (wide) RF_LAUNCH(16, 8);
    else RF_LAUNCH(16, 4);
  } else {
    if (wide) RF_LAUNCH(4, 8);
    else RF_LAUNCH(4, 4);
  }
#undef RF_LAUNCH
  return true;
}

template <typename T>
static void rs_launch(const T *input, T *output, const RsArgs &a, bool adjoint, hipStream_t st) {
  const long long Vt = (long long)a.nt[0] * a.nt[1] * a.nt[2];
  const long long nthreads = (long long)a.N * Vt;
  if (adjoint) {
    const long long ns = (long long)a.N * a.C * a.ns[0] * a.ns[1] * a.ns[2];
    hipLaunchKernelGGL(rs_fill<T>, dim3(rs_blocks(ns)), dim3(RS_BLOCK), 0, st, output, ns, T(0));
    hipLaunchKernelGGL((resize_kernel<T, true>), dim3(rs_blocks(nthreads)), dim3(RS_BLOCK), 0, st, input, output, a);
  } else if (!rs_fused<T>(input, output, a, st) && !rs_separable<T>(input, output, a, st)) {
    hipLaunchKernelGGL((resize_kernel<T, false>), dim3(rs_blocks(nthreads)), dim3(RS_BLOCK), 0, st, input, output, a);
  }
}

}  // namespace ni_amd

using namespace ni_amd;

extern "C" {

int ni_resize(int32_t dtype, int32_t dim, int64_t N, int64_t C, const int64_t *in_shape, const int64_t *out_shape,
              const double *factor, const int32_t *bound, const int32_t *order, const int32_t *mode,
              int32_t do_adjoint, int32_t normalize, int32_t accumulate, const void *input, void *output,
              void *stream) {
  set_error("");
  NI_CHECK(in_shape && out_shape && factor && bound && order && mode && input && output, "resize: missing argument");
  NI_CHECK(dim >= 1 && dim <= 3, "resize: expected a 1D, 2D or 3D tensor (got %d spatial dims)", dim);
  NI_CHECK(dtype == NI_FLOAT32 || dtype == NI_FLOAT64, "resize: unsupported dtype %d", dtype);
  NI_CHECK(N > 0 && C > 0, "resize: expected a non empty tensor");
  RsArgs a;
  a.N = (int)N;
  a.C = (int)C;
  // the isotropic nearest / linear kernels (and quadratic in 3-D) overwrite
  // a given output, the others add into it (resize_common.cpp:440-530)
  const bool iso = order[0] == order[1] && order[0] == order[2];
  const bool overwrite = iso && (order[0] <= 1 || (order[0] == 2 && dim == 3));
  a.accumulate = (do_adjoint || overwrite) ? 0 : (accumulate != 0);
  a.nearest_dbl = iso && order[0] == 0;
  // source / target (resize.cpp:52-53)
  const int64_t *ss = do_adjoint ? out_shape : in_shape;
  const int64_t *ts = do_adjoint ? in_shape : out_shape;
  double f[3], shift[3], scale[3];
  f[0] = factor[0]; f[1] = factor[1]; f[2] = factor[2];
  for (int d = 0; d < 3; ++d) {
    if (do_adjoint) f[d] = 1. / f[d];
    const double Ds = d < dim ? (double)ss[d] : 1., Dt = d < dim ? (double)ts[d] : 1.;
    NI_CHECK(Ds > 0 && Dt > 0, "resize: expected a non empty tensor");
    rs_affine(f[d], Ds, Dt, mode[d], shift[d], scale[d]);
    NI_CHECK(order[d] >= 0 && order[d] <= 7, "resize: interpolation order %d not in 0..7", order[d]);
    if (d < dim) {
      a.ns[d] = (int)ss[d];
      a.nt[d] = (int)ts[d];
      a.bound[d] = bound[d];
      a.order[d] = order[d];
      a.shift[d] = shift[d];
      a.scale[d] = scale[d];
    } else {
      // axes the reference's 1-D / 2-D kernels do not touch: identity
      a.ns[d] = a.nt[d] = 1;
      a.bound[d] = B_DCT2;
      a.order[d] = 0;
      a.shift[d] = 0.;
      a.scale[d] = 1.;
    }
  }
  hipStream_t st = (hipStream_t)stream;
  if (dtype == NI_FLOAT32) rs_launch<float>((const float *)input, (float *)output, a, do_adjoint != 0, st);
  else rs_launch<double>((const double *)input, (double *)output, a, do_adjoint != 0, st);
  NI_HIP_CHECK(hipGetLastError());
  if (normalize) {
    double m = scale[0] * scale[1] * scale[2];   // 3-D (the switch's default)
    if (dim == 2) m *= scale[0] * scale[1];
    if (dim == 1) m *= scale[0] * (scale[0] * scale[1]);
    const int64_t *os = do_adjoint ? ss : ts;
    long long n = N * C;
    for (int d = 0; d < dim; ++d) n *= os[d];
    if (dtype == NI_FLOAT32)
      hipLaunchKernelGGL(rs_scale<float>, dim3(rs_blocks(n)), dim3(RS_BLOCK), 0, st, (float *)output, n, (float)m);
    else
      hipLaunchKernelGGL(rs_scale<double>, dim3(rs_blocks(n)), dim3(RS_BLOCK), 0, st, (double *)output, n, m);
    NI_HIP_CHECK(hipGetLastError());
  }
  return 0;
}

int ni_affine_grid(int32_t dtype, int64_t nbatch, const int64_t *shape, const void *mat, void *out, void *stream) {
  set_error("");
  NI_CHECK(shape && mat && out, "affine_grid: missing argument");
  NI_CHECK(dtype == NI_FLOAT32 || dtype == NI_FLOAT64, "affine_grid: unsupported dtype %d", dtype);
  long long V = 1;
  for (int d = 0; d < 3; ++d) {
    NI_CHECK(shape[d] >= 0 && shape[d] < (1LL << 31), "affine_grid: bad size %lld", (long long)shape[d]);
    V *= shape[d];
    NI_CHECK(V < (1LL << 31), "affine_grid: lattice too large");
  }
  const long long n = nbatch * V;
  if (n <= 0) return 0;
  NI_CHECK(launch_fits((n + RS_BLOCK - 1) / RS_BLOCK, RS_BLOCK), "affine_grid: lattice too large");
  hipStream_t st = (hipStream_t)stream;
  if (dtype == NI_FLOAT32)
    hipLaunchKernelGGL(affine_lattice<float>, dim3(rs_blocks(n)), dim3(RS_BLOCK), 0, st, (const float *)mat,
                       (float *)out, (int)shape[0], (int)shape[1], (int)shape[2], n);
  else
    hipLaunchKernelGGL(affine_lattice<double>, dim3(rs_blocks(n)), dim3(RS_BLOCK), 0, st, (const double *)mat,
                       (double *)out, (int)shape[0], (int)shape[1], (int)shape[2], n);
  NI_HIP_CHECK(hipGetLastError());
  return 0;
}

}  // extern "C"
