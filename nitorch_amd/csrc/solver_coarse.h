// The coarse end of the multigrid pyramid in one launch.
//
// Levels of at most CoarseCfg<T>::LIM voxels hold too little work to fill a
// chip: run kernel by kernel, a relaxation of one (14 launches for 4 PCG
// steps) takes about 5 us a launch whatever its size, and a full multigrid
// pass visits these levels most often.  Here one work-group a batch element
// keeps the level it works on in LDS and registers and runs every V-cycle
// below the first such level -- relaxation, residual, restriction,
// prolongation -- between barriers.  PCG: 160 x 192 x 160 (four such
// levels), 2 cycles of 4 steps: 15.8 -> 11.4 ms a solve, of which 2.4 ms here (9
// launches instead of about 1500).  Gauss-Seidel: 63 x 77 x 58, 2 cycles of 2
// sweeps: 6.00 -> 5.16 ms, of which 2.2 ms here: a class step (about 1.1 us)
// is one wavefront's 25 taps and their latency; reading what the next class
// needs beside the solution before the barrier took it from 5.38 to 5.16.
//
// Formulas are those of the per-level kernels (pcg_*, relax_small,
// reg_kernel, transfer_kernel); sums over voxels differ by their order.
#pragma once

#define CO_LEVELS 5     // levels a launch handles
#define CO_CLASSES 128  // Gauss-Seidel classes of a level, at most
#define CO_AXES 64      // X + Y + Z of a level, at most (transfer tables)
#define CO_WORDS 13     // words of a voxel's stencil: 25 neighbours, 16 bits each

// Voxels of a level (the stencil tables and, with Gauss-Seidel, g and H of the
// level fit LDS), and threads: few enough that a thread's voxels' PCG state
// and a stencil's 75 values fit its registers.
template <typename T>
struct CoarseCfg {
  static constexpr int LIM = sizeof(T) == 4 ? 1200 : 600;
  static constexpr int NTH = sizeof(T) == 4 ? 512 : 256;
  static constexpr int VPT = (LIM + NTH - 1) / NTH;
  static constexpr int TAB = LIM + LIM / 4 + CO_LEVELS;   // voxels of all levels (each at most ceil(1/2) an axis)
};

template <typename T>
struct CoarseLevel {
  int X, Y, Z;
  const T *h;       // [N, CC, V]
  T *g, *x;         // [N, 3, V]
  StencilT<T> S;
};

// What every launch on a pyramid needs, in device memory (scalar loads; as a
// kernel argument, indexing it by level would copy it to scratch).
template <typename T>
struct CoarseArgs {
  int nl, CC, nb_iter;
  int b[3];
  CoarseLevel<T> L[CO_LEVELS];
  ColourPlan P[CO_LEVELS];   // Gauss-Seidel
};

template <typename T>
__global__ void coarse_write(CoarseArgs<T> *dst, CoarseArgs<T> src) {
  *dst = src;
}

// Shared state of a work-group.  `u` holds the field that the next stencil or
// transfer reads, a voxel's components together (one 16-byte read); `nb` the
// neighbours of every voxel of every level ((voxel << 2) | (sign + 1), two a
// word), folded once a launch: computing them at each use took four times the
// stencil's own arithmetic.  With Gauss-Seidel, `gh` holds the level's g and
// H, mem / cls the members of each class of every level.
template <typename T>
struct __align__(4 * sizeof(T)) Co4 {
  T x, y, z, w;
};

// Taps of the transfers between levels l and l + 1 along each axis (x, y, z
// coordinates in turn): weights and (offset << 2) | (sign + 1) in the source
// level.  Their double divisions, at each use, took longer than a relaxation.
template <typename T>
struct CoTaps {
  T dw[CO_AXES][4], uw[CO_AXES][3];                       // down: restriction, up: prolongation
  unsigned short df[CO_AXES][4], uf[CO_AXES][3];
};

template <typename T, bool CG>
struct CoarseLds {
  Co4<T> u[CoarseCfg<T>::LIM];
  CoTaps<T> taps[CO_LEVELS - 1];
  unsigned nb[CO_WORDS * CoarseCfg<T>::TAB];
  double red[2][CoarseCfg<T>::NTH / 64];
  T gh[CG ? 1 : 9 * CoarseCfg<T>::LIM];
  unsigned short mem[CG ? 1 : CoarseCfg<T>::TAB];
  int cls[CG ? 1 : CO_LEVELS][CG ? 1 : CO_CLASSES + 1];
  int cnt[CG ? 1 : CO_CLASSES];
};

// Place of displacement (i, j, k) among the 25 of the stencil.
__host__ __device__ constexpr int co_place(int i, int j, int k) {
  if (j == 0 && k == 0) return i == 0 ? 0 : i == -1 ? 1 : i == 1 ? 2 : i == -2 ? 7 : 8;
  if (i == 0 && k == 0) return j == -1 ? 3 : j == 1 ? 4 : j == -2 ? 9 : 10;
  if (i == 0 && j == 0) return k == -1 ? 5 : k == 1 ? 6 : k == -2 ? 11 : 12;
  if (k == 0) return 13 + (i > 0) + 2 * (j > 0);
  if (j == 0) return 17 + (i > 0) + 2 * (k > 0);
  return 21 + (j > 0) + 2 * (k > 0);
}

// Neighbour words of voxel v of a level (written at nb[word * TAB + at]).
template <typename T>
__device__ __forceinline__ void co_neighbours(unsigned *nb, const CoarseLevel<T> &L, const int *bound, int v) {
  const int sz[3] = {L.X, L.Y, L.Z}, st[3] = {L.Y * L.Z, L.Z, 1};
  const int co[3] = {v / st[0], (v / L.Z) % L.Y, v % L.Z};
  int of[3][5], sg[3][5];
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int t = 0; t < 5; ++t) of[d][t] = fold<int>(bound[d], co[d] + t - 2, sz[d], sg[d][t]) * st[d];
  unsigned e[2 * CO_WORDS];
  e[25] = 0;
#pragma unroll
  for (int i = -2; i <= 2; ++i)
#pragma unroll
    for (int j = -2; j <= 2; ++j)
#pragma unroll
      for (int k = -2; k <= 2; ++k) {
        const int ai = i < 0 ? -i : i, aj = j < 0 ? -j : j, ak = k < 0 ? -k : k;
        if (ai + aj + ak > 2 || (ai && aj && ak)) continue;
        const int s = sg[0][i + 2] * sg[1][j + 2] * sg[2][k + 2];
        e[co_place(i, j, k)] = (unsigned)(((of[0][i + 2] + of[1][j + 2] + of[2][k + 2]) << 2) | (s + 1));
      }
#pragma unroll
  for (int w = 0; w < CO_WORDS; ++w) nb[w * CoarseCfg<T>::TAB] = e[2 * w] | (e[2 * w + 1] << 16);
}

// Work-group sum of v in double (two buffers in turn: a barrier a call).
template <int NTH>
__device__ __forceinline__ double co_sum(double v, double (*red)[NTH / 64], int &flip) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) red[flip][threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0;
#pragma unroll
  for (int k = 0; k < NTH / 64; ++k) s += red[flip][k];
  flip ^= 1;
  return s;
}

// (L u) of the voxel with neighbour words e, its own values in own.
template <typename T>
__device__ __forceinline__ void co_stencil(const Co4<T> *u, const unsigned (&e)[CO_WORDS], bool signs,
                                           const StencilT<T> &S, T (&own)[3], T (&out)[3]) {
  T val[25][3];
#pragma unroll
  for (int w = 0; w < CO_WORDS; ++w) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int q = 2 * w + h;
      if (q >= 25) break;
      const unsigned f = h ? e[w] >> 16 : e[w] & 0xffffu;
      const Co4<T> c = u[f >> 2];
      val[q][0] = c.x;
      val[q][1] = c.y;
      val[q][2] = c.z;
      if (signs && q) {
        const int s = (int)(f & 3u) - 1;
#pragma unroll
        for (int d = 0; d < 3; ++d) val[q][d] = s == 0 ? T(0) : (s < 0 ? -val[q][d] : val[q][d]);
      }
    }
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) own[d] = val[0][d];
  auto at = [&](int c, int i, int j, int k) -> T { return val[co_place(i, j, k)][c]; };
  apply_L_core<T>(at, S, out);
}

// The same, the words read from nb.
template <typename T>
__device__ __forceinline__ void co_words(const unsigned *nb, unsigned (&e)[CO_WORDS]) {
#pragma unroll
  for (int w = 0; w < CO_WORDS; ++w) e[w] = nb[w * CoarseCfg<T>::TAB];
}
template <typename T>
__device__ __forceinline__ void co_stencil(const Co4<T> *u, const unsigned *nb, bool signs, const StencilT<T> &S,
                                           T (&own)[3], T (&out)[3]) {
  unsigned e[CO_WORDS];
  co_words<T>(nb, e);
  co_stencil<T>(u, e, signs, S, own, out);
}

// Tables of the transfer from level I to level O (NT = 4: restriction, 3:
// prolongation), as transfer_kernel's taps.
template <typename T, int NT>
__device__ __forceinline__ void co_tables(T (*wt)[NT], unsigned short (*of)[NT], const CoarseLevel<T> &I, const CoarseLevel<T> &O,
                          const int *bound) {
  for (int c = threadIdx.x; c < O.X + O.Y + O.Z; c += CoarseCfg<T>::NTH) {
    const int d = c < O.X ? 0 : (c < O.X + O.Y ? 1 : 2);
    const int w = c - (d == 0 ? 0 : (d == 1 ? O.X : O.X + O.Y));
    const int ni = d == 0 ? I.X : (d == 1 ? I.Y : I.Z), no = d == 0 ? O.X : (d == 1 ? O.Y : O.Z);
    const int st = d == 0 ? I.Y * I.Z : (d == 1 ? I.Z : 1);
    const double sc = (double)ni / (double)no, inv = (double)no / (double)ni;
    const double xc = (w + 0.5) * sc - 0.5;
    const int lo = NT == 4 ? (int)floor(xc) - 1 : (int)floor(xc + 0.5) - 1;
#pragma unroll
    for (int k = 0; k < NT; ++k) {
      const double dd = xc - (double)(lo + k);
      int sg;
      const int j = fold<int>(d == 0 ? bound[0] : (d == 1 ? bound[1] : bound[2]), lo + k, ni, sg) * st;
      wt[c][k] = T(NT == 4 ? w_lin(dd * inv) * inv : w_quad(dd));
      of[c][k] = (unsigned short)((j << 2) | (sg + 1));
    }
  }
}

// The three channels of a transfer at output voxel o, from an input field in
// LDS; the order of the sums is transfer_kernel's.
template <typename T, int NT>
__device__ __forceinline__ void co_transfer(const Co4<T> *u, const T (*wt)[NT], const unsigned short (*of)[NT],
                                            bool signs, const CoarseLevel<T> &O, const T (&f)[3], int o, T (&out)[3]) {
  const int x = o / (O.Y * O.Z), y = O.X + (o / O.Z) % O.Y, z = O.X + O.Y + o % O.Z;
  T acc[3] = {T(0), T(0), T(0)};
  T wy[NT], wz[NT];
  int oy[NT], oz[NT];
#pragma unroll
  for (int k = 0; k < NT; ++k) {
    wy[k] = wt[y][k];
    wz[k] = wt[z][k];
    oy[k] = of[y][k];
    oz[k] = of[z][k];
  }
#pragma unroll 1
  for (int a = 0; a < NT; ++a) {
    const int ox = of[x][a];
    T accy[3] = {T(0), T(0), T(0)};
#pragma unroll
    for (int b = 0; b < NT; ++b) {
      T accz[3] = {T(0), T(0), T(0)};
#pragma unroll
      for (int e = 0; e < NT; ++e) {
        const Co4<T> c = u[(ox >> 2) + (oy[b] >> 2) + (oz[e] >> 2)];
        const int s = signs ? ((ox & 3) - 1) * ((oy[b] & 3) - 1) * ((oz[e] & 3) - 1) : 1;
        if (s) {
          accz[0] += (s < 0 ? -c.x : c.x) * wz[e];
          accz[1] += (s < 0 ? -c.y : c.y) * wz[e];
          accz[2] += (s < 0 ? -c.z : c.z) * wz[e];
        }
      }
#pragma unroll
      for (int c = 0; c < 3; ++c) accy[c] += accz[c] * wy[b];
    }
    const T wx = wt[x][a];
#pragma unroll
    for (int c = 0; c < 3; ++c) acc[c] += accy[c] * wx;
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) out[c] = acc[c] * f[c];   // displacement scaling
}

template <typename T, bool CG>
struct Coarse {
  using Cfg = CoarseCfg<T>;
  static constexpr int NTH = Cfg::NTH, VPT = Cfg::VPT;
  const CoarseArgs<T> &a;
  CoarseLds<T, CG> &m;
  int n, flip;
  bool signs;
  T xv[VPT][3];   // this thread's voxels (t + k NTH) of the current level's solution

  __device__ __forceinline__ Coarse(const CoarseArgs<T> &a_, CoarseLds<T, CG> &m_) : a(a_), m(m_), n((int)blockIdx.x), flip(0) {
    signs = false;
    for (int d = 0; d < 3; ++d) signs = signs || bound_signs(a.b[d]);
  }
  __device__ __forceinline__ int vox(const CoarseLevel<T> &L) const { return L.X * L.Y * L.Z; }

  // u <- the threads' values (every thread is past its reads of u)
  __device__ __forceinline__ void publish(int V, const T (&v)[VPT][3]) {
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int i = threadIdx.x + k * NTH;
      if (i < V) m.u[i] = Co4<T>{v[k][0], v[k][1], v[k][2], T(0)};
    }
    __syncthreads();
  }
  // first voxel of level l in the tables
  __device__ __forceinline__ int first(int l) const {
    int at = 0;
    for (int q = 0; q < l; ++q) at += vox(a.L[q]);
    return at;
  }
  __device__ __forceinline__ void load3(const T *p, int V, int i, T (&o)[3]) const {
    const T *q = p + (size_t)n * 3 * V;
    o[0] = q[i];
    o[1] = q[V + i];
    o[2] = q[2 * V + i];
  }
  __device__ __forceinline__ void store3(T *p, int V, int i, const T (&v)[3]) const {
    T *q = p + (size_t)n * 3 * V;
    q[i] = v[0];
    q[V + i] = v[1];
    q[2 * V + i] = v[2];
  }
  __device__ __forceinline__ void hess(const CoarseLevel<T> &L, int V, int i, T (&M)[6]) const {
    load_H<T>(L.h ? L.h + (size_t)n * a.CC * V : nullptr, L.h ? a.CC : 0, V, i, M);
  }
  // M u + L u
  static __device__ __forceinline__ void op(const T (&M)[6], const T (&Lu)[3], const T (&u)[3], T (&o)[3]) {
    o[0] = Lu[0] + M[0] * u[0] + M[3] * u[1] + M[4] * u[2];
    o[1] = Lu[1] + M[3] * u[0] + M[1] * u[1] + M[5] * u[2];
    o[2] = Lu[2] + M[4] * u[0] + M[5] * u[1] + M[2] * u[2];
  }
  static __device__ __forceinline__ void jacobi(const T (&M)[6], const T (&dg)[3], const T (&v)[3], T (&o)[3]) {
    const T opt = T(1.000001);
    const T a0 = M[0] * opt + dg[0], b0 = M[1] * opt + dg[1], c0 = M[2] * opt + dg[2];
    const T p = M[3], q = M[4], s = M[5];
    const T idt = T(1) / (a0 * b0 * c0 - a0 * s * s - b0 * q * q - c0 * p * p + T(2) * p * q * s);
    o[0] = idt * (v[0] * (b0 * c0 - s * s) + v[1] * (q * s - p * c0) + v[2] * (p * s - q * b0));
    o[1] = idt * (v[0] * (q * s - p * c0) + v[1] * (a0 * c0 - q * q) + v[2] * (p * q - a0 * s));
    o[2] = idt * (v[0] * (p * s - q * b0) + v[1] * (p * q - a0 * s) + v[2] * (a0 * b0 - p * p));
  }

  // nb_iter PCG steps on level l from xv; u holds the solution afterwards.
  __device__ __forceinline__ void relax_cg(int l) {
    const CoarseLevel<T> &L = a.L[l];
    const int V = vox(L);
    const T dg[3] = {L.S.diag[0], L.S.diag[1], L.S.diag[2]};
    const unsigned *nb = m.nb + first(l);
    T r[VPT][3], p[VPT][3], M[VPT][6], own[3];
    publish(V, xv);
    double acc = 0;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int i = threadIdx.x + k * NTH;
#pragma unroll
      for (int c = 0; c < 3; ++c) r[k][c] = p[k][c] = T(0);
      if (i >= V) continue;
      T Lu[3], Au[3], g[3];
      hess(L, V, i, M[k]);
      load3(L.g, V, i, g);
      co_stencil<T>(m.u, nb + i, signs, L.S, own, Lu);
      op(M[k], Lu, xv[k], Au);
#pragma unroll
      for (int c = 0; c < 3; ++c) r[k][c] = g[c] - Au[c];
      jacobi(M[k], dg, r[k], p[k]);
      acc += (double)r[k][0] * p[k][0] + (double)r[k][1] * p[k][1] + (double)r[k][2] * p[k][2];
    }
    double rz = co_sum<NTH>(acc, m.red, flip);
#pragma unroll 1
    for (int it = 0; it < a.nb_iter; ++it) {
      publish(V, p);
      T Ap[VPT][3];
      acc = 0;
#pragma unroll
      for (int k = 0; k < VPT; ++k) {
        const int i = threadIdx.x + k * NTH;
        if (i >= V) continue;
        T Lu[3];
        co_stencil<T>(m.u, nb + i, signs, L.S, own, Lu);
        op(M[k], Lu, p[k], Ap[k]);
        acc += (double)p[k][0] * Ap[k][0] + (double)p[k][1] * Ap[k][1] + (double)p[k][2] * Ap[k][2];
      }
      const double pap = co_sum<NTH>(acc, m.red, flip);
      const T alpha = T(rz / (pap > 1e-12 ? pap : 1e-12));
      if (it + 1 == a.nb_iter) {   // nothing reads the last residual and direction
#pragma unroll
        for (int k = 0; k < VPT; ++k)
#pragma unroll
          for (int c = 0; c < 3; ++c) xv[k][c] += alpha * p[k][c];
        break;
      }
      T z[VPT][3];
      acc = 0;
#pragma unroll
      for (int k = 0; k < VPT; ++k) {
        if ((int)threadIdx.x + k * NTH >= V) continue;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          xv[k][c] += alpha * p[k][c];
          r[k][c] -= alpha * Ap[k][c];
        }
        jacobi(M[k], dg, r[k], z[k]);
        acc += (double)r[k][0] * z[k][0] + (double)r[k][1] * z[k][1] + (double)r[k][2] * z[k][2];
      }
      const double rzn = co_sum<NTH>(acc, m.red, flip);
      const T beta = T(rzn / (rz > 1e-12 ? rz : 1e-12));
      rz = rzn;
#pragma unroll
      for (int k = 0; k < VPT; ++k)
        if ((int)threadIdx.x + k * NTH < V)
#pragma unroll
          for (int c = 0; c < 3; ++c) p[k][c] = z[k][c] + beta * p[k][c];
    }
    publish(V, xv);
  }

  // nb_iter Gauss-Seidel sweeps on level l from xv; u and xv hold the solution
  // afterwards.
  __device__ __forceinline__ void relax_gs(int l) {
    const CoarseLevel<T> &L = a.L[l];
    const int V = vox(L);
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int i = threadIdx.x + k * NTH;
      if (i >= V) continue;
      T M[6], g[3];
      hess(L, V, i, M);
      load3(L.g, V, i, g);
#pragma unroll
      for (int c = 0; c < 3; ++c) m.gh[c * V + i] = g[c];
#pragma unroll
      for (int c = 0; c < 6; ++c) m.gh[(3 + c) * V + i] = M[c];
    }
    publish(V, xv);
    const int base = first(l);
    const int *cls = m.cls[l];
    // a class's first NTH members, one a thread: what does not depend on the
    // solution is read before the barrier that the class waits for
    unsigned e[CO_WORDS];
    T g[3], M[6];
    int v = -1;
    auto fetch = [&](int k, int end) {
      v = -1;
      if (k >= end) return;
      v = m.mem[base + k];
      co_words<T>(m.nb + base + v, e);
#pragma unroll
      for (int c = 0; c < 3; ++c) g[c] = m.gh[c * V + v];
#pragma unroll
      for (int c = 0; c < 6; ++c) M[c] = m.gh[(3 + c) * V + v];
    };
    auto update = [&]() {
      if (v < 0) return;
      T Lx[3], x[3];
      co_stencil<T>(m.u, e, signs, L.S, x, Lx);
      gs_update<T>(Lx, L.S.diag, g[0], g[1], g[2], M, x[0], x[1], x[2]);
      m.u[v] = Co4<T>{x[0], x[1], x[2], T(0)};
    };
    fetch(threadIdx.x, cls[1]);
#pragma unroll 1
    for (int it = 0; it < a.nb_iter; ++it)
#pragma unroll 1
      for (int col = 0; cls[col] < V; ++col) {
        const int c1 = cls[col + 1];
        update();
#pragma unroll 1
        for (int k = cls[col] + NTH + (int)threadIdx.x; k < c1; k += NTH) {
          fetch(k, c1);
          update();
        }
        const int nx = c1 < V ? col + 1 : 0;
        fetch(cls[nx] + (int)threadIdx.x, cls[nx + 1]);
        __syncthreads();
      }
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int i = threadIdx.x + k * NTH;
      if (i < V) {
        const Co4<T> c = m.u[i];
        xv[k][0] = c.x;
        xv[k][1] = c.y;
        xv[k][2] = c.z;
      }
    }
  }

  __device__ __forceinline__ void relax(int l) {
    if constexpr (CG) relax_cg(l);
    else relax_gs(l);
  }

  __device__ __forceinline__ void zero_x() {
#pragma unroll
    for (int k = 0; k < VPT; ++k) xv[k][0] = xv[k][1] = xv[k][2] = T(0);
  }
  __device__ __forceinline__ void load_x(int l) {
    const CoarseLevel<T> &L = a.L[l];
    const int V = vox(L);
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int i = threadIdx.x + k * NTH;
      if (i < V) load3(L.x, V, i, xv[k]);
    }
  }
  __device__ __forceinline__ void store_x(int l) {
    const CoarseLevel<T> &L = a.L[l];
    const int V = vox(L);
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int i = threadIdx.x + k * NTH;
      if (i < V) store3(L.x, V, i, xv[k]);
    }
  }

  // g of level l + 1 <- restriction of the residual of level l (u: its solution)
  __device__ __forceinline__ void descend(int l) {
    const CoarseLevel<T> &L = a.L[l], &D = a.L[l + 1];
    const int V = vox(L), W = vox(D);
    const unsigned *nb = m.nb + first(l);
    T r[VPT][3];
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
      const int i = threadIdx.x + k * NTH;
      if (i >= V) continue;
      T Lu[3], Au[3], g[3], M[6], own[3];
      hess(L, V, i, M);
      load3(L.g, V, i, g);
      co_stencil<T>(m.u, nb + i, signs, L.S, own, Lu);
      op(M, Lu, xv[k], Au);
#pragma unroll
      for (int c = 0; c < 3; ++c) r[k][c] = g[c] - Au[c];
    }
    __syncthreads();
    publish(V, r);
    // fine / coarse size ratio of each channel's axis
    const T f[3] = {T((double)L.X / (double)D.X), T((double)L.Y / (double)D.Y),
                    T((double)L.Z / (double)D.Z)};
    for (int i = threadIdx.x; i < W; i += NTH) {
      T o[3];
      co_transfer<T, 4>(m.u, m.taps[l].dw, m.taps[l].df, signs, D, f, i, o);
      store3(D.g, W, i, o);
    }
    __syncthreads();   // g is read, and u written, by other threads next
  }
  // xv of level l <- its stored x (with `add`) + prolongation of level l + 1 (u: its solution)
  __device__ __forceinline__ void ascend(int l, bool add) {
    const CoarseLevel<T> &L = a.L[l], &D = a.L[l + 1];
    const int V = vox(L);
    const T f[3] = {T((double)L.X / (double)D.X), T((double)L.Y / (double)D.Y),
                    T((double)L.Z / (double)D.Z)};
#pragma unroll 1
    for (int k = 0; k < VPT; ++k) {
      const int i = threadIdx.x + k * NTH;
      T o[3] = {T(0), T(0), T(0)};
      if (i < V) {
        co_transfer<T, 3>(m.u, m.taps[l].uw, m.taps[l].uf, signs, L, f, i, o);
        if (add) {
          T old[3];
          load3(L.x, V, i, old);
#pragma unroll
          for (int c = 0; c < 3; ++c) o[c] += old[c];
        }
      }
      // (rolled: VPT shifts put value k in place k)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
#pragma unroll
        for (int q = 0; q + 1 < VPT; ++q) xv[q][c] = xv[q + 1][c];
        xv[VPT - 1][c] = o[c];
      }
    }
    __syncthreads();   // every thread is past its reads of u
  }

  // one V-cycle from level `base`, whose solution is in xv on entry and exit
  // (u: the solution too on exit)
  __device__ __forceinline__ void vcycle(int base) {
    const int down = a.nl - 1 - base;
#pragma unroll 1
    for (int s = 0; s <= 2 * down; ++s) {
      const int l = s <= down ? base + s : base + 2 * down - s;
      if (s > down) ascend(l, true);
      relax(l);
      if (s < down) {
        store_x(l);
        descend(l);
        zero_x();
      }
    }
  }
};

template <typename T, bool CG>
__global__ __launch_bounds__(CoarseCfg<T>::NTH) void coarse_kernel(const CoarseArgs<T> *__restrict__ args, int start,
                                                                   int nb_cycles, int zero) {
  // start: the full-multigrid start on these levels, else one V-cycle from the
  // first, whose solution starts from zero (zero) or from x
  const CoarseArgs<T> &a = *args;
  extern __shared__ __align__(16) char co_smem[];
  CoarseLds<T, CG> &m = *(CoarseLds<T, CG> *)co_smem;
  constexpr int NTH = CoarseCfg<T>::NTH;
  // neighbours of every level's voxels; Gauss-Seidel: members of every class
  int base = 0;
  for (int l = 0; l < a.nl; ++l) {
    const int Y = a.L[l].Y, Z = a.L[l].Z, V = a.L[l].X * Y * Z;
    for (int v = threadIdx.x; v < V; v += NTH) co_neighbours<T>(m.nb + base + v, a.L[l], a.b, v);
    if (l + 1 < a.nl) {
      co_tables<T, 4>(m.taps[l].dw, m.taps[l].df, a.L[l], a.L[l + 1], a.b);
      co_tables<T, 3>(m.taps[l].uw, m.taps[l].uf, a.L[l + 1], a.L[l], a.b);
    }
    if constexpr (!CG) {
      const ColourPlan &Q = a.P[l];
      const int ncls = plan_classes(Q);
      for (int i = threadIdx.x; i < ncls; i += NTH) m.cnt[i] = 0;
      __syncthreads();
      for (int v = threadIdx.x; v < V; v += NTH)
        atomicAdd(&m.cnt[plan_class(Q, v / (Y * Z), (v / Z) % Y, v % Z)], 1);
      __syncthreads();
      if (threadIdx.x == 0) {
        int acc = 0;
        for (int k = 0; k < ncls; ++k) {
          m.cls[l][k] = acc;
          acc += m.cnt[k];
          m.cnt[k] = 0;
        }
        for (int k = ncls; k <= CO_CLASSES; ++k) m.cls[l][k] = acc;
      }
      __syncthreads();
      for (int v = threadIdx.x; v < V; v += NTH) {
        const int k = plan_class(Q, v / (Y * Z), (v / Z) % Y, v % Z);
        m.mem[base + m.cls[l][k] + atomicAdd(&m.cnt[k], 1)] = (unsigned short)v;
      }
      __syncthreads();
    }
    base += V;
  }
  __syncthreads();
  Coarse<T, CG> c(a, m);
  const int last = a.nl - 1, top = start ? last : 0;
  if (zero) c.zero_x();
  else c.load_x(top);
#pragma unroll 1
  for (int l = top; l >= 0; --l) {
    if (l < top) c.ascend(l, false);
    const int cycles = l < top ? nb_cycles : 1;   // (the start's first: a relaxation of the last level)
#pragma unroll 1
    for (int q = 0; q < cycles; ++q) c.vcycle(l);
    if (cycles <= 0) c.publish(c.vox(a.L[l]), c.xv);
  }
  c.store_x(0);
}
