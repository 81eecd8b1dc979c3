// Push / count of the tiles that tile_kernel's box does not hold but one or two
// larger ones do: rotated, zoomed and moderately deformed grids of 3-D float
// fields.
//
// A work-group owns a tile of tile_kernel's, one part of 4 x 8 x 8 samples (2 x
// 8 x 8 above order 5) a wave.  The parts are taken together as far as the
// bounding box of their taps fits the box in LDS (all eight; four, two or one
// at a time), accumulated into it by FP64 LDS atomics, and the box is added to
// the output once, folded and signed, with one FP32 global atomic per non-zero
// element.  Products and sums are FP64: gfx950 runs FP64 and unpacked FP32
// multiply-adds at one rate (50 and 56 lanes a clock and CU).
//
// What bounds it are the LDS atomics (at best 7.4 lanes a clock and CU; 16
// lanes are served at once when their elements differ mod 16) and the
// instructions that feed them.  Samples consecutive along z whose first taps
// are consecutive too (a run, of at most G samples) first sum their splats in
// registers: length + ORD atomics a tap row instead of length * (ORD + 1).  On
// these grids the runs are short and of all lengths, and a wave whose lanes
// each walked their own would take as many passes as its busiest lane has
// runs; so the runs of all waves are listed by length, and each wave takes 64
// of one length at a time: no lane waits, and the code for a length has no
// predicates.  A sample's weights are evaluated again for every channel, as
// the list does not tie the runs to lanes; on a smooth grid that, and not
// reusing them, makes this slower than tile_kernel (181 x 217 x 181, 8
// channels, order 3: 1.72 ms against 1.26).
//
// Against the binned pass, which took these tiles before (181 x 217 x 181,
// order 3): rotation by 15 degrees and zoom 1.1, one channel 0.55 -> 0.35 ms,
// eight 2.84 -> 1.61; smooth warp of 2 voxels RMS 0.69 -> 0.47 and 3.71 -> 2.47.
// An FP32 global atomic a tap instead of the boxes was 3 to 15 times slower.
//
// Weights, the out-of-bound rule and the splat order of each sample are
// those of pp_sample (nitorch/_C/src/impl/pushpull_common.cpp: OOB :926-974,
// splat3d :1235-1290, linear :1653-1858, nearest :2314-2341); folding and
// signs follow bounds_common.h:28-219.
#pragma once

namespace ni_amd {

template <int ORD>
struct STile {
  using D = TileBox<ORD>;                                   // the tiles of tile_kernel
  static constexpr int NTH = D::NTH, NWV = NTH / 64;
  static constexpr int LV = NWV == 8 ? 3 : 2;               // log2 of the parts
  static constexpr int NS = D::R;                           // samples of a lane: x rows of its part
  static constexpr int PX = NS, PY = 8, PZ = 8;             // part of a wave
  // longest run: its weights (z in double) and sums fit 128 registers
  static constexpr int G = ORD == 0 ? 1 : ORD <= 4 ? 4 : ORD == 5 ? 3 : 2;
  static constexpr int CAP = 9216;                          // box elements (72 KB; two work-groups a CU)
  static constexpr int MAXAX = 128;                         // box extent per axis
  static_assert(NWV == 1 << LV && D::TZ == 2 * PZ && D::TX * D::TY == (NWV / 2) * PX * PY, "a part a wave");
};

// The splats of one run of GS samples, this lane's.  gp: grid at its first
// sample (z step gz, coordinate step gD); tp: its values (z step tz).
template <int ORD, bool COUNT, int GS>
__device__ __forceinline__ void st_splat(double *box, const float *gp, int gz, int gD, const float *tp, int tz, int m0,
                                         int m1, int m2, int DYZ, int DZ) {
  constexpr int NT = ORD + 1, WS = GS + ORD;
  float wx[GS][NT], wy[GS][NT];
  double wz[GS][NT], v[GS];
  int off = 0;
#pragma unroll
  for (int i = 0; i < GS; ++i) {
    float t[NT], g[NT];
    const int l0 = tl_taps<ORD>(gp[i * gz], wx[i], g);
    const int l1 = tl_taps<ORD>(gp[i * gz + gD], wy[i], g);
    const int l2 = tl_taps<ORD>(gp[i * gz + 2 * gD], t, g);
    if (i == 0) off = (l0 - m0) * DYZ + (l1 - m1) * DZ + (l2 - m2);
#pragma unroll
    for (int k = 0; k < NT; ++k) wz[i][k] = (double)t[k];
    v[i] = COUNT ? 1.0 : (double)tp[i * tz];
  }
  double *bp = box + off;
#pragma unroll 1
  for (int kx = 0; kx < NT; ++kx, bp += DYZ) {
    double xv[GS];
#pragma unroll
    for (int i = 0; i < GS; ++i) {
      xv[i] = (double)wx[i][0] * v[i];
      tl_rot(wx[i]);
      tl_opaque(wy[i]);   // converted where used: hoisted, the doubles would not fit the registers
    }
    double *bq = bp;
#pragma unroll
    for (int ky = 0; ky < NT; ++ky, bq += DZ) {
      double acc[WS];
#pragma unroll
      for (int i = 0; i < GS; ++i) {
        const double cw = xv[i] * (double)wy[i][ky];
#pragma unroll
        for (int kz = 0; kz < NT; ++kz)
          acc[i + kz] = (i == 0 || kz == NT - 1) ? cw * wz[i][kz] : fma(cw, wz[i][kz], acc[i + kz]);
      }
#pragma unroll
      for (int s = 0; s < WS; ++s) atomicAdd(bq + s, acc[s]);
      __builtin_amdgcn_sched_barrier(0);   // one row's sums live at a time
    }
  }
}

// tiles: their count, the count of the tiles already in fb, their ids.  fb: a
// count, then the ids of the tiles left to the binned pass; it gets those with
// a part that does not fit the box by itself, and all when it has more than
// 1 / ST_FAR as many already.
template <int ORD, bool COUNT>
__global__ __launch_bounds__((STile<ORD>::NTH), 4) void scatter_kernel(PPArgs<float> a, int ntx, int nty, int ntz,
                                                                       const int *tiles, int *fb) {
  using B = STile<ORD>;
  using D = TileBox<ORD>;
  constexpr int NT = ORD + 1, G = B::G, NS = B::NS, NTH = B::NTH, NWV = B::NWV, LV = B::LV;
  __shared__ double box[B::CAP];
  __shared__ unsigned short list[NTH * NS];
  __shared__ int fofs[3 * B::MAXAX];
  __shared__ float fsg[3 * B::MAXAX];
  __shared__ int part[NWV][6];
  __shared__ int wcnt[NWV][G];        // runs of length g + 1 of each wave
  __shared__ int blk[2 * NWV - 1][6]; // first tap and extent of each aligned group of 8, 4, 4, 2, ... parts
  __shared__ unsigned fits;

  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int ntiles = tiles[0];
  if ((int64_t)tiles[1] * ST_FAR > ntiles) {
    for (int j = blockIdx.x * NTH + threadIdx.x; j < ntiles; j += gridDim.x * NTH)
      fb[1 + atomicAdd(fb, 1)] = tiles[2 + j];
    return;
  }
  for (int j = blockIdx.x; j < ntiles; j += gridDim.x) {
    const int tile = tiles[2 + j];
    __syncthreads();   // the previous tile is done with the shared state
    int r = tile;
    const int tz = r % ntz; r /= ntz;
    const int ty = r % nty; r /= nty;
    const int tx = r % ntx;
    const int n = r / ntx;
    const int sz[3] = {(int)a.sX, (int)a.sY, (int)a.sZ};
    // sample i of this lane within the tile: (sx + i, sy, sz0); groups of
    // parts halve z first, then y, then x
    const int wx = LV == 3 || D::TX > B::PX ? w & 1 : 0, wy = D::TY > B::PY ? (w >> (LV - 2)) & 1 : 0;
    const int sx = wx * B::PX, sy = wy * B::PY + (lane >> 3), sz0 = (w >> (LV - 1)) * B::PZ + (lane & 7);
    const int g1 = (int)a.grid_s[1], g2 = (int)a.grid_s[2], g3 = (int)a.grid_s[3], gD = (int)a.grid_s[4];
    const float *gt = a.grid + (int)(n * a.grid_s[0] + (int64_t)tx * D::TX * a.grid_s[1] +
                                     (int64_t)ty * D::TY * a.grid_s[2] + (int64_t)tz * D::TZ * a.grid_s[3]);
    const float tol = (a.extrap & 2) ? 0.55f : 0.05f;

    // ---- first taps: the part's bounding box, and the lanes' runs ----
    int mn[3] = {INT_MAX, INT_MAX, INT_MAX}, mx[3] = {INT_MIN, INT_MIN, INT_MIN};
    unsigned runs = 0;   // sample i, 3 bits: length of the run it starts (0: none)
    int cnt[G];
#pragma unroll
    for (int g = 0; g < G; ++g) cnt[g] = 0;
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      int lo[3] = {0, 0, 0};
      bool ok = tx * D::TX + sx + i < (int)a.tX && ty * D::TY + sy < (int)a.tY && tz * D::TZ + sz0 < (int)a.tZ;
      if (ok) {
        const float *gp = gt + (sx + i) * g1 + sy * g2 + sz0 * g3;
        const float xs[3] = {gp[0], gp[gD], gp[2 * gD]};
        if (!(a.extrap & 1))
#pragma unroll
          for (int d = 0; d < 3; ++d) ok = ok && (xs[d] >= -tol && xs[d] < (float)(sz[d] - 1) + tol);
        if (ok) {
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            lo[d] = tl_first<ORD>(xs[d]);
            mn[d] = min(mn[d], lo[d]);
            mx[d] = max(mx[d], lo[d]);
          }
        }
      }
      // does this sample continue the run of the previous one (z - 1, the lane before)?
      const int z = lane & 7;
      const int p0 = __shfl_up(lo[0], 1, 64), p1 = __shfl_up(lo[1], 1, 64), p2 = __shfl_up(lo[2], 1, 64);
      const unsigned long long in = __ballot(ok);
      const bool cont = ok && z && ((in >> ((lane - 1) & 63)) & 1) && lo[0] == p0 && lo[1] == p1 &&
                        (unsigned)lo[2] == (unsigned)p2 + 1u;
      // the z row's breaks: where a run starts or a sample is out of bounds;
      // runs are cut into pieces of G
      const unsigned row = (unsigned)(__ballot(!cont) >> (lane & ~7)) & 0xffu;
      const unsigned before = row & ((2u << z) - 1u), after = row >> (z + 1);
      const int pos = before ? z - (31 - __clz((int)before)) : 0;
      const int left = after ? __ffs((int)after) : 8 - z;   // samples from here to the next break
      const int len = ok && pos % G == 0 ? min(G, left) : 0;
      runs |= (unsigned)len << (3 * i);
#pragma unroll
      for (int g = 0; g < G; ++g) cnt[g] += __popcll(__ballot(len == g + 1));
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      mn[d] = wave_min(mn[d]);
      mx[d] = wave_max(mx[d]);
    }
    if (lane == 0) {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        part[w][d] = mn[d];
        part[w][3 + d] = mx[d];
      }
#pragma unroll
      for (int g = 0; g < G; ++g) wcnt[w][g] = cnt[g];
    }
    __syncthreads();
    // ---- groups of parts whose box fits ----
    if (w == 0) {
      bool fit = false;
      if (lane < 2 * NWV - 1) {
        const int lv = 31 - __clz(lane + 1), np = NWV >> lv, q0 = (lane + 1 - (1 << lv)) * np;
        int m[3] = {INT_MAX, INT_MAX, INT_MAX}, M[3] = {INT_MIN, INT_MIN, INT_MIN};
        for (int q = q0; q < q0 + np; ++q)
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            m[d] = min(m[d], part[q][d]);
            M[d] = max(M[d], part[q][3 + d]);
          }
        fit = true;
        int64_t vol = 1;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const int64_t e = m[0] > M[0] ? 0 : (int64_t)M[d] - (int64_t)m[d] + NT;   // 0: no sample in bounds
          fit = fit && e <= B::MAXAX;
          blk[lane][d] = m[d];
          blk[lane][3 + d] = (int)(fit ? e : 0);
          vol *= fit ? (d == 2 ? e | 1 : e) : 0;
        }
        fit = fit && vol <= B::CAP;
      }
      const unsigned long long f = __ballot(fit);
      if (lane == 0) fits = (unsigned)f;
    }
    __syncthreads();
    const unsigned fm = (unsigned)__builtin_amdgcn_readfirstlane((int)fits);
    auto ident = [&](int p, int lv) { return (1 << lv) - 1 + (p >> (LV - lv)); };
    // largest aligned group that starts at part p and fits
    auto group = [&](int p) {
      int lv = p == 0 ? 0 : LV - __builtin_ctz(p);
      while (lv < LV && !((fm >> ident(p, lv)) & 1u)) ++lv;
      return lv;
    };
    if ((fm >> (NWV - 1)) != (1u << NWV) - 1u) {
      if (threadIdx.x == 0) fb[1 + atomicAdd(fb, 1)] = tile;
      continue;
    }

    const int C = COUNT ? 1 : (int)a.C;
    const int t1 = COUNT ? 0 : (int)a.trgt_s[2], t2 = COUNT ? 0 : (int)a.trgt_s[3], t3 = COUNT ? 0 : (int)a.trgt_s[4];
    const float *tt = COUNT ? nullptr
                            : a.trgt + (int)(n * a.trgt_s[0] + (int64_t)tx * D::TX * a.trgt_s[2] +
                                             (int64_t)ty * D::TY * a.trgt_s[3] + (int64_t)tz * D::TZ * a.trgt_s[4]);
    float *out = a.out + (int)(n * a.out_s[0]);
    const int oC = (int)a.out_s[1];

    for (int p = 0; p < NWV;) {
      const int lv = group(p), id = ident(p, lv), pe = p + (NWV >> lv);
      const int m0 = __builtin_amdgcn_readfirstlane(blk[id][0]), m1 = __builtin_amdgcn_readfirstlane(blk[id][1]),
                m2 = __builtin_amdgcn_readfirstlane(blk[id][2]);
      const int e0 = __builtin_amdgcn_readfirstlane(blk[id][3]), e1 = __builtin_amdgcn_readfirstlane(blk[id][4]),
                e2 = __builtin_amdgcn_readfirstlane(blk[id][5]);
      const int p0 = p;
      p = pe;
      if (e0 <= 0) continue;
      const int DZ = e2 | 1, DYZ = e1 * DZ;
      __syncthreads();   // the previous group is done with box, list and tables
      for (int q = threadIdx.x; q < e0 * DYZ; q += NTH) box[q] = 0.0;
      for (int q = threadIdx.x; q < e0 + e1 + e2; q += NTH) {
        const int d = q < e0 ? 0 : (q < e0 + e1 ? 1 : 2);
        const int b = q - (d == 0 ? 0 : (d == 1 ? e0 : e0 + e1));
        int sg = 0;
        const int j = fold<int>(d == 0 ? a.bound[0] : (d == 1 ? a.bound[1] : a.bound[2]),
                                tap_at(d == 0 ? m0 : (d == 1 ? m1 : m2), b), d == 0 ? sz[0] : (d == 1 ? sz[1] : sz[2]), sg);
        fofs[q] = j * (int)(d == 0 ? a.out_s[2] : (d == 1 ? a.out_s[3] : a.out_s[4]));
        fsg[q] = (float)sg;
      }
      // list of the group's runs, longest first
      int tot[G];
#pragma unroll
      for (int g = 0; g < G; ++g) tot[g] = 0;
      int mine[G];
#pragma unroll
      for (int g = 0; g < G; ++g) mine[g] = 0;
      for (int q = p0; q < pe; ++q)
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const int k = wcnt[q][g];
          tot[g] += k;
          mine[g] += q < w ? k : 0;
        }
      if (w >= p0 && w < pe) {
        const unsigned long long below = (1ull << lane) - 1ull;
        int first = 0;
#pragma unroll
        for (int g = G - 1; g >= 0; --g) {
          int at = first + mine[g];
          first += tot[g];
#pragma unroll
          for (int i = 0; i < NS; ++i) {
            const bool is = ((runs >> (3 * i)) & 7u) == (unsigned)(g + 1);
            const unsigned long long m = __ballot(is);
            if (is) list[at + __popcll(m & below)] = (unsigned short)(((sx + i) << 8) | (sy << 4) | sz0);
            at += __popcll(m);
          }
        }
      }
      __syncthreads();
      for (int c = 0; c < C; ++c) {
        // 64 runs of one length a wave at a time
        const float *tc = COUNT ? nullptr : tt + c * (int)a.trgt_s[1];
        auto chunk = [&](auto len, int s0, int s1) {
          constexpr int GS = decltype(len)::value;
          const int at = s0 + lane;
          if (at >= s1) return;
          const int code = list[at];
          const int x = code >> 8, y = (code >> 4) & 15, z = code & 15;
          st_splat<ORD, COUNT, GS>(box, gt + x * g1 + y * g2 + z * g3, g3, gD,
                                   COUNT ? nullptr : tc + x * t1 + y * t2 + z * t3, t3, m0, m1, m2, DYZ, DZ);
        };
        int ch = w;   // chunk of the list, over all lengths
        int s0 = 0;
        auto length = [&](auto len) {
          const int k = tot[decltype(len)::value - 1], nch = (k + 63) >> 6;
          for (; ch < nch; ch += NWV) chunk(len, s0 + 64 * ch, s0 + k);
          ch -= nch;
          s0 += k;
        };
        if constexpr (G >= 4) length(std::integral_constant<int, G >= 4 ? 4 : 1>{});
        if constexpr (G >= 3) length(std::integral_constant<int, G >= 3 ? 3 : 1>{});
        if constexpr (G >= 2) length(std::integral_constant<int, G >= 2 ? 2 : 1>{});
        length(std::integral_constant<int, 1>{});
        __syncthreads();
        // add the box to the output, folded and signed; clear it for the next channel
        float *oc = out + c * oC;
        const float r2 = 1.f / (float)e2;
        for (int q = threadIdx.x; q < e1 * e2; q += NTH) {
          const int by = tl_div(q, e2, r2), bz = q - by * e2;
          double *bq = box + by * DZ + bz;
          float *op = oc + fofs[e0 + by] + fofs[e0 + e1 + bz];
          const float sg = fsg[e0 + by] * fsg[e0 + e1 + bz];
          for (int bx = 0; bx < e0; bx += 4) {
            double d[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) d[u] = bx + u < e0 ? bq[(bx + u) * DYZ] : 0.0;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              if (d[u] == 0.0) continue;
              bq[(bx + u) * DYZ] = 0.0;
              const float f = (float)d[u], s = fsg[bx + u] * sg;
              if (f != 0.f && s != 0.f) atomic_add(op + fofs[bx + u], f * s);
            }
          }
        }
        if (c + 1 < C) __syncthreads();
      }
    }
  }
}

}  // namespace ni_amd
