// mlp_features.hip -- stencil features of the learned Newton predictor
// (training rows; the inference forms them in registers, mlp_infer.hip).
//
// Features of a node (3D: 27 neighbours, clamped at the boundary; 2D: the z
// offsets repeat the plane).  For the fields f = c, mu, sum eta^2, eta_{i1},
// eta_{i2} of neighbour s:
//   x[s*10 + f]     = f(t_n)
//   x[s*10 + 5 + f] = (f(t_n) - f(t_{n-1})) / ls
// with (i1, i2) the two largest order parameters at the node at t_n and ls
// the node's local increment scale, the RMS of the 135 increments plus a
// floor; x[270] = dt * dt_scale, x[271] = log10(ls * inc_scale) (the local
// scale relative to the global one, 1 / inc_scale).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "mlp.hpp"
#include "mlp_net.hpp"

namespace hps
{
  // A workgroup of 8 waves owns 8 x 8 nodes (x, y) and marches along z over
  // zc node planes.  A ring of 3 planes of its 10 x 10 halo holds, per node,
  // what every stencil around it needs and only once: the increments of
  // (c, mu, sum eta^2, eta_i) in FP64 and the bf16 roundings of their values
  // at t_n.  The next plane's u rows are in flight while a plane is worked on.
  // 161^3 nodes, 12 order parameters: 1.2 ms (the rows alone are 2.3 GB, 0.47
  // ms at the copy rate); 6.8 ms when each stencil point summed eta^2 again
  // from a halo of raw components.
  constexpr int ST_TX = 8, ST_TY = 8, ST_TN = ST_TX * ST_TY;
  constexpr int ST_HX = ST_TX + 2, ST_HN = ST_HX * (ST_TY + 2);
  constexpr int ST_NC_MAX = 14;
  constexpr int ST_HALF = 32; // rows formed at a time
  constexpr int ST_NT   = 512;
  // rows in LDS: padded to an odd number of 16-byte pieces (bank spread)
  constexpr int ST_XS = FEAT_STRIDE + 8;

  struct StencilArgs
  {
    FeatParams      fp;
    const double   *u_prev, *u_cur;
    int            *top2;
    float          *lscale;
    uint16_t       *X;
    int             zc; // node planes per march
  };

  // strides per halo node (odd numbers of 8 and 4 bytes: bank spread)
  __host__ __device__ constexpr int st_ds(int nc)
  {
    return (nc + 1) | 1;
  }
  __host__ __device__ constexpr int st_bs(int nc)
  {
    return 2 * (((nc + 2) / 2) | 1);
  }
  // byte offsets of the LDS arrays (a plane as read shares the rows' space)
  struct StencilLds
  {
    int dring, ils, tail, tops, bring, total;
  };
  __host__ __device__ constexpr StencilLds stencil_lds(int nc)
  {
    const int  rows = ST_HALF * ST_XS * 2, raw = 2 * ST_HN * nc * 8;
    StencilLds l{};
    l.dring = rows > raw ? rows : raw;             // increments [3][ST_HN][st_ds]
    l.ils   = l.dring + 3 * ST_HN * st_ds(nc) * 8; // 1 / ls [ST_TN]
    l.tail  = l.ils + ST_TN * 8;                   // features 270, 271 [ST_TN]
    l.tops  = l.tail + ST_TN * 4;                  // i1 | i2 << 8 [3][ST_TN]
    l.bring = l.tops + 3 * ST_TN * 4;              // bf16 values [3][ST_HN][st_bs]
    l.total = l.bring + 3 * ST_HN * st_bs(nc) * 2;
    return l;
  }
  static_assert(stencil_lds(ST_NC_MAX).total <= 80 * 1024, "LDS of two workgroups");

  template <int nc>
  __global__ void __launch_bounds__(ST_NT, 4) k_features(StencilArgs a)
  {
    constexpr int ST_ITEMS = (2 * ST_HN * nc + ST_NT - 1) / ST_NT; // u entries per thread and plane
    extern __shared__ __align__(16) unsigned char st_smem[];
    const FeatParams &fp = a.fp;
    constexpr int     G = nc - 2, DS = st_ds(nc), BS = st_bs(nc);
    constexpr StencilLds L = stencil_lds(nc);
    uint16_t *xr    = (uint16_t *)st_smem; // [ST_HALF][ST_XS]
    double   *raw   = (double *)st_smem;   // a plane as read: [2][ST_HN][nc]
    double   *dring = (double *)(st_smem + L.dring);
    double   *ils   = (double *)(st_smem + L.ils);
    uint32_t *tail  = (uint32_t *)(st_smem + L.tail);
    int      *tops  = (int *)(st_smem + L.tops);
    uint16_t *bring = (uint16_t *)(st_smem + L.bring);

    const int tid = threadIdx.x;
    const int nsx = (fp.nn[0] + ST_TX - 1) / ST_TX, nsy = (fp.nn[1] + ST_TY - 1) / ST_TY;
    const int x0 = (int)(blockIdx.x % nsx) * ST_TX;
    const int y0 = (int)((blockIdx.x / nsx) % nsy) * ST_TY;
    const int z0 = (int)(blockIdx.x / (nsx * nsy)) * a.zc;
    const int z1 = min(z0 + a.zc, fp.nn[2]);
    const int64_t plane = (int64_t)fp.nn[0] * fp.nn[1] * nc;
    const int64_t base  = ((int64_t)y0 * fp.nn[0] + x0) * nc; // the tile's first node

    // this thread's entries of a raw plane: i = tid + 512 j over [t][node][c]
    constexpr int n_raw = ST_HN * nc;
    int64_t    off[ST_ITEMS];
#pragma unroll
    for (int j = 0; j < ST_ITEMS; ++j)
      {
        int i = tid + ST_NT * j;
        i     = i < n_raw ? i : i - n_raw;
        const int h = i / nc, c = i - h * nc;
        const int x = min(max(x0 + h % ST_HX - 1, 0), fp.nn[0] - 1) - x0;
        const int y = min(max(y0 + h / ST_HX - 1, 0), fp.nn[1] - 1) - y0;
        off[j]      = ((int64_t)y * fp.nn[0] + x) * nc + c;
      }
    double val[ST_ITEMS];
    auto   request = [&](int v) {
      const int64_t z  = min(max(v, 0), fp.nn[2] - 1);
      const double *pc = a.u_cur + z * plane + base;
      const double *pp = a.u_prev + z * plane + base;
#pragma unroll
      for (int j = 0; j < ST_ITEMS; ++j)
        {
          const int i = tid + ST_NT * j;
          if (i < 2 * n_raw)
            val[j] = (i < n_raw ? pc : pp)[off[j]];
        }
    };

    request(z0 - 1);
    for (int v = z0 - 1; v <= z1; ++v)
      {
        // ---- plane v into the ring
        const int slot = (v - z0 + 1) % 3;
#pragma unroll
        for (int j = 0; j < ST_ITEMS; ++j)
          if (tid + ST_NT * j < 2 * n_raw)
            raw[tid + ST_NT * j] = val[j];
        __syncthreads();
        if (v < z1)
          request(v + 1);
        {
          // four lanes per halo node: each the sum of squares of one time
          // level and every fourth component
          const int h = tid >> 2, p = tid & 3;
          if (h < ST_HN)
            {
              const double *rc = raw + h * nc, *rp = raw + (ST_HN + h) * nc;
              const double *rt = (p & 1) ? rp : rc;
              double        s  = 0.0;
#pragma unroll
              for (int i = 2; i < nc; ++i)
                s += rt[i] * rt[i];
              const double other = __shfl_xor(s, 1, 64);
              double      *d     = dring + (slot * ST_HN + h) * DS;
              uint16_t    *b     = bring + (slot * ST_HN + h) * BS;
              if (p == 2)
                {
                  d[2] = s - other;
                  b[2] = f2bf((float)s);
                }
#pragma unroll
              for (int j = 0; j < (nc + 3) / 4; ++j)
                {
                  const int c = p + 4 * j;
                  if (c >= nc)
                    break;
                  const int    q = c < 2 ? c : c + 1;
                  const double e = rc[c];
                  d[q]           = e - rp[c];
                  b[q]           = f2bf((float)e);
                }
              const int hx = h % ST_HX - 1, hy = h / ST_HX - 1;
              if (p == 3 && hx >= 0 && hx < ST_TX && hy >= 0 && hy < ST_TY)
                {
                  int    i1 = 0, i2 = G > 1 ? 1 : 0;
                  double e1 = -1e300, e2 = -1e300;
                  for (int i = 0; i < G; ++i)
                    {
                      const double e = rc[2 + i];
                      if (e > e1)
                        {
                          e2 = e1;
                          i2 = i1;
                          e1 = e;
                          i1 = i;
                        }
                      else if (e > e2)
                        {
                          e2 = e;
                          i2 = i;
                        }
                    }
                  if (G == 1)
                    i2 = 0;
                  tops[slot * ST_TN + hy * ST_TX + hx] = i1 | (i2 << 8);
                }
            }
        }
        __syncthreads();
        if (v < z0 + 1)
          continue;

        // ---- the nodes of plane z = v - 1; ring offsets of z - 1, z, z + 1
        const int z      = v - 1;
        const int n0     = ((v - z0 + 2) % 3) * ST_HN; // plane z - 1
        const int n1     = ((v - z0) % 3) * ST_HN;     // plane z
        const int n2     = slot * ST_HN;               // plane z + 1
        const int *ztops = tops + ((v - z0) % 3) * ST_TN;
        // ring node of stencil point s of tile node n
        auto at = [&](int n, int s) {
          const int q = s / 9, r = s - 9 * q;
          const int b = q == 0 ? n0 : (q == 1 ? n1 : n2);
          return b + (n / ST_TX + r / 3) * ST_HX + n % ST_TX + r % 3;
        };
        {
          // local increment scale, 8 lanes per node
          const int sub = tid & 7, n = tid >> 3;
          const int i1 = ztops[n] & 255, i2 = ztops[n] >> 8;
          double    ss = 0.0;
#pragma unroll
          for (int j = 0; j < 4; ++j)
            {
              const int s = sub + 8 * j;
              if (s >= 27)
                break;
              const double *d = dring + at(n, s) * DS;
              ss += d[0] * d[0];
              ss += d[1] * d[1];
              ss += d[2] * d[2];
              ss += d[3 + i1] * d[3 + i1];
              ss += d[3 + i2] * d[3 + i2];
            }
          // fixed order over the node's lanes
          ss += __shfl_xor(ss, 1, 64);
          ss += __shfl_xor(ss, 2, 64);
          ss += __shfl_xor(ss, 4, 64);
          if (sub == 0)
            {
              const double ls = sqrt(ss / 135.0) + fp.inc_floor;
              ils[n]          = 1.0 / ls;
              tail[n]         = f2bf((float)(fp.dt * fp.dt_scale)) |
                        ((uint32_t)f2bf((float)log10(ls * fp.inc_scale)) << 16);
              const int gx = x0 + n % ST_TX, gy = y0 + n / ST_TX;
              if (gx < fp.nn[0] && gy < fp.nn[1])
                {
                  const int64_t node = ((int64_t)z * fp.nn[1] + gy) * fp.nn[0] + gx;
                  a.lscale[node]     = (float)ls;
                  a.top2[2 * node]     = i1;
                  a.top2[2 * node + 1] = i2;
                }
            }
        }
        __syncthreads();
        for (int half = 0; half < ST_TN / ST_HALF; ++half)
          {
            // feature rows: a lane takes one node and every 16th stencil point
            {
              const int    r = tid & (ST_HALF - 1), n = half * ST_HALF + r;
              const int    i1 = ztops[n] & 255, i2 = ztops[n] >> 8;
              const double s = ils[n];
#pragma unroll
              for (int k = 0; k < 2; ++k)
                {
                  const int sp = (tid >> 5) + 16 * k;
                  if (sp >= 27)
                    break;
                  const int       h = at(n, sp);
                  const double   *d = dring + h * DS;
                  const uint16_t *b = bring + h * BS;
                  uint32_t       *x = (uint32_t *)(xr + r * ST_XS + sp * 10);
                  auto inc = [&](int q) { return (uint32_t)f2bf((float)(d[q] * s)); };
                  x[0] = *(const uint32_t *)b;
                  x[1] = b[2] | ((uint32_t)b[3 + i1] << 16);
                  x[2] = b[3 + i2] | (inc(0) << 16);
                  x[3] = inc(1) | (inc(2) << 16);
                  x[4] = inc(3 + i1) | (inc(3 + i2) << 16);
                }
            }
            if (tid < ST_HALF)
              *(uint32_t *)(xr + tid * ST_XS + 270) = tail[half * ST_HALF + tid];
            __syncthreads();
            constexpr int CH = FEAT_STRIDE / 8; // 16-byte pieces of a row
            for (int i = tid; i < ST_HALF * CH; i += ST_NT)
              {
                const int r = i / CH, ch = i - CH * r;
                const int gx = x0 + r % ST_TX;
                const int gy = y0 + half * (ST_HALF / ST_TX) + r / ST_TX;
                if (gx < fp.nn[0] && gy < fp.nn[1])
                  {
                    const int64_t node = ((int64_t)z * fp.nn[1] + gy) * fp.nn[0] + gx;
                    *(uint4 *)(a.X + node * FEAT_STRIDE + ch * 8) =
                      *(const uint4 *)(xr + r * ST_XS + ch * 8);
                  }
              }
            __syncthreads();
          }
      }
  }

  // node planes per march: deep marches stage fewer halo planes (zc + 2 for
  // zc), but the grid should keep about 1024 workgroups (2 per CU at once,
  // two rounds) while the mesh has them
  static int stencil_planes(const FeatParams &fp, int64_t &nwg)
  {
    const int64_t cols = (int64_t)((fp.nn[0] + ST_TX - 1) / ST_TX) *
                         ((fp.nn[1] + ST_TY - 1) / ST_TY);
    int64_t zc = cols * fp.nn[2] / 1024;
    zc         = zc < 2 ? 2 : (zc > 32 ? 32 : zc);
    const int64_t chunks = (fp.nn[2] + zc - 1) / zc;
    nwg                  = cols * chunks;
    return (int)((fp.nn[2] + chunks - 1) / chunks);
  }

  void mlp_features(hipStream_t s, const FeatParams &fp, const double *u_prev,
                    const double *u_cur, uint16_t *X, int *top2, float *lscale)
  {
    StencilArgs a{};
    a.fp        = fp;
    a.u_prev    = u_prev;
    a.u_cur     = u_cur;
    a.X         = X;
    a.top2      = top2;
    a.lscale    = lscale;
    int64_t nwg = 0;
    a.zc        = stencil_planes(fp, nwg);
    switch (fp.n_comp)
      {
#define HPS_NC(N)                                                                    \
  case N:                                                                            \
    k_features<N><<<(unsigned)nwg, ST_NT, stencil_lds(N).total, s>>>(a);             \
    break;
        HPS_NC(3) HPS_NC(4) HPS_NC(5) HPS_NC(6) HPS_NC(7) HPS_NC(8)
        HPS_NC(9) HPS_NC(10) HPS_NC(11) HPS_NC(12) HPS_NC(13) HPS_NC(14)
#undef HPS_NC
      }
  }
} // namespace hps
