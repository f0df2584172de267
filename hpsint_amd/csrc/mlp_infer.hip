// mlp_infer.hip -- fused inference of the learned Newton predictor: stencil
// features, the 272-128-128-128-4 network and the corrected extrapolation.
//
// Two kernels.  k_fields reads u_prev and u_cur once and leaves, per node,
// what the 27 stencils around it read: the FP64 increments of (c, mu, sum
// eta^2, eta_i) and the bf16 roundings of their values at t_n, component by
// component, so that consecutive nodes are consecutive in memory.  k_infer
// gives each wave 32 nodes and keeps everything of theirs in registers: the
// features are formed in the matrix cores' operand layout, and a layer's
// result layout is the next layer's operand layout once the weights' columns
// are permuted to match (done when they are copied to LDS), so no
// activation goes through LDS and no wave waits for another.
//
// Measured at 161^3 nodes, 12 order parameters, with the increment norm: 1.97
// ms (k_fields 0.32, at 4.9 TB/s; k_infer 1.45, 0.88 of it VALU issue, most
// of that the 384 tanh per node; its MFMA 0.24; the rest is waiting for the
// gathers at 2 waves/SIMD).  Feature, layer and
// correction kernels one after the other, with a row of 272 features per node
// in memory, took 13.4 ms; one kernel whose waves shared a tile's features
// and activations through LDS 3.1 ms (15 barriers per tile, 2 waves/SIMD).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "mlp.hpp"
#include "mlp_net.hpp"

namespace hps
{
  // workspace arrays (byte offsets), N nodes
  struct InferWs
  {
    int64_t d2, ds, v4, de, be, total;
  };
  static InferWs infer_ws(int64_t N, int G)
  {
    InferWs w{};
    w.d2    = 0;                    // double2 (dc, dmu) [N]
    w.ds    = w.d2 + 16 * N;        // double d(sum eta^2) [N]
    w.v4    = w.ds + 8 * N;         // bf16 c, mu, sum eta^2, 0 [N]
    w.de    = w.v4 + 8 * N;         // double d(eta_g) [G][N]
    w.be    = w.de + 8 * N * G;     // bf16 eta_g [G][N]
    w.total = w.be + 2 * N * G;
    return w;
  }

  struct InferArgs
  {
    FeatParams      fp;
    const double   *u_prev, *u_cur;
    const uint16_t *W[4];
    const float    *b[4];
    const float    *out_scale;
    int            *top2;
    float          *lscale;
    double         *out;
    char           *ws;
    InferWs         l;
  };

  constexpr int FLD_NODES = 128; // nodes per workgroup of 256 lanes

  template <int NC>
  __global__ void __launch_bounds__(256) k_fields(InferArgs a)
  {
    constexpr int     G = NC - 2;
    __shared__ double raw[2][FLD_NODES * NC];
    const int64_t     N = a.fp.n_nodes, n0 = (int64_t)blockIdx.x * FLD_NODES;
    const int         n_here = (int)(N - n0 < FLD_NODES ? N - n0 : FLD_NODES);
    constexpr int     PER    = FLD_NODES * NC / 256 + (FLD_NODES * NC % 256 != 0);
    double            v[2][PER];
#pragma unroll
    for (int j = 0; j < PER; ++j)
      {
        const int i = threadIdx.x + 256 * j;
        if (i < n_here * NC)
          {
            v[0][j] = a.u_cur[n0 * NC + i];
            v[1][j] = a.u_prev[n0 * NC + i];
          }
      }
#pragma unroll
    for (int j = 0; j < PER; ++j)
      {
        const int i = threadIdx.x + 256 * j;
        if (i < n_here * NC)
          {
            raw[0][i] = v[0][j];
            raw[1][i] = v[1][j];
          }
      }
    __syncthreads();
    // two threads per node, half a workgroup apart: consecutive lanes write
    // consecutive nodes
    const int r = threadIdx.x & (FLD_NODES - 1), p = threadIdx.x / FLD_NODES;
    if (r >= n_here)
      return;
    const int64_t n  = n0 + r;
    const double *rc = raw[0] + r * NC, *rp = raw[1] + r * NC;
    double       *de = (double *)(a.ws + a.l.de);
    uint16_t     *be = (uint16_t *)(a.ws + a.l.be);
    if (p == 0)
      {
        double s = 0.0, t = 0.0;
#pragma unroll
        for (int i = 2; i < NC; ++i)
          {
            s += rc[i] * rc[i];
            t += rp[i] * rp[i];
          }
        ((double2 *)(a.ws + a.l.d2))[n] = make_double2(rc[0] - rp[0], rc[1] - rp[1]);
        ((double *)(a.ws + a.l.ds))[n]  = s - t;
        ((uint2 *)(a.ws + a.l.v4))[n] =
          make_uint2(f2bf((float)rc[0]) | ((uint32_t)f2bf((float)rc[1]) << 16),
                     f2bf((float)s));
      }
    else
      {
        int    i1 = 0, i2 = G > 1 ? 1 : 0;
        double e1 = -1e300, e2 = -1e300;
#pragma unroll
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
        a.top2[2 * n]     = i1;
        a.top2[2 * n + 1] = G == 1 ? 0 : i2;
      }
    for (int g = p; g < G; g += 2)
      {
        const double e  = rc[2 + g];
        de[g * N + n]   = e - rp[2 + g];
        be[g * N + n]   = f2bf((float)e);
      }
  }

  // k_infer: 8 waves per workgroup, one workgroup per CU (its LDS holds all
  // weights), each wave 32 nodes at a time.  Lanes l and l + 32 share node
  // l: half 0 forms the features of stencil points 0..12 (slot i: point i),
  // half 1 of points 26..14 (slot i: point 26 - i), and of the centre point
  // half 0 takes the values and half 1 the increments.
  constexpr int INF_NT = 512, INF_WAVES = INF_NT / 64;
  constexpr int INF_K0 = NET_IN / 16, INF_K = NET_H / 16, INF_RT = NET_H / 32;
  // one fragment: 64 lanes x 8 bf16
  constexpr int FRAG = 64 * 8;
  struct InferLds
  {
    static constexpr int w0 = 0, w1 = w0 + INF_RT * INF_K0 * FRAG * 2,
                         w2 = w1 + INF_RT * INF_K * FRAG * 2,
                         w3 = w2 + INF_RT * INF_K * FRAG * 2, bias = w3 + INF_K * FRAG * 2,
                         y = bias + (3 * NET_H + 2 * NET_OUT) * 4,
                         total = y + INF_WAVES * 32 * 8 * 4;
  };
  static_assert(InferLds::total <= 160 * 1024, "weights and outputs in one CU's LDS");

  // feature of entry q (0..135) of half h's operand
  __device__ __forceinline__ int feature_of(int h, int q)
  {
    if (q < 130)
      return (h ? 26 - q / 10 : q / 10) * 10 + q % 10;
    return q < 135 ? 130 + 5 * h + (q - 130) : 270 + h;
  }
  // input of the next layer at k-step k, half h, entry j: the output that a
  // lane of half h holds there (32x32 result: output 8 (r >> 2) + 4 h + (r &
  // 3) of a 32-row tile in register r)
  __device__ __forceinline__ int hidden_of(int k, int h, int j)
  {
    return 32 * (k >> 1) + 8 * (2 * (k & 1) + (j >> 2)) + 4 * h + (j & 3);
  }

  // the 128 outputs of a hidden layer: x holds KS k-steps of operands, the
  // result (tanh, bf16) INF_K k-steps of the next layer's operands
  template <int KS>
  __device__ __forceinline__ void infer_layer(const char *w, const float *bias,
                                              const uint4 *x, uint4 *out, int lane)
  {
    const int h = lane >> 5;
#pragma unroll
    for (int t = 0; t < INF_RT; ++t)
      {
        f32x16 acc;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          acc[r] = 0.f;
        const uint4 *f = (const uint4 *)(w + t * KS * FRAG * 2) + lane;
#pragma unroll
        for (int k = 0; k < KS; ++k)
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, f[64 * k]),
                                                        __builtin_bit_cast(bf16x8, x[k]), acc, 0,
                                                        0, 0);
#pragma unroll
        for (int q = 0; q < 2; ++q)
          {
            bf16x8 o;
#pragma unroll
            for (int g = 0; g < 2; ++g)
              {
                const f32x4 b = *(const f32x4 *)(bias + 32 * t + 8 * (2 * q + g) + 4 * h);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                  o[4 * g + r] = (__bf16)tanh_fast(acc[4 * (2 * q + g) + r] + b[r]);
              }
            out[2 * t + q] = __builtin_bit_cast(uint4, o);
          }
      }
  }

  template <int NC>
  __global__ void __launch_bounds__(INF_NT, 2) k_infer(InferArgs a)
  {
    extern __shared__ __align__(16) char inf_smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    float    *bias = (float *)(inf_smem + InferLds::bias);

    // ---- weights into LDS, fragment by fragment
    for (int i = tid; i < INF_RT * INF_K0 * 64; i += INF_NT)
      {
        const int l = i & 63, k = (i >> 6) % INF_K0, t = (i >> 6) / INF_K0;
        const uint16_t *row = a.W[0] + (32 * t + (l & 31)) * NET_IN;
        uint16_t       *dst = (uint16_t *)(inf_smem + InferLds::w0) + i * 8;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          dst[j] = row[feature_of(l >> 5, 8 * k + j)];
      }
    for (int i = tid; i < INF_RT * INF_K * 64; i += INF_NT)
      {
        const int l = i & 63, k = (i >> 6) % INF_K, t = (i >> 6) / INF_K;
        const int row = (32 * t + (l & 31)) * NET_H;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          {
            const int c = row + hidden_of(k, l >> 5, j);
            ((uint16_t *)(inf_smem + InferLds::w1))[i * 8 + j] = a.W[1][c];
            ((uint16_t *)(inf_smem + InferLds::w2))[i * 8 + j] = a.W[2][c];
          }
      }
    for (int i = tid; i < INF_K * 64; i += INF_NT)
      {
        const int l = i & 63, k = i >> 6;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          ((uint16_t *)(inf_smem + InferLds::w3))[i * 8 + j] =
            (l & 31) < NET_OUT ? a.W[3][(l & 31) * NET_H + hidden_of(k, l >> 5, j)] : 0;
      }
    for (int i = tid; i < 3 * NET_H; i += INF_NT)
      bias[i] = a.b[i / NET_H][i % NET_H];
    if (tid < NET_OUT)
      {
        bias[3 * NET_H + tid]           = a.b[3][tid];
        bias[3 * NET_H + NET_OUT + tid] = a.out_scale[tid];
      }
    __syncthreads();

    const uint32_t N = (uint32_t)a.fp.n_nodes;
    const int      h = lane >> 5, sg = h ? -1 : 1;
    const uint32_t nx = a.fp.nn[0], ny = a.fp.nn[1], nz = a.fp.nn[2];
    // 32-bit byte offsets into each array (mlp_infer_covers)
    const char *d2 = a.ws + a.l.d2, *ds = a.ws + a.l.ds, *v4 = a.ws + a.l.v4;
    const char *de = a.ws + a.l.de, *be = a.ws + a.l.be;
    float(*ysh)[8] = (float(*)[8])(inf_smem + InferLds::y) + 32 * wave;

    // each XCD (blockIdx % 8) works through a contiguous eighth of the nodes:
    // the planes that its stencils share stay in its L2
    const uint32_t tiles = (N + 31) / 32, per = (tiles + 7) / 8;
    for (uint32_t t = (blockIdx.x / 8) * INF_WAVES + wave; t < per;
         t += gridDim.x / 8 * INF_WAVES)
      {
        const uint32_t tile = (blockIdx.x % 8) * per + t;
        if (tile >= tiles)
          break;
        const uint32_t first = tile * 32;
        const uint32_t node  = min(first + (uint32_t)(lane & 31), N - 1);
        const uint32_t row = node / nx, x = node - row * nx, z = row / ny, y = row - z * ny;
        // neighbours towards the half's side of the stencil, clamped
        auto step = [](uint32_t i, int d, uint32_t n) {
          return (uint32_t)min(max((int)i + d, 0), (int)n - 1);
        };
        uint32_t xs[3], rows[5];
#pragma unroll
        for (int d = 0; d < 3; ++d)
          {
            xs[d]   = step(x, sg * (d - 1), nx);
            rows[d] = (step(z, -sg, nz) * ny + step(y, sg * (d - 1), ny)) * nx;
          }
        rows[3] = (z * ny + step(y, -sg, ny)) * nx;
        rows[4] = row * nx;
        const int      i1 = a.top2[2 * (int64_t)node], i2 = a.top2[2 * (int64_t)node + 1];
        const uint32_t p1 = (uint32_t)i1 * N, p2 = (uint32_t)i2 * N;

        // ---- the half's share of the stencil
        constexpr int PTS = 13;
        double        d[PTS + 1][5];
        uint32_t      w[PTS + 1][3]; // bf16 (c, mu), (s, eta_i1), (eta_i2, -)
#pragma unroll
        for (int i = 0; i < PTS + 1; ++i)
          {
            const uint32_t q  = rows[i / 3] + xs[i % 3];
            const double2  dm = *(const double2 *)(d2 + 16 * q);
            d[i][0]           = dm.x;
            d[i][1]           = dm.y;
            d[i][2]           = *(const double *)(ds + 8 * q);
            d[i][3]           = *(const double *)(de + 8 * (p1 + q));
            d[i][4]           = *(const double *)(de + 8 * (p2 + q));
            const uint2 v     = *(const uint2 *)(v4 + 8 * q);
            const uint32_t e1 = *(const uint16_t *)(be + 2 * (p1 + q));
            w[i][0]           = v.x;
            w[i][1]           = v.y | (e1 << 16);
            w[i][2]           = *(const uint16_t *)(be + 2 * (p2 + q));
          }
        double ss = 0.0;
#pragma unroll
        for (int i = 0; i < PTS; ++i)
#pragma unroll
          for (int f = 0; f < 5; ++f)
            ss += d[i][f] * d[i][f];
        double sc = 0.0; // the centre once per node
#pragma unroll
        for (int f = 0; f < 5; ++f)
          sc += d[PTS][f] * d[PTS][f];
        ss += h ? sc : 0.0;
        ss += __shfl_xor(ss, 32, 64);
        const double ls  = sqrt(ss / 135.0) + a.fp.inc_floor;
        const double inv = 1.0 / ls;

        // ---- operands of the first layer: 10 entries per point, then the
        // centre's 5 and feature 270 or 271
        uint32_t xw[4 * INF_K0];
        auto     pack = [](float lo, float hi) {
          typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
          bf16x2         v;
          v[0] = (__bf16)lo;
          v[1] = (__bf16)hi;
          return __builtin_bit_cast(uint32_t, v);
        };
#pragma unroll
        for (int i = 0; i < PTS; ++i)
          {
            xw[5 * i]     = w[i][0];
            xw[5 * i + 1] = w[i][1];
            xw[5 * i + 2] = w[i][2] | (pack((float)(d[i][0] * inv), 0.f) << 16);
            xw[5 * i + 3] = pack((float)(d[i][1] * inv), (float)(d[i][2] * inv));
            xw[5 * i + 4] = pack((float)(d[i][3] * inv), (float)(d[i][4] * inv));
          }
        {
          const float extra = h ? (float)log10(ls * a.fp.inc_scale) :
                                  (float)(a.fp.dt * a.fp.dt_scale);
          const uint32_t x270 = pack(extra, 0.f);
          const double  *c    = d[PTS];
          xw[5 * PTS]         = h ? pack((float)(c[0] * inv), (float)(c[1] * inv)) : w[PTS][0];
          xw[5 * PTS + 1]     = h ? pack((float)(c[2] * inv), (float)(c[3] * inv)) : w[PTS][1];
          xw[5 * PTS + 2] = (h ? pack((float)(c[4] * inv), 0.f) : w[PTS][2]) | (x270 << 16);
        }
        uint4 x0[INF_K0], x1[INF_K], x2[INF_K];
#pragma unroll
        for (int k = 0; k < INF_K0; ++k)
          x0[k] = make_uint4(xw[4 * k], xw[4 * k + 1], xw[4 * k + 2], xw[4 * k + 3]);

        infer_layer<INF_K0>(inf_smem + InferLds::w0, bias, x0, x1, lane);
        infer_layer<INF_K>(inf_smem + InferLds::w1, bias + NET_H, x1, x2, lane);
        infer_layer<INF_K>(inf_smem + InferLds::w2, bias + 2 * NET_H, x2, x1, lane);
        f32x16 acc;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          acc[r] = 0.f;
#pragma unroll
        for (int k = 0; k < INF_K; ++k)
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            __builtin_bit_cast(bf16x8, ((const uint4 *)(inf_smem + InferLds::w3))[64 * k + lane]),
            __builtin_bit_cast(bf16x8, x1[k]), acc, 0, 0, 0);

        // ---- u_pred of the 32 nodes: the corrections go to the wave's rows
        // in LDS (lanes 0..31 hold outputs 0..3), then one entry per lane
        if (h == 0)
          {
#pragma unroll
            for (int k = 0; k < NET_OUT; ++k)
              ysh[lane][k] = bias[3 * NET_H + NET_OUT + k] * (acc[k] + bias[3 * NET_H + k]);
            ysh[lane][4]                 = (float)ls;
            ((int *)ysh[lane])[5]        = i1;
            ((int *)ysh[lane])[6]        = i2;
            if (first + lane < N)
              a.lscale[node] = (float)ls;
          }
        __builtin_amdgcn_wave_barrier();
        const int64_t e0 = (int64_t)first * NC;
#pragma unroll
        for (int j = 0; j < NC / 2; ++j)
          {
            const int     i  = lane + 64 * j;
            const int     r  = i / NC, c = i - r * NC;
            if (first + r < N)
              {
                double    u  = 2.0 * a.u_cur[e0 + i] - a.u_prev[e0 + i];
                const int j1 = ((const int *)ysh[r])[5], j2 = ((const int *)ysh[r])[6];
                // with one order parameter i1 = i2: output 2 only
                const int k = c < 2 ? c : (c == 2 + j1 ? 2 : (c == 2 + j2 ? 3 : -1));
                if (k >= 0)
                  u += (double)ysh[r][4] * (double)ysh[r][k];
                a.out[e0 + i] = u;
              }
          }
        if constexpr (NC % 2 != 0)
          {
            const int i = lane + 64 * (NC / 2), r = i / NC, c = i - r * NC;
            if (i < 32 * NC && first + r < N)
              {
                double    u  = 2.0 * a.u_cur[e0 + i] - a.u_prev[e0 + i];
                const int j1 = ((const int *)ysh[r])[5], j2 = ((const int *)ysh[r])[6];
                const int k  = c < 2 ? c : (c == 2 + j1 ? 2 : (c == 2 + j2 ? 3 : -1));
                if (k >= 0)
                  u += (double)ysh[r][4] * (double)ysh[r][k];
                a.out[e0 + i] = u;
              }
          }
        __builtin_amdgcn_wave_barrier();
      }
  }

  // feature rows (mlp_features.hip) of the nodes of the last k_fields, from its
  // arrays instead of u: for programs that look at the rows of a prediction.  32
  // nodes per workgroup, 8 lanes per node; the sums of squares in k_features'
  // order, so that both give the same bits.
  constexpr int ROW_NODES = 32;
  __global__ void __launch_bounds__(256) k_rows(InferArgs a, uint16_t *__restrict__ X)
  {
    constexpr int XS = NET_IN + 8;
    __shared__ __align__(16) uint16_t rows[ROW_NODES * XS];
    const int64_t N = a.fp.n_nodes, n0 = (int64_t)blockIdx.x * ROW_NODES;
    const int     r = threadIdx.x >> 3, sub = threadIdx.x & 7;
    const int64_t node = min(n0 + r, N - 1);
    const int     nx = a.fp.nn[0], ny = a.fp.nn[1], nz = a.fp.nn[2];
    const int     x = (int)(node % nx), y = (int)(node / nx % ny), z = (int)(node / nx / ny);
    const double   *d2 = (const double *)(a.ws + a.l.d2), *ds = (const double *)(a.ws + a.l.ds);
    const uint16_t *v4 = (const uint16_t *)(a.ws + a.l.v4), *be = (const uint16_t *)(a.ws + a.l.be);
    const double   *de = (const double *)(a.ws + a.l.de);
    auto            plane = [&](int i) { return min(max(i, 0), a.fp.n_comp - 3) * N; };
    const int64_t   p1 = plane(a.top2[2 * node]), p2 = plane(a.top2[2 * node + 1]);
    auto            at = [&](int s) {
      const int xx = min(max(x + s % 3 - 1, 0), nx - 1), yy = min(max(y + s / 3 % 3 - 1, 0), ny - 1);
      const int zz = min(max(z + s / 9 - 1, 0), nz - 1);
      return ((int64_t)zz * ny + yy) * nx + xx;
    };
    double ss = 0.0;
    for (int s = sub; s < 27; s += 8)
      {
        const int64_t q    = at(s);
        const double  d[5] = {d2[2 * q], d2[2 * q + 1], ds[q], de[p1 + q], de[p2 + q]};
#pragma unroll
        for (int f = 0; f < 5; ++f)
          ss += d[f] * d[f];
      }
    ss += __shfl_xor(ss, 1, 64);
    ss += __shfl_xor(ss, 2, 64);
    ss += __shfl_xor(ss, 4, 64);
    const double ls = sqrt(ss / 135.0) + a.fp.inc_floor, inv = 1.0 / ls;
    uint16_t    *row = rows + r * XS;
    for (int s = sub; s < 27; s += 8)
      {
        const int64_t q  = at(s);
        uint16_t     *o  = row + 10 * s;
        o[0] = v4[4 * q];
        o[1] = v4[4 * q + 1];
        o[2] = v4[4 * q + 2];
        o[3] = be[p1 + q];
        o[4] = be[p2 + q];
        o[5] = f2bf((float)(d2[2 * q] * inv));
        o[6] = f2bf((float)(d2[2 * q + 1] * inv));
        o[7] = f2bf((float)(ds[q] * inv));
        o[8] = f2bf((float)(de[p1 + q] * inv));
        o[9] = f2bf((float)(de[p2 + q] * inv));
      }
    if (sub == 0)
      {
        row[270] = f2bf((float)(a.fp.dt * a.fp.dt_scale));
        row[271] = f2bf((float)log10(ls * a.fp.inc_scale));
      }
    __syncthreads();
    constexpr int CH = NET_IN / 8; // 16-byte pieces of a row
    for (int i = threadIdx.x; i < ROW_NODES * CH; i += 256)
      {
        const int m = i / CH, c = i - CH * m;
        if (n0 + m < N)
          *(uint4 *)(X + (n0 + m) * NET_IN + 8 * c) = *(const uint4 *)(rows + m * XS + 8 * c);
      }
  }

  int64_t mlp_infer_workspace(const FeatParams &fp)
  {
    // k_infer's 32-bit byte offsets must reach every array of the workspace
    const int64_t most = 8 * fp.n_nodes * (fp.n_comp - 2 < 2 ? 2 : fp.n_comp - 2);
    if (most >= (int64_t)1 << 32 || fp.n_nodes >= (int64_t)1 << 28)
      return 0;
    return infer_ws(fp.n_nodes, fp.n_comp - 2).total;
  }

  void mlp_infer(hipStream_t s, const FeatParams &fp, const double *u_prev, const double *u_cur,
                 const uint16_t *const *W, const float *const *b, const float *out_scale,
                 int *top2, float *lscale, double *out, void *ws)
  {
    InferArgs a{};
    a.fp     = fp;
    a.u_prev = u_prev;
    a.u_cur  = u_cur;
    a.top2   = top2;
    a.lscale = lscale;
    for (int l = 0; l < 4; ++l)
      {
        a.W[l] = W[l];
        a.b[l] = b[l];
      }
    a.out_scale = out_scale;
    a.out       = out;
    a.ws        = (char *)ws;
    a.l         = infer_ws(fp.n_nodes, fp.n_comp - 2);
    const unsigned nf    = (unsigned)((fp.n_nodes + FLD_NODES - 1) / FLD_NODES);
    // one workgroup per CU, the same number on each of the 8 XCDs
    const int64_t  per = (fp.n_nodes + 255) / 256, wgs = (per + INF_WAVES - 1) / INF_WAVES;
    const unsigned ni  = 8 * (unsigned)(wgs < 32 ? wgs : 32);
    switch (fp.n_comp)
      {
#define HPS_NC(N)                                             \
  case N:                                                     \
    k_fields<N><<<nf, 256, 0, s>>>(a);                        \
    k_infer<N><<<ni, INF_NT, InferLds::total, s>>>(a);        \
    break;
        HPS_NC(3) HPS_NC(4) HPS_NC(5) HPS_NC(6) HPS_NC(7) HPS_NC(8)
        HPS_NC(9) HPS_NC(10) HPS_NC(11) HPS_NC(12) HPS_NC(13) HPS_NC(14)
#undef HPS_NC
      }
  }

  void mlp_infer_rows(hipStream_t s, const FeatParams &fp, const int *top2, const void *ws,
                      uint16_t *X)
  {
    InferArgs a{};
    a.fp   = fp;
    a.top2 = const_cast<int *>(top2);
    a.ws   = (char *)const_cast<void *>(ws);
    a.l    = infer_ws(fp.n_nodes, fp.n_comp - 2);
    k_rows<<<(unsigned)((fp.n_nodes + ROW_NODES - 1) / ROW_NODES), 256, 0, s>>>(a, X);
  }
} // namespace hps
