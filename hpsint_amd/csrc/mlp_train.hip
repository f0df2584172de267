// mlp_train.hip -- one training step of the learned Newton predictor's
// 272-128-128-128-4 network in three launches.
//
//   k_train   forward, MSE loss and the backward pass down to every layer's
//             pre-activation gradient, 64 rows per workgroup;
//   k_wgrad   all weight gradients, split over the rows;
//   k_update  sums of the splits, bias gradients and the Adam step of every
//             parameter.
// The roundings to bf16 are those of the layer-by-layer kernels (mlp.hip):
// activations, dY and the back-propagated gradients; accumulation in FP32.
//
// A batch of 16384 rows took 0.91 ms in 31 launches: 0.69 in the four
// weight-gradient products, whose 48 workgroups loaded both operands 2 bytes
// at a time along the contraction, 0.09 in column sums of one workgroup per
// column.  Now 0.077 ms: k_train 0.024, k_wgrad 0.028, k_update 0.005 and the
// wait for the loss.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "mlp.hpp"
#include "mlp_net.hpp"

namespace hps
{
  typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
  typedef short  short4v __attribute__((ext_vector_type(4)));

  constexpr int TR_ROWS = 64, TR_NT = 512, TR_TILES = TR_ROWS / 16;
  // LDS rows: padded to an odd number of 16-byte pieces (bank spread)
  constexpr int TR_XS = NET_IN + 8, TR_HS = NET_H + 8;
  constexpr int TR_HB = TR_ROWS * TR_HS; // entries of an activation tile

  // workspace: activations and gradients of the batch, bf16
  struct TrainWs
  {
    int64_t h[3], dz[3], dy, wpart, bpart, lpart, total; // byte offsets
    int     nwg, splits;
  };
  constexpr int TR_NW = NET_IN * NET_H + 2 * NET_H * NET_H + NET_H * NET_OUT; // weights
  constexpr int TR_NB = 3 * NET_H + NET_OUT;                                  // biases

  // splits of the weight gradients' contraction: 512 rows each (11 column
  // tiles then make 352 workgroups at 16384 rows), at most 32 (their partial
  // sums are 280 KB each)
  static TrainWs train_ws(int M)
  {
    TrainWs       w{};
    const int64_t act = (int64_t)M * NET_H * 2;
    w.nwg             = (M + TR_ROWS - 1) / TR_ROWS;
    w.splits          = (M + 511) / 512;
    w.splits          = w.splits < 1 ? 1 : (w.splits > 32 ? 32 : w.splits);
    int64_t o         = 0;
    for (int l = 0; l < 3; ++l)
      {
        w.h[l] = o;
        o += act;
        w.dz[l] = o;
        o += act;
      }
    w.dy = o;
    o += (int64_t)M * NET_OUT * 2;
    o       = (o + 15) & ~(int64_t)15;
    w.wpart = o;
    o += (int64_t)w.splits * TR_NW * 4;
    w.bpart = o;
    o += (int64_t)w.nwg * TR_NB * 4;
    w.lpart = o;
    o += (int64_t)w.nwg * 4;
    w.total = o;
    return w;
  }

  struct TrainArgs
  {
    int             M;
    const uint16_t *X;
    const float    *T;
    const uint16_t *W[4]; // bf16
    const float    *b[4];
    char           *ws;
    TrainWs         l;
  };

  // A operands of v_mfma_f32_16x16x32_bf16 for this wave's 16 rows: lane l
  // holds row l & 15, inputs 8 (l >> 4) .. + 7 of each 32
  template <int K>
  __device__ __forceinline__ void load_rows(const uint16_t *__restrict__ W, int wave, int lane,
                                            bf16x8 *f)
  {
    const uint16_t *row = W + (16 * wave + (lane & 15)) * K + 8 * (lane >> 4);
#pragma unroll
    for (int k = 0; k < K / 32; ++k)
      f[k] = __builtin_bit_cast(bf16x8, *(const uint4 *)(row + 32 * k));
  }
  // the same of W^T (128 x 128): row = input, contraction over the outputs
  __device__ __forceinline__ void load_cols(const uint16_t *__restrict__ W, int wave, int lane,
                                            bf16x8 *f)
  {
    const uint16_t *col = W + 16 * wave + (lane & 15) + 8 * (lane >> 4) * NET_H;
#pragma unroll
    for (int k = 0; k < NET_H / 32; ++k)
      {
        uint16_t e[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          e[j] = col[(32 * k + j) * NET_H];
        f[k] = __builtin_bit_cast(bf16x8, make_uint4(e[0] | ((uint32_t)e[1] << 16),
                                                     e[2] | ((uint32_t)e[3] << 16),
                                                     e[4] | ((uint32_t)e[5] << 16),
                                                     e[6] | ((uint32_t)e[7] << 16)));
      }
  }

  // acc[n]: of tile rows 16 n + (l & 15), this wave's outputs 4 (l >> 4) + r
  template <int K>
  __device__ __forceinline__ void product(const bf16x8 *f, const uint16_t *src, int stride,
                                          int lane, f32x4 *acc)
  {
    const uint16_t *row = src + (lane & 15) * stride + 8 * (lane >> 4);
#pragma unroll
    for (int k = 0; k < K / 32; ++k)
#pragma unroll
      for (int n = 0; n < TR_TILES; ++n)
        acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          f[k], __builtin_bit_cast(bf16x8, *(const uint4 *)(row + 16 * n * stride + 32 * k)),
          acc[n], 0, 0, 0);
  }
  __device__ __forceinline__ void clear(f32x4 *acc)
  {
#pragma unroll
    for (int n = 0; n < TR_TILES; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        acc[n][r] = 0.f;
  }

  __global__ void __launch_bounds__(TR_NT, 2) k_train(TrainArgs a)
  {
    extern __shared__ __align__(16) char tr_smem[];
    uint16_t *xr = (uint16_t *)tr_smem;             // [64][TR_XS] features, later dz1
    uint16_t *h  = xr + TR_ROWS * TR_XS;            // [3][64][TR_HS]
    uint16_t *dz = h + 3 * TR_HB;                   // [2][64][TR_HS]: dz3, dz2
    uint16_t *dy = dz + 2 * TR_HB;                  // [64][NET_OUT]
    float    *lsum = (float *)(dy + TR_ROWS * NET_OUT);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m0 = (int)blockIdx.x * TR_ROWS, rows = min(TR_ROWS, a.M - m0);

    // weights of the wave's 16 rows of every product
    bf16x8  w0[NET_IN / 32], w1[NET_H / 32], w2[NET_H / 32], w2t[NET_H / 32], w1t[NET_H / 32];
    bf16x4  w0t, w3t; // inputs 256..271 of layer 0; W3^T
    load_rows<NET_IN>(a.W[0], wave, lane, w0);
    w0t = __builtin_bit_cast(bf16x4, *(const uint2 *)(a.W[0] + (16 * wave + (lane & 15)) * NET_IN +
                                                      256 + 4 * (lane >> 4)));
    for (int i = tid; i < TR_ROWS * (NET_IN / 8); i += TR_NT)
      {
        const int r = i / (NET_IN / 8), c = i - r * (NET_IN / 8);
        uint4     v = make_uint4(0, 0, 0, 0);
        if (r < rows)
          v = *(const uint4 *)(a.X + (int64_t)(m0 + r) * NET_IN + 8 * c);
        *(uint4 *)(xr + r * TR_XS + 8 * c) = v;
      }
    load_rows<NET_H>(a.W[1], wave, lane, w1);
    load_rows<NET_H>(a.W[2], wave, lane, w2);
    load_cols(a.W[2], wave, lane, w2t);
    load_cols(a.W[1], wave, lane, w1t);
    {
      uint16_t e[4] = {0, 0, 0, 0};
      if (lane < 16)
#pragma unroll
        for (int j = 0; j < NET_OUT; ++j)
          e[j] = a.W[3][j * NET_H + 16 * wave + lane];
      w3t = __builtin_bit_cast(bf16x4, make_uint2(e[0] | ((uint32_t)e[1] << 16),
                                                  e[2] | ((uint32_t)e[3] << 16)));
    }
    const int o = 16 * wave + 4 * (lane >> 4); // the lane's 4 outputs
    __syncthreads();

    // ---- forward
    f32x4 acc[TR_TILES];
    auto  hidden = [&](const float *bias, uint16_t *dst) {
#pragma unroll
      for (int n = 0; n < TR_TILES; ++n)
        {
          bf16x4 v;
#pragma unroll
          for (int r = 0; r < 4; ++r)
            v[r] = (__bf16)tanh_fast(acc[n][r] + bias[o + r]);
          *(bf16x4 *)(dst + (16 * n + (lane & 15)) * TR_HS + o) = v;
        }
    };
    clear(acc);
    product<NET_IN>(w0, xr, TR_XS, lane, acc);
#pragma unroll
    for (int n = 0; n < TR_TILES; ++n)
      acc[n] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
        __builtin_bit_cast(short4v, w0t),
        __builtin_bit_cast(short4v, *(const uint2 *)(xr + (16 * n + (lane & 15)) * TR_XS + 256 +
                                                     4 * (lane >> 4))),
        acc[n], 0, 0, 0);
    hidden(a.b[0], h);
    __syncthreads();
    clear(acc);
    product<NET_H>(w1, h, TR_HS, lane, acc);
    hidden(a.b[1], h + TR_HB);
    __syncthreads();
    clear(acc);
    product<NET_H>(w2, h + TR_HB, TR_HS, lane, acc);
    hidden(a.b[2], h + 2 * TR_HB);
    __syncthreads();
    // ---- output layer, loss and dY: wave n < 4 takes tile rows 16 n ...
    if (wave < TR_TILES)
      {
        f32x4           y    = {0.f, 0.f, 0.f, 0.f};
        const uint16_t *row  = h + 2 * TR_HB + (16 * wave + (lane & 15)) * TR_HS + 8 * (lane >> 4);
        const uint16_t *wrow = a.W[3] + (lane & (NET_OUT - 1)) * NET_H + 8 * (lane >> 4);
#pragma unroll
        for (int k = 0; k < NET_H / 32; ++k)
          {
            uint4 w = *(const uint4 *)(wrow + 32 * k);
            if ((lane & 15) >= NET_OUT)
              w = make_uint4(0, 0, 0, 0);
            y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, w),
              __builtin_bit_cast(bf16x8, *(const uint4 *)(row + 32 * k)), y, 0, 0, 0);
          }
        float s = 0.f;
        if (lane < 16) // outputs 0..3 of tile row 16 wave + lane
          {
            const int   r   = 16 * wave + lane;
            const float inv = 1.f / (float)((int64_t)a.M * NET_OUT);
            bf16x4      v;
#pragma unroll
            for (int k = 0; k < NET_OUT; ++k)
              {
                float d = 0.f;
                if (r < rows)
                  d = (y[k] + a.b[3][k]) - a.T[(int64_t)(m0 + r) * NET_OUT + k];
                s += d * d;
                v[k] = (__bf16)(2.f * d * inv);
              }
            *(bf16x4 *)(dy + r * NET_OUT) = v;
            s *= inv;
          }
#pragma unroll
        for (int m = 8; m > 0; m >>= 1)
          s += __shfl_down(s, m, 16);
        if (lane == 0)
          lsum[wave] = s;
      }
    __syncthreads();
    // ---- backward: dz_l = (dz_{l+1} W) (1 - h_l^2)
    auto slope = [&](const uint16_t *hl, uint16_t *dst) {
#pragma unroll
      for (int n = 0; n < TR_TILES; ++n)
        {
          const int    r = 16 * n + (lane & 15);
          const bf16x4 v = *(const bf16x4 *)(hl + r * TR_HS + o);
          bf16x4       g;
#pragma unroll
          for (int k = 0; k < 4; ++k)
            {
              const float t = (float)v[k];
              g[k]          = (__bf16)(acc[n][k] * (1.f - t * t));
            }
          *(bf16x4 *)(dst + r * TR_HS + o) = g;
        }
    };
    clear(acc);
#pragma unroll
    for (int n = 0; n < TR_TILES; ++n)
      {
        uint2 v = make_uint2(0, 0);
        if (lane < 16)
          v = *(const uint2 *)(dy + (16 * n + lane) * NET_OUT);
        acc[n] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
          __builtin_bit_cast(short4v, w3t), __builtin_bit_cast(short4v, v), acc[n], 0, 0, 0);
      }
    slope(h + 2 * TR_HB, dz);
    __syncthreads();
    clear(acc);
    product<NET_H>(w2t, dz, TR_HS, lane, acc);
    slope(h + TR_HB, dz + TR_HB);
    __syncthreads();
    clear(acc);
    product<NET_H>(w1t, dz + TR_HB, TR_HS, lane, acc);
    slope(h, xr); // the features are no longer needed
    __syncthreads();

    // ---- to memory: activations and gradients (16-byte pieces), bias
    // gradients and loss of the tile
    constexpr int PC = NET_H / 8;
    for (int i = tid; i < 6 * TR_ROWS * PC; i += TR_NT)
      {
        const int t = i / (TR_ROWS * PC), q = i - t * (TR_ROWS * PC);
        const int r = q / PC, c = q - r * PC;
        if (r >= rows)
          continue;
        const uint16_t *src = t < 3 ? h + t * TR_HB : (t == 3 ? xr : dz + (5 - t) * TR_HB);
        const int64_t   off = t == 0 ? a.l.h[0] :
                                       (t == 1 ? a.l.h[1] :
                                                 (t == 2 ? a.l.h[2] :
                                                           (t == 3 ? a.l.dz[0] :
                                                                     (t == 4 ? a.l.dz[1] :
                                                                               a.l.dz[2]))));
        *(uint4 *)(a.ws + off + ((int64_t)(m0 + r) * NET_H + 8 * c) * 2) =
          *(const uint4 *)(src + r * TR_HS + 8 * c);
      }
    if (tid < rows)
      *(uint2 *)(a.ws + a.l.dy + (int64_t)(m0 + tid) * NET_OUT * 2) =
        *(const uint2 *)(dy + tid * NET_OUT);
    float *bpart = (float *)(a.ws + a.l.bpart) + (int64_t)blockIdx.x * TR_NB;
    if (tid < TR_NB)
      {
        const uint16_t *src = tid < NET_H     ? xr + tid :
                              tid < 2 * NET_H ? dz + TR_HB + (tid - NET_H) :
                              tid < 3 * NET_H ? dz + (tid - 2 * NET_H) :
                                                dy + (tid - 3 * NET_H);
        const int       st  = tid < 3 * NET_H ? TR_HS : NET_OUT;
        float           s   = 0.f;
#pragma unroll 16
        for (int r = 0; r < TR_ROWS; ++r)
          s += bf2f(src[r * st]);
        bpart[tid] = s;
      }
    if (tid == 0)
      ((float *)(a.ws + a.l.lpart))[blockIdx.x] = (lsum[0] + lsum[1]) + (lsum[2] + lsum[3]);
  }

  // k_wgrad: gW_l = dz_l^T a_l.  A workgroup of 4 waves forms 128 outputs x 64
  // inputs (a wave 32 x 64) over its split of the rows, 64 rows at a time:
  // row pairs are loaded 16 bytes wide, packed and stored transposed, so that
  // the operands' contraction runs along LDS rows.
  constexpr int WG_MB = 64, WG_NB = 64, WG_S = WG_MB + 8;
  constexpr int WG_TILES = (NET_IN + WG_NB - 1) / WG_NB + 3 * (NET_H / WG_NB);
  __global__ void __launch_bounds__(256) k_wgrad(TrainArgs a)
  {
    __shared__ __align__(16) uint16_t As[NET_H][WG_S], Bs[WG_NB][WG_S];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // layer and first input of this column tile
    int           t  = (int)blockIdx.x, l = 0;
    constexpr int T0 = (NET_IN + WG_NB - 1) / WG_NB;
    if (t >= T0)
      {
        l = 1 + (t - T0) / (NET_H / WG_NB);
        t = (t - T0) % (NET_H / WG_NB);
      }
    const int       c0 = t * WG_NB, n_in = l == 0 ? NET_IN : NET_H;
    const int       n_out = l == 3 ? NET_OUT : NET_H;
    const int       ncol  = min(WG_NB, n_in - c0);
    const int64_t   zo = l == 0 ? a.l.dz[0] : (l == 1 ? a.l.dz[1] : (l == 2 ? a.l.dz[2] : a.l.dy));
    const uint16_t *Z  = (const uint16_t *)(a.ws + zo);
    const uint16_t *B  = l == 0 ? a.X :
                                  (const uint16_t *)(a.ws + (l == 1 ? a.l.h[0] :
                                                                      (l == 2 ? a.l.h[1] : a.l.h[2])));
    const int per   = ((a.M + a.l.splits - 1) / a.l.splits + WG_MB - 1) / WG_MB * WG_MB;
    const int mbeg  = (int)blockIdx.y * per, mend = min(a.M, mbeg + per);

    // staged units: (row pair, 8 columns); A: 32 pairs x 16, B: 32 pairs x 8
    uint4 ra[2][2], rb[2];
    auto  load8 = [](const uint16_t *p, bool ok) {
      return ok ? *(const uint4 *)p : make_uint4(0, 0, 0, 0);
    };
    auto fetch = [&](int m) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
        {
          const int unit = tid + 256 * u, pr = unit >> 4, oc = unit & 15;
#pragma unroll
          for (int e = 0; e < 2; ++e)
            {
              const int r = m + 2 * pr + e;
              if (l < 3)
                ra[u][e] = load8(Z + (int64_t)r * NET_H + 8 * oc, r < mend);
              else // dY: rows of 4 values
                {
                  ra[u][e] = make_uint4(0, 0, 0, 0);
                  if (oc == 0 && r < mend)
                    {
                      const uint2 v = *(const uint2 *)(Z + (int64_t)r * NET_OUT);
                      ra[u][e]      = make_uint4(v.x, v.y, 0, 0);
                    }
                }
            }
        }
      const int pr = tid >> 3, oc = tid & 7;
#pragma unroll
      for (int e = 0; e < 2; ++e)
        {
          const int r = m + 2 * pr + e;
          rb[e]       = load8(B + (int64_t)r * n_in + c0 + 8 * oc, r < mend && 8 * oc < ncol);
        }
    };
    // rows 2 p, 2 p + 1 of 8 columns as 8 pairs, transposed
    auto stage = [&](uint16_t (*S)[WG_S], int pr, int oc, const uint4 &v0, const uint4 &v1) {
      const uint32_t x0[4] = {v0.x, v0.y, v0.z, v0.w}, x1[4] = {v1.x, v1.y, v1.z, v1.w};
#pragma unroll
      for (int j = 0; j < 4; ++j)
        {
          *(uint32_t *)&S[8 * oc + 2 * j][2 * pr] = (x0[j] & 0xFFFFu) | (x1[j] << 16);
          *(uint32_t *)&S[8 * oc + 2 * j + 1][2 * pr] = (x0[j] >> 16) | (x1[j] & 0xFFFF0000u);
        }
    };
    f32x16 acc[2];
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[n][r] = 0.f;
    if (mbeg < mend)
      fetch(mbeg);
    for (int m = mbeg; m < mend; m += WG_MB)
      {
#pragma unroll
        for (int u = 0; u < 2; ++u)
          stage(As, (tid + 256 * u) >> 4, (tid + 256 * u) & 15, ra[u][0], ra[u][1]);
        stage(Bs, tid >> 3, tid & 7, rb[0], rb[1]);
        __syncthreads();
        if (m + WG_MB < mend)
          fetch(m + WG_MB);
        if (32 * wave < n_out)
#pragma unroll
          for (int k = 0; k < WG_MB / 16; ++k)
            {
              const bf16x8 f = __builtin_bit_cast(
                bf16x8, *(const uint4 *)&As[32 * wave + (lane & 31)][16 * k + 8 * (lane >> 5)]);
#pragma unroll
              for (int n = 0; n < 2; ++n)
                acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                  f,
                  __builtin_bit_cast(
                    bf16x8, *(const uint4 *)&Bs[32 * n + (lane & 31)][16 * k + 8 * (lane >> 5)]),
                  acc[n], 0, 0, 0);
            }
        __syncthreads();
      }
    // this split's partial sums: layers back to back, row-major
    const int first = l == 0 ? 0 : NET_IN * NET_H + (l - 1) * NET_H * NET_H;
    float    *out = (float *)(a.ws + a.l.wpart) + (int64_t)blockIdx.y * TR_NW + first;
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        {
          const int row = 32 * wave + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
          const int col = 32 * n + (lane & 31);
          if (row < n_out && col < ncol)
            out[row * n_in + c0 + col] = acc[n][r];
        }
  }

  struct UpdateArgs
  {
    const float *wpart, *bpart;
    int          splits, nwg;
    float       *p[8], *m1[8], *m2[8]; // weights of the 4 layers, then biases
    uint16_t    *Wb[4];
    float        lr, b1, b2, eps, c1, c2;
  };

  // one weight per thread in the first blocks, then one bias per wave
  constexpr int UP_WBLK = (TR_NW + 255) / 256;
  __global__ void __launch_bounds__(256) k_update(UpdateArgs a)
  {
    int   layer = 0, i = 0;
    float g = 0.f;
    if (blockIdx.x < UP_WBLK)
      {
        i = (int)blockIdx.x * 256 + threadIdx.x;
        if (i >= TR_NW)
          return;
        const float *p = a.wpart + i;
#pragma unroll 8
        for (int s = 0; s < a.splits; ++s)
          g += p[(int64_t)s * TR_NW];
        constexpr int w1 = NET_IN * NET_H, w = NET_H * NET_H;
        layer = i < w1 ? 0 : (i < w1 + w ? 1 : (i < w1 + 2 * w ? 2 : 3));
        i -= layer == 0 ? 0 : w1 + (layer - 1) * w;
      }
    else
      {
        const int lane = threadIdx.x & 63;
        i = ((int)blockIdx.x - UP_WBLK) * 4 + (threadIdx.x >> 6);
        if (i >= TR_NB)
          return;
#pragma unroll 4
        for (int s = lane; s < a.nwg; s += 64)
          g += a.bpart[(int64_t)s * TR_NB + i];
#pragma unroll
        for (int m = 32; m > 0; m >>= 1)
          g += __shfl_xor(g, m, 64);
        if (lane)
          return;
        layer = 4 + i / NET_H;
        i     = i % NET_H;
      }
    // Adam on the FP32 master values (pointers selected, not indexed: the
    // arguments stay in scalar registers)
    float *p = nullptr, *m1 = nullptr, *m2 = nullptr;
#pragma unroll
    for (int l = 0; l < 8; ++l)
      if (layer == l)
        {
          p  = a.p[l];
          m1 = a.m1[l];
          m2 = a.m2[l];
        }
    const float x = a.b1 * m1[i] + (1.f - a.b1) * g;
    const float y = a.b2 * m2[i] + (1.f - a.b2) * g * g;
    m1[i]         = x;
    m2[i]         = y;
    const float w = p[i] - a.lr * (x / a.c1) / (sqrtf(y / a.c2) + a.eps);
    p[i]          = w;
#pragma unroll
    for (int l = 0; l < 4; ++l)
      if (layer == l)
        a.Wb[l][i] = f2bf(w);
  }

  int64_t mlp_train_workspace(int M, int *n_loss)
  {
    const TrainWs w = train_ws(M);
    if (n_loss)
      *n_loss = w.nwg;
    return w.total;
  }

  const float *mlp_train_step(hipStream_t s, const MlpTrain &t)
  {
    constexpr size_t lds = (TR_ROWS * TR_XS + 5 * TR_HB + TR_ROWS * NET_OUT) * 2 + 64;
    TrainArgs        a{};
    a.M  = t.M;
    a.X  = t.X;
    a.T  = t.T;
    a.ws = (char *)t.ws;
    a.l  = train_ws(t.M);
    UpdateArgs u{};
    for (int l = 0; l < 4; ++l)
      {
        a.W[l]     = t.Wb[l];
        a.b[l]     = t.b[l];
        u.Wb[l]    = t.Wb[l];
        u.p[l]     = t.W[l];
        u.m1[l]    = t.mW[l];
        u.m2[l]    = t.vW[l];
        u.p[4 + l] = t.b[l];
        u.m1[4 + l] = t.mb[l];
        u.m2[4 + l] = t.vb[l];
      }
    u.wpart  = (const float *)(a.ws + a.l.wpart);
    u.bpart  = (const float *)(a.ws + a.l.bpart);
    u.splits = a.l.splits;
    u.nwg    = a.l.nwg;
    u.lr     = t.lr;
    u.b1     = t.b1;
    u.b2     = t.b2;
    u.eps    = t.eps;
    u.c1     = t.c1;
    u.c2     = t.c2;
    k_train<<<a.l.nwg, TR_NT, lds, s>>>(a);
    k_wgrad<<<dim3(WG_TILES, a.l.splits), 256, 0, s>>>(a);
    k_update<<<UP_WBLK + (TR_NB + 3) / 4, 256, 0, s>>>(u);
    return (const float *)(a.ws + a.l.lpart);
  }
} // namespace hps
