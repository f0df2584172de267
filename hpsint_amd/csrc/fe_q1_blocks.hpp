// fe_q1_blocks.hpp -- all node blocks of the 3D Q1 tangent with scalar
// mobility in one pass over the linearisation cache.
//
// The n_c x n_c block of node j is sum_q JxW psi_m'(q) M(q) psi_m(q) over the
// Gauss points of the node's cells (the blocks of
// InverseComponentBlockDiagonalMatrix::do_update, I/lac/preconditioners.h:
// 254-318, from SinteringOperatorGenericQuad, S/operator_sintering_generic.h:
// 104-190).  With scalar mobility its entries are a few sums per node:
//   mass fields, sum JxW f psi^2, of
//     f''_cc, f''_c,eta_i, f''_eta_i,eta_i, eta_i eta_j (i > j);
//   flux fields, sum JxW s psi (grad mu . grad psi), of
//     dM/dc and 2 Mgb (sum_j eta_j - eta_i);
//   the mobility field, sum JxW M |grad psi|^2;
// and the constants sum JxW psi^2 and sum JxW |grad psi|^2.  Applying the
// tangent to one unit input per block column (q1_probe) forms n_c (n_c + 12)
// sums instead, n_c times over the cache.
#pragma once

#include <type_traits>

#include "fe_q1.hpp"

namespace hps
{
  template <int G>
  struct BlockFields
  {
    static constexpr int NC = G + 2;
    // field numbers
    static constexpr int cc = 0, ci = 1, ii = 1 + G, ij = 1 + 2 * G;
    static constexpr int mass = ij + G * (G - 1) / 2; // mass fields before this
    static constexpr int xc = mass, xi = mass + 1, mob = mass + 1 + G;
    static constexpr int count = mob + 1;
    // One sweep over the cache forms the fields [f, sweep_end(f)): their node
    // sums share a workgroup's LDS (49 nodes, 4 lanes per node) and their
    // sums towards the next node plane stay in registers (1 per mass field, 3
    // per flux field, 2 for the mobility field), of which this many fit
    // without spills; the sweeps share them evenly
    static constexpr int held(int f)
    {
      return f < mass ? 1 : (f < mob ? 3 : 2);
    }
    template <typename T>
    static constexpr int sweep_end(int f0)
    {
      constexpr int most = sizeof(T) == 4 ? 76 : 38;
      int           all  = 0;
      for (int f = 0; f < count; ++f)
        all += held(f);
      const int per = (all + (all + most - 1) / most - 1) / ((all + most - 1) / most);
      int       n = 0, f = f0;
      while (f < count && (f == f0 || n + held(f) <= per + 1))
        n += held(f++);
      return f;
    }
  };

  // f(integral_constant 0) ... f(N - 1)
  template <int N, typename F, int I = 0>
  __device__ __forceinline__ void each_grain(F &&f)
  {
    if constexpr (I < N)
      {
        f(std::integral_constant<int, I>{});
        each_grain<N, F, I + 1>(static_cast<F &&>(f));
      }
  }

  namespace blk
  {
    constexpr int WX = 8, WY = 8;           // cells of a workgroup
    constexpr int OX = WX - 1, OY = WY - 1; // nodes it completes per plane
    constexpr int ON = OX * OY;
    constexpr int OS = ON + 2;              // their LDS row (odd: bank spread)
    constexpr int NT = WX * WY * 4;
  } // namespace blk

  // A workgroup completes the blocks of 7 x 7 nodes (x, y) on the node planes
  // z0 .. z0 + zn - 1 and visits all 8 x 8 cells around them, layer by layer,
  // so no node's sum is shared with another workgroup (a cell is visited 1.3
  // times; partial sums would have to be written, read and added for 100
  // entries per node).  Lanes as in the z-column tangent: 4 lanes per cell
  // (x/y Gauss points and corners), both z Gauss points in the lane; z sums
  // in registers, x and y by DPP butterflies, the four cells around a node
  // through LDS.  Sweep [F0, F1) forms those fields and writes the entries
  // made of them.
  // Bound: VALU issue (slots 71 % busy) and HBM (3.7 of a copy's 4.8 TB/s) at 2
  // waves/SIMD; 1.88 M nodes, 8 order parameters, FP32:
  // 0.78 ms where ten q1_probe launches, their fix-ups and the conversion to
  // FP64 took 4.1 ms (the 1.5 GB written take 0.31 ms at the copy rate).
  template <int G, typename T, int F0, int F1>
  __global__ void __launch_bounds__(blk::NT) __attribute__((amdgpu_waves_per_eu(2)))
    q1_blocks(const KParams kp, const T *__restrict__ cache, double *__restrict__ blocks, int zn)
  {
    using BF           = BlockFields<G>;
    using CL           = CacheLayout<3, G, false>;
    constexpr int NC   = G + 2, NF = CL::n_fields, NE = NC * NC;
    constexpr int NS   = F1 - F0;
    constexpr int EPL  = (NE + 63) / 64; // entries per lane
    constexpr int CNT  = 8 * 4 * 8;      // lanes of a cache tile
    constexpr auto in  = [](int f) { return f >= F0 && f < F1; };
    // (the lanes whose node is not completed here write past the 49)
    __shared__ T slots[4][NS][blk::OS];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int bx = tid & 1, by = (tid >> 1) & 1, cx = (tid >> 2) & 7, cy = tid >> 5;
    const int nwx = (kp.nn[0] + blk::OX - 1) / blk::OX, nwy = (kp.nn[1] + blk::OY - 1) / blk::OY;
    const int X0 = (int)(blockIdx.x % nwx) * blk::OX;
    const int Y0 = (int)((blockIdx.x / nwx) % nwy) * blk::OY;
    const int z0 = (int)(blockIdx.x / (nwx * nwy)) * zn, z1 = min(z0 + zn, kp.nn[2]);
    const int gx = X0 - 1 + cx, gy = Y0 - 1 + cy; // the lane's cell
    const bool valid = gx >= 0 && gx < kp.nc[0] && gy >= 0 && gy < kp.nc[1];
    // its corner's node among the completed ones
    const int  ox = cx - 1 + bx, oy = cy - 1 + by;
    const bool owned = ox >= 0 && ox < blk::OX && oy >= 0 && oy < blk::OY;
    T         *slot  = &slots[bx | (by << 1)][0][owned ? oy * blk::OX + ox : blk::ON];
    const int64_t layer = (int64_t)NF * CNT;
    const T      *ccol =
      cache + (valid ? ((int64_t)(gy >> 2) * kp.nt[0] + (gx >> 3)) * kp.tz * layer +
                         (((gx & 7) + 8 * (gy & 3)) * 8 + (bx | (by << 1))) :
                       0);
    const int64_t tile_z = (int64_t)kp.nt[0] * kp.nt[1] * kp.tz * layer;

    // Levels along one direction, with psi = sa, sb at a node's near and far
    // Gauss point and psi' = +-1/h: psi^2 gives sa^2 (near + r far), psi psi'
    // gives +-(sa / h) (near + r1 far), psi'^2 gives (near + far) / h^2.  A
    // factor sa^2 per direction is left to the entries' factors.
    const T r1 = Q1Hat<T>::r, r = T(0.07179676972449082589); // sb / sa and its square
    const T is = T(1.2679491924311227065), iaa = T(1.6076951545867362); // 1 / sa, 1 / sa^2
    const T hx = T(kp.inv_h[0]), hy = T(kp.inv_h[1]), hz = T(kp.inv_h[2]);
    const T ex = bx ? hx * is : -(hx * is), ey = by ? hy * is : -(hy * is), ez = hz * is;
    const T kx = hx * hx * iaa, ky = hy * hy * iaa, kz = hz * hz * iaa;

    // this lane's entries e = lane + 64 j (column by column): field and its
    // factor, factors of the mass and of the stiffness (FP64 also in FP32
    // assembly: w0 times the mass is the largest part of most diagonals)
    int    ef[EPL];
    double eg[EPL], em[EPL], ek[EPL];
#pragma unroll
    for (int j = 0; j < EPL; ++j)
      {
        const int e = lane + 64 * j, b = e / NC, a = e - b * NC; // column, row
        int       f = -1;
        double    g = 1.0, m = 0.0, k = 0.0;
        if (a == 0)
          {
            f = b == 0 ? BF::xc : (b == 1 ? BF::mob : BF::xi + b - 2);
            m = b == 0 ? kp.pp.w0 : 0.0;
          }
        else if (a == 1)
          {
            f = b == 0 ? BF::cc : (b == 1 ? -1 : BF::ci + b - 2);
            g = -1.0;
            m = b == 1 ? kp.pp.w_alg : 0.0;
            k = b == 0 ? -kp.pp.kappa_c : 0.0;
          }
        else if (b == 0)
          {
            f = BF::ci + a - 2;
            g = kp.pp.L;
          }
        else if (b == a)
          {
            f = BF::ii + a - 2;
            g = kp.pp.L;
            m = kp.pp.w0;
            k = kp.pp.L * kp.pp.kappa_p;
          }
        else if (b > 1)
          {
            const int hi = max(a, b) - 2, lo = min(a, b) - 2;
            f            = BF::ij + hi * (hi - 1) / 2 + lo;
            g            = kp.pp.L * 24.0 * kp.pp.B;
          }
        // -1: no field (constant entries go with the first sweep), -2: not
        // of this sweep
        const bool mine = e < NE && (f < 0 ? F0 == 0 : in(f));
        ef[j]           = mine ? (f < 0 ? -1 : f - F0) : -2;
        eg[j]           = g * kp.jxw * 0.24065167645154237;
        em[j]           = m * kp.jxw;
        ek[j]           = k * kp.jxw;
      }

    // sums towards the layer's upper node plane, before the x and y levels:
    // one per mass field, three (d/dx, d/dy, d/dz part) per flux field, two
    // for the mobility field
    constexpr int NM = (BF::mass < F1 ? BF::mass : F1) - F0;     // mass fields here
    constexpr int X0F = BF::mass > F0 ? BF::mass : F0;           // first flux field here
    constexpr int NX = (BF::mob < F1 ? BF::mob : F1) - X0F;      // flux fields here
    T up_m[NM > 0 ? NM : 1], up_x[NX > 0 ? NX : 1][3], up_k[2];
#pragma unroll
    for (int i = 0; i < (NM > 0 ? NM : 1); ++i)
      up_m[i] = T(0);
#pragma unroll
    for (int i = 0; i < (NX > 0 ? NX : 1); ++i)
      up_x[i][0] = up_x[i][1] = up_x[i][2] = T(0);
    up_k[0] = up_k[1] = T(0);

    // FP32: the next layer's cache fields arrive during the current layer
    // (FP64 allocations spill with them).  Fields are zero outside the mesh
    // (which makes every node field zero but those that `on` masks).
    constexpr bool PF = sizeof(T) == 4;
    T    next[2][NF];
    auto request = [&](int k) {
      if (k >= 0 && k < kp.nc[2])
        {
          const T *c = ccol + (int64_t)(k / kp.tz) * tile_z + (int64_t)(k % kp.tz) * layer;
#pragma unroll
          for (int f = 0; f < NF; ++f)
            {
              next[0][f] = valid ? c[f * CNT] : T(0);
              next[1][f] = valid ? c[f * CNT + 4] : T(0);
            }
        }
      else
#pragma unroll
        for (int f = 0; f < NF; ++f)
          next[0][f] = next[1][f] = T(0);
    };
    if constexpr (PF)
      request(z0 - 1);
    for (int k = z0 - 1; k < z1; ++k)
      {
        // ---- cell layer k, between the node planes k and k + 1
        const bool on = valid && k >= 0 && k < kp.nc[2];
        if constexpr (!PF)
          request(k);
        T lin[2][NF];
#pragma unroll
        for (int f = 0; f < NF; ++f)
          {
            lin[0][f] = next[0][f];
            lin[1][f] = next[1][f];
          }
        if (PF && k + 1 < z1)
          request(k + 1);
        // ---- node plane k: what the layer below left plus this layer's
        // lower half; its upper half stays for the next plane.  mass and
        // flux take the field's values at the two Gauss points.
        auto put_slot = [&](int f, T v) { slot[f * blk::OS] = v; };
        auto mass = [&](auto F, T v0, T v1) {
          constexpr int f = F;
          if constexpr (in(f))
            {
              T lo         = up_m[f - F0] + (v0 + r * v1);
              up_m[f - F0] = r * v0 + v1;
              lo += r * xshfl<1>(lo);
              lo += r * xshfl<2>(lo);
              put_slot(f - F0, lo);
            }
        };
        auto flux = [&](auto F, T v0, T v1) {
          constexpr int f = F;
          if constexpr (in(f))
            {
              constexpr int i = f - X0F;
              T             l[3];
#pragma unroll
              for (int d = 0; d < 3; ++d)
                {
                  const T a = v0 * lin[0][CL::grad_mu + d], b = v1 * lin[1][CL::grad_mu + d];
                  if (d < 2)
                    {
                      l[d]       = up_x[i][d] + (a + r * b);
                      up_x[i][d] = r * a + b;
                    }
                  else // psi' of the lower node is -1/h, of the upper 1/h
                    {
                      l[d]       = up_x[i][d] - ez * (a + r1 * b);
                      up_x[i][d] = ez * (r1 * a + b);
                    }
                }
              l[0] = ex * (l[0] + r1 * xshfl<1>(l[0]));
              l[1] += r * xshfl<1>(l[1]);
              l[2] += r * xshfl<1>(l[2]);
              const T p = l[0] + l[2];
              put_slot(f - F0, (p + r * xshfl<2>(p)) + ey * (l[1] + r1 * xshfl<2>(l[1])));
            }
        };
        T S2[2], sum[2], M[2], cc[2], dM[2];
#pragma unroll
        for (int q = 0; q < 2; ++q)
          {
            const T  c = lin[q][CL::c];
            const T *e = lin[q] + CL::eta;
            const T  A = T(kp.pp.A), B = T(kp.pp.B);
            T        pairs = T(0);
            S2[q] = sum[q] = T(0);
#pragma unroll
            for (int i = 0; i < G; ++i)
              {
                S2[q] += e[i] * e[i];
                pairs += e[i] * sum[q]; // sum_{j < i} eta_j
                sum[q] += e[i];
              }
            const T c1 = T(1) - c, c2 = c * c * (c1 * c1);
            const T phi = phi_clamped(c);
            M[q]        = T(kp.pp.Mvol) * phi + T(kp.pp.Mvap) * (T(1) - phi) +
                   T(kp.pp.Msurf) * T(4.0) * c2 + (T(2.0) * T(kp.pp.Mgb)) * pairs;
            M[q]  = on ? M[q] : T(0);
            cc[q] = T(2.0) * A * (c * c) + T(4.0) * A * c * (T(2.0) * c - T(2.0)) +
                    T(2.0) * A * (c1 * c1) + T(2.0) * B;
            dM[q] = (T(kp.pp.Mvol) - T(kp.pp.Mvap)) * (T(30.0) * c2) +
                    T(kp.pp.Msurf) * T(8.0) * c * (T(1.0) - T(3.0) * c + T(2.0) * c * c);
          }
        mass(std::integral_constant<int, BF::cc>{}, on ? cc[0] : T(0), on ? cc[1] : T(0));
        flux(std::integral_constant<int, BF::xc>{}, dM[0], dM[1]);
        each_grain<G>([&](auto I) {
          constexpr int i = I;
          const T       B = T(kp.pp.B);
          const T       e0 = lin[0][CL::eta + i], e1 = lin[1][CL::eta + i];
          const T       c0 = lin[0][CL::c], c1 = lin[1][CL::c];
          mass(std::integral_constant<int, BF::ci + i>{}, (B * T(12.0)) * e0 * (e0 - T(1.0)),
               (B * T(12.0)) * e1 * (e1 - T(1.0)));
          auto dee = [&](T c, T e, T s2) {
            return B * (T(12.0) - T(12.0) * c + T(2.0) * e * (T(12.0) * c - T(24.0)) +
                        T(24.0) * (e * e) + T(12.0) * s2);
          };
          mass(std::integral_constant<int, BF::ii + i>{}, on ? dee(c0, e0, S2[0]) : T(0),
               on ? dee(c1, e1, S2[1]) : T(0));
          flux(std::integral_constant<int, BF::xi + i>{}, (T(2.0) * T(kp.pp.Mgb)) * (sum[0] - e0),
               (T(2.0) * T(kp.pp.Mgb)) * (sum[1] - e1));
          each_grain<i>([&](auto J) {
            constexpr int j = J;
            mass(std::integral_constant<int, BF::ij + i * (i - 1) / 2 + j>{},
                 e0 * lin[0][CL::eta + j], e1 * lin[1][CL::eta + j]);
          });
        });
        if constexpr (in(BF::mob))
          {
            T       xy = up_k[0] + (M[0] + r * M[1]); // d/dx and d/dy parts
            T       zz = up_k[1] + kz * (M[0] + M[1]);
            up_k[0]    = r * M[0] + M[1];
            up_k[1]    = kz * (M[0] + M[1]);
            const T px = xshfl<1>(xy), pz = xshfl<1>(zz);
            const T p  = kx * (xy + px) + (zz + r * pz);
            xy += r * px;
            put_slot(BF::mob - F0, (p + r * xshfl<2>(p)) + ky * (xy + xshfl<2>(xy)));
          }
        __syncthreads();
        if (k >= z0)
          {
            const double two3 = 2.0 / 3.0;
            const double nz   = (k > 0) + (k < kp.nc[2]);
            for (int n = wave; n < blk::ON; n += blk::NT / 64)
              {
                const int x = X0 + n % blk::OX, y = Y0 + n / blk::OX;
                if (x >= kp.nn[0] || y >= kp.nn[1])
                  continue;
                // 1D sums over the node's 1 or 2 cells: psi^2 gives 2/3 per
                // cell, psi'^2 gives 2 / h^2 (times JxW)
                const double nx = (x > 0) + (x < kp.nc[0]), ny = (y > 0) + (y < kp.nc[1]);
                const double mx = two3 * nx, my = two3 * ny, mz = two3 * nz;
                const double sx = 2.0 * nx * (kp.inv_h[0] * kp.inv_h[0]);
                const double sy = 2.0 * ny * (kp.inv_h[1] * kp.inv_h[1]);
                const double sz = 2.0 * nz * (kp.inv_h[2] * kp.inv_h[2]);
                const double mass  = mx * my * mz;
                const double stiff = sx * my * mz + mx * sy * mz + mx * my * sz;
                double *out = blocks + (((int64_t)k * kp.nn[1] + y) * kp.nn[0] + x) * NE;
#pragma unroll
                for (int j = 0; j < EPL; ++j)
                  if (ef[j] != -2)
                    {
                      double v = em[j] * mass + ek[j] * stiff;
                      if (ef[j] >= 0)
                        v += eg[j] * (double)((slots[0][ef[j]][n] + slots[1][ef[j]][n]) +
                                              (slots[2][ef[j]][n] + slots[3][ef[j]][n]));
                      out[lane + 64 * j] = v;
                    }
              }
          }
        __syncthreads();
      }
  }
} // namespace hps
