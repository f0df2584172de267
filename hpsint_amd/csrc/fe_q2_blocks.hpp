// fe_q2_blocks.hpp -- all node blocks of the Q2 tangent in one pass over the
// linearisation cache.
//
// The block of node j is sum_q JxW psi_m'(q) M(q) psi_m(q) over its cells
// (InverseComponentBlockDiagonalMatrix::do_update, I/lac/preconditioners.h:
// 254-318).  Its entries are made of
//   mass sums, w phi^2, of f''_cc, f''_c,eta_i, f''_eta_i,eta_i and
//     eta_i eta_j (i > j);
//   flux sums, w phi (V . grad phi), with V the c row's flux per unit value of
//     c or eta_i;
//   two stiffness sums, w grad phi . (D grad phi), with D the c row's flux per
//     unit gradient of c (tensorial mobility) and of mu;
// and the constants sum w phi^2, sum w |grad phi|^2: with 10 order parameters
// 66 + 11 + 2 sums.  (Applying the tangent to one unit input per column took
// 24 sums for each of the 12 columns and the cache 12 times.)
#pragma once

#include <type_traits>
#include <utility>

#include "fe_q2.hpp"

namespace hps
{
  template <int G>
  struct Q2BlockFields
  {
    static constexpr int cc = 0, ci = 1, ii = 1 + G, ij = 1 + 2 * G;
    static constexpr int mass = ij + G * (G - 1) / 2;
    // pair p: i (i - 1) / 2 + j, i > j
    static constexpr int pair_i(int p)
    {
      int i = 1;
      while ((i + 1) * i / 2 <= p)
        ++i;
      return i;
    }
  };

  template <typename F, int... I>
  __device__ __forceinline__ void q2_each(std::integer_sequence<int, I...>, F &&f)
  {
    (f(std::integral_constant<int, I>{}), ...);
  }

  // Lanes, colours and the store/add rule as the other Q2 kernels.  Sums run
  // through LDS in batches of R fields (6: with 12 the 36 reads in flight of a
  // pass take 72 registers; 9 and 12 measured the same), one pass per
  // direction; the results of a lane's node stay in registers until its block
  // is written.  The flux and stiffness sums come first, while the cache
  // fields are held; the mass sums need c and eta_i only.
  // Bound: latency at 2 waves/SIMD, of the LDS passes (1000 LDS of 8 k
  // instructions per wave; VALU slots 21 % busy) and of the blocks that the colour
  // passes read back; 40 x 45 x 37 cells, 10 order parameters, FP64 tensorial:
  // 1.6 ms, 4.6 GB moved (0.96 ms at the copy rate; one write is 0.64 GB) (3.7 ms
  // with one column at a time; 1.95 ms with every lane storing its own block,
  // 16 bytes per line).
  template <int DIM, int G, bool TENS, typename T>
  __global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
    q2_blocks(const Q2Params kp, const T *__restrict__ cache, double *__restrict__ blocks)
  {
    using CL         = CacheLayout<DIM, G, TENS>;
    using LN         = Q2Lane<DIM>;
    using BF         = Q2BlockFields<G>;
    constexpr int NC = G + 2, NF = CL::n_fields, LP = LN::LP;
    constexpr int R  = 6;
    __shared__ T  A[R * 64], B[R * 64];

    const LN  L(kp);
    const int l  = L.l;
    const T  *cl = cache + ((kp.wg_base + blockIdx.x) * NF) * LP + l;
    auto      in = [&](int f) { return L.valid ? cl[f * LP] : T(0); };

    // The sums over the cell's Gauss points of the N batched fields in A,
    // whose weight along d is type(r, d), into out(r, value).  1D weights of
    // the lane's node: K[0] phi phi, [1] phi' phi, [2] phi' phi' (times w_q),
    // formed again for each pass (the lane's index goes through an empty asm
    // statement) instead of held in 54 registers across the kernel.
    auto sums = [&](auto N, auto type, auto out) {
      constexpr int n = N;
      T             K[3][3];
      auto          coefs = [&](int d) {
        int t = L.t[d];
        asm volatile("" : "+v"(t));
        T sc[3], ec[3];
        q2_s_col(t, sc);
        q2_e_col(t, ec);
#pragma unroll
        for (int q = 0; q < 3; ++q)
          {
            const T w = q2_w<T>(q);
            const T e = ec[q] * T(kp.inv_h[d]);
            K[0][q]   = w * sc[q] * sc[q];
            K[1][q]   = w * sc[q] * e;
            K[2][q]   = w * e * e;
          }
      };
      __syncthreads();
      coefs(0);
#pragma unroll
      for (int r = 0; r < n; ++r)
        B[r * 64 + l] = q2_pass(A + r * 64, L.base(0), 1, K[type(r, 0)]);
      __syncthreads();
      coefs(1);
      if constexpr (DIM == 3)
        {
#pragma unroll
          for (int r = 0; r < n; ++r)
            A[r * 64 + l] = q2_pass(B + r * 64, L.base(1), 3, K[type(r, 1)]);
          __syncthreads();
          coefs(2);
#pragma unroll
          for (int r = 0; r < n; ++r)
            out(r, q2_pass(A + r * 64, L.base(2), 9, K[type(r, DIM - 1)]));
        }
      else
#pragma unroll
        for (int r = 0; r < n; ++r)
          out(r, q2_pass(B + r * 64, L.base(1), 3, K[type(r, 1)]));
      __syncthreads();
    };

    const T c = in(CL::c);
    T       eta[G], sum = T(0), S2 = T(0);
#pragma unroll
    for (int i = 0; i < G; ++i)
      {
        eta[i] = in(CL::eta + i);
        sum += eta[i];
        S2 += eta[i] * eta[i];
      }

    // ---- flux sums: V of c, then of eta_i, FB vectors at a time
    T lin[TENS && G > 1 ? CL::gb_q : NF]; // (Q_i are read where they are used)
#pragma unroll
    for (int f = 0; f < (TENS && G > 1 ? CL::gb_q : NF); ++f)
      lin[f] = in(f);
    const T zero[3] = {T(0), T(0), T(0)};
    T       v[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k)
      v[k] = T(0);
    T flux[G + 1];
    {
      T V[DIM];
      v[0] = T(1);
      tangent_grad_c<DIM, G, TENS>(kp.pp, lin, v, zero, zero, V, zero);
      v[0] = T(0);
#pragma unroll
      for (int d = 0; d < DIM; ++d)
        A[d * 64 + l] = V[d];
    }
    constexpr int FB = R / DIM;
    q2_each(std::make_integer_sequence<int, (G + 1 + FB - 1) / FB>{}, [&](auto Q) {
      constexpr int b0 = Q * FB, n = b0 + FB <= G + 1 ? FB : G + 1 - b0;
#pragma unroll
      for (int k = 0; k < n; ++k)
        if (b0 + k > 0)
          {
            const int i = b0 + k - 1;
#pragma unroll
            for (int d = 0; d < DIM; ++d)
              {
                T x = (sum - eta[i]) * lin[CL::grad_mu + d];
                if constexpr (TENS && G > 1)
                  x -= in(CL::gb_q + i * DIM + d);
                if constexpr (TENS && G == 1)
                  x = T(0);
                A[(k * DIM + d) * 64 + l] = T(2.0) * T(kp.pp.Mgb) * x;
              }
          }
      T acc[n];
#pragma unroll
      for (int k = 0; k < n; ++k)
        acc[k] = T(0);
      sums(std::integral_constant<int, n * DIM>{},
           [](int r, int d) { return r % DIM == d ? 1 : 0; }, [&](int r, T x) { acc[r / DIM] += x; });
#pragma unroll
      for (int k = 0; k < n; ++k)
        {
          flux[b0 + k] = acc[k];
          asm volatile("" : "+v"(flux[b0 + k]));
        }
    });

    // ---- stiffness sums of (c, mu) and, tensorial, (c, c): D symmetrised
    T stiff[2] = {T(0), T(0)}; // c, mu
    q2_each(std::make_integer_sequence<int, 2>{}, [&](auto P) {
      constexpr int p = P;
      if constexpr (p == 1 || TENS)
        {
          constexpr int np = DIM * (DIM + 1) / 2;
          T             D[DIM][DIM];
#pragma unroll
          for (int d = 0; d < DIM; ++d)
            {
              T u[3] = {T(0), T(0), T(0)};
              u[d]   = T(1);
              tangent_grad_c<DIM, G, TENS>(kp.pp, lin, v, p == 0 ? u : zero, p == 1 ? u : zero,
                                           D[d], zero);
            }
#pragma unroll
          for (int a = 0; a < DIM; ++a)
#pragma unroll
            for (int b = a; b < DIM; ++b)
              A[sym_index<DIM>(a, b) * 64 + l] = a == b ? D[a][a] : D[a][b] + D[b][a];
          T x = T(0);
          sums(std::integral_constant<int, np>{},
               [](int r, int d) {
                 int t = 0;
                 for (int a = 0; a < DIM; ++a)
                   for (int b = a; b < DIM; ++b)
                     if (sym_index<DIM>(a, b) == r)
                       t = (a == d ? 1 : 0) + (b == d ? 1 : 0);
                 return t;
               },
               [&](int, T s) { x += s; });
          stiff[p] = x;
          asm volatile("" : "+v"(stiff[p]));
        }
    });

    // ---- mass sums
    T       mass[BF::mass];
    const T a_ee = T(kp.pp.B) * (T(12.0) * ((T(1.0) - c) + S2));
    const T b_ee = T(kp.pp.B) * (T(24.0) * (c - T(2.0)));
    auto    field = [&](auto F) -> T {
      constexpr int f = F;
      if constexpr (f == BF::cc)
        return T(12.0) * T(kp.pp.A) * (c * (c - T(1.0))) + T(2.0) * (T(kp.pp.A) + T(kp.pp.B));
      else if constexpr (f < BF::ii)
        return T(12.0) * T(kp.pp.B) * (eta[f - BF::ci] * (eta[f - BF::ci] - T(1.0)));
      else if constexpr (f < BF::ij)
        {
          const T e = eta[f - BF::ii];
          return a_ee + e * (b_ee + T(24.0) * T(kp.pp.B) * e);
        }
      else
        {
          constexpr int i = BF::pair_i(f - BF::ij), j = f - BF::ij - i * (i - 1) / 2;
          return eta[i] * eta[j];
        }
    };
    constexpr int NB = (BF::mass + R - 1) / R;
    q2_each(std::make_integer_sequence<int, NB>{}, [&](auto Q) {
      constexpr int f0 = Q * R, n = f0 + R <= BF::mass ? R : BF::mass - f0;
      q2_each(std::make_integer_sequence<int, n>{}, [&](auto I) {
        constexpr int r = I;
        A[r * 64 + l]   = field(std::integral_constant<int, f0 + r>{});
      });
      sums(std::integral_constant<int, n>{}, [](int, int) { return 0; },
           [&](int r, T v) {
             mass[f0 + r] = v;
             asm volatile("" : "+v"(mass[f0 + r]));
           });
    });

    // ---- the blocks: RB rows (of column entries) of every node at a time go
    // through LDS, so that the wave writes runs of RB n_c entries instead of
    // 16 bytes per line
    constexpr int W = NC % 2 == 0 ? 2 : 1; // (rows of an even n_c are 16-byte aligned)
    using V         = std::conditional_t<W == 2, double2, double>;
    constexpr int RB = 2, RL = RB * NC / W + 1; // LDS row of a node, in V
    __shared__ V       rows[LP * RL];
    __shared__ int64_t where[LP]; // 2 node + (this colour is the first to reach it)
    if (L.valid)
      where[l] = 2 * LN::node(kp, L.cc, L.p) + (LN::first(kp, L.cc, L.p) ? 1 : 0);
    const int64_t left  = kp.n_col - (int64_t)blockIdx.x * LN::CPW;
    const int     nodes = LN::NP * (left < LN::CPW ? (int)left : LN::CPW);
    // 1D: sum w phi^2 = 2/15 (end nodes), 8/15 (middle); sum w phi'^2 = 7/3,
    // 16/3 over h^2
    double m = kp.h_prod, k = 0.0;
    {
      double m1[DIM], k1[DIM];
#pragma unroll
      for (int d = 0; d < DIM; ++d)
        {
          m1[d] = L.t[d] == 1 ? 8.0 / 15.0 : 2.0 / 15.0;
          k1[d] = (L.t[d] == 1 ? 16.0 / 3.0 : 7.0 / 3.0) * (kp.inv_h[d] * kp.inv_h[d]);
          m *= m1[d];
        }
#pragma unroll
      for (int d = 0; d < DIM; ++d)
        {
          double x = kp.h_prod * k1[d];
#pragma unroll
          for (int e = 0; e < DIM; ++e)
            x *= e == d ? 1.0 : m1[e];
          k += x;
        }
    }
    const double  hp = kp.h_prod, Lm = kp.pp.L, w0 = kp.pp.w0;
    V            *out = reinterpret_cast<V *>(blocks);
    // entry of column b, row a
    auto entry = [&](auto IB, auto IA) -> double {
      constexpr int b = IB, a = IA;
      if constexpr (b == 0 && a == 0)
        return w0 * m + hp * (double)(flux[0] + stiff[0]);
      else if constexpr (b == 0 && a == 1)
        return -hp * (double)mass[BF::cc] - kp.pp.kappa_c * k;
      else if constexpr (b == 0)
        return Lm * hp * (double)mass[BF::ci + (a - 2)];
      else if constexpr (b == 1)
        return a == 0 ? hp * (double)stiff[1] : (a == 1 ? kp.pp.w_alg * m : 0.0);
      else if constexpr (a == 0)
        return hp * (double)flux[b - 1];
      else if constexpr (a == 1)
        return -hp * (double)mass[BF::ci + (b - 2)];
      else if constexpr (a == b)
        return w0 * m + Lm * hp * (double)mass[BF::ii + (a - 2)] + Lm * kp.pp.kappa_p * k;
      else
        {
          constexpr int hi = (a > b ? a : b) - 2, lo = (a > b ? b : a) - 2;
          return Lm * 24.0 * kp.pp.B * hp * (double)mass[BF::ij + hi * (hi - 1) / 2 + lo];
        }
    };
    __syncthreads();
    q2_each(std::make_integer_sequence<int, (NC + RB - 1) / RB>{}, [&](auto Q) {
      constexpr int b0 = Q * RB, nb = b0 + RB <= NC ? RB : NC - b0;
      constexpr int RV = nb * NC / W, ST = (LP * RV + 63) / 64;
      // what the earlier colours left there, requested before the exchange
      V o[ST];
#pragma unroll
      for (int i = 0; i < ST; ++i)
        {
          const int x = l + 64 * i, n = x / RV;
          o[i]        = V{};
          if (n < nodes)
            if (const int64_t f = where[n]; !(f & 1))
              o[i] = out[(f >> 1) * (NC * NC / W) + b0 * NC / W + (x - n * RV)];
        }
      q2_each(std::make_integer_sequence<int, nb * NC / W>{}, [&](auto E) {
        constexpr int e = E * W, b = b0 + e / NC, a = e % NC;
        if (l < LP)
          {
            double *d = reinterpret_cast<double *>(&rows[l * RL + E]);
            d[0]      = entry(std::integral_constant<int, b>{}, std::integral_constant<int, a>{});
            if constexpr (W == 2)
              d[1] = entry(std::integral_constant<int, b>{}, std::integral_constant<int, a + 1>{});
          }
      });
      __syncthreads();
      int l2 = l; // (the addresses are formed again, not held)
      asm volatile("" : "+v"(l2));
#pragma unroll
      for (int i = 0; i < ST; ++i)
        {
          const int x = l2 + 64 * i, n = x / RV;
          if (n < nodes)
            {
              V r = rows[n * RL + (x - n * RV)];
              if constexpr (W == 2)
                {
                  r.x = o[i].x + r.x;
                  r.y = o[i].y + r.y;
                }
              else
                r = o[i] + r;
              out[(where[n] >> 1) * (NC * NC / W) + b0 * NC / W + (x - n * RV)] = r;
            }
        }
      __syncthreads();
    });
  }
} // namespace hps
