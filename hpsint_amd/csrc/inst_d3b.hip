// Instantiations: node blocks of the 3D Q1 scalar-mobility tangent in one
// pass over the cache, FP64 and FP32, 1-12 order parameters.
#include "fe_q1_blocks.hpp"
#include "ops.hpp"

namespace hps
{
  template <int G, typename T, int F0>
  static void sweeps(unsigned nwg, int zn, const KParams &kp, const T *cache, double *blocks,
                     hipStream_t s)
  {
    using BF         = BlockFields<G>;
    constexpr int F1 = BF::template sweep_end<T>(F0);
    q1_blocks<G, T, F0, F1><<<nwg, blk::NT, 0, s>>>(kp, cache, blocks, zn);
    if constexpr (F1 < BF::count)
      sweeps<G, T, F1>(nwg, zn, kp, cache, blocks, s);
  }

  template <typename T>
  static bool node_blocks(int n_grains, const KParams &kp, const T *cache, double *blocks,
                          hipStream_t s)
  {
    // planes per march: a march visits one more cell layer than it completes
    // planes, so deep ones waste less, but the grid should hold four rounds
    // of the 512 workgroups that run at once while the mesh allows it
    const int64_t cols = (int64_t)((kp.nn[0] + blk::OX - 1) / blk::OX) *
                         ((kp.nn[1] + blk::OY - 1) / blk::OY);
    int64_t zn = cols * kp.nn[2] / 2048;
    zn         = zn < 4 ? 4 : (zn > 32 ? 32 : zn);
    const int64_t chunks = (kp.nn[2] + zn - 1) / zn;
    zn                   = (kp.nn[2] + chunks - 1) / chunks;
    const unsigned nwg   = (unsigned)(cols * chunks);
    switch (n_grains)
      {
#define HPS_CASE(G)                                                \
  case G:                                                          \
    sweeps<G, T, 0>(nwg, (int)zn, kp, cache, blocks, s);           \
    return true;
        HPS_CASE(1)
        HPS_CASE(2)
        HPS_CASE(3)
        HPS_CASE(4)
        HPS_CASE(5)
        HPS_CASE(6)
        HPS_CASE(7)
        HPS_CASE(8)
        HPS_CASE(9)
        HPS_CASE(10)
        HPS_CASE(11)
        HPS_CASE(12)
#undef HPS_CASE
        default:
          return false;
      }
  }

  bool node_blocks_d3(int n_grains, const KParams &kp, const double *cache, double *blocks,
                      hipStream_t s)
  {
    return node_blocks<double>(n_grains, kp, cache, blocks, s);
  }
  bool node_blocks_d3(int n_grains, const KParams &kp, const float *cache, double *blocks,
                      hipStream_t s)
  {
    return node_blocks<float>(n_grains, kp, cache, blocks, s);
  }
} // namespace hps
