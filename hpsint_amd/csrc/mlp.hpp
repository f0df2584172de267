// mlp.hpp -- launchers of the learned-predictor kernels (mlp.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace hps
{
  enum MlpEpilogue
  {
    EPI_F32       = 0, // store the FP32 product (split-K partials)
    EPI_BIAS_TANH = 1, // bf16 tanh(C + bias)
    EPI_BIAS_F32  = 2, // FP32 C + bias
    EPI_DTANH     = 3, // bf16 C * (1 - H^2)
  };

  constexpr int FEAT_STRIDE = 272; // 27 neighbours x 10 + dt + 1

  struct FeatParams
  {
    int64_t n_nodes;
    int     nn[3];
    int     n_comp;
    double  dt, dt_scale, inc_scale, inc_floor;
  };

  void mlp_gemm(hipStream_t, int ta, int tb, int epi, int M, int N, int K, const uint16_t *A,
                int lda, const uint16_t *B, int ldb, void *C, int ldc, const float *bias,
                const uint16_t *H, int nsplit, int64_t split_stride);
  void mlp_sum_splits(hipStream_t, int64_t n, int nsplit, const float *part, float *out);
  void mlp_colsum(hipStream_t, int M, int N, const uint16_t *X, float *out);
  void mlp_loss(hipStream_t, int64_t n, const float *Y, const float *T, uint16_t *dY,
                float *partial, int nblocks);
  void mlp_adam(hipStream_t, int n_out, int n_in, float *W, float *m1, float *m2, const float *g,
                float lr, float b1, float b2, float eps, float c1, float c2, uint16_t *Wb,
                uint16_t *WTb);
  void mlp_features(hipStream_t, const FeatParams &, const double *u_prev, const double *u_cur,
                    uint16_t *X, int *top2, float *lscale);
  // features, the 272-128-128-128-4 network and u_pred (also writes top2 and
  // lscale); out must not overlap u_prev or u_cur.  ws: mlp_infer_workspace
  // bytes of 16-byte aligned device memory (0 bytes: mesh not covered)
  int64_t mlp_infer_workspace(const FeatParams &);
  void    mlp_infer(hipStream_t, const FeatParams &, const double *u_prev, const double *u_cur,
                    const uint16_t *const *W, const float *const *b, const float *out_scale,
                    int *top2, float *lscale, double *out, void *ws);
  // the feature rows (as mlp_features) that the last mlp_infer on ws formed
  void    mlp_infer_rows(hipStream_t, const FeatParams &, const int *top2, const void *ws,
                         uint16_t *X);
  // one Adam step of the 272-128-128-128-4 network on M rows; returns the
  // device address of the loss' partial sums (n_loss of them).  X, Wb and ws
  // 16-byte aligned
  struct MlpTrain
  {
    int             M;
    const uint16_t *X;
    const float    *T;
    float          *W[4], *b[4], *mW[4], *vW[4], *mb[4], *vb[4];
    uint16_t       *Wb[4];
    float           lr, b1, b2, eps, c1, c2;
    void           *ws;
  };
  int64_t      mlp_train_workspace(int M, int *n_loss);
  const float *mlp_train_step(hipStream_t, const MlpTrain &);
  void mlp_predict(hipStream_t, int64_t n_nodes, int nc, const double *u_prev,
                   const double *u_cur, const float *Y, const int *top2, const float *out_scale,
                   const float *lscale, double *u_pred);
  void mlp_targets(hipStream_t, int64_t n_nodes, int nc, const double *u_prev,
                   const double *u_cur, const double *u_next, const int *top2,
                   const float *out_scale, const float *lscale, float *T);
} // namespace hps
