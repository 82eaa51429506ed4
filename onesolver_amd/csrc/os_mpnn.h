// os_mpnn.h -- launchers of the warm-start network's kernels (mpnn.hip).
#pragma once

#include "os_kernels.h"

namespace os {

// The head of the last layer: its weights (wo [64], bo behind them), the
// labels (null: prediction only) and what it writes.
struct MpHead {
  const float *wo = nullptr;
  const uint8_t *labels = nullptr;
  float inv_count = 0.0f;
  float *p = nullptr;
  float *dlogit = nullptr;
  double *lossblock = nullptr;  // one per 64 rows
};

void mp_launch_features(hipStream_t st, int B, int n, int Np, const double *q, double *rowstat,
                        double *scale, uint16_t *A, float *X0, uint16_t *XT0);
// A null: M is given (sparse instances).  head: the last layer.
void mp_launch_layer_fwd(hipStream_t st, int B, int n, int Np, const uint16_t *A,
                         const uint16_t *XT, const float *Hin, float *M, const float *wl,
                         float *Z, float *H, uint16_t *HT, const MpHead *head);
// head: the last layer; dHprev null: the first.
void mp_launch_layer_bwd(hipStream_t st, int B, int Np, const uint16_t *A,
                         const uint16_t *dMsgTin, const float *dHin, const MpHead *head,
                         const float *Z, const float *wl, const float *Hin, const float *M,
                         float *dHprev, uint16_t *dMsgT, float *partial, float *head_partial);
void mp_launch_grad_sum(hipStream_t st, int layers, int groups, const float *partial,
                        const float *head_partial, float *grad);
void mp_launch_loss_sum(hipStream_t st, size_t count, const double *terms, double *out);
void mp_launch_adam(hipStream_t st, int P, const float *grad, const uint8_t *kind, float *w,
                    float *m, float *v, float *wc, float lr, float b1, float b2, float eps,
                    int step);
void mp_launch_csr_features(hipStream_t st, int I, int max_n, const CsrInst *inst,
                            const int32_t *row_ptr, const double *val, const double *diag,
                            const int32_t *scale_rows, double *scale, float *X0);
void mp_launch_csr_agg(hipStream_t st, int I, int max_n, const CsrInst *inst,
                       const int32_t *row_ptr, const int32_t *col, const double *val,
                       const double *scale, const float *Hin, float *M);
void mp_launch_compute_copy(hipStream_t st, int P, const uint8_t *kind, const float *w,
                            float *wc);

}  // namespace os
