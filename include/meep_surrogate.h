/*
 * meep_surrogate.h -- C ABI of the spectral neural-operator kernels in
 * libmeepfdtd.so (BF16 matrix-core GEMM and the elementwise pieces of
 * training and inference).
 *
 * The reference has no learned component: these entry points have no
 * counterpart in it.  They serve the surrogate-assisted inverse-design loop
 * (meep_torch_amd.surrogate), which predicts transmission spectra and their
 * density gradients and falls back to the FDTD engine when a verification
 * solve disagrees.
 *
 * Conventions as in meep_fdtd.h: device pointers, 0 on success, negative
 * code plus mt_last_error() on failure, all work enqueued on `stream`.
 * BF16 buffers hold raw bfloat16 bit patterns (uint16, round-to-nearest-even
 * from FP32).
 */
#ifndef MEEP_SURROGATE_H
#define MEEP_SURROGATE_H

#ifdef __cplusplus
extern "C" {
#endif

/* C[z] = alpha * sum_{r<R} A[z,r] (M x K) * B[z,r] (K x N) + beta * C[z],
 * z < batch.  A, B: BF16; C: FP32.  Element (i, k) of A[z,r] sits at
 * A + z*a_b + r*a_r + i*a_m + k*a_k, and likewise for B and C (no r axis).
 * The reduction space R x ceil(K/32) is cut into `splits` contiguous parts
 * over grid.z; for splits > 1, `work` holds splits*batch*M*N floats of
 * partial tiles, summed in split order (deterministic). */
typedef struct {
  int M, N, K, R, batch, splits;
  const void* A;
  long long a_m, a_k, a_b, a_r;
  const void* B;
  long long b_k, b_n, b_b, b_r;
  float* C;
  long long c_m, c_n, c_b;
  float* work;
  float alpha, beta;
} mt_gemm;

int mt_gemm_bf16(const mt_gemm* g, void* stream);

/* y[i] = bf16(x[i]), i < n. */
int mt_cast_bf16(const float* x, void* y, long long n, void* stream);

/* x viewed as (rows, C, P): x += bias[c] (pre-activation, stored in place);
 * act = gelu(x) if `act` else x, written to act16 (BF16) and/or act32
 * (FP32) when non-NULL.  gelu is the exact erf form. */
int mt_bias_act(float* x, const float* bias, int C, int P, long long n, int act, void* act16, float* act32,
                void* stream);

/* d = dy * gelu'(pre) (or dy if !act); with row_bcast, dy is one value per
 * row of length P, times `scale` (backward of a mean).  Written to d32
 * and/or d16 when non-NULL. */
int mt_act_grad(const float* dy, const float* pre, long long n, int act, int P, int row_bcast, float scale,
                float* d32, void* d16, void* stream);

/* out[c] = scale * sum_{b<B, p<P} x[b, c, p] (fixed-order, deterministic).
 * work: device scratch of B*C floats (the per-(b, c) row sums). */
int mt_channel_sum(const float* x, float* out, float* work, int B, int C, int P, float scale, void* stream);

/* out[r] = scale * sum_{p<P} x[r, p]. */
int mt_row_sum(const float* x, float* out, long long rows, int P, float scale, void* stream);

/* Spectral weights W[i, o, m] = wre + i*wim (Ci x Co x Mo, FP32) -> per-mode
 * BF16 real block matrices wp[m] (2Ci x 2Co) = [[Wre, Wim], [-Wim, Wre]]. */
int mt_pack_spectral(const float* wre, const float* wim, void* wp, int Ci, int Co, int Mo, void* stream);

/* Gradient of mt_pack_spectral: dwre = d11 + d22, dwim = d12 - d21. */
int mt_unpack_spectral_grad(const float* dwp, float* dwre, float* dwim, int Ci, int Co, int Mo, void* stream);

/* Adam (with decoupled-from-nothing L2 term wd*w added to the gradient):
 * m = b1 m + (1-b1) g; v = b2 v + (1-b2) g^2;
 * w -= lr * (m / (1-b1^step)) / (sqrt(v / (1-b2^step)) + eps). */
int mt_adam(float* w, const float* g, float* m, float* v, long long n, float lr, float b1, float b2, float eps,
            int step, float wd, void* stream);

/* Fused passes of the operator with 64 channels, 128 modes, 128 head units and
 * P = n*n points, P % 16 == 0 (matrix-core size; other sizes use the calls
 * above).  Activations are (B, 64, P) BF16, spectra (B, 256, 64) BF16 with row
 * 2 m + re/im, FP32 partial sums are folded in a fixed order.  16-byte aligned
 * BF16 pointers.
 *
 * lift: x16 (B, 3, P) = [rho, (i+0.5)/n, (j+0.5)/n], v16 = w x16 + bias.
 * lift_back: drho = w[:, 0]^T dv16. */
int mt_fno_lift(const float* rho, const void* w, const float* bias, void* x16, void* v16, int B, int n,
                void* stream);
int mt_fno_lift_back(const void* dv16, const void* w, float* drho, int B, int P, void* stream);

/* part (splits, B, 256, 64) = x16 against the 256 rows of basis (256, P), the
 * points split in order; with y16 also wpart (splits, B, 64, 64) =
 * sum_p x16[c'] y16[c]. */
int mt_fno_dft(const void* x16, const void* basis, const void* y16, float* part, float* wpart, int B, int P,
               int splits, void* stream);

/* Per mode m: in16[b] = BF16 of the summed partials (row pair 2m, 2m+1: 128
 * values), out16[b][n] = sum_k in16[b][k] w[m][n][k]. */
int mt_fno_mix(const float* part, int splits, const void* w, void* in16, void* out16, int B, int Mo, void* stream);

/* u = basis_t u16 + w (64 x 64) x16 + bias -> pre (if not NULL); y16 = gelu(u)
 * or u.  basis_t: rows p of (P, 256) in fragment order, [ceil(P/128) * 4]
 * 32-point tiles x [16] steps of 16 x [64] lanes x [8]: lane 32 h + i holds
 * point 32 t + i, values 16 q + 8 h .. + 7. */
int mt_fno_out(const void* u16, const void* basis_t, const void* w, const void* x16, const float* bias, float* pre,
               void* y16, int B, int P, int act, void* stream);

/* d = (basis_t u16 + w x16) (* gelu'(pre) with act) -> y16; part (B,
 * ceil(P/128), 64) = sums of d over each 128 points (if not NULL). */
int mt_fno_out_back(const void* u16, const void* basis_t, const void* w, const void* x16, const float* pre,
                    void* y16, float* part, int B, int P, int act, void* stream);

/* out = wo mean_P gelu(wq v16 + bq) + bo; part: scratch of B * chunks * 128. */
int mt_fno_head(const void* v16, const void* wq, const float* bq, const void* wo, const float* bo, float* part,
                int chunks, void* hm16, float* out, int B, int P, int n_out, void* stream);

/* Backward of mt_fno_head: dv16; with dwo also dwo, dbo and the partial sums
 * (B * chunks, ...) of dbq (128), of dv's channels (64) and of dwq (128, 64).
 * wq_t (64, 128) is wq transposed. */
int mt_fno_head_back(const float* dout, const void* v16, const void* wq, const void* wq_t, const float* bq,
                     const void* wo, const void* hm16, float* dwo, float* dbo, float* dhm, void* dv16,
                     float* qbpart, float* vbpart, float* qwpart, int chunks, int B, int P, int n_out,
                     void* stream);

/* out[i] = sum_{q<Q} part[q][i], i < n (part is overwritten). */
int mt_fno_fold(float* part, int Q, int n, float* out, void* stream);

/* mt_pack_spectral for Ci = Co = C, and its per-mode transpose wp_t. */
int mt_fno_pack(const float* wre, const float* wim, void* wp, void* wp_t, int C, int Mo, void* stream);

/* y_t (C, R) = BF16 of x (R, C) transposed, and y (R, C) = BF16 of x unless NULL. */
int mt_cast_transpose_bf16(const float* x, void* y, void* y_t, int R, int C, void* stream);
/* The same without y. */
int mt_transpose_bf16(const float* x, void* y, int R, int C, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* MEEP_SURROGATE_H */
