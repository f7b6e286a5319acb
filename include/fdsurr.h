/* fdsurr.h - C ABI of the gfx950 BF16 MFMA kernels of the convolutional
 * surrogate (3x3 convolutions of a U-Net over the coarse phase field).
 *
 * No reference counterpart: the reference has no learned model.  These are
 * the building blocks of the surrogate that fast-forwards the coarse phase
 * field of the lattice-Boltzmann solver (libfdlbm.so).
 *
 * Conventions
 *   activations  NHWC, bfloat16 (raw uint16 bit patterns), C % 8 == 0
 *   weights      [Cout][3][3][Cin] bfloat16, Cout % 16 == 0
 *   padding      1 (zeros), stride 1: output H x W equals the input's
 *   accumulation FP32 (MFMA v_mfma_f32_16x16x32_bf16)
 *   pointers     device memory owned by the caller; `stream` is a
 *                hipStream_t (NULL: the default stream); every call is
 *                asynchronous on it
 *   returns      0, or a negative code with a message from fds_last_error()
 */
#ifndef FDSURR_H
#define FDSURR_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define FDS_OK 0
#define FDS_E_ARG (-1)
#define FDS_E_HIP (-2)

/* y = act(conv3x3(x, w) + bias): y32 (float NHWC) and/or y16 (bf16 NHWC),
 * either may be NULL; bias may be NULL; relu != 0 applies max(0, .). */
int fds_conv3x3_fwd(const uint16_t* x, const uint16_t* w, const float* bias, float* y32, uint16_t* y16,
                    int32_t N, int32_t H, int32_t W, int32_t Cin, int32_t Cout, int32_t relu, void* stream);

/* wt[ci][tap][co] = w[co][8 - tap][ci]: the weights of the transposed
 * convolution, so that conv3x3(dy, wt) is the gradient of the input. */
int fds_flip_weights(const uint16_t* w, uint16_t* wt, int32_t Cin, int32_t Cout, void* stream);

/* For n <= 16 layers at once, in one launch: w16[l] = w[l] rounded to bf16
 * (nearest even) and wt[l] = fds_flip_weights of it, from the FP32 weights
 * w[l] [cout[l]][3][3][cin[l]].  w, w16, wt, cin and cout are host arrays of
 * n entries (device pointers in the first three). */
int fds_cast_flip(int32_t n, const float* const* w, uint16_t* const* w16, uint16_t* const* wt, const int32_t* cin,
                  const int32_t* cout, void* stream);

/* dx = conv3x3(dy', wt) with wt from fds_flip_weights (dy has Cout
 * channels, dx has Cin).  dy' = dy where relu_y > 0 and 0 elsewhere when
 * relu_y (the bf16 output of a ReLU forward, same shape as dy) is given,
 * dy otherwise.  dx32 and/or dx16 may be NULL. */
int fds_conv3x3_bwd_data(const uint16_t* dy, const uint16_t* wt, const uint16_t* relu_y, float* dx32,
                         uint16_t* dx16, int32_t N, int32_t H, int32_t W, int32_t Cin, int32_t Cout, void* stream);

/* Number of floats of scratch fds_conv3x3_bwd_weight needs. */
int64_t fds_bwd_weight_scratch(int32_t N, int32_t H, int32_t W, int32_t Cin, int32_t Cout);

/* dw[co][tap][ci] = sum over pixels of dy'[p][co] * x[p + d(tap)][ci]
 * (float, overwritten); dbias[co] = sum over pixels of dy'[p][co] (float,
 * overwritten, may be NULL); dy' as for fds_conv3x3_bwd_data (relu_y may
 * be NULL).  scratch: fds_bwd_weight_scratch floats.  Deterministic:
 * fixed-order partial sums, no atomics. */
int fds_conv3x3_bwd_weight(const uint16_t* x, const uint16_t* dy, const uint16_t* relu_y, float* dw, float* dbias,
                           float* scratch, int32_t N, int32_t H, int32_t W, int32_t Cin, int32_t Cout, void* stream);

/* Decoder input of the U-Net: out[n][h][w][0:C1] = lo[n][h/2][w/2][:]
 * (nearest-neighbour upsampling, lo is N x H/2 x W/2 x C1) and
 * out[n][h][w][C1:C1+C2] = skip[n][h][w][:]; bf16 NHWC, H and W even, C1
 * and C2 multiples of 8.  Replaces torch.cat([up(lo), skip], dim=3). */
int fds_up_cat(const uint16_t* lo, const uint16_t* skip, uint16_t* out, int32_t N, int32_t H, int32_t W,
               int32_t C1, int32_t C2, void* stream);

/* Gradients of fds_up_cat: dlo (N x H/2 x W/2 x C1) = the sum of dout over
 * each 2 x 2 block of its first C1 channels, the two columns of each row
 * summed and rounded to bf16 first, then the two rows (the order of the
 * gradients of two nearest-neighbour repeats, along w then h); dskip = the
 * last C2 channels of dout. */
int fds_up_cat_bwd(const uint16_t* dout, uint16_t* dlo, uint16_t* dskip, int32_t N, int32_t H, int32_t W,
                   int32_t C1, int32_t C2, void* stream);

/* fds_up_cat_bwd with dlo zeroed where lo (the coarse input, the bf16 output
 * of a ReLU, N x H/2 x W/2 x C1) is not > 0: that ReLU's backward.  lo may
 * be NULL (then fds_up_cat_bwd).  dskip may be NULL: it is then not formed,
 * and the caller reads the skip gradient as the channels C1 .. C1 + C2 - 1
 * of dout in place. */
int fds_up_cat_bwd_masked(const uint16_t* dout, const uint16_t* lo, uint16_t* dlo, uint16_t* dskip, int32_t N,
                          int32_t H, int32_t W, int32_t C1, int32_t C2, void* stream);

/* out = dy where y > 0 (bf16 values as floats: -0 and NaN are not), else 0:
 * the backward mask of a ReLU whose bf16 output is y; n values, n % 8 == 0;
 * out may be dy. */
int fds_relu_mask(const uint16_t* dy, const uint16_t* y, uint16_t* out, int64_t n, void* stream);

/* Gradient of s (N x H x W x C bf16, H and W even, C a multiple of 8), the
 * output of a ReLU that feeds a 2 x 2 average pool (gradient dp, N x H/2 x
 * W/2 x C) and a skip connection (gradient dskip, N x H x W x C with pixels
 * dskip_ld channels apart, dskip_ld >= C a multiple of 8, so that a channel
 * slice of the decoder input's gradient is read in place):
 * out = 0 where s is not > 0, else bf16(bf16(dp[n][h/2][w/2][c] / 4) +
 * dskip[n][h][w][c]) -- the mean's backward, the sum of the two gradients
 * and the ReLU's backward, each rounded as torch rounds them. */
int fds_pool_skip_bwd(const uint16_t* dp, const uint16_t* dskip, int32_t dskip_ld, const uint16_t* s, uint16_t* out,
                      int32_t N, int32_t H, int32_t W, int32_t C, void* stream);

/* y = the mean of x over each 2 x 2 block (x N x H x W x C, H and W even, C a
 * multiple of 8; y N x H/2 x W/2 x C; bf16): the four values added in float,
 * row by row, times 1/4, rounded - torch's mean over the two axes. */
int fds_avg_pool2(const uint16_t* x, uint16_t* y, int32_t N, int32_t H, int32_t W, int32_t C, void* stream);

/* The U-Net's input, N x H x W x 8 bf16: psi, ux * scale, uy * scale, solid,
 * lm, th, 0, 0.  psi, ux, uy: N x H x W floats; solid the same, or H x W for
 * every sample (solid_per_sample 0); lm and th: lm_n, th_n = 1 or N floats. */
int fds_net_inputs(const float* psi, const float* ux, const float* uy, const float* solid, int32_t solid_per_sample,
                   const float* lm, int32_t lm_n, const float* th, int32_t th_n, float scale, uint16_t* out, int32_t N,
                   int32_t H, int32_t W, void* stream);

/* Bytes of scratch fds_unet_fwd needs (-1: bad arguments). */
int64_t fds_unet_scratch(int32_t N, int32_t H, int32_t W, const int32_t* c);

/* Forward pass of the whole U-Net in one call: y (N x H x W x 8 floats, the
 * head's output) from x (N x H x W x 8 bf16; H and W multiples of 8).  c:
 * the widths of the four levels (multiples of 8); w and bias: device pointers
 * of the FP32 weights and biases of the 15 layers, encoder then decoder then
 * head (e0a e0b e1a e1b e2a e2b e3a e3b d2a d2b d1a d1b d0a d0b head), in
 * host arrays.  The same kernels as the calls above, launch by launch. */
int fds_unet_fwd(const uint16_t* x, const float* const* w, const float* const* bias, float* y, void* scratch,
                 int32_t N, int32_t H, int32_t W, const int32_t* c, void* stream);

/* The training loss over n pixels: with o the network's output (pixels ld >= 3
 * floats apart), d = psi0 + o[0] - psi1 and x = v0 + o[1..2] - v1 (v0, v1: two
 * floats a pixel, 8-byte aligned), loss = sum(d^2 wf) / w + lambda sum(|x|^2
 * wf) / w; w: one float.  scratch: fds_net_loss_scratch doubles.
 * Deterministic.  res (3 floats a pixel, or NULL): d and x, from which
 * fds_net_loss_bwd forms dout (3 floats a pixel) = g (one float) times the
 * gradient of the loss in o, in the order of products of PyTorch's autograd
 * for that expression. */
int64_t fds_net_loss_scratch(void);
int fds_net_loss(const float* out, int32_t ld, const float* psi0, const float* psi1, const float* v0, const float* v1,
                 const float* wf, const float* w, float lambda, double* scratch, float* loss, float* res, int64_t n,
                 void* stream);
int fds_net_loss_bwd(const float* res, const float* wf, const float* w, float lambda, const float* g, float* dout,
                     int64_t n, void* stream);

/* Message of the last failed call on this thread. */
const char* fds_last_error(void);

#ifdef __cplusplus
}
#endif

#endif /* FDSURR_H */
