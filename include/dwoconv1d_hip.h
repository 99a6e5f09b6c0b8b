/*
 * libdwoconv1d_hip.so -- C ABI of the MI355X (gfx950) depthwise oriented 1D convolution.
 *
 * This is the boundary a binding of the reference's operator module would call in place
 * of the five functions its JIT-built extension exports
 * (models/dwoconv1d/dwoconv1d_kernel.py:29-36,54-60: fprop, dgrad, wgrad, nhwc_to_nchw,
 * nchw_to_nhwc).  Plain pointers and sizes only; the library never allocates, frees or
 * retains device memory: the caller owns inputs, outputs and scratch.  Every launch is
 * asynchronous on the stream passed in (the reference launches on the current stream,
 * models/dwoconv1d/kernels/kernels.cu:25).
 *
 * First use.  The first launch of a kernel on a device queries its occupancy and sets its
 * dynamic-LDS attribute, which a stream capture does not allow.  Call dwo_init() once per
 * device (with that device current) before capturing calls into a graph; without it the set-up
 * happens lazily inside the first call of each entry point on each shape class.  Each launching
 * entry point clears the calling thread's HIP last-error state on entry, so the positive
 * status it returns always belongs to its own launches.
 *
 * Tap blobs.  `taps` arguments are device copies of a blob built by dwo_build_taps for the
 * same C and K as the call; the kernels index the blob with the call's C and K and cannot
 * verify its header, so a blob of another size leads to out-of-range reads.  The caller checks
 * the size (dwo_taps_bytes) before launching.
 *
 * Operator definition (models/dwoconv1d_reference/kernels/kernels.cpp:36-52,71-90,111-126),
 * pad = K/2, P = ceil(H/stride), Q = ceil(W/stride):
 *   dh(s) = (int)(-sinf(theta_c) * (s - pad)),  dw(s) = (int)(cosf(theta_c) * (s - pad))
 *   fprop: y[n,c,p,q]  = sum_s x[n,c,p*stride+dh(s),q*stride+dw(s)] * w[c,s]   (taps outside = 0)
 *   dgrad: dx[n,c,h,w] = sum_s dy[n,c,(h-dh(s))/stride,(w-dw(s))/stride] * w[c,s]
 *                        (only taps whose two numerators are divisible by stride and in range)
 *   wgrad: dw[c,s]     = sum_{n,p,q} x[n,c,p*stride+dh(s),q*stride+dw(s)] * dy[n,c,p,q]
 *
 * Layouts: DWO_NCHW tensors are [N,C,H,W]; DWO_NHWC tensors are [N,H,W,C].  The NHWC entry
 * points read and write NHWC directly, which replaces the reference's transpose passes
 * (models/dwoconv1d/kernels/kernels.cu:56-68, nhwc_utils.h:46-110).
 * Element types: activations x, y, dy, dx are fp32, bf16 or fp16; weights, bias, dw and db
 * are always passed as fp32 and all accumulation is fp32.  With 16-bit activations the
 * row-direction orientations of the stride-1 plane kernels multiply through a two-element dot
 * product whose operands are both in the activation type: there the weights are rounded to
 * that type first (the reference holds the weights in the activation type throughout,
 * models/dwoconv1d/kernels/kernels.cu:25); the error stays within the 16-bit tolerance.
 */
#ifndef DWOCONV1D_HIP_H
#define DWOCONV1D_HIP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* status codes: 0 ok, negative = argument error, positive = hipError_t of the launch */
#define DWO_OK 0
#define DWO_ERR_NULL_POINTER (-1)
#define DWO_ERR_BAD_SHAPE (-2)    /* N,C,H,W < 1 or sizes overflow int32 indexing */
#define DWO_ERR_BAD_KERNEL (-3)   /* K even, < 1 or > DWO_MAX_K */
#define DWO_ERR_BAD_STRIDE (-4)   /* stride not in {1,2,4} */
#define DWO_ERR_BAD_DTYPE (-5)
#define DWO_ERR_BAD_LAYOUT (-6)
#define DWO_ERR_SCRATCH_TOO_SMALL (-7)
#define DWO_ERR_BAD_TAPS (-8)     /* host-side tap blob does not match C,K */
#define DWO_ERR_STATIC_SCRATCH_LIMIT (-9) /* dwo_wgrad_static: partial sums exceed the static scratch */

#define DWO_MAX_K 63

#define DWO_F32 0
#define DWO_BF16 1
#define DWO_F16 2

#define DWO_NCHW 0
#define DWO_NHWC 1
/* Added to DWO_NHWC: dwo_taps_grouped() returned 1 for the tap table and this element type, i.e. the channels
 * of every aligned 16 bytes share one orientation.  Such calls may take kernels that work on whole
 * pieces (other results' rounding, same precision); a table it does not hold for is slow, not wrong.  The
 * scratch of dwo_wgrad is sized with the layout of the call. */
#define DWO_GROUPED 2

/* Library version (major*10000 + minor*100 + patch). */
int dwo_version(void);

/* Human-readable text for a status returned by any entry point. */
const char *dwo_status_string(int status);

/*
 * One-time set-up of every kernel on the current device (occupancy queries, dynamic-LDS
 * attributes), so that later calls only launch kernels and can be captured into a graph.
 * Replaces nothing the reference's extension exports: there the set-up is the JIT build plus
 * the cudaFuncSetAttribute of every launcher call (models/dwoconv1d/kernels/kernels.h:520-531).
 * Idempotent and thread-safe; call once per device with that device current.
 */
int dwo_init(void);

/*
 * Host-side tap table.  Replaces the per-thread sincosf + truncation of the reference
 * kernels (models/dwoconv1d/kernels/kernels.h:240-241,285-287) with one table computed
 * on the host in fp32 exactly as kernels.cpp:37,43-44 does.  `theta_host` holds C angles
 * in radians.  The caller copies the `dwo_taps_bytes(C,K)`-byte blob to device memory and
 * passes that device pointer as `taps` below; the blob's layout is private to the library.
 */
size_t dwo_taps_bytes(int C, int K);
int dwo_build_taps(const float *theta_host, int C, int K, void *taps_host);

/* 1 when every run of `channels` channels (aligned, C a multiple) of a host blob shares one of the eight
 * compile-time orientations, else 0; channels = 16 / element size for DWO_GROUPED. */
int dwo_taps_grouped(const void *taps_host, int channels);

/* Debug/inspection helper: (dh,dw) of channel c, tap s from a host blob. */
int dwo_taps_get(const void *taps_host, int c, int s, int *dh, int *dw);

/*
 * fprop -- replaces `fprop(x, w, theta)` (models/dwoconv1d/kernels/kernels.cu:15-27) plus
 * the separate bias add of models/dwoconv1d/dwoconv1d.py:34-35 when `bias` is non-NULL.
 * x: [N,C,H,W] or [N,H,W,C] `dtype`; w: [C,K] fp32; bias: [C] fp32 or NULL;
 * y: [N,C,P,Q] or [N,P,Q,C] `dtype`.
 */
int dwo_fprop(const void *x, const float *w, const float *bias, const void *taps, void *y,
              int N, int C, int H, int W, int K, int stride, int dtype, int layout,
              void *stream);

/*
 * dgrad -- replaces `dgrad(dy, w, theta)` (models/dwoconv1d/kernels/kernels.cu:29-40).
 * dy: [N,C,P,Q] / [N,P,Q,C]; dx: [N,C,H,W] / [N,H,W,C]; H,W are the input extents.
 */
int dwo_dgrad(const void *dy, const float *w, const void *taps, void *dx,
              int N, int C, int H, int W, int K, int stride, int dtype, int layout,
              void *stream);

/*
 * wgrad -- replaces `wgrad(dy, x, theta)` (models/dwoconv1d/kernels/kernels.cu:42-54) and,
 * when `db` is non-NULL, the bias gradient `dy.sum([0,2,3])` of dwoconv1d.py:66-67.
 * Deterministic: workgroups write partial sums into `scratch` (`dwo_wgrad_scratch_bytes`
 * bytes, caller-allocated, contents undefined on entry and exit) and the partial sums of a
 * channel are added in a fixed order -- no floating-point atomics, unlike
 * models/dwoconv1d/kernels/kernels.h:504-517.  For the stride-1 plane shapes that addition
 * happens inside the same kernel (the last workgroup of a channel to finish does it, found by
 * an integer counter in device memory the library owns); otherwise, and always under stream
 * capture, a second small kernel does it.  Both give the same bits.
 * dw: [C,K] fp32 (fully overwritten); db: [C] fp32 or NULL.
 *
 * Concurrency.  Calls on one stream are ordered.  Calls on different streams may overlap as long
 * as they do not share `scratch` (or `dw`/`db`): the library's counters belong to the stream
 * (the first 64 streams that call wgrad on a device each get a set; calls on further streams,
 * on hipStreamPerThread and under capture use the second kernel instead), so no two launches
 * that can run at the same time count on the same counters.  A captured graph contains no
 * reference to library-owned memory.
 */
size_t dwo_wgrad_scratch_bytes(int N, int C, int H, int W, int K, int stride, int dtype,
                               int layout);
int dwo_wgrad(const void *dy, const void *x, const void *taps, float *dw, float *db,
              void *scratch, size_t scratch_bytes,
              int N, int C, int H, int W, int K, int stride, int dtype, int layout,
              void *stream);

/*
 * wgrad without any device allocation by caller or library -- no counterpart in the reference.
 * It is for callers that cannot allocate: code under stream capture, tight serving loops,
 * harnesses that forbid hipMalloc.  Same results as dwo_wgrad (bit for bit: the same kernels),
 * with the partial sums kept in a DWO_STATIC_SCRATCH_BYTES array in device memory that is part
 * of the library image (one copy per GPU, held until the process ends).  Shapes whose
 * dwo_wgrad_scratch_bytes exceed it are refused with DWO_ERR_STATIC_SCRATCH_LIMIT.  Every call on a
 * GPU shares that GPU's array: calls that overlap in time on one GPU (different streams or
 * threads) race; calls on one stream are ordered.  Nothing in the array has to survive between
 * calls and nothing in it has to be cleared.
 */
#define DWO_STATIC_SCRATCH_BYTES (8u << 20)
int dwo_wgrad_static(const void *dy, const void *x, const void *taps, float *dw, float *db,
                     int N, int C, int H, int W, int K, int stride, int dtype, int layout,
                     void *stream);

/*
 * Where the partial sums of the stride-1 plane wgrad kernels are added up: in_kernel != 0 (the
 * default) inside the kernel that produced them, 0 in a second kernel.  The results are
 * bit-identical; the switch exists so that both paths can be exercised and compared.  No
 * counterpart in the reference.  Process-wide; returns the previous setting.
 */
int dwo_set_wgrad_reduction(int in_kernel);

/*
 * fprop of a pointwise-projected NHWC tensor without materialising it: y = fprop(pw(x)) with
 * pw(x)[n,h,w,c] = pw_b[c] + sum_k x[n,h,w,k] * pw_w[c,k], rounded to the activation type as the
 * separate layer's output would be.  The stem's first two layers of the reference
 * (models/convnext.py:143,177-178: pw1 = nn.Linear(3, 64) then the stride-2 oriented
 * convolution) in one pass: the 64-channel full-resolution tensor never goes to memory.
 * x is [N,H,W,Cin] with Cin in {1,2,3,4}; pw_w [C,Cin] and pw_b [C] (may be null) are fp32; C must
 * be a multiple of 4; the other arguments are those of dwo_fprop with layout DWO_NHWC.
 */
int dwo_pointwise_fprop_nhwc(const void *x, const float *pw_w, const float *pw_b, const float *w,
                             const float *bias, const void *taps, void *y, int N, int Cin, int C,
                             int H, int W, int K, int stride, int dtype, void *stream);
/* The same with a layout code: DWO_NHWC, or DWO_NHWC | DWO_GROUPED as dwo_fprop takes it. */
int dwo_pointwise_fprop(const void *x, const float *pw_w, const float *pw_b, const float *w,
                        const float *bias, const void *taps, void *y, int N, int Cin, int C, int H,
                        int W, int K, int stride, int dtype, int layout, void *stream);

/*
 * Forward-only glue of a ConvNeXt-1D block, each one pass over HBM in place of the PyTorch
 * passes the reference spends around the operator (no counterpart in the reference's
 * extension; they replace models/convnext.py:306-318 -- permute + LayerNorm before the
 * pointwise layers, layer scale + permute + residual after them -- and the channels-last
 * LayerNorm + GELU of the stem, :176-190).  LayerNorm is over the channel dimension, biased
 * variance, fp32 statistics; gamma, beta and scale are fp32 [C]; C must be even.
 *
 * dwo_layernorm_nhwc:      out[r,:] = act(LN(x[r,:]) * gamma + beta) for rows of C contiguous
 *                          channels (act = exact GELU when gelu != 0), C <= 2048.
 * dwo_nchw_layernorm_nhwc: x [N,C,H,W] -> out [N,H,W,C] = LN over C * gamma + beta, C <= 1536.
 * dwo_nhwc_scale_add_nchw: y [N,H,W,C] -> out [N,C,H,W] = res + scale[c] * y; scale and res
 *                          (an [N,C,H,W] tensor) may be null.
 */
int dwo_layernorm_nhwc(const void *x, const float *gamma, const float *beta, void *out,
                       size_t rows, int C, float eps, int gelu, int dtype, void *stream);
int dwo_nchw_layernorm_nhwc(const void *x, const float *gamma, const float *beta, void *out, int N,
                            int C, int H, int W, float eps, int dtype, void *stream);
int dwo_nhwc_scale_add_nchw(const void *y, const float *scale, const void *res, void *out, int N,
                            int C, int H, int W, int dtype, void *stream);

/*
 * Parameter gradients of a pointwise layer with few inputs (the stem's first layer,
 * models/convnext.py:143,177): dw[c,k] = sum_p dy[p,c] * x[p,k], db[c] = sum_p dy[p,c] (db may be
 * null), fp32, for x [rows,Cin], dy [rows,C] of one type, Cin in {1,2,3,4}.  dy is 16-byte aligned and C a
 * multiple of 16 bytes' worth of channels, at most 256 such pieces.  scratch holds at least
 * dwo_pointwise_wgrad_scratch_bytes(Cin, C) bytes.
 */
size_t dwo_pointwise_wgrad_scratch_bytes(int Cin, int C);
/* The layer itself: y[p,c] = b[c] + sum_k x[p,k] * w[c,k] (b may be null), all of one 16-bit type, summed in fp32; y is
 * 16-byte aligned, C a multiple of 64. */
int dwo_pointwise_forward(const void *x, const void *w, const void *b, void *y, size_t rows, int Cin, int C, int dtype,
                          void *stream);
int dwo_pointwise_wgrad(const void *dy, const void *x, float *dw, float *db, void *scratch, size_t scratch_bytes,
                        size_t rows, int Cin, int C, int dtype, void *stream);

/*
 * The passes around the operator and the pointwise layers of a block (models/convnext.py:306-318) and of the stem
 * (:176-190) with their backward passes; no counterpart in the reference's extension.  LayerNorm is over C with the
 * biased variance; gamma, beta and scale are fp32 [C]; C is a multiple of 8 up to 1024; tensors are dense and 16-byte
 * aligned; in_dtype and out_dtype are equal or one of them is DWO_F32; stats receives (mean, 1 / deviation) per row, what the
 * backward pass takes (forward only: may be null); dgamma, dbeta and dscale are written as grad_dtype and may be null;
 * scratch holds at least dwo_block_scratch_bytes(C) bytes.
 *
 * dwo_ln_rows:     out[r,:] = act(LN(x[r,:])) for rows of C channels (act = exact GELU where gelu & 1; where gelu & 2 what it
 *                  takes, and its gradient in the backward pass, are rounded to out_dtype as separate passes round them);
 *                  _backward also takes dout [rows,C] (out_dtype) and writes dx (in_dtype).
 * dwo_ln_tile:     x [N,C,H,W] -> out [N,H,W,C] = LN over C; _backward: dout [N,H,W,C] -> dx [N,C,H,W].
 * dwo_ln_patch:    x [N,C,H,W] -> LN over C -> out [N,H/2,W/2,4C], patches [C][2][2] (H, W at least 2; an odd last row or
 *                  column is in no patch); stats [N,H/2,W/2,2,2]; _backward writes dx of the pixels in patches.
 * dwo_block_tail:  out [N,C,H,W] = res + scale[c] * y for y [N,H,W,C] of y_dtype, out of dtype (y's type or DWO_F32) and
 *                  res of res_dtype (either); scale and res may be null; where rounded != 0 scale[c] * y is rounded to y_dtype
 *                  before the sum.  _backward: dout [N,C,H,W] (dtype) ->
 *                  dy [N,H,W,C] (y_dtype) and, where y is not null, dscale.  (The gradient of res is dout.)
 */
size_t dwo_block_scratch_bytes(int C);
int dwo_ln_rows(const void *x, const float *gamma, const float *beta, void *out, float *stats, size_t rows, int C,
                float eps, int gelu, int in_dtype, int out_dtype, void *stream);
int dwo_ln_rows_backward(const void *dout, const void *x, const float *stats, const float *gamma, const float *beta,
                         void *dx, void *dgamma, void *dbeta, void *scratch, size_t scratch_bytes, size_t rows, int C,
                         int gelu, int in_dtype, int out_dtype, int grad_dtype, void *stream);
int dwo_ln_tile(const void *x, const float *gamma, const float *beta, void *out, float *stats, int N, int C, int H,
                int W, float eps, int in_dtype, int out_dtype, void *stream);
int dwo_ln_tile_backward(const void *dout, const void *x, const float *stats, const float *gamma, void *dx,
                         void *dgamma, void *dbeta, void *scratch, size_t scratch_bytes, int N, int C, int H, int W,
                         int in_dtype, int out_dtype, int grad_dtype, void *stream);
int dwo_ln_patch(const void *x, const float *gamma, const float *beta, void *out, float *stats, int N, int C, int H,
                 int W, float eps, int in_dtype, int out_dtype, void *stream);
int dwo_ln_patch_backward(const void *dout, const void *x, const float *stats, const float *gamma, void *dx,
                          void *dgamma, void *dbeta, void *scratch, size_t scratch_bytes, int N, int C, int H, int W,
                          int in_dtype, int out_dtype, int grad_dtype, void *stream);
int dwo_block_tail(const void *y, const float *scale, const void *res, void *out, int N, int C, int H, int W,
                   int rounded, int y_dtype, int res_dtype, int dtype, void *stream);
int dwo_block_tail_backward(const void *dout, const void *y, const float *scale, void *dy, void *dscale, void *scratch,
                            size_t scratch_bytes, int N, int C, int H, int W, int y_dtype, int dtype, int grad_dtype,
                            void *stream);

/*
 * Parameter gradients of a pointwise layer K -> N over 16-bit activations (the blocks' linear layers,
 * models/convnext.py:296-298): dw[n,k] = sum_m dy[m,n] * x[m,k], db[n] = sum_m dy[m,n] (db may be null), for
 * dy [rows,N] and x [rows,K] of type dtype (DWO_BF16 or DWO_F16), summed in fp32 and written as grad_dtype.  N and
 * K are multiples of 8 up to 65536, rows at most 2^31; dy, x and scratch are 16-byte aligned and scratch holds at least
 * dwo_linear_wgrad_scratch_bytes(rows, N, K) bytes (0: sizes that are not accepted).
 */
size_t dwo_linear_wgrad_scratch_bytes(size_t rows, int N, int K);
int dwo_linear_wgrad(const void *dy, const void *x, void *dw, void *db, void *scratch, size_t scratch_bytes,
                     size_t rows, int N, int K, int dtype, int grad_dtype, void *stream);

/*
 * A pointwise layer K -> N at inference with what follows it in a block (models/convnext.py:306-318), for 16-bit
 * types (DWO_BF16, DWO_F16): y[m,n] = bias[n] + sum_k x[m,k] * w[n,k], summed in fp32; w [N,K] and bias [N] (may be
 * null) have the activations' type.  N and K are multiples of 8 up to 65536, rows below 2^31; tensors are 16-byte aligned.
 *
 * dwo_linear_rows:   out [rows,N] = act(y), act = exact GELU when gelu != 0.
 * dwo_linear_planes: x [images,HW,K] -> out [images,N,HW] = res + scale[n] * y; scale [N] and res (like out) may be
 *                    null and have the activations' type.
 */
int dwo_linear_rows(const void *x, const void *w, const void *bias, void *out, size_t rows, int N, int K, int gelu,
                    int dtype, void *stream);
int dwo_linear_planes(const void *x, const void *w, const void *bias, const void *scale, const void *res, void *out,
                      int images, int HW, int N, int K, int dtype, void *stream);

/*
 * Both pointwise layers of a block at inference in one kernel (models/convnext.py:306-318), for 16-bit types and C = 96, 128,
 * 192 or 384: out [images,C,HW] = res + scale[c] * (b2 + w2 gelu(b1 + w1 x)) for x [images,HW,C], w1 [4C,C], w2 [C,4C], all
 * of the activations' type, 16-byte aligned, images * HW below 2^31; scale [C] may be null.
 */
int dwo_block_mlp(const void *x, const void *w1, const void *b1, const void *w2, const void *b2, const void *scale,
                  const void *res, void *out, int images, int HW, int C, int dtype, void *stream);

/*
 * The stem's last layers at inference in one kernel (models/convnext.py:184-190), for 16-bit types, K = 64 and N = 96 or
 * 128: out [images,N,HW] = LayerNorm over n of (bias[n] + sum_k w[n][k] z[image][p][k]), where z is GELU(LayerNorm over k of
 * x) in x's type, x [images,HW,K].  x, w [N,K] and bias [N] (or null) have the activations' type, x, w and out are 16-byte
 * aligned, images * HW is below 2^31; the norms' parameters (gamma_in, beta_in [K]; gamma, beta [N]) are fp32.
 */
int dwo_linear_norm_planes(const void *x, const float *gamma_in, const float *beta_in, float eps_in, const void *w,
                           const void *bias, const float *gamma, const float *beta, float eps, void *out, int images, int HW,
                           int N, int K, int dtype, void *stream);

#ifdef __cplusplus
}
#endif
#endif /* DWOCONV1D_HIP_H */
