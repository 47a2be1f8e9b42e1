/*
 * exl3_layer.h — C-ABI of the MI355X (gfx950) kernels of the layer pipeline
 * around the trellis encoder (alpha2beta/EXL3_Intel_Arc_quantizer's
 * exl3_quant/hadamard.py, regularize.py and ldlq.py, which do this work with
 * torch tensor operations). Same conventions as exl3_encoder.h: device
 * buffers owned by the caller, nothing allocated, work enqueued on `stream`
 * (a hipStream_t, NULL = the null stream), 0 on success and a message in
 * exl3_last_error() otherwise. Matrices are float32, row-major, contiguous.
 */
#ifndef EXL3_LAYER_H
#define EXL3_LAYER_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Replaces preapply_had_l / preapply_had_r (hadamard.py:73-96) and their
 * in-place forms (hadamard.py:99-126): the orthonormal Sylvester matrix of
 * order 128, H[i][j] = (-1)^popcount(i & j) / sqrt(128), applied blockwise.
 * side = 0: out = H @ in on every 128-row block (rows % 128 == 0);
 * side = 1: out = in @ H on every 128-column block (cols % 128 == 0).
 * Computed as a fast Walsh-Hadamard transform in fp32; in == out is allowed. */
int exl3_hadamard128(const float* in, float* out, int64_t rows, int64_t cols, int side,
                     void* stream);

/* Division by a scale vector and the blockwise Hadamard transform in one pass
 * over HBM, the arithmetic of a division (correctly rounded fp32) followed by
 * exl3_hadamard128: the single steps that exl3_rotate and exl3_row_energy
 * join (regularize.py:171-181), for a caller that wants them apart.
 * side = 1: out = (in / divisor[col]) @ H, divisor of `cols` floats (the
 *           fold of sv before H_r); slice_sumsq, if not NULL, receives the
 *           sum of squares of every 32-element slice of every output row,
 *           slice_sumsq[row * (cols / 32) + slice] (the first pass of the
 *           row RMS that regularize takes next).
 * side = 0: out = H @ (in / divisor[row]), divisor of `rows` floats (the
 *           fold of su before H_l); slice_sumsq must be NULL.
 * divisor may be NULL (no division); in == out is allowed. */
int exl3_hadamard128_scaled(const float* in, float* out, int64_t rows, int64_t cols, int side,
                            const float* divisor, float* slice_sumsq, void* stream);

/* The two matrix passes of regularize (regularize.py:159-181) for a matrix of
 * multiples of 128, each one read of `in`: sums[row * (cols / 128) + segment] =
 * the sum of squares of every 128-element segment of the rows of (in / sv) H,
 * and out = H (((in / sv) H) / su). H is orthonormal, so the sums are taken
 * without it; out has the values of exl3_hadamard128_scaled side 1 (divisor
 * sv) and then side 0 (divisor su). sv holds `cols` floats, su `rows`; out
 * does not overlap in. */
int exl3_row_energy(const float* in, const float* sv, float* sums, int64_t rows, int64_t cols,
                    void* stream);
int exl3_rotate(const float* in, const float* sv, const float* su, float* out, int64_t rows,
                int64_t cols, void* stream);

/* Replaces weight_from_quantized (hadamard.py:129-140): out = (H (in) * su)
 * H * sv with the blockwise transforms of exl3_hadamard128, su of `rows`
 * floats (one per row), sv of `cols` floats, in one pass over HBM; the same
 * fp32 operations as the separate transforms and scalings. rows and cols are
 * multiples of 128; out and sv are 8-byte aligned; out does not overlap in. */
int exl3_unrotate(const float* in, const float* su, const float* sv, float* out, int64_t rows,
                  int64_t cols, void* stream);

/* Replaces decode_weight_from_storage (serialization.py:223-266): the weight
 * of a stored projection, exl3_unrotate of the codebook values of its packed
 * tiles (uint16 [rows / 16][cols / 16][16 K], the words exl3_pack_trellis
 * writes, 4-byte aligned) with codebook cb, in one pass. */
int exl3_decode_weight(const uint16_t* packed, const float* su, const float* sv, float* out,
                       int64_t rows, int64_t cols, int K, int cb, void* stream);

/* Second pass of block_rms (regularize.py:41-56) over slice sums made
 * elsewhere: out[o] = sqrt(S_o / n), S_o the sum of slice_sumsq[o * slices
 * + s] over s = 0 .. slices - 1 taken in slice order. */
int exl3_block_rms_from_slices(const float* slice_sumsq, float* out, int64_t outputs, int64_t n,
                               int64_t slices, void* stream);

/* The input-channel step of regularize (regularize.py:171-181): scales[r] as
 * exl3_block_rms_from_slices, 0.1 where that is below 1e-30, and su_out[r] =
 * su[r] * scales[r] / -1.24371088 + 1e-10. */
int exl3_input_scales(const float* slice_sumsq, const float* su, float* scales, float* su_out,
                      int64_t rows, int64_t n, int64_t slices, void* stream);

/* The output-channel step of regularize (regularize.py:102-168) for a
 * rows x cols matrix x: scales = its column RMS (32-row slices, as
 * exl3_block_rms) divided by their mean unless that is below 1e-30 (no
 * energy); where the scales apply, columns whose scale is below 1e-30 get
 * 0.1 and divisor[c] = sv[c] * scales[c] + 1e-10, elsewhere divisor = sv;
 * sv_out = divisor with 0 for those columns. decide: 0 the scales do not
 * apply, 1 they do, 2 they do if the skew is below 0.15; forced != 0: they
 * also apply to a matrix without energy. With diag (diag_len values,
 * diag_stride apart; may be NULL) the skew is the share of sum(sqrt(diag))
 * that its largest diag_len / 50 values hold and is written to flags[1];
 * without it flags[1] is read when decide = 2. flags (device doubles):
 * {has energy, skew, applied}. workspace: exl3_block_rms_workspace(rows,
 * cols, 0, 32) floats. */
int exl3_output_scales(const float* x, int64_t rows, int64_t cols, const float* diag,
                       int64_t diag_stride, int64_t diag_len, const float* sv, int decide,
                       int forced, float* workspace, int64_t workspace_elems, float* scales,
                       float* divisor, float* sv_out, double* flags, void* stream);

/* The sum of hessian_from_activations (calibration.py:337-357): h = scale *
 * X^T X for X of `tokens` rows (row stride ldx elements) and d columns, bf16
 * (bf16 != 0) or fp16, products and sums in float32, h float32 d x d
 * contiguous and exactly symmetric. d and ldx are multiples of 8, x is
 * 16-byte aligned. No float32 sum runs over more than chunk_tokens tokens
 * (>= 1; taken down to a multiple of 64, or 64): the chunks' sums are added
 * in float32, in token order. exl3_gram is exl3_gram_chunked with 8192.
 * workspace: exl3_gram_workspace floats (0 where the tokens are not shared
 * out). */
int exl3_gram_chunked(const uint16_t* x, int bf16, int64_t tokens, int64_t ldx, int64_t d,
                      float scale, int64_t chunk_tokens, float* h, float* workspace,
                      int64_t workspace_elems, void* stream);
int exl3_gram(const uint16_t* x, int bf16, int64_t tokens, int64_t ldx, int64_t d, float scale,
              float* h, float* workspace, int64_t workspace_elems, void* stream);

/* Floats of workspace exl3_gram needs on the current device, or -1 for a
 * shape it does not take. */
int64_t exl3_gram_workspace(int64_t tokens, int64_t d);

/* The damping of hessian_from_activations (calibration.py:359-385) on the
 * diagonal of h (row stride ld): adds max(1e-8, lambda * mean(diagonal)),
 * then replaces values below floor_value in magnitude by it. mean (device)
 * receives the mean. */
int exl3_damp_diagonal(float* h, int64_t d, int64_t ld, double lambda, float floor_value,
                       float* mean, void* stream);

/* Replaces block_rms (regularize.py:41-56): out = sqrt(S / n), S the sum of
 * squares along `dim` (0: over rows, one output per column; 1: over
 * columns, one per row) taken in slices of `blocksize` whose sums are
 * accumulated in slice order. workspace: device floats, at least
 * exl3_block_rms_workspace(rows, cols, dim, blocksize) of them (the slice
 * sums). */
int exl3_block_rms(const float* x, float* out, int64_t rows, int64_t cols, int dim, int blocksize,
                   float* workspace, int64_t workspace_elems, void* stream);

/* Floats of workspace exl3_block_rms needs (outputs x slices), or -1 for
 * invalid arguments. */
int64_t exl3_block_rms_workspace(int64_t rows, int64_t cols, int dim, int blocksize);

/* The diagonal-block step of a blocked Cholesky factorisation, which
 * replaces torch.linalg.cholesky_ex in block_ldl (ldlq.py:76-142): factors
 * the nb x nb block at `a` (leading dimension lda, lower triangle read,
 * nb <= exl3_cholesky_block_order()) in place into L (zeros above the
 * diagonal). A non-positive or NaN pivot k sets *info (device int32) to
 * offset + k + 1 unless it is already non-zero. */
int exl3_cholesky_diag_block(float* a, int64_t lda, int nb, int64_t offset, int32_t* info,
                             void* stream);

/* Replaces torch.linalg.cholesky_ex in block_ldl (ldlq.py:76-142): factors
 * the n x n matrix at `a` (contiguous, lower triangle read) in place into L;
 * the entries above the diagonal outside the diagonal blocks of order 128
 * are not touched, those inside become 0. inverses receives the inverses of
 * L's 16 x 16 diagonal tiles, [ceil(n / 16)][16][16] (a last tile that n
 * cuts is completed by an identity). A non-positive or NaN pivot k sets
 * *info (device int32) to k + 1 unless it is already non-zero. Two launches
 * per 128 columns, no host synchronisation. */
int exl3_cholesky(float* a, int64_t n, float* inverses, int32_t* info, void* stream);

/* Floats of `inverses` exl3_cholesky needs, or -1 for n < 1. */
int64_t exl3_cholesky_inverse_elems(int64_t n);

/* The fold of block_ldl (ldlq.py:120-142) for 16-wide blocks: out's block
 * column b = l's block column b times inverses[b] below the diagonal tile,
 * an identity in it, zeros above. n is a multiple of 16, l lower
 * triangular; out does not overlap l. */
int exl3_block_fold(const float* l, const float* inverses, float* out, int64_t n, void* stream);

/* Largest block order exl3_cholesky_diag_block accepts (128). */
int exl3_cholesky_block_order(void);

/* One 16-row block of an LDLQ traversal inside an encoder call: device
 * addresses (as integers) of the block's first row in W, in its
 * compensation rows, in Wq and in E = W - Wq (all float, row stride n), of
 * its (n / 16, 256) int16 states, and the block's first tile in the call's
 * batch. A call's blocks are listed in batch order, back to back
 * (tile0 of block b + 1 = tile0 + n / 16 of block b). The table itself is
 * read by the kernels, so it lives in device memory. */
typedef struct exl3_ldlq_block {
  int64_t w;
  int64_t comp;
  int64_t wq;
  int64_t err;
  int64_t states;
  int64_t n;
  int64_t tile0;
  int64_t reserved;
} exl3_ldlq_block;

/* Replaces the tile formation of one LDLQ step (ldlq.py:276-287) for every
 * block of an encoder call: x[tile0 + t][p] = W[r][16 t + c] + comp[r][16 t + c]
 * with (r, c) the row and column of tensor_core_perm(p) in a 16 x 16 tile.
 * x is f32 [tiles][256]; tiles = the sum of the blocks' n / 16. */
int exl3_ldlq_gather(const exl3_ldlq_block* blocks, int nblocks, int64_t tiles, float* x,
                     void* stream);

/* Replaces the write-back of one LDLQ step (ldlq.py:289-300) for every
 * block of an encoder call, from the encoder's tensor-core-order outputs
 * recon (f32 [tiles][256]) and idx (int16 [tiles][256]): Wq[r][16 t + c] =
 * recon, E[r][16 t + c] = W - recon at the same position, and the block's
 * states[t][p] = idx[tile0 + t][p]. */
int exl3_ldlq_scatter(const exl3_ldlq_block* blocks, int nblocks, int64_t tiles,
                      const float* recon, const int16_t* idx, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* EXL3_LAYER_H */
