// MI355X (gfx950) kernels of the layer pipeline around the trellis encoder
// (reference: exl3_quant/hadamard.py, regularize.py, ldlq.py):
//
//   had128_right_kernel / had128_left_kernel
//       the blockwise orthonormal Sylvester transform of order 128 as a fast
//       Walsh-Hadamard transform: 7 butterfly levels of fp32 add/sub and one
//       scale instead of a 128-term dot product per output. HBM-bound: one
//       read and one write of the matrix. Right (x @ H per 128-column
//       block): one wave per 128-element row segment, two elements per lane,
//       levels 2..7 across lanes. Left (H @ x per 128-row block): one thread
//       per column of a row block, the 128 values in registers; loads and
//       stores are coalesced across the wave's 64 columns.
//   unrotate_kernel
//       the way back from the encoder's basis (both transforms and both
//       scales) in one pass, from a matrix or straight from packed tiles.
//   row_energy_kernel / rotate_kernel
//       the way there (regularize): row energies, then both divisions and
//       both transforms in one pass.
//   block_rms_slices_kernel / block_rms_reduce_{columns,rows}_kernel
//       sqrt(sum of squares / n) along one dimension: one thread per slice
//       of `blocksize` sums its squares in order, then one thread per output
//       accumulates the slice sums in slice order.
//   column_slices_kernel / output_scales_kernel
//       regularize's column slice sums, and the output-channel scales from
//       the column RMS, with the skew decision on the device.
//   cholesky_diag_kernel, cholesky_solve_kernel, cholesky_update_kernel
//       a blocked right-looking Cholesky factorisation on the fp32 matrix
//       cores, 128 columns a panel.
//   block_fold_kernel
//       the block columns of the factor times the inverses of its 16 x 16
//       diagonal tiles (a block LDL's factor).
//   ldlq_gather_kernel / ldlq_scatter_kernel
//       one LDLQ step's tile formation and write-back for every 16-row block
//       of an encoder call, one 256-thread workgroup per tile: thread p moves
//       tensor-core element p between the tile and row r, column 16 t + c of
//       the block (W + compensation in; Wq, E = W - Wq and the states out).
#include <hip/hip_runtime.h>

#include <stdint.h>

#include "../../include/exl3_layer.h"
#include "exl3_codebook.h"
#include "exl3_errors.h"
#include "exl3_layout.h"

using exl3::check_launch;
using exl3::set_error;

namespace {

// 1 / sqrt(128), rounded to fp32.
constexpr float kHadScale = 0.088388347648318440550f;

hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

// ---------------------------------------------------------------- Hadamard

constexpr int HAD_N = 128;
constexpr int HAD_RIGHT_WAVES = 4;

__device__ __forceinline__ float flip(float v, uint32_t sign) {
  return __uint_as_float(__float_as_uint(v) ^ sign);
}
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}

// Butterfly of lane distance h: the lane without bit h holds the lower
// element a of each pair (a, b) and keeps a + b, its partner keeps a - b.
// Partners are reached without the LDS crossbar: DPP quad_perm (1, 2), quad
// reversal then row_half_mirror (4: i ^ 3 ^ 7), row_ror:8 (8), and
// v_permlane16_swap / v_permlane32_swap (16, 32), which leave the lower
// element of every pair in one register and the upper in the other. Through
// ds_bpermute the 12 exchanges a row takes were the transform kernels' LDS
// traffic (decoding a 4096 x 4096 projection took 38 us, 28 so). h must fold
// to a constant; every lane of the wave must be active.
__device__ __forceinline__ float had_level(float v, int lane, int h) {
  const uint32_t sign = (lane & h) ? 0x80000000u : 0u;
  switch (h) {
    case 1: return dpp<0xB1>(v) + flip(v, sign);
    case 2: return dpp<0x4E>(v) + flip(v, sign);
    case 4: return dpp<0x141>(dpp<0x1B>(v)) + flip(v, sign);
    case 8: return dpp<0x128>(v) + flip(v, sign);
    case 16: {
      const uint32_t u = __float_as_uint(v);
      const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
      return __uint_as_float(r[0]) + flip(__uint_as_float(r[1]), sign);
    }
    default: {
      const uint32_t u = __float_as_uint(v);
      const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
      return __uint_as_float(r[0]) + flip(__uint_as_float(r[1]), sign);
    }
  }
}

// DIV: every element of column c is divided by div[c] before the transform
// (regularize's fold of sv into the weight). SUMSQ: the sum of squares of
// each 32-element slice of the transformed row goes to
// sumsq[row * (cols / 32) + slice] (the first pass of the row RMS that
// follows the transform); lanes 16 j .. 16 j + 15 hold slice j of the
// segment and add their squares in a butterfly.
template <bool DIV, bool SUMSQ>
__global__ void __launch_bounds__(64 * HAD_RIGHT_WAVES)
    had128_right_kernel(const float* __restrict__ in, float* __restrict__ out, int64_t segments,
                        int64_t seg_per_row, const float* __restrict__ div,
                        float* __restrict__ sumsq) {
  const int lane = threadIdx.x & 63;
  const int64_t stride = (int64_t)gridDim.x * HAD_RIGHT_WAVES;
  for (int64_t seg = (int64_t)blockIdx.x * HAD_RIGHT_WAVES + (threadIdx.x >> 6); seg < segments;
       seg += stride) {
    // Lane l holds elements 2l and 2l + 1 of the segment.
    float2 v = reinterpret_cast<const float2*>(in + seg * HAD_N)[lane];
    if (DIV) {
      const float2 d =
          reinterpret_cast<const float2*>(div + (seg % seg_per_row) * HAD_N)[lane];
      v.x = v.x / d.x;
      v.y = v.y / d.y;
    }
    float lo = v.x + v.y, hi = v.x - v.y;
#pragma unroll
    for (int h = 1; h < 64; h <<= 1) {
      lo = had_level(lo, lane, h);
      hi = had_level(hi, lane, h);
    }
    lo = lo * kHadScale;
    hi = hi * kHadScale;
    reinterpret_cast<float2*>(out + seg * HAD_N)[lane] = make_float2(lo, hi);
    if (SUMSQ) {
      float q = lo * lo + hi * hi;
#pragma unroll
      for (int h = 1; h < 16; h <<= 1) q = q + __shfl_xor(q, h, 64);
      if ((lane & 15) == 0) sumsq[seg * (HAD_N / 32) + (lane >> 4)] = q;
    }
  }
}

// DIV: every element of row r is divided by div[r] before the transform
// (the fold of su).
template <bool DIV>
__global__ void __launch_bounds__(256)
    had128_left_kernel(const float* __restrict__ in, float* __restrict__ out, int64_t cols,
                       const float* __restrict__ div) {
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c >= cols) return;
  const int64_t row0 = (int64_t)blockIdx.y * HAD_N;
  const int64_t base = row0 * cols + c;
  float v[HAD_N];
#pragma unroll
  for (int r = 0; r < HAD_N; ++r) {
    v[r] = in[base + r * cols];
    if (DIV) v[r] = v[r] / div[row0 + r];
  }
#pragma unroll
  for (int h = 1; h < HAD_N; h <<= 1) {
#pragma unroll
    for (int i = 0; i < HAD_N; ++i) {
      if (!(i & h)) {
        const float a = v[i], b = v[i + h];
        v[i] = a + b;
        v[i + h] = a - b;
      }
    }
  }
#pragma unroll
  for (int r = 0; r < HAD_N; ++r) out[base + r * cols] = v[r] * kHadScale;
}

// H_l, x su per row, H_r, x sv per column (hadamard.py:129-140) of one
// 128 x 128 block per workgroup: the block is closed under both transforms,
// so the whole way back is one read and one write of the matrix, where the
// two transforms and two scalings by themselves are four of each. PACKED
// reads the block's 64 tiles of stored trellis words instead of a matrix
// (state, codebook value and tensor-core position computed in the kernel),
// so a stored projection is decoded in one pass of K / 8 + 4 bytes per
// weight. The fp32 operations and their order are those of the separate
// passes: results are bit-identical to them.
//
// Eight waves. First half: wave w takes rows 32 (w / 2) .. + 31 of 64
// columns, one column per lane, the 32 values in registers (butterfly
// distances 1 .. 16), and leaves them in LDS. Second half: each wave takes
// rows g, g + 32, g + 64, g + 96 (distances 32 and 64), two columns per
// lane, scales them and transforms the four rows across the wave. 64 KiB of
// LDS, two workgroups per CU. A 4096 x 4096 projection at K = 4 (75 MB)
// decodes in 28 us; unpacking, a table lookup, the un-permutation, two
// transforms and two scalings took 390 us.
constexpr int UN_THREADS = 512;

template <bool PACKED, int CB>
__global__ void __launch_bounds__(UN_THREADS, 4)
    unrotate_kernel(const float* __restrict__ in, const uint32_t* __restrict__ packed, int K,
                    const float* __restrict__ su, const float* __restrict__ sv,
                    float* __restrict__ out, int64_t cols) {
  __shared__ __attribute__((aligned(16))) float s[HAD_N * HAD_N];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int half = wave & 1, r0 = (wave >> 1) * 32;
  const int64_t row0 = (int64_t)blockIdx.y * HAD_N, col0 = (int64_t)blockIdx.x * HAD_N;

  float v[32];
  int c;  // the lane's column
  if constexpr (PACKED) {
    // Tile row `wave` of the block is 8 tiles, 64 K words, contiguous.
    uint32_t* s_words = reinterpret_cast<uint32_t*>(s);
    const uint32_t* src =
        packed + ((row0 / 16 + wave) * (cols / 16) + col0 / 16) * (int64_t)(8 * K);
    // Word j sits at j ^ (j / 64 % 8): the lanes of a read are K words apart,
    // so that those in one bank are whole 64-word blocks apart.
    auto at = [](int j) { return j ^ ((j >> 6) & 7); };
    for (int j = 0; j < K; ++j) s_words[at((wave * K + j) * 64 + lane)] = src[j * 64 + lane];
    __syncthreads();
    // Column 8 half + lane % 8 of tile column lane / 8. Row 2 q + (e & 1) +
    // 8 (e >> 1) of tile column cc + 8 half is encoded element i = 32 cc +
    // 8 q + 4 half + e, whose state is the 16 bits of the tile's stream
    // ending at bit (i + 1) K: the same bit offset in every lane, from word
    // cc K on (a stored uint32 is 32 stream bits, most significant first).
    const int cc = lane & 7, tc = lane >> 3;
    c = tc * 16 + half * 8 + cc;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int tile = ((r0 / 16 + t) * 8 + tc) * 8 * K;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int last = (8 * q + 4 * half + e + 1) * K - 1;  // the window's last bit
          const int word = cc * K + (last >> 5);
          const uint32_t lo = s_words[at(tile + word)];
          const uint32_t hi = s_words[at(tile + (word > 0 ? word - 1 : 8 * K - 1))];
          const uint32_t state = __builtin_amdgcn_alignbit(hi, lo, 31 - (last & 31)) & 0xFFFFu;
          v[16 * t + 2 * q + (e & 1) + 8 * (e >> 1)] = (float)decode_state(CB, state);
        }
      }
    }
    __syncthreads();
  } else {
    c = half * 64 + lane;
    const float* src = in + (row0 + r0) * cols + col0 + c;
#pragma unroll
    for (int r = 0; r < 32; ++r) v[r] = src[r * cols];
  }
#pragma unroll
  for (int h = 1; h < 32; h <<= 1) {
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      if (!(i & h)) {
        const float a = v[i], b = v[i + h];
        v[i] = a + b;
        v[i + h] = a - b;
      }
    }
  }
#pragma unroll
  for (int r = 0; r < 32; ++r) s[(r0 + r) * HAD_N + c] = v[r];
  __syncthreads();

  const float2 d = reinterpret_cast<const float2*>(sv + col0)[lane];
#pragma unroll 1
  for (int g = wave; g < 32; g += 8) {
    float2 x[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      x[j] = reinterpret_cast<const float2*>(s + (g + 32 * j) * HAD_N)[lane];
#pragma unroll
    for (int h = 1; h < 4; h <<= 1) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (!(j & h)) {
          const float2 a = x[j], b = x[j + h];
          x[j] = make_float2(a.x + b.x, a.y + b.y);
          x[j + h] = make_float2(a.x - b.x, a.y - b.y);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float u = su[row0 + g + 32 * j];
      const float a = (x[j].x * kHadScale) * u, b = (x[j].y * kHadScale) * u;
      x[j] = make_float2(a + b, a - b);
    }
#pragma unroll
    for (int h = 1; h < 64; h <<= 1) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        x[j].x = had_level(x[j].x, lane, h);
        x[j].y = had_level(x[j].y, lane, h);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      reinterpret_cast<float2*>(out + (row0 + g + 32 * j) * cols + col0)[lane] =
          make_float2((x[j].x * kHadScale) * d.x, (x[j].y * kHadScale) * d.y);
  }
}

// Row energies of (in / sv) H_r without the transform: it is orthonormal, so
// a 128-element segment keeps its sum of squares (and in float32 this one has
// the fewer roundings). One read of the matrix and 1/128 of it written. A wave
// takes two rows of a segment at a time, 16 bytes a lane, EN_LOADS of them
// issued together. In a segment with two infinities the transform would meet
// inf - inf, and its energy is NaN.
constexpr int EN_LOADS = 8, EN_WAVES = 4, EN_ROWS = 2 * EN_LOADS * EN_WAVES;

// Sum over the lane's half of the wave.
__device__ __forceinline__ float half_wave_sum(float q) {
  q = q + dpp<0xB1>(q);
  q = q + dpp<0x4E>(q);
  q = q + dpp<0x141>(dpp<0x1B>(q));
  q = q + dpp<0x128>(q);
  const uint32_t u = __float_as_uint(q);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

__global__ void __launch_bounds__(64 * EN_WAVES)
    row_energy_kernel(const float* __restrict__ in, int64_t cols, const float* __restrict__ sv,
                      float* __restrict__ sums) {
  const int lane = threadIdx.x & 63, half = lane >> 5;
  // Workgroups along the columns first.
  const uint32_t segments = (uint32_t)(cols / HAD_N), seg = blockIdx.x % segments;
  const int64_t row0 = (int64_t)(blockIdx.x / segments) * EN_ROWS +
                       (int64_t)(threadIdx.x >> 6) * (2 * EN_LOADS) + half;
  const float* src = in + row0 * cols + (int64_t)seg * HAD_N;
  float4 x[EN_LOADS];
#pragma unroll
  for (int j = 0; j < EN_LOADS; ++j)
    x[j] = reinterpret_cast<const float4*>(src + 2 * j * cols)[lane & 31];
  const float4 d = reinterpret_cast<const float4*>(sv + (int64_t)seg * HAD_N)[lane & 31];
#pragma unroll
  for (int j = 0; j < EN_LOADS; ++j) {
    const float v[4] = {x[j].x / d.x, x[j].y / d.y, x[j].z / d.z, x[j].w / d.w};
    const float q =
        half_wave_sum((v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]));
    int infinities = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint64_t all = __ballot(__builtin_isinf(v[e]));
      infinities += __popc((uint32_t)(half ? all >> 32 : all));
    }
    if ((lane & 31) == 0)
      sums[(row0 + 2 * j) * segments + seg] = infinities > 1 ? __builtin_nanf("") : q;
  }
}

// H_l (((in / sv) H_r) / su) of one 128 x 128 block per workgroup: both
// transforms and both divisions of regularize in one read and one write,
// once the row scales are known. The fp32 operations and their order are
// those of the separate passes: results are bit-identical to them.
//
// The mirror image of unrotate_kernel. First half: each wave takes rows 4 g
// .. 4 g + 3 for four g, two columns per lane, all its loads issued together;
// the right transform runs across the wave, the left one starts with row
// distances 1 and 2. Second half: wave w takes rows w / 2, w / 2 + 4, .. of
// 64 columns, one column per lane (distances 4 .. 64). 64 KiB of LDS, two
// workgroups per CU. A 4096 matrix (134 MB) takes 33 us, about half of it the
// cross-lane butterflies' and the divisions' instructions, and 15 us in
// row_energy_kernel; storing the right transform and reading it again for the
// left one took 61.
constexpr int RO_THREADS = 512, RO_WAVES = RO_THREADS / 64, RO_GROUPS = HAD_N / 4 / RO_WAVES;

__global__ void __launch_bounds__(RO_THREADS, 4)
    rotate_kernel(const float* __restrict__ in, const float* __restrict__ sv,
                  const float* __restrict__ su, float* __restrict__ out, int64_t cols) {
  __shared__ __attribute__((aligned(16))) float s[HAD_N * HAD_N];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t row0 = (int64_t)blockIdx.y * HAD_N, col0 = (int64_t)blockIdx.x * HAD_N;

  float2 x[RO_GROUPS][4];
#pragma unroll
  for (int g = 0; g < RO_GROUPS; ++g) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      x[g][j] = reinterpret_cast<const float2*>(
          in + (row0 + 4 * (wave + RO_WAVES * g) + j) * cols + col0)[lane];
  }
  const float2 d = reinterpret_cast<const float2*>(sv + col0)[lane];
#pragma unroll
  for (int g = 0; g < RO_GROUPS; ++g) {
    const int r0 = 4 * (wave + RO_WAVES * g);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float a = x[g][j].x / d.x, b = x[g][j].y / d.y;
      float lo = a + b, hi = a - b;
#pragma unroll
      for (int h = 1; h < 64; h <<= 1) {
        lo = had_level(lo, lane, h);
        hi = had_level(hi, lane, h);
      }
      const float u = su[row0 + r0 + j];
      x[g][j] = make_float2((lo * kHadScale) / u, (hi * kHadScale) / u);
    }
#pragma unroll
    for (int h = 1; h < 4; h <<= 1) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (!(j & h)) {
          const float2 a = x[g][j], b = x[g][j + h];
          x[g][j] = make_float2(a.x + b.x, a.y + b.y);
          x[g][j + h] = make_float2(a.x - b.x, a.y - b.y);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) reinterpret_cast<float2*>(s + (r0 + j) * HAD_N)[lane] = x[g][j];
  }
  __syncthreads();

  const int q = wave >> 1, c = (wave & 1) * 64 + lane;
  float v[32];
#pragma unroll
  for (int r = 0; r < 32; ++r) v[r] = s[(q + 4 * r) * HAD_N + c];
#pragma unroll
  for (int h = 1; h < 32; h <<= 1) {
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      if (!(i & h)) {
        const float a = v[i], b = v[i + h];
        v[i] = a + b;
        v[i + h] = a - b;
      }
    }
  }
  float* dst = out + (row0 + q) * cols + col0 + c;
#pragma unroll
  for (int r = 0; r < 32; ++r) dst[4 * r * cols] = v[r] * kHadScale;
}

// --------------------------------------------------------------- block RMS

// Output o reduces x[o * so + t * st] over t < n, in ns slices of bs.
// Pass 1: one thread per (output, slice) sums the slice's squares in order
// into ws: slice-major (ws[s * outputs + o]) when dim = 0, so that threads
// of a wave read adjacent columns, output-major (ws[o * ns + s]) when
// dim = 1, so that they read adjacent slices of one row.
__global__ void __launch_bounds__(256)
    block_rms_slices_kernel(const float* __restrict__ x, float* __restrict__ ws, int64_t outputs,
                            int64_t n, int64_t so, int64_t st, int bs, int64_t ns, int dim) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= outputs * ns) return;
  const int64_t o = dim == 0 ? idx % outputs : idx / ns;
  const int64_t s = dim == 0 ? idx / outputs : idx % ns;
  const int64_t t0 = s * bs, t1 = t0 + bs < n ? t0 + bs : n;
  const float* p = x + o * so;
  float slice = 0.0f;
  for (int64_t t = t0; t < t1; ++t) {
    const float v = p[t * st];
    const float sq = v * v;
    slice = slice + sq;
  }
  ws[idx] = slice;
}

// Pass 2: one thread per output accumulates its slice sums in slice order.
// The additions are one dependent chain, the loads are not: RMS_BATCH of
// them are issued together, so a chain of 128 slices waits for memory 4
// times instead of 128 (4096 outputs, 128 slices: 18.7 us one load at a
// time).
constexpr int RMS_BATCH = 32;

template <class Load>
__device__ __forceinline__ float ordered_sum(int64_t ns, Load load) {
  float acc = 0.0f;
  int64_t s = 0;
  for (; s + RMS_BATCH <= ns; s += RMS_BATCH) {
    float v[RMS_BATCH];
#pragma unroll
    for (int j = 0; j < RMS_BATCH; ++j) v[j] = load(s + j);
#pragma unroll
    for (int j = 0; j < RMS_BATCH; ++j) acc = (s + j == 0) ? v[j] : acc + v[j];
  }
  for (; s < ns; ++s) {
    const float v = load(s);
    acc = (s == 0) ? v : acc + v;
  }
  return acc;
}

// dim = 0: ws[s * outputs + o], coalesced over the outputs.
__global__ void __launch_bounds__(64)
    block_rms_reduce_columns_kernel(const float* __restrict__ ws, float* __restrict__ out,
                                    int64_t outputs, int64_t n, int64_t ns) {
  const int64_t o = (int64_t)blockIdx.x * 64 + threadIdx.x;
  if (o >= outputs) return;
  out[o] = sqrtf(ordered_sum(ns, [&](int64_t s) { return ws[s * outputs + o]; }) / (float)n);
}

// dim = 1: ws[o * ns + s]. A workgroup's ROWS_RED outputs are contiguous in
// ws, so their slice sums pass through LDS in chunks of ROWS_CHUNK, loaded
// along the rows (coalesced) and summed down them by one lane per output
// (a row stride of ROWS_CHUNK + 1: 64 different banks). 4096 outputs, 128
// slices: 37.6 us with strided loads from HBM, 4.0 us here.
// su != NULL: the output is an input-channel scale and the row's sign-folded
// divisor goes to su_out (regularize.py:171-181): a scale that is zero
// becomes 0.1, su_out = su * scale / -1.24371088 + 1e-10, where the division
// by the constant is a multiplication by its reciprocal, as torch divides by
// a host scalar.
constexpr int ROWS_RED = 64, ROWS_CHUNK = 128;

constexpr float kTiny = 1e-30f;       // below this an RMS counts as zero
constexpr float kZeroFloor = 0.1f;    // scale of an all-zero row or column
constexpr float kScaleEps = 1e-10f;   // added to every scale
constexpr float kCodebookScale = 1.24371088f;
constexpr float kSkewCutoff = 0.15f;  // output scales only below this skew
constexpr int kSkewFraction = 50;     // the skew looks at the top 1/50 of the diagonal

__global__ void __launch_bounds__(256)
    block_rms_reduce_rows_kernel(const float* __restrict__ ws, float* __restrict__ out,
                                 int64_t outputs, int64_t n, int64_t ns,
                                 const float* __restrict__ su, float* __restrict__ su_out) {
  __shared__ float s_v[ROWS_RED][ROWS_CHUNK + 1];
  const int64_t o0 = (int64_t)blockIdx.x * ROWS_RED;
  const int rows = outputs - o0 < ROWS_RED ? (int)(outputs - o0) : ROWS_RED;
  float acc = 0.0f;
  for (int64_t s0 = 0; s0 < ns; s0 += ROWS_CHUNK) {
    const int len = ns - s0 < ROWS_CHUNK ? (int)(ns - s0) : ROWS_CHUNK;
#pragma unroll 8
    for (int i = threadIdx.x; i < rows * ROWS_CHUNK; i += 256) {
      const int r = i / ROWS_CHUNK, c = i % ROWS_CHUNK;
      if (c < len) s_v[r][c] = ws[(o0 + r) * ns + s0 + c];
    }
    __syncthreads();
    if ((int)threadIdx.x < rows) {
      const float* row = s_v[threadIdx.x];
      const float part = ordered_sum(len, [&](int64_t c) {
        return c == 0 && s0 > 0 ? acc + row[0] : row[c];
      });
      acc = part;
    }
    __syncthreads();
  }
  if ((int)threadIdx.x >= rows) return;
  const int64_t o = o0 + threadIdx.x;
  float v = sqrtf(acc / (float)n);
  if (su != nullptr) {
    if (fabsf(v) < kTiny) v = kZeroFloor;
    su_out[o] = (su[o] * v) * (1.0f / -kCodebookScale) + kScaleEps;
  }
  out[o] = v;
}

// ----------------------------------------------------------- output scales

constexpr int SC_THREADS = 1024;

// Sum over the workgroup, in every thread.
__device__ __forceinline__ double block_sum(double v, double* s_red) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < SC_THREADS / 64; ++w) t += s_red[w];
  return t;
}

// Share of sum(sqrt(diag)) held by its largest len / 50 entries
// (regularize.py:102-118), by one workgroup: the m-th largest value is found
// by radix selection over the bits of the (non-negative) roots, eight bits a
// pass, so nothing is sorted. Sums in double. A NaN root makes the skew NaN.
__device__ float diagonal_skew(const float* __restrict__ diag, int64_t stride, int64_t len,
                               uint32_t* s_hist, uint32_t* s_pick, double* s_red) {
  const int64_t m = len / kSkewFraction;
  auto root = [&](int64_t i) { return sqrtf(diag[i * stride]) + 0.0f; };
  uint32_t prefix = 0, left = (uint32_t)m;
  for (int shift = 24; m > 0 && shift >= 0; shift -= 8) {
    for (int b = threadIdx.x; b < 256; b += SC_THREADS) s_hist[b] = 0;
    __syncthreads();
    for (int64_t i = threadIdx.x; i < len; i += SC_THREADS) {
      const uint32_t bits = __float_as_uint(root(i));
      if (shift == 24 || (bits >> (shift + 8)) == prefix)
        atomicAdd(&s_hist[(bits >> shift) & 255u], 1u);
    }
    __syncthreads();
    if (threadIdx.x < 64) {
      // Lane l holds bins 255 - 4 l .. 252 - 4 l; the bin where the count
      // from the top reaches `left` is the next byte.
      const int lane = threadIdx.x;
      uint32_t c[4], own = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) own += c[j] = s_hist[255 - 4 * lane - j];
      uint32_t upto = own;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = (uint32_t)__shfl_up((int)upto, d, 64);
        if (lane >= d) upto += o;
      }
      uint32_t before = upto - own;
      if (before < left && upto >= left) {
        int j = 0;
        while (before + c[j] < left) before += c[j++];
        s_pick[0] = (prefix << 8) | (uint32_t)(255 - 4 * lane - j);
        s_pick[1] = left - before;
      }
    }
    __syncthreads();
    prefix = s_pick[0];
    left = s_pick[1];
    __syncthreads();
  }
  double all = 0.0, top = 0.0;
  for (int64_t i = threadIdx.x; i < len; i += SC_THREADS) {
    const float r = root(i);
    all += (double)r;
    if (m > 0 && __float_as_uint(r) > prefix) top += (double)r;
  }
  all = block_sum(all, s_red);
  top = block_sum(top, s_red);
  if (m > 0) top += (double)left * (double)__uint_as_float(prefix);
  // A NaN root is in `all`; the quotient is NaN whatever was selected.
  return (float)top / (float)all;
}

// First pass of the column RMS (block_rms_slices_kernel's sums for dim = 0 and
// 32-row slices), and in workgroup 0 the skew of the Hessian diagonal into
// flags[1]: its four histogram passes over a few thousand values take 10 us
// and wait for nothing here, so they run under the matrix's read (67 MB: 15
// us) and not after it.
constexpr int COL_SLICE = 32;

__global__ void __launch_bounds__(SC_THREADS)
    column_slices_kernel(const float* __restrict__ x, float* __restrict__ ws, int64_t cols,
                         int64_t rows, int64_t ns, const float* __restrict__ diag,
                         int64_t diag_stride, int64_t diag_len, double* __restrict__ flags) {
  __shared__ uint32_t s_hist[256];
  __shared__ uint32_t s_pick[2];
  __shared__ double s_red[SC_THREADS / 64];
  int64_t b = blockIdx.x;
  if (diag != nullptr) {
    if (b == 0) {
      const float skew = diagonal_skew(diag, diag_stride, diag_len, s_hist, s_pick, s_red);
      if (threadIdx.x == 0) flags[1] = (double)skew;
      return;
    }
    --b;
  }
  const int64_t idx = b * SC_THREADS + threadIdx.x;
  if (idx >= cols * ns) return;
  const int64_t o = idx % cols, t0 = idx / cols * COL_SLICE;
  const float* p = x + t0 * cols + o;
  float slice = 0.0f;
  if (t0 + COL_SLICE <= rows) {
    float v[COL_SLICE];
#pragma unroll
    for (int t = 0; t < COL_SLICE; ++t) v[t] = p[t * cols];
#pragma unroll
    for (int t = 0; t < COL_SLICE; ++t) slice = slice + v[t] * v[t];
  } else {
    for (int64_t t = 0; t < rows - t0; ++t) {
      const float v = p[t * cols];
      slice = slice + v * v;
    }
  }
  ws[idx] = slice;
}

// The output-channel scales of regularize (regularize.py:136-168) from the
// column RMS, in one workgroup: normalised by their mean unless W has no
// energy, zero columns floored and sv folded where the scales apply. decide:
// 0 never, 1 always, 2 where the skew (flags[1]) is below the cutoff; forced:
// they also apply where W has no energy. divisor is what W's columns are
// divided by, sv_out the same with zeros for the dead columns. flags =
// {any energy, skew, applied}.
__global__ void __launch_bounds__(SC_THREADS)
    output_scales_kernel(float* __restrict__ scales, int64_t cols,
                         const float* __restrict__ sv, int decide, int forced,
                         float* __restrict__ divisor, float* __restrict__ sv_out,
                         double* __restrict__ flags) {
  __shared__ double s_red[SC_THREADS / 64];
  double sum = 0.0;
  for (int64_t i = threadIdx.x; i < cols; i += SC_THREADS) sum += (double)scales[i];
  const float mean = (float)(block_sum(sum, s_red) / (double)cols);
  const bool live = mean > kTiny;
  const bool apply = (forced && !live) || decide == 1 ||
                     (decide == 2 && (float)flags[1] < kSkewCutoff);
  for (int64_t i = threadIdx.x; i < cols; i += SC_THREADS) {
    float v = scales[i] / (live ? mean : 1.0f);
    const bool dead = fabsf(v) < kTiny;
    float d = sv[i];
    if (apply) {
      if (dead) v = kZeroFloor;
      d = d * v + kScaleEps;
    }
    scales[i] = v;
    divisor[i] = d;
    sv_out[i] = dead ? 0.0f : d;
  }
  if (threadIdx.x == 0) {
    flags[0] = live ? 1.0 : 0.0;
    flags[2] = apply ? 1.0 : 0.0;
  }
}

// -------------------------------------------------------------- Cholesky
//
// Blocked right-looking factorisation in panels of 128 columns, two launches
// a panel: the panel's rows below its diagonal block are solved against it
// (cholesky_solve_kernel), then every 128 x 128 tile of the trailing lower
// triangle loses X_i X_j^T (cholesky_update_kernel), whose first workgroup
// takes the next diagonal block and goes on to factor it while the others
// update. What bounds a 4096 matrix is the chain of its 32 panels, each the
// update and factorisation of one diagonal block by one workgroup plus one
// solve; the 23 GFLOP of updates run beside it on the fp32 matrix cores
// (v_mfma_f32_16x16x4: fp32 products and sums).
//
// A diagonal block is factored in 16-column steps: one wave factors the
// 16 x 16 diagonal tile in registers, four columns at a time, and inverts
// it, the tiles below it are multiplied by that inverse, and while the
// trailing tiles are updated the first wave already takes the next diagonal
// tile.
// The 16 x 16 inverses are kept: the panel solve multiplies by them, and
// they are what a block LDL folds into the factor's columns.
// A 128-block took 87 us with one barrier per column, 26 us here (of which
// 16 columns take about 2 us); a panel of a 4096 matrix takes 41 us (update
// and next diagonal block 34, solve 7.5) where the diagonal kernel, a library
// triangular solve and a library GEMM took 170.
//
// Fragments. For v_mfma_f32_16x16x4 lane l gives A[l % 16][l / 16] and
// B[l / 16][l % 16] and holds D[4 (l / 16) + r][l % 16] in register r. Over
// 16 values of k, lane l's step-t value may be k = 4 (l / 16) + t, in A and
// B alike, so a lane's four values are one 16-byte load along k.

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int CH_NB = 128;               // panel width, largest block order
constexpr int CH_T = 16;                 // tile
constexpr int CH_TILES = CH_NB / CH_T;
constexpr int CH_LD = CH_NB + 4;         // LDS row stride: 16-byte aligned, rows 4 banks apart
constexpr int CH_WLD = CH_T + 4;
constexpr int CH_THREADS = 256;
constexpr int CH_KC = 32, CH_KLD = CH_KC + 4;  // columns staged at a time by the update

// acc += A B over 16 values of k.
__device__ __forceinline__ f32x4 mfma16(f32x4 a, f32x4 b, f32x4 acc) {
#pragma unroll
  for (int t = 0; t < 4; ++t) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t], b[t], acc, 0, 0, 0);
  return acc;
}

// 1 / sqrt(p) to an ulp, from the hardware estimate; p below 2^-100 is scaled,
// since the estimate takes a subnormal for zero.
__device__ __forceinline__ float inverse_sqrt(float p) {
  const float plain = __builtin_amdgcn_rsqf(p);
  const float tiny = __builtin_amdgcn_rsqf(p * 0x1p64f) * 0x1p32f;
  return p < 0x1p-100f ? tiny : plain;
}

// The value of `v` in lane `src` of the wave.
__device__ __forceinline__ float lane_value(float v, int src) {
  return __int_as_float(__builtin_amdgcn_ds_bpermute(4 * src, __float_as_int(v)));
}
__device__ __forceinline__ float uniform_value(float v, int src) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), src));
}
// v[i] of four registers. By value: a choice between array elements becomes a
// choice between addresses, and the array then lives in scratch memory or LDS.
__device__ __forceinline__ float pick(float v0, float v1, float v2, float v3, int i) {
  const float lo = i & 1 ? v1 : v0, hi = i & 1 ? v3 : v2;
  return i & 2 ? hi : lo;
}

// Factors a 16 x 16 tile held in m (the whole symmetric tile in D layout:
// m[t] = element [4 (l / 16) + t][l % 16]). Writes the factor to d (LDS, row
// stride CH_LD, zeros above the diagonal) and its inverse to s_inv. One wave,
// and no global store in it: each would be waited for on the way.
//
// Four columns at a time: rows 4 p .. 4 p + 3 of the symmetric remainder are
// columns 4 p .. 4 p + 3, one row per lane, in lanes 16 p .. 16 p + 15; every
// 16-lane group takes a copy and factors them (6 multiply-adds against a
// scalar), and the remainder loses their product in one matrix instruction
// whose two operands are the same register. The inverse advances beside it:
// rows 4 p .. of the remainder of I are divided by the 4 x 4 diagonal part
// in place, and the rest loses the columns times those rows. Entries of
// finished rows and columns are garbage that no later one reads.
__device__ __forceinline__ void factor_tile(f32x4 m, float* d, float* s_inv, int lane,
                                            int64_t index, int32_t* info) {
  const int r = lane & 15, g = lane >> 4;
  f32x4 w;
#pragma unroll
  for (int t = 0; t < 4; ++t) w[t] = 4 * g + t == r ? 1.0f : 0.0f;
  int bad = 0;
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    float v[4], rs[4], x[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) v[c] = lane_value(m[c], 16 * p + r);
    float l[4][4];  // the 4 x 4 diagonal part, uniform
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float pivot = uniform_value(v[c], 4 * p + c);
      rs[c] = inverse_sqrt(pivot);
      // The column times 1 / root (LAPACK's potf2 scaling); the diagonal,
      // which no other entry waits for, is the root with one correction (its
      // residual is exact in fp32).
      const float scaled = v[c] * rs[c];
#pragma unroll
      for (int e = c + 1; e < 4; ++e) {
        l[e][c] = uniform_value(scaled, 4 * p + e);
        v[e] = fmaf(-l[e][c], scaled, v[e]);
      }
      const float root = pivot * rs[c];
      const float fixed = fmaf(fmaf(-root, root, pivot), 0.5f * rs[c], root);
      v[c] = r == 4 * p + c ? fixed : scaled;
      // One scalar test for all that is not positive and finite, since this
      // is the chain. An infinite pivot is its own root, which 0 = 1 / root
      // does not give; its column is zero.
      const uint32_t bits = __float_as_uint(pivot);
      if (__builtin_expect(bits - 1u >= 0x7F7FFFFFu, 0)) {
        if (bits == 0x7F800000u) {
          if (r == 4 * p + c) v[c] = pivot;
        } else if (bad == 0) {
          bad = 4 * p + c + 1;
        }
      }
    }
    if (g == 0) {
      f32x4 q;
#pragma unroll
      for (int c = 0; c < 4; ++c) q[c] = 4 * p + c <= r ? v[c] : 0.0f;
      *reinterpret_cast<f32x4*>(d + r * CH_LD + 4 * p) = q;
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      float y = w[c];
#pragma unroll
      for (int e = 0; e < c; ++e) y = fmaf(-l[c][e], x[e], y);
      x[c] = y * rs[c];
    }
    if (g == p) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        // The inverse is lower triangular: nothing above the diagonal.
        s_inv[(4 * p + c) * CH_WLD + r] = 4 * p + c >= r ? x[c] : 0.0f;
      }
    }
    if (p < 3) {
      const float a = pick(v[0], v[1], v[2], v[3], g);  // column 4 p + g, row r: A and, transposed, B
      float rows[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) rows[c] = lane_value(x[c], 16 * p + r);
      m = __builtin_amdgcn_mfma_f32_16x16x4f32(-a, a, m, 0, 0, 0);
      const float b = pick(rows[0], rows[1], rows[2], rows[3], g);
      w = __builtin_amdgcn_mfma_f32_16x16x4f32(-a, b, w, 0, 0, 0);
    }
  }
  if (bad != 0 && lane == 0) atomicCAS(info, 0, (int32_t)(index + bad));
}

// X_i X_j^T, X the 16 columns from column k0 of the block in LDS.
__device__ __forceinline__ f32x4 tile_product(const float* s, int i, int j, int k0, int lane) {
  const int r = lane & 15, g = lane >> 4;
  const f32x4 a = *reinterpret_cast<const f32x4*>(s + (16 * i + r) * CH_LD + k0 + 4 * g);
  const f32x4 b = *reinterpret_cast<const f32x4*>(s + (16 * j + r) * CH_LD + k0 + 4 * g);
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  return mfma16(a, b, zero);
}

// Diagonal tile t of the block in LDS, its lower triangle mirrored.
__device__ __forceinline__ f32x4 symmetric_tile(const float* s, int t, int lane) {
  const int r = lane & 15, g = lane >> 4;
  const float* d = s + 16 * t * (CH_LD + 1);
  f32x4 m;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int row = 4 * g + q;
    m[q] = row >= r ? d[row * CH_LD + r] : d[r * CH_LD + row];
  }
  return m;
}

// Factors the 128 x 128 block in LDS (its lower triangle; tiles past
// `tiles` are left alone). inv receives the inverses of its 16 x 16 diagonal
// tiles, back to back (may be NULL). All four waves.
__device__ __forceinline__ void factor_block(float* s, float* s_inv, int tiles, float* __restrict__ inv,
                             int64_t offset, int32_t* info) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  auto store_inverse = [&](int t) {
    static_assert(CH_T * CH_T == CH_THREADS, "one element of a tile per thread");
    if (inv)
      inv[t * CH_THREADS + threadIdx.x] =
          s_inv[(threadIdx.x / CH_T) * CH_WLD + threadIdx.x % CH_T];
  };
  if (wave == 0) factor_tile(symmetric_tile(s, 0, lane), s, s_inv, lane, offset, info);
  __syncthreads();
  for (int kb = 0; kb + 1 < tiles; ++kb) {
    const int k0 = 16 * kb;
    store_inverse(kb);
    // X_t = S_t inverse^T for the tiles below the diagonal one.
    const int r = lane & 15, g = lane >> 4;
    const f32x4 w = *reinterpret_cast<const f32x4*>(s_inv + r * CH_WLD + 4 * g);
    for (int t = kb + 1 + wave; t < tiles; t += 4) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(s + (16 * t + r) * CH_LD + k0 + 4 * g);
      const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
      const f32x4 d = mfma16(x, w, zero);
      // Every lane's loads above are done before any lane of the wave
      // stores: one wave owns the tile and its instructions are in order.
#pragma unroll
      for (int q = 0; q < 4; ++q) s[(16 * t + 4 * g + q) * CH_LD + k0 + r] = d[q];
    }
    __syncthreads();
    if (wave == 0) {
      const f32x4 m = symmetric_tile(s, kb + 1, lane) - tile_product(s, kb + 1, kb + 1, k0, lane);
      factor_tile(m, s + (k0 + 16) * (CH_LD + 1), s_inv, lane, offset + k0 + 16, info);
    } else {
      // The other trailing tiles, lower triangle, dealt over waves 1 .. 3.
      const int left = tiles - kb - 2;  // tile rows below the next diagonal tile
      for (int u = wave - 1; u < left * (left + 3) / 2; u += 3) {
        // Tile row i has i + 2 tiles, tile columns kb + 1 .. kb + 2 + i.
        int i = 0, j = u;
        while (j > i + 1) j -= i++ + 2;
        const int ti = kb + 2 + i, tj = kb + 1 + j;
        const f32x4 d = tile_product(s, ti, tj, k0, lane);
        float* c = s + (16 * ti + 4 * g) * CH_LD + 16 * tj + r;
#pragma unroll
        for (int t = 0; t < 4; ++t) c[t * CH_LD] -= d[t];
      }
    }
    __syncthreads();
  }
  store_inverse(tiles - 1);
}

// The lower triangle of the factored block to a (leading dimension lda),
// zeros above the diagonal, the first nb rows and columns only.
__device__ __forceinline__ void store_block(const float* s, float* __restrict__ a, int64_t lda,
                                            int nb) {
#pragma unroll 16
  for (int e = 0; e < CH_NB * CH_NB / CH_THREADS; ++e) {
    const int i = threadIdx.x + e * CH_THREADS, r = i / CH_NB, c = i % CH_NB;
    const float v = c <= r ? s[r * CH_LD + c] : 0.0f;
    if (r < nb && c < nb) a[r * lda + c] = v;
  }
}

// Factors the nb x nb block at `a` (row-major, leading dimension lda, lower
// triangle read) in place: L on and below the diagonal, zeros above.
// Positions past nb act as an identity block and are never stored. A pivot
// that is not positive (or NaN) sets *info to offset + k + 1 if *info is
// still 0; the factorisation then carries on and its result is meaningless,
// as LAPACK's potrf leaves it.
__global__ void __launch_bounds__(CH_THREADS)
    cholesky_diag_kernel(float* __restrict__ a, int64_t lda, int nb, int64_t offset,
                         float* __restrict__ inv, int32_t* __restrict__ info) {
  __shared__ __attribute__((aligned(16))) float s[CH_NB * CH_LD];
  __shared__ __attribute__((aligned(16))) float s_inv[CH_T * CH_WLD];
  // Loads at clamped positions, none behind a branch, so that they are in
  // flight together.
#pragma unroll 32
  for (int e = 0; e < CH_NB * CH_NB / CH_THREADS; ++e) {
    const int i = threadIdx.x + e * CH_THREADS, r = i / CH_NB, c = i % CH_NB;
    const float v = a[(int64_t)(r < nb ? r : nb - 1) * lda + (c < nb ? c : nb - 1)];
    s[r * CH_LD + c] = (r < nb && c <= r) ? v : (r == c ? 1.0f : 0.0f);
  }
  __syncthreads();
  factor_block(s, s_inv, (nb + CH_T - 1) / CH_T, inv, offset, info);
  store_block(s, a, lda, nb);
}

// Rows [r0, n) of panel column j0 (128 wide): X = A L11^-T against the
// factored block L11 at (j0, j0), 16 columns at a time: X_c = (A_c -
// sum_{k < c} X_k L_ck^T) W_c^T, W_c the inverse of L11's diagonal tile c.
// One wave per 16 rows, its 16 x 128 strip in registers; X_c passes through
// a wave-private LDS tile to become an operand.
__global__ void __launch_bounds__(CH_THREADS)
    cholesky_solve_kernel(float* __restrict__ a, int64_t n, int64_t j0,
                          const float* __restrict__ inv) {
  __shared__ __attribute__((aligned(16))) float s_l[CH_NB * CH_LD];
  __shared__ __attribute__((aligned(16))) float s_x[CH_THREADS / 64][CH_T * CH_WLD];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const float* l11 = a + j0 * n + j0;
#pragma unroll 32
  for (int e = 0; e < CH_NB * CH_NB / CH_THREADS; ++e) {
    const int i = threadIdx.x + e * CH_THREADS;
    s_l[i / CH_NB * CH_LD + i % CH_NB] = l11[i / CH_NB * n + i % CH_NB];
  }
  const int64_t row0 = j0 + CH_NB + (int64_t)blockIdx.x * 64 + wave * 16 + 4 * g;
  float* strip = a + row0 * n + j0 + r;
  f32x4 acc[CH_TILES];
#pragma unroll
  for (int c = 0; c < CH_TILES; ++c) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      // Rows past the matrix read its last row; they are never stored, and
      // rows of a strip do not mix.
      const int64_t past = row0 + q < n ? 0 : row0 + q - (n - 1);
      acc[c][q] = strip[(q - past) * n + 16 * c];
    }
  }
  f32x4 w[CH_TILES];
#pragma unroll
  for (int c = 0; c < CH_TILES; ++c) {
#pragma unroll
    for (int t = 0; t < 4; ++t) w[c][t] = inv[c * CH_T * CH_T + r * CH_T + 4 * g + t];
  }
  __syncthreads();
  float* x = s_x[wave];
  auto operand = [&](f32x4 d) {
    // D layout to A layout through the wave's own tile.
#pragma unroll
    for (int q = 0; q < 4; ++q) x[(4 * g + q) * CH_WLD + r] = d[q];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const f32x4 v = *reinterpret_cast<const f32x4*>(x + r * CH_WLD + 4 * g);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    return v;
  };
#pragma unroll
  for (int c = 0; c < CH_TILES; ++c) {
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    acc[c] = mfma16(operand(acc[c]), w[c], zero);
    if (c + 1 < CH_TILES) {
      const f32x4 xa = -operand(acc[c]);
#pragma unroll
      for (int d = c + 1; d < CH_TILES; ++d)
        acc[d] = mfma16(
            xa, *reinterpret_cast<const f32x4*>(s_l + (16 * d + r) * CH_LD + 16 * c + 4 * g),
            acc[d]);
    }
  }
#pragma unroll
  for (int c = 0; c < CH_TILES; ++c) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (row0 + q < n) strip[q * n + 16 * c] = acc[c][q];
    }
  }
}

// Workgroup 0's share of a trailing update: the next diagonal block (order
// nb at `a`, leading dimension lda) loses X X^T, X its rows of the finished
// panel at x, and is factored. This is the chain that a factorisation waits
// for, so it is not the general tile below: X is one operand, staged once
// and whole, only the 36 tiles on and below the diagonal are computed, nine a
// wave (tile rows w and 7 - w), and its waves go first on their CU. Through
// the general tile the launch took 40 us, 34 so.
__device__ __forceinline__ void factor_next(float* s, float* s_inv, const float* __restrict__ x,
                                            float* __restrict__ a, int64_t lda, int nb,
                                            float* __restrict__ inv, int64_t offset,
                                            int32_t* info) {
  __builtin_amdgcn_s_setprio(3);
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int r = lane & 15, g = lane >> 4;
  auto clamp = [&](int i) { return i < nb ? i : nb - 1; };
#pragma unroll 32
  for (int e = 0; e < CH_NB * CH_NB / CH_THREADS; ++e) {
    const int i = threadIdx.x + e * CH_THREADS;
    s[i / CH_NB * CH_LD + i % CH_NB] = x[clamp(i / CH_NB) * lda + i % CH_NB];
  }
  constexpr int OWN = CH_TILES + 1;
  auto tile_row = [&](int u) { return u <= w ? w : CH_TILES - 1 - w; };
  auto tile_col = [&](int u) { return u <= w ? u : u - w - 1; };
  f32x4 acc[OWN] = {}, old[OWN];
#pragma unroll
  for (int u = 0; u < OWN; ++u) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
      old[u][t] = a[clamp(16 * tile_row(u) + 4 * g + t) * lda + clamp(16 * tile_col(u) + r)];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < CH_NB; k += 16) {
    auto fragment = [&](int tile) {
      return *reinterpret_cast<const f32x4*>(s + (16 * tile + r) * CH_LD + k + 4 * g);
    };
    const f32x4 lo = fragment(w), hi = fragment(CH_TILES - 1 - w);
#pragma unroll
    for (int u = 0; u < OWN; ++u)
      acc[u] = mfma16(u <= w ? lo : hi, fragment(tile_col(u)), acc[u]);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < OWN; ++u) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int row = 16 * tile_row(u) + 4 * g + t, col = 16 * tile_col(u) + r;
      // Above the diagonal nothing is read.
      s[row * CH_LD + col] =
          row < nb && col < nb ? old[u][t] - acc[u][t] : (row == col ? 1.0f : 0.0f);
    }
  }
  __syncthreads();
  factor_block(s, s_inv, (nb + CH_T - 1) / CH_T, inv, offset, info);
  store_block(s, a, lda, nb);
}

// Tile (i, j) of the trailing lower triangle (128 x 128 tiles from row and
// column j0 + 128): C -= X_i X_j^T, X the panel at column j0. Workgroup 0 is
// the next diagonal block, which it factors (rows past n act as an identity
// there).
__global__ void __launch_bounds__(CH_THREADS)
    cholesky_update_kernel(float* __restrict__ a, int64_t n, int64_t j0, float* __restrict__ inv,
                           int32_t* __restrict__ info) {
  __shared__ __attribute__((aligned(16))) float s[CH_NB * CH_LD];
  __shared__ __attribute__((aligned(16))) float s_inv[CH_T * CH_WLD];
  static_assert(2 * CH_NB * CH_KLD <= CH_NB * CH_LD, "both operands fit where the block goes");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  // Tile b of the triangle in row order: i (i + 1) / 2 + j.
  const int b = blockIdx.x;
  const int64_t base = j0 + CH_NB;
  if (b == 0) {
    factor_next(s, s_inv, a + base * n + j0, a + base * n + base, n,
                n - base < CH_NB ? (int)(n - base) : CH_NB, inv, base, info);
    return;
  }
  int ti = (int)((sqrtf(8.0f * (float)b + 1.0f) - 1.0f) * 0.5f);
  while ((ti + 1) * (ti + 2) / 2 <= b) ++ti;
  while (ti * (ti + 1) / 2 > b) --ti;
  const int tj = b - ti * (ti + 1) / 2;
  const int64_t i0 = base + (int64_t)ti * CH_NB, c0 = base + (int64_t)tj * CH_NB;

  float* s_a = s;
  float* s_b = s + CH_NB * CH_KLD;
  const int wi = (wave >> 1) * 64, wj = (wave & 1) * 64;
  // The wave's 64 x 64 part of C. The products are summed by themselves and
  // subtracted once: summed onto C, 128 roundings at C's size made the
  // factor's error six times as large. Loads are at clamped positions, none
  // behind a branch: rows and columns past the matrix are never stored.
  auto clamp = [&](int64_t x) { return x < n ? x : n - 1; };
  f32x4 acc[4][4] = {}, old[4][4];
  auto fetch_c = [&]() {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const float* c = a + clamp(i0 + wi + 16 * p + 4 * g + t) * n;
#pragma unroll
        for (int q = 0; q < 4; ++q) old[p][q][t] = c[clamp(c0 + wj + 16 * q + r)];
      }
    }
  };
  // Panel columns k0 .. k0 + 31 of both row ranges, one chunk in registers
  // ahead of the one in LDS.
  constexpr int PER = CH_NB * CH_KC / CH_THREADS;
  float na[PER], nb_[PER];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int x = threadIdx.x + e * CH_THREADS;
      const int64_t col = j0 + k0 + x % CH_KC;
      na[e] = a[clamp(i0 + x / CH_KC) * n + col];
      nb_[e] = a[clamp(c0 + x / CH_KC) * n + col];
    }
  };
  fetch(0);
#pragma unroll
  for (int k0 = 0; k0 < CH_NB; k0 += CH_KC) {
    __syncthreads();
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int x = threadIdx.x + e * CH_THREADS;
      s_a[x / CH_KC * CH_KLD + x % CH_KC] = na[e];
      s_b[x / CH_KC * CH_KLD + x % CH_KC] = nb_[e];
    }
    __syncthreads();
    if (k0 + CH_KC < CH_NB) {
      fetch(k0 + CH_KC);
    } else {
      fetch_c();
    }
#pragma unroll
    for (int kk = 0; kk < CH_KC; kk += 16) {
      f32x4 fa[4], fb[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        fa[t] = *reinterpret_cast<const f32x4*>(s_a + (wi + 16 * t + r) * CH_KLD + kk + 4 * g);
        fb[t] = *reinterpret_cast<const f32x4*>(s_b + (wj + 16 * t + r) * CH_KLD + kk + 4 * g);
      }
#pragma unroll
      for (int p = 0; p < 4; ++p) {
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[p][q] = mfma16(fa[p], fb[q], acc[p][q]);
      }
    }
  }
#pragma unroll
  for (int p = 0; p < 4; ++p) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int64_t row = i0 + wi + 16 * p + 4 * g + t, col = c0 + wj + 16 * q + r;
        if (row < n && col <= row) a[row * n + col] = old[p][q][t] - acc[p][q][t];
      }
    }
  }
}

// Block column c of a block LDL factor (ldlq.py:130-142 of the reference):
// the factor's 16 columns times the inverse of their diagonal tile, an
// identity in the tile's own rows, zeros above. One wave per block column
// and 64 rows; HBM-bound (the lower triangle in, the matrix out).
__global__ void __launch_bounds__(256)
    block_fold_kernel(const float* __restrict__ l, const float* __restrict__ inv,
                      float* __restrict__ out, int64_t n) {
  const int lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  const int64_t c = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (16 * c >= n) return;
  f32x4 w;
#pragma unroll
  for (int t = 0; t < 4; ++t) w[t] = inv[c * CH_T * CH_T + (4 * g + t) * CH_T + r];
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int64_t tile = (int64_t)blockIdx.y * 4 + p;
    if (16 * tile >= n) return;
    f32x4 d;
    if (tile > c) {
      f32x4 x;
      const float* src = l + (16 * tile + r) * n + 16 * c + 4 * g;
#pragma unroll
      for (int t = 0; t < 4; ++t) x[t] = src[t];
      const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
      d = mfma16(x, w, zero);
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t) d[t] = tile == c && r == 4 * g + t ? 1.0f : 0.0f;
    }
    float* dst = out + (16 * tile + 4 * g) * n + 16 * c + r;
#pragma unroll
    for (int t = 0; t < 4; ++t) dst[t * n] = d[t];
  }
}

// ------------------------------------------------------------ LDLQ steps

// Index of the block holding batch tile `tile` (blocks sorted by tile0).
__device__ __forceinline__ int ldlq_block_of(const exl3_ldlq_block* __restrict__ blocks,
                                             int nblocks, int64_t tile) {
  int b = 0;
  while (b + 1 < nblocks && blocks[b + 1].tile0 <= tile) ++b;
  return b;
}

__global__ void __launch_bounds__(256)
    ldlq_gather_kernel(const exl3_ldlq_block* __restrict__ blocks, int nblocks,
                       float* __restrict__ x) {
  const int64_t tile = blockIdx.x;
  const exl3_ldlq_block blk = blocks[ldlq_block_of(blocks, nblocks, tile)];
  const int64_t t = tile - blk.tile0;
  // A table that does not cover this tile writes nothing (the host checks
  // the table before it is uploaded).
  if (t < 0 || t >= blk.n / 16) return;
  const int p = threadIdx.x;
  const int e = exl3::tc_perm(p);
  const int64_t off = (int64_t)(e >> 4) * blk.n + t * 16 + (e & 15);
  const float* w = reinterpret_cast<const float*>(blk.w);
  const float* comp = reinterpret_cast<const float*>(blk.comp);
  x[tile * 256 + p] = w[off] + comp[off];
}

__global__ void __launch_bounds__(256)
    ldlq_scatter_kernel(const exl3_ldlq_block* __restrict__ blocks, int nblocks,
                        const float* __restrict__ recon, const int16_t* __restrict__ idx) {
  const int64_t tile = blockIdx.x;
  const exl3_ldlq_block blk = blocks[ldlq_block_of(blocks, nblocks, tile)];
  const int64_t t = tile - blk.tile0;
  if (t < 0 || t >= blk.n / 16) return;
  const int p = threadIdx.x;
  const int e = exl3::tc_perm(p);
  const int64_t off = (int64_t)(e >> 4) * blk.n + t * 16 + (e & 15);
  const float v = recon[tile * 256 + p];
  const float w = reinterpret_cast<const float*>(blk.w)[off];
  reinterpret_cast<float*>(blk.wq)[off] = v;
  reinterpret_cast<float*>(blk.err)[off] = w - v;
  reinterpret_cast<int16_t*>(blk.states)[t * 256 + p] = idx[tile * 256 + p];
}

// Checks the shape and launches the Hadamard kernel variant for (side,
// divisor present, sums of squares wanted).
int launch_hadamard(const float* in, float* out, int64_t rows, int64_t cols, int side,
                    const float* div, float* sumsq, void* stream, const char* what) {
  if (!in || !out) return set_error("%s: NULL buffer", what);
  if (rows <= 0 || cols <= 0) return set_error("%s: empty matrix (%lld x %lld)", what,
                                                (long long)rows, (long long)cols);
  if (side != 0 && side != 1) return set_error("%s: side must be 0 or 1, got %d", what, side);
  if (side == 0 && rows % HAD_N)
    return set_error("%s: rows (%lld) must be divisible by 128", what, (long long)rows);
  if (side == 1 && cols % HAD_N)
    return set_error("%s: columns (%lld) must be divisible by 128", what, (long long)cols);
  hipStream_t st = as_stream(stream);
  if (side == 1) {
    const int64_t seg_per_row = cols / HAD_N;
    const int64_t segments = rows * seg_per_row;
    const int64_t want = (segments + HAD_RIGHT_WAVES - 1) / HAD_RIGHT_WAVES;
    // Grid-stride beyond 65536 workgroups (several segments per wave).
    const int64_t blocks = want < 65536 ? want : 65536;
    const dim3 grid((unsigned)blocks), block(64 * HAD_RIGHT_WAVES);
    if (div && sumsq)
      hipLaunchKernelGGL((had128_right_kernel<true, true>), grid, block, 0, st, in, out, segments,
                         seg_per_row, div, sumsq);
    else if (div)
      hipLaunchKernelGGL((had128_right_kernel<true, false>), grid, block, 0, st, in, out,
                         segments, seg_per_row, div, sumsq);
    else if (sumsq)
      hipLaunchKernelGGL((had128_right_kernel<false, true>), grid, block, 0, st, in, out,
                         segments, seg_per_row, div, sumsq);
    else
      hipLaunchKernelGGL((had128_right_kernel<false, false>), grid, block, 0, st, in, out,
                         segments, seg_per_row, div, sumsq);
  } else {
    const int64_t gx = (cols + 255) / 256, gy = rows / HAD_N;
    if (gx > INT32_MAX || gy > 65535) return set_error("%s: matrix too large", what);
    const dim3 grid((unsigned)gx, (unsigned)gy), block(256);
    if (div)
      hipLaunchKernelGGL((had128_left_kernel<true>), grid, block, 0, st, in, out, cols, div);
    else
      hipLaunchKernelGGL((had128_left_kernel<false>), grid, block, 0, st, in, out, cols, div);
  }
  return check_launch(what);
}

// Whole 128 x 128 blocks of a matrix and the grid that takes one each.
int block_grid(int64_t rows, int64_t cols, dim3* grid, const char* what) {
  if (rows <= 0 || cols <= 0 || rows % HAD_N || cols % HAD_N)
    return set_error("%s: both dimensions must be positive multiples of 128, got %lld x %lld",
                     what, (long long)rows, (long long)cols);
  if (cols / HAD_N > INT32_MAX || rows / HAD_N > 65535)
    return set_error("%s: matrix too large", what);
  *grid = dim3((unsigned)(cols / HAD_N), (unsigned)(rows / HAD_N));
  return 0;
}

// Checks and grid of the unrotate kernel: whole 128 x 128 blocks, out and sv
// read and written as float2.
int unrotate_grid(const void* in, const float* su, const float* sv, const float* out,
                  int64_t rows, int64_t cols, dim3* grid, const char* what) {
  if (!in || !su || !sv || !out) return set_error("%s: NULL buffer", what);
  if (((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(sv)) & 7) != 0)
    return set_error("%s: out and sv must be 8-byte aligned", what);
  return block_grid(rows, cols, grid, what);
}

}  // namespace

// ------------------------------------------------------------------- C-ABI

extern "C" {

int exl3_hadamard128(const float* in, float* out, int64_t rows, int64_t cols, int side,
                     void* stream) {
  return launch_hadamard(in, out, rows, cols, side, nullptr, nullptr, stream, "hadamard128");
}

int exl3_hadamard128_scaled(const float* in, float* out, int64_t rows, int64_t cols, int side,
                            const float* divisor, float* slice_sumsq, void* stream) {
  if (slice_sumsq && side != 1)
    return set_error("hadamard128_scaled: slice sums of squares need side = 1");
  return launch_hadamard(in, out, rows, cols, side, divisor, slice_sumsq, stream,
                         "hadamard128_scaled");
}

int exl3_row_energy(const float* in, const float* sv, float* sums, int64_t rows, int64_t cols,
                    void* stream) {
  if (!in || !sv || !sums) return set_error("row_energy: NULL buffer");
  dim3 grid;
  if (block_grid(rows, cols, &grid, "row_energy")) return 1;
  static_assert(HAD_N % EN_ROWS == 0, "whole workgroups to a row block");
  unsigned b;
  if (exl3::grid_1d(rows * (cols / HAD_N), EN_ROWS, &b, "row_energy")) return 1;
  hipLaunchKernelGGL(row_energy_kernel, dim3(b), dim3(64 * EN_WAVES), 0, as_stream(stream), in,
                     cols, sv, sums);
  return check_launch("row_energy");
}

int exl3_rotate(const float* in, const float* sv, const float* su, float* out, int64_t rows,
                int64_t cols, void* stream) {
  if (!in || !sv || !su || !out) return set_error("rotate: NULL buffer");
  dim3 grid;
  if (block_grid(rows, cols, &grid, "rotate")) return 1;
  hipLaunchKernelGGL(rotate_kernel, grid, dim3(RO_THREADS), 0, as_stream(stream), in, sv, su, out,
                     cols);
  return check_launch("rotate");
}

int exl3_unrotate(const float* in, const float* su, const float* sv, float* out, int64_t rows,
                  int64_t cols, void* stream) {
  dim3 grid;
  if (unrotate_grid(in, su, sv, out, rows, cols, &grid, "unrotate")) return 1;
  hipLaunchKernelGGL((unrotate_kernel<false, 0>), grid, dim3(UN_THREADS), 0, as_stream(stream), in,
                     nullptr, 0, su, sv, out, cols);
  return check_launch("unrotate");
}

int exl3_decode_weight(const uint16_t* packed, const float* su, const float* sv, float* out,
                       int64_t rows, int64_t cols, int K, int cb, void* stream) {
  if (K < 1 || K > 8) return set_error("decode_weight: K must be in 1..8, got %d", K);
  if (cb < 0 || cb > 2) return set_error("decode_weight: cb must be 0, 1, or 2, got %d", cb);
  dim3 grid;
  if (unrotate_grid(packed, su, sv, out, rows, cols, &grid, "decode_weight")) return 1;
  if (reinterpret_cast<uintptr_t>(packed) & 3)
    return set_error("decode_weight: the words must be 4-byte aligned");
  const uint32_t* words = reinterpret_cast<const uint32_t*>(packed);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(UN_THREADS), 0, as_stream(stream), nullptr, words, K, su,
                       sv, out, cols);
  };
  switch (cb) {
    case 0: launch(unrotate_kernel<true, 0>); break;
    case 1: launch(unrotate_kernel<true, 1>); break;
    default: launch(unrotate_kernel<true, 2>); break;
  }
  return check_launch("decode_weight");
}

int exl3_block_rms_from_slices(const float* slice_sumsq, float* out, int64_t outputs, int64_t n,
                               int64_t slices, void* stream) {
  if (!slice_sumsq || !out) return set_error("block_rms_from_slices: NULL buffer");
  if (outputs <= 0 || n <= 0 || slices <= 0)
    return set_error("block_rms_from_slices: empty shape (%lld outputs, n %lld, %lld slices)",
                     (long long)outputs, (long long)n, (long long)slices);
  unsigned b;
  if (exl3::grid_1d(outputs, ROWS_RED, &b, "block_rms_from_slices")) return 1;
  hipLaunchKernelGGL(block_rms_reduce_rows_kernel, dim3(b), dim3(256), 0, as_stream(stream),
                     slice_sumsq, out, outputs, n, slices, nullptr, nullptr);
  return check_launch("block_rms_from_slices");
}

int exl3_input_scales(const float* slice_sumsq, const float* su, float* scales, float* su_out,
                      int64_t rows, int64_t n, int64_t slices, void* stream) {
  if (!slice_sumsq || !su || !scales || !su_out) return set_error("input_scales: NULL buffer");
  if (rows <= 0 || n <= 0 || slices <= 0)
    return set_error("input_scales: empty shape (%lld rows, n %lld, %lld slices)",
                     (long long)rows, (long long)n, (long long)slices);
  unsigned b;
  if (exl3::grid_1d(rows, ROWS_RED, &b, "input_scales")) return 1;
  hipLaunchKernelGGL(block_rms_reduce_rows_kernel, dim3(b), dim3(256), 0, as_stream(stream),
                     slice_sumsq, scales, rows, n, slices, su, su_out);
  return check_launch("input_scales");
}

int exl3_output_scales(const float* x, int64_t rows, int64_t cols, const float* diag,
                       int64_t diag_stride, int64_t diag_len, const float* sv, int decide,
                       int forced, float* workspace, int64_t workspace_elems, float* scales,
                       float* divisor, float* sv_out, double* flags, void* stream) {
  if (!x || !sv || !workspace || !scales || !divisor || !sv_out || !flags)
    return set_error("output_scales: NULL buffer");
  if (rows <= 0 || cols <= 0) return set_error("output_scales: empty matrix");
  if (decide < 0 || decide > 2) return set_error("output_scales: decide must be 0, 1 or 2");
  if (diag && (diag_len <= 0 || diag_len > INT32_MAX || diag_stride < 1))
    return set_error("output_scales: bad diagonal (%lld values, stride %lld)",
                     (long long)diag_len, (long long)diag_stride);
  const int64_t ns = (rows + COL_SLICE - 1) / COL_SLICE;
  if (workspace_elems < cols * ns)
    return set_error("output_scales: workspace holds %lld floats, %lld needed",
                     (long long)workspace_elems, (long long)(cols * ns));
  unsigned b1, b2;
  if (exl3::grid_1d(cols * ns, SC_THREADS, &b1, "output_scales")) return 1;
  if (exl3::grid_1d(cols, 64, &b2, "output_scales")) return 1;
  hipStream_t sm = as_stream(stream);
  hipLaunchKernelGGL(column_slices_kernel, dim3(b1 + (diag ? 1 : 0)), dim3(SC_THREADS), 0, sm, x,
                     workspace, cols, rows, ns, diag, diag_stride, diag_len, flags);
  hipLaunchKernelGGL(block_rms_reduce_columns_kernel, dim3(b2), dim3(64), 0, sm, workspace, scales,
                     cols, rows, ns);
  hipLaunchKernelGGL(output_scales_kernel, dim3(1), dim3(SC_THREADS), 0, sm, scales, cols, sv,
                     decide, forced, divisor, sv_out, flags);
  return check_launch("output_scales");
}

int64_t exl3_block_rms_workspace(int64_t rows, int64_t cols, int dim, int blocksize) {
  if (rows <= 0 || cols <= 0 || (dim != 0 && dim != 1) || blocksize <= 0) return -1;
  const int64_t outputs = dim == 0 ? cols : rows, n = dim == 0 ? rows : cols;
  return outputs * ((n + blocksize - 1) / blocksize);
}

int exl3_block_rms(const float* x, float* out, int64_t rows, int64_t cols, int dim, int blocksize,
                   float* workspace, int64_t workspace_elems, void* stream) {
  if (!x || !out || !workspace) return set_error("block_rms: NULL buffer");
  if (rows <= 0 || cols <= 0) return set_error("block_rms: empty matrix");
  if (dim != 0 && dim != 1) return set_error("block_rms: dim must be 0 or 1, got %d", dim);
  if (blocksize <= 0) return set_error("block_rms: blocksize must be positive, got %d", blocksize);
  const int64_t need = exl3_block_rms_workspace(rows, cols, dim, blocksize);
  if (workspace_elems < need)
    return set_error("block_rms: workspace holds %lld floats, %lld needed",
                     (long long)workspace_elems, (long long)need);
  const int64_t outputs = dim == 0 ? cols : rows;
  const int64_t n = dim == 0 ? rows : cols;
  const int64_t so = dim == 0 ? 1 : cols, st = dim == 0 ? cols : 1;
  const int64_t ns = (n + blocksize - 1) / blocksize;
  unsigned b1, b2;
  if (exl3::grid_1d(outputs * ns, 256, &b1, "block_rms")) return 1;
  if (exl3::grid_1d(outputs, 64, &b2, "block_rms")) return 1;
  static_assert(ROWS_RED == 64, "both reductions take 64 outputs to a workgroup");
  hipStream_t sm = as_stream(stream);
  hipLaunchKernelGGL(block_rms_slices_kernel, dim3(b1), dim3(256), 0, sm, x, workspace, outputs, n,
                     so, st, blocksize, ns, dim);
  if (check_launch("block_rms")) return 1;
  if (dim == 0)
    hipLaunchKernelGGL(block_rms_reduce_columns_kernel, dim3(b2), dim3(64), 0, sm, workspace, out,
                       outputs, n, ns);
  else
    hipLaunchKernelGGL(block_rms_reduce_rows_kernel, dim3(b2), dim3(256), 0, sm, workspace, out,
                       outputs, n, ns, nullptr, nullptr);
  return check_launch("block_rms");
}

int exl3_cholesky_diag_block(float* a, int64_t lda, int nb, int64_t offset, int32_t* info,
                             void* stream) {
  if (!a || !info) return set_error("cholesky_diag_block: NULL buffer");
  if (nb < 1 || nb > CH_NB)
    return set_error("cholesky_diag_block: block order must be in 1..%d, got %d", CH_NB, nb);
  if (lda < nb) return set_error("cholesky_diag_block: lda (%lld) < block order (%d)",
                                 (long long)lda, nb);
  if (offset < 0) return set_error("cholesky_diag_block: negative offset");
  hipLaunchKernelGGL(cholesky_diag_kernel, dim3(1), dim3(CH_THREADS), 0, as_stream(stream), a, lda,
                     nb, offset, nullptr, info);
  return check_launch("cholesky_diag_block");
}

int exl3_cholesky(float* a, int64_t n, float* inverses, int32_t* info, void* stream) {
  if (!a || !inverses || !info) return set_error("cholesky: NULL buffer");
  // The tiles of a trailing triangle are counted in 32 bits.
  if (n < 1 || n > (int64_t)CH_NB * 46000)
    return set_error("cholesky: bad order %lld", (long long)n);
  hipStream_t st = as_stream(stream);
  const int first = n < CH_NB ? (int)n : CH_NB;
  hipLaunchKernelGGL(cholesky_diag_kernel, dim3(1), dim3(CH_THREADS), 0, st, a, n, first, 0,
                     inverses, info);
  for (int64_t j0 = 0; j0 + CH_NB < n; j0 += CH_NB) {
    const int64_t rows = n - j0 - CH_NB;
    const int64_t tiles = (rows + CH_NB - 1) / CH_NB;
    hipLaunchKernelGGL(cholesky_solve_kernel, dim3((unsigned)((rows + 63) / 64)),
                       dim3(CH_THREADS), 0, st, a, n, j0, inverses + j0 * CH_T);
    hipLaunchKernelGGL(cholesky_update_kernel, dim3((unsigned)(tiles * (tiles + 1) / 2)),
                       dim3(CH_THREADS), 0, st, a, n, j0, inverses + (j0 + CH_NB) * CH_T, info);
  }
  return check_launch("cholesky");
}

int64_t exl3_cholesky_inverse_elems(int64_t n) {
  return n < 1 ? -1 : (n + CH_T - 1) / CH_T * CH_T * CH_T;
}

int exl3_block_fold(const float* l, const float* inverses, float* out, int64_t n, void* stream) {
  if (!l || !inverses || !out) return set_error("block_fold: NULL buffer");
  if (n < CH_T || n % CH_T)
    return set_error("block_fold: order %lld is not a positive multiple of 16", (long long)n);
  const int64_t tiles = n / CH_T;
  if ((tiles + 3) / 4 > 65535) return set_error("block_fold: matrix too large");
  hipLaunchKernelGGL(block_fold_kernel, dim3((unsigned)((tiles + 3) / 4), (unsigned)((tiles + 3) / 4)),
                     dim3(256), 0, as_stream(stream), l, inverses, out, n);
  return check_launch("block_fold");
}

int exl3_cholesky_block_order(void) { return CH_NB; }

int exl3_ldlq_gather(const exl3_ldlq_block* blocks, int nblocks, int64_t tiles, float* x,
                     void* stream) {
  if (!blocks || !x) return set_error("ldlq_gather: NULL buffer");
  if (nblocks < 1) return set_error("ldlq_gather: no blocks");
  if (tiles < 1 || tiles > INT32_MAX) return set_error("ldlq_gather: bad tile count %lld",
                                                       (long long)tiles);
  hipLaunchKernelGGL(ldlq_gather_kernel, dim3((unsigned)tiles), dim3(256), 0, as_stream(stream),
                     blocks, nblocks, x);
  return check_launch("ldlq_gather");
}

int exl3_ldlq_scatter(const exl3_ldlq_block* blocks, int nblocks, int64_t tiles,
                      const float* recon, const int16_t* idx, void* stream) {
  if (!blocks || !recon || !idx) return set_error("ldlq_scatter: NULL buffer");
  if (nblocks < 1) return set_error("ldlq_scatter: no blocks");
  if (tiles < 1 || tiles > INT32_MAX) return set_error("ldlq_scatter: bad tile count %lld",
                                                       (long long)tiles);
  hipLaunchKernelGGL(ldlq_scatter_kernel, dim3((unsigned)tiles), dim3(256), 0, as_stream(stream),
                     blocks, nblocks, recon, idx);
  return check_launch("ldlq_scatter");
}

}  // extern "C"
