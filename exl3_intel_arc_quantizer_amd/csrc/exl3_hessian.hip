// MI355X (gfx950) kernels of the calibration Hessian H = X^T X / tokens
// (reference: exl3_quant/calibration.py:337-385) from half-precision
// activations X (tokens, d):
//
//   gram_kernel         one lower tile of X^T X per workgroup (and per share
//                       of the tokens) on the matrix cores
//   gram_reduce_kernel  the sum over the shares, where there are several
//   damp_kernel         mean of the diagonal, damping and floor
//
// X^T X is symmetric: only tiles on and below the diagonal are computed and
// each is stored twice, so a 4096-wide Hessian of 8192 tokens is 153 GFLOP
// (253 whole tiles of 192; the triangle alone is 137) instead of the 275 of a
// general product, and the division by the token count (a product with its
// reciprocal, as torch divides by a host number) rides on the store instead
// of passes of its own.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "../../include/exl3_layer.h"
#include "exl3_errors.h"

using exl3::check_launch;
using exl3::set_error;

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Tokens staged at a time and a workgroup's threads: eight waves, two by four
// over the tile.
constexpr int GR_K = 64, GR_THREADS = 512, GR_OCTS = GR_K / 8;

template <bool BF16>
__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (BF16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
}

// Tile b of the lower triangle in row order: b = i (i + 1) / 2 + j, j <= i.
__device__ __forceinline__ void lower_tile(int b, int& i, int& j) {
  i = (int)((sqrtf(8.0f * (float)b + 1.0f) - 1.0f) * 0.5f);
  while ((i + 1) * (i + 2) / 2 <= b) ++i;
  while (i * (i + 1) / 2 > b) --i;
  j = b - i * (i + 1) / 2;
}

// One TS x TS tile (rows i0.., columns j0.. of X^T X) over the token chunks
// [c0, c1) of GR_K. v_mfma_f32_16x16x32 wants eight consecutive tokens of one
// column in a lane, and X holds consecutive columns: a thread loads 8 tokens
// x 8 columns (16-byte loads, coalesced along the columns; with 8-byte loads
// an 8192 x 4096 Gram matrix took 30 us more), turns them with one v_perm
// per dword and stores eight 16-byte vectors (8 tokens of a column). Column
// 8 q + j of an operand sits at vector j (TS / 8 + 2) + q of its token octet:
// the stores of a wave are contiguous and the 16 lanes of a load phase hit 16
// different bank groups. Loads are in flight for two chunks; two LDS buffers,
// one barrier a chunk. Two waves a SIMD, so that one's staging and waits run
// beside the other's products: with one wave a SIMD (quarters of the tile,
// 32 x 32 products) a chunk of a 192 tile took 2.0 us, 1.4 here (1.0 with the
// GPU to itself), of which the products are 0.48; the rest is staging and
// LDS traffic. A library product of 8192 x 4096 bf16 activations took 262-300
// us, and clearing, adding and dividing 60 more.
//
// An accumulator takes `run` chunks at most. A float32 sum loses up to half a
// place of its total with every matrix instruction, so one accumulator over
// all tokens loses in proportion to their number: 65,536 tokens x 4096, one
// share, had a root mean square error of 1.26e-6 on the diagonal, where sums
// over 8192 tokens, added in float32, have 1.6e-7. RUNS, for shares longer
// than that: a run's sum is added to the tile's total, which its workgroup
// alone reads and writes, in the partial tiles or, where there are none, in h
// below the diagonal. That costs 7 % (8192 tokens a run: 65,536 x 4096 1337
// us without it, 1431 with it, 16,384 x 4096 307 and 321); shorter shares,
// which the loop around the runs made 1 % slower, take the kernel without it.
template <int TS, bool BF16, bool RUNS>
__global__ void __launch_bounds__(GR_THREADS, 2)
    gram_kernel(const uint16_t* __restrict__ x, int64_t ldx, int64_t tokens, int64_t d,
                float scale, float* h, float* parts, int tiles, int chunks, int share, int run) {
  constexpr int WI = TS / 32, WJ = TS / 64;          // 16 x 16 blocks of a wave
  constexpr int QP = TS / 8 + 2;                     // vectors of one column residue
  constexpr int OCT = 8 * QP;                        // vectors of one token octet
  constexpr int UNITS = GR_OCTS * TS / 8;            // 8 x 8 units of one operand
  // One unit a thread, in the first waves.
  static_assert(2 * UNITS <= GR_THREADS && 2 * UNITS % 64 == 0, "whole waves stage");
  __shared__ u32x4 s[2][2][GR_OCTS * OCT];           // buffer, operand

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool stages = wave < 2 * UNITS / 64;
  int ti, tj;
  lower_tile((int)blockIdx.x % tiles, ti, tj);
  const int split = (int)blockIdx.x / tiles;
  const int c0 = split * share, c1 = c0 + share < chunks ? c0 + share : chunks;
  const int64_t i0 = (int64_t)ti * TS, j0 = (int64_t)tj * TS;

  // The thread's unit: operand (0: rows of the tile, 1: its columns), octet
  // and column group. Columns past d read the last group: they only reach
  // results that are not stored.
  const int unit = stages ? tid : 0;
  const int op = unit / UNITS, oct = unit % UNITS / (TS / 8), q8 = unit % UNITS % (TS / 8);
  const int64_t col8 = (op ? j0 : i0) + 8 * q8;
  // Bytes from the chunk's first token.
  const uint32_t off = (uint32_t)((oct * 8 * ldx + (col8 < d ? col8 : d - 8)) * 2);
  u32x4 raw[2][8];
  // Whole chunk c: a uniform row base plus the thread's offset.
  auto fetch = [&](int c, u32x4 (&to)[8]) {
    if (!stages) return;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const char* row = reinterpret_cast<const char*>(x + ((int64_t)c * GR_K + r) * ldx);
      to[r] = *reinterpret_cast<const u32x4*>(row + off);
    }
  };
  // A chunk that the tokens end in: those past the end read the last one and
  // count as zero.
  auto fetch_end = [&](int c, u32x4 (&to)[8]) {
    if (!stages) return;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int64_t t = (int64_t)c * GR_K + 8 * oct + r;
      const int64_t back = t < tokens ? 0 : t - (tokens - 1);
      const char* row = reinterpret_cast<const char*>(x + ((int64_t)c * GR_K + r - back) * ldx);
      const u32x4 v = *reinterpret_cast<const u32x4*>(row + off);
      to[r] = back ? u32x4{0u, 0u, 0u, 0u} : v;
    }
  };
  auto stage = [&](const u32x4 (&from)[8], int buf) {
    if (!stages) return;
    u32x4* out = s[buf][op] + oct * OCT + q8;
#pragma unroll
    for (int pair = 0; pair < 4; ++pair) {
      u32x4 lo, hi;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const uint32_t a = from[2 * m][pair], b = from[2 * m + 1][pair];
        lo[m] = __builtin_amdgcn_perm(b, a, 0x05040100u);
        hi[m] = __builtin_amdgcn_perm(b, a, 0x07060302u);
      }
      out[(2 * pair) * QP] = lo;
      out[(2 * pair + 1) * QP] = hi;
    }
  };

  f32x4 acc[WI][WJ];
  const int wi = (wave >> 2) * (TS / 2), wj = (wave & 3) * (TS / 4);
  auto vector_of = [&](int col) { return (col & 7) * QP + (col >> 3); };
  // Columns 16 apart are 2 vectors apart.
  const int fa = vector_of(wi + (lane & 15)) + (lane >> 4) * OCT;
  const int fb = vector_of(wj + (lane & 15)) + (lane >> 4) * OCT;
  // The chunk in buffer `buf`; `between` (the next chunk's staging) goes
  // beside the last step's products and not earlier: it waits for loads.
  auto multiply = [&](int buf, auto between) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < GR_K / 32; ++k) {
      u32x4 a[WI], b[WJ];
#pragma unroll
      for (int v = 0; v < WI; ++v) a[v] = s[buf][0][fa + 2 * v + 4 * k * OCT];
#pragma unroll
      for (int v = 0; v < WJ; ++v) b[v] = s[buf][1][fb + 2 * v + 4 * k * OCT];
      if (k + 1 == GR_K / 32) {
        __builtin_amdgcn_sched_barrier(0);
        between();
      }
#pragma unroll
      for (int p = 0; p < WI; ++p) {
#pragma unroll
        for (int q = 0; q < WJ; ++q) acc[p][q] = mfma16<BF16>(a[p], b[q], acc[p][q]);
      }
    }
  };

  // The sum over chunks [r0, r1): the whole chunks, loads two chunks ahead of
  // the products and no branch around them (past the end they repeat the last
  // chunk), then the chunk that the tokens end in.
  auto sum_run = [&](int r0, int r1) {
#pragma unroll
    for (int p = 0; p < WI; ++p) {
#pragma unroll
      for (int q = 0; q < WJ; ++q) acc[p][q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    const int whole = (int64_t)r1 * GR_K <= tokens ? r1 : r1 - 1;
    if (r0 < whole) {
      const int last = whole - 1;
      auto at = [&](int c) { return c < last ? c : last; };
      fetch(r0, raw[0]);
      fetch(at(r0 + 1), raw[1]);
      stage(raw[0], 0);
      __syncthreads();
      int c = r0;
      for (; c + 1 < whole; c += 2) {
        fetch(at(c + 2), raw[0]);
        multiply(0, [&] { stage(raw[1], 1); });
        __syncthreads();
        fetch(at(c + 3), raw[1]);
        multiply(1, [&] { stage(raw[0], 0); });
        __syncthreads();
      }
      if (c < whole) multiply(0, [] {});
      __syncthreads();
    }
    if (whole < r1) {
      fetch_end(whole, raw[0]);
      stage(raw[0], 0);
      __syncthreads();
      multiply(0, [] {});
      if constexpr (RUNS) __syncthreads();
    }
  };

  // Lane l holds rows 4 (l / 16) + t of column l % 16 of a block in element
  // t; d is a multiple of 8, so a lane's four rows are in the matrix or past
  // it together.
  const int row0 = wi + 4 * (lane >> 4), col0 = wj + (lane & 15);
  auto inside = [&](int p, int q) { return i0 + row0 + 16 * p < d && j0 + col0 + 16 * q < d; };
  if constexpr (!RUNS) {
    sum_run(c0, c1);
  } else {
    auto with_total = [&](auto f) {
      float* total = parts ? parts + (int64_t)blockIdx.x * TS * TS : h + i0 * d + j0;
      int64_t ld = parts ? TS : d;
      // Not known to be the same in every run: the addresses of 4 WI WJ
      // elements would otherwise stay in registers through the products. (So
      // h and parts are not restrict: this is another pointer to them.)
      asm volatile("" : "+s"(total), "+s"(ld));
      float* own = total + row0 * ld + col0;
#pragma unroll
      for (int p = 0; p < WI; ++p) {
#pragma unroll
        for (int q = 0; q < WJ; ++q) {
          if (parts || inside(p, q)) f(own + 16 * p * ld + 16 * q, ld, acc[p][q]);
        }
      }
    };
    for (int r0 = c0;;) {
      const int r1 = c1 - r0 > run ? r0 + run : c1;
      sum_run(r0, r1);
      if (r0 > c0)
        with_total([](const float* total, int64_t ld, f32x4& sum) {
          f32x4 v;
#pragma unroll
          for (int t = 0; t < 4; ++t) v[t] = total[t * ld];
          sum = v + sum;
        });
      r0 = r1;
      if (r0 >= c1) break;
      with_total([](float* total, int64_t ld, const f32x4& sum) {
#pragma unroll
        for (int t = 0; t < 4; ++t) total[t * ld] = sum[t];
      });
    }
  }

  float* part = parts ? parts + (int64_t)blockIdx.x * TS * TS : nullptr;
#pragma unroll
  for (int p = 0; p < WI; ++p) {
#pragma unroll
    for (int q = 0; q < WJ; ++q) {
      const int col = col0 + 16 * q, row = row0 + 16 * p;
      if (part) {
#pragma unroll
        for (int t = 0; t < 4; ++t) part[(row + t) * TS + col] = acc[p][q][t];
      } else if (inside(p, q)) {
#pragma unroll
        for (int t = 0; t < 4; ++t) h[(i0 + row + t) * d + j0 + col] = acc[p][q][t] * scale;
        if (ti != tj) {
#pragma unroll
          for (int t = 0; t < 4; ++t) h[(j0 + col) * d + i0 + row + t] = acc[p][q][t] * scale;
        }
      }
    }
  }
}

// H from the shares' partial tiles, added in token order: one 32 x 32 block
// of a tile per workgroup, its mirror image through LDS.
__global__ void __launch_bounds__(256)
    gram_reduce_kernel(const float* __restrict__ parts, int ts, int tiles, int splits,
                       float scale, float* __restrict__ h, int64_t d) {
  __shared__ float s[32][33];
  int ti, tj;
  lower_tile((int)blockIdx.x, ti, tj);
  const int side = ts / 32, bi = (int)blockIdx.y / side, bj = (int)blockIdx.y % side;
  const int64_t i0 = (int64_t)ti * ts + 32 * bi, j0 = (int64_t)tj * ts + 32 * bj;
  const int c = threadIdx.x & 31, r0 = threadIdx.x >> 5;
#pragma unroll
  for (int r = r0; r < 32; r += 8) {
    const float* p = parts + (int64_t)blockIdx.x * ts * ts + (32 * bi + r) * ts + 32 * bj + c;
    float v = p[0];
    for (int k = 1; k < splits; ++k) v += p[(int64_t)k * tiles * ts * ts];
    v *= scale;
    s[r][c] = v;
    if (i0 + r < d && j0 + c < d) h[(i0 + r) * d + j0 + c] = v;
  }
  if (ti == tj) return;
  __syncthreads();
#pragma unroll
  for (int r = r0; r < 32; r += 8) {
    if (j0 + r < d && i0 + c < d) h[(j0 + r) * d + i0 + c] = s[c][r];
  }
}

// diag += max(1e-8, lambda * mean(diag)), then values below floor in
// magnitude become floor; the mean goes to mean_out. One workgroup.
__global__ void __launch_bounds__(1024)
    damp_kernel(float* __restrict__ h, int64_t d, int64_t ld, double lambda, float floor_value,
                float* __restrict__ mean_out) {
  __shared__ double s_red[16];
  double sum = 0.0;
#pragma unroll 8
  for (int64_t i = threadIdx.x; i < d; i += 1024) sum += (double)h[i * (ld + 1)];
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) sum += __shfl_xor(sum, m, 64);
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = sum;
  __syncthreads();
  sum = 0.0;
  for (int w = 0; w < 16; ++w) sum += s_red[w];
  const float mean = (float)(sum / (double)d);
  const double damp = lambda * (double)mean;
  // A NaN mean stays NaN only where max(1e-8, NaN) would: it does not.
  const float add = (float)(damp > 1e-8 ? damp : 1e-8);
#pragma unroll 4
  for (int64_t i = threadIdx.x; i < d; i += 1024) {
    const float v = h[i * (ld + 1)] + add;
    h[i * (ld + 1)] = fabsf(v) < floor_value ? floor_value : v;
  }
  if (threadIdx.x == 0) *mean_out = mean;
}

// How a Gram matrix is cut: tile side, shares of the tokens per tile and the
// chunks of a share.
struct GramPlan {
  int ts, tiles, splits, share, chunks;
};

// The cut with the least estimated time on `cus` compute units (one
// workgroup each): rounds of workgroups times a share's chunks times a
// chunk's cycles (measured at 1.0-1.4 us for 192 and 0.9 us for 128), plus
// writing and reading the partial tiles where the tokens are shared out.
// Measured, us a call back to back, 192 / 128 at their best share count: 500 x
// 4096 25 / 37, 8192 x 4096 164 / 297, 16384 x 5120 578 / 962, 2048 x 2048
// 31 / 34, 8192 x 1024 36 / 32, 16384 x 512 47 / 40.
//
// Partial tiles take no more memory than H itself, which a product and a sum
// by a library would take as well, or 128 MiB. The bound costs wide inputs
// alone, and those a few percent: 262,144 x 11,008 would share the tokens out
// in four, 962 MiB beside an H of 462, for an estimated 34.0 ms against 34.7.
constexpr int64_t GRAM_WORKSPACE = (int64_t)32 << 20;  // floats

GramPlan gram_plan(int64_t tokens, int64_t d, int cus) {
  GramPlan best{};
  double least = 0.0;
  const int chunks = (int)((tokens + GR_K - 1) / GR_K);
  for (int ts : {192, 128}) {
    const int64_t side = (d + ts - 1) / ts;
    const int64_t tiles = side * (side + 1) / 2;
    const double cycles = ts == 192 ? 2900.0 : 2100.0;
    for (int splits = 1; splits <= 32 && splits <= chunks; ++splits) {
      const int share = (chunks + splits - 1) / splits;
      if ((int64_t)share * (splits - 1) >= chunks) continue;  // an empty share
      if (splits > 1 && splits * tiles * ts * ts > std::max(d * d, GRAM_WORKSPACE)) break;
      const double rounds = (double)((tiles * splits + cus - 1) / cus);
      double us = rounds * (share * cycles + 6000.0) / 2400.0;
      if (splits > 1) us += 5.0 + tiles * (double)ts * ts * 4.0 * 2.0 * splits / 4.0e6;
      if (best.ts == 0 || us < least) {
        least = us;
        best = GramPlan{ts, (int)tiles, splits, share, chunks};
      }
    }
  }
  return best;
}

int current_cus() {
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
    return 256;
  return n;
}

bool gram_shape_ok(int64_t tokens, int64_t d) {
  // The tiles of the triangle and the chunks are counted in 32 bits.
  return tokens >= 1 && tokens <= ((int64_t)1 << 32) && d >= 8 && d % 8 == 0 && d <= 1 << 20;
}

}  // namespace

extern "C" {

int64_t exl3_gram_workspace(int64_t tokens, int64_t d) {
  if (!gram_shape_ok(tokens, d)) return -1;
  const GramPlan p = gram_plan(tokens, d, current_cus());
  return p.splits > 1 ? (int64_t)p.splits * p.tiles * p.ts * p.ts : 0;
}

int exl3_gram(const uint16_t* x, int bf16, int64_t tokens, int64_t ldx, int64_t d, float scale,
              float* h, float* workspace, int64_t workspace_elems, void* stream) {
  return exl3_gram_chunked(x, bf16, tokens, ldx, d, scale, 8192, h, workspace, workspace_elems,
                           stream);
}

int exl3_gram_chunked(const uint16_t* x, int bf16, int64_t tokens, int64_t ldx, int64_t d,
                      float scale, int64_t chunk_tokens, float* h, float* workspace,
                      int64_t workspace_elems, void* stream) {
  if (!x || !h) return set_error("gram: NULL buffer");
  if (!gram_shape_ok(tokens, d) || ldx < d || ldx % 8 || ldx > 1 << 24)
    return set_error("gram: bad shape (%lld tokens, d %lld, row stride %lld)", (long long)tokens,
                     (long long)d, (long long)ldx);
  if (reinterpret_cast<uintptr_t>(x) & 15) return set_error("gram: x must be 16-byte aligned");
  if (chunk_tokens < 1)
    return set_error("gram: chunk_tokens must be positive, got %lld", (long long)chunk_tokens);
  const GramPlan p = gram_plan(tokens, d, current_cus());
  const int64_t need = p.splits > 1 ? (int64_t)p.splits * p.tiles * p.ts * p.ts : 0;
  if (need && (!workspace || workspace_elems < need))
    return set_error("gram: workspace holds %lld floats, %lld needed",
                     (long long)(workspace ? workspace_elems : 0), (long long)need);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  float* parts = need ? workspace : nullptr;
  // Whole chunks of the kernel, at least one; all of them for one sum.
  const int run = chunk_tokens >= tokens
                      ? p.chunks
                      : (int)std::clamp<int64_t>(chunk_tokens / GR_K, 1, p.chunks);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(p.tiles * p.splits)), dim3(GR_THREADS), 0, st, x,
                       ldx, tokens, d, scale, h, parts, p.tiles, p.chunks, p.share, run);
  };
  auto launch_tile = [&](auto side, auto runs) {
    if (bf16) launch(gram_kernel<side(), true, runs()>);
    else launch(gram_kernel<side(), false, runs()>);
  };
  auto launch_runs = [&](auto runs) {
    if (p.ts == 192) launch_tile(std::integral_constant<int, 192>{}, runs);
    else launch_tile(std::integral_constant<int, 128>{}, runs);
  };
  if (p.share > run) launch_runs(std::true_type{});
  else launch_runs(std::false_type{});
  if (parts)
    hipLaunchKernelGGL(gram_reduce_kernel, dim3((unsigned)p.tiles, (p.ts / 32) * (p.ts / 32)),
                       dim3(256), 0, st, parts, p.ts, p.tiles, p.splits, scale, h, d);
  return check_launch("gram");
}

int exl3_damp_diagonal(float* h, int64_t d, int64_t ld, double lambda, float floor_value,
                       float* mean, void* stream) {
  if (!h || !mean) return set_error("damp_diagonal: NULL buffer");
  if (d < 1 || ld < d) return set_error("damp_diagonal: bad shape (%lld, stride %lld)",
                                        (long long)d, (long long)ld);
  hipLaunchKernelGGL(damp_kernel, dim3(1), dim3(1024), 0, reinterpret_cast<hipStream_t>(stream), h,
                     d, ld, lambda, floor_value, mean);
  return check_launch("damp_diagonal");
}

}  // extern "C"
