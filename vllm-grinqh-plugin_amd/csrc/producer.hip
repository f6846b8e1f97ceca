// Producer fusion: the operations that feed a GRINQH linear in a Llama-style
// block also emit the batch statistic the union grading needs, so the
// product does not read x once more to build it.
//
//   rmsnorm_sigma:  h = x (+ residual_in; h to residual_out), y = RNE(h * rsqrt(mean(h^2) + eps)) * w
//   silu_mul_sigma: y = RNE(silu(g)) * u for gate_up = [g | u]
//
// Both write y and, for every chunk of kSigmaChunkRows rows, the column maxima
// sigma_chunks[chunk][k] = max over the chunk's rows of |y[m][k]| (fmaxf: NaN
// ignored unless every value is NaN, as the products' own statistic does).
// The maximum over the chunks is sigma_k = max_m |y[m][k]|, the statistic of
// grinqh/kernel.py:249; the products take the chunk maxima directly.
//
// Arithmetic follows vLLM's fused_add_rms_norm and SiluAndMul kernels (the
// operations these replace in the model): the residual sum is rounded to the
// activation dtype and its fp32 square enters the variance; the normalised
// value is rounded to the dtype before the weight multiply; silu is computed
// in fp32 and rounded before the multiply by the up half.
#include <type_traits>

#include "grinqh_common.h"
#include "grinqh_launch.h"

namespace grinqh {

constexpr int kProducerCols = 512;                      // columns per piece: 8 per lane of a wave
constexpr int kProducerThreads = 64 * kSigmaChunkRows;  // one wave per row of the chunk

// Pieces of 512 columns per block.  One when the grid is small (at decode
// sizes the block's own latency is all there is); towards two blocks of 1024
// threads per CU otherwise, so that a prefill's blocks repeat the variance
// less often and overlap one piece's loads with the last one's maxima.
inline int producer_pieces(int M, int cols) {
  const int64_t per_row = (cols + kProducerCols - 1) / kProducerCols;
  const int64_t blocks = per_row * ((M + kSigmaChunkRows - 1) / kSigmaChunkRows);
  const int64_t p = blocks / (2 * kTargetBlocks);
  return (int)(p < 1 ? 1 : (p < per_row ? p : per_row));
}

// |y| of one piece: one wave's row per slot, NaN where the chunk has no row.
typedef float ProducerRows[kSigmaChunkRows][kProducerCols];

// Column maxima of the chunk (fmaxf: NaN ignored unless every value is NaN)
// for columns c0 .. c0 + kProducerCols - 1 below `cols`: each wave leaves its
// row's |y| in LDS, then one thread per column takes the maximum.  The caller
// alternates two buffers, so that one barrier per piece is enough.
__device__ __forceinline__ void store_chunk_maxima(ProducerRows& s_abs, const float (&av)[8],
                                                   float* __restrict__ sigma_chunks, int c0, int cols) {
  const int lane = threadIdx.x & 63, row = threadIdx.x >> 6;
#pragma unroll
  for (int e = 0; e < 8; e += 4)
    *reinterpret_cast<f32x4_t*>(&s_abs[row][8 * lane + e]) = f32x4_t{av[e], av[e + 1], av[e + 2], av[e + 3]};
  __syncthreads();
  const int cc = threadIdx.x;
  if (cc >= kProducerCols || c0 + cc >= cols) return;
  float v = s_abs[0][cc];
#pragma unroll
  for (int r = 1; r < kSigmaChunkRows; ++r) v = fmaxf(v, s_abs[r][cc]);
  sigma_chunks[(int64_t)blockIdx.y * cols + c0 + cc] = v;
}

// Block = kSigmaChunkRows rows x `pieces` runs of 512 columns, one wave per
// row.  Bound by latency at decode sizes (32 rows x 4096 columns are 0.5 MB), so each wave
// has all it reads in flight at once: first its own 512 columns of the row
// (and the weight), then the whole row in batches of eight 16-byte loads per
// lane for the variance, which every column block of the chunk repeats (L2
// reads only); the sum stays in the wave (butterfly), so the rows meet only for
// the column maxima.  32 rows x 4096 with the residual: 21.0 ->
// 6.6 us (256 threads, 16 of them sharing a row and walking it with one load
// in flight); 4096 rows x 8192: 138 -> 62 us (4.3 TB/s).
// BATCH: runs of 512 columns in flight for the variance.  Rows of up to 1024
// columns take 2, and of up to 512 the one run that the block's piece has loaded
// already: with 8 they summed up to 7 runs of zeros, and the 64 registers of
// those left one block per CU.  The loop is written once with and once without
// the residual.  Without it, us: 16 rows x 256 5.6 -> 3.5, 8192 x 256 11.1 ->
// 6.2, 4096 x 1024 12.6 -> 8.0, 16 x 4096 6.0 -> 5.0.
// Since every column block reads whole rows of residual_in, the sum goes to a
// separate residual_out (writing it back in place would race with those reads).
template <typename DT, int BATCH>
__global__ __launch_bounds__(kProducerThreads) void rmsnorm_sigma_kernel(
    const uint16_t* __restrict__ x, int64_t ldx, const uint16_t* __restrict__ residual,
    uint16_t* __restrict__ residual_out, const uint16_t* __restrict__ weight, float eps, uint16_t* __restrict__ y,
    float* __restrict__ sigma_chunks, int M, int K, int pieces) {
  __shared__ ProducerRows s_abs[2];
  const int lane = threadIdx.x & 63;
  const int row = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m = blockIdx.y * kSigmaChunkRows + row;
  const int c_begin = blockIdx.x * pieces * kProducerCols;
  const int c_end = min(c_begin + pieces * kProducerCols, K);
  const u32x4_t zero = u32x4_t{0u, 0u, 0u, 0u};
  const bool live = m < M;  // wave-uniform
  const uint16_t* xr = x + (int64_t)m * ldx;
  const uint16_t* rr = residual != nullptr ? residual + (int64_t)m * K : nullptr;
  u32x4_t a = zero, r = zero, wv = zero;
  auto load_piece = [&](int k) {
    if (!live || k >= K) return;  // K % 8 == 0: a lane's 8 columns are all in or all out
    a = *reinterpret_cast<const u32x4_t*>(xr + k);
    wv = *reinterpret_cast<const u32x4_t*>(weight + k);
    if (rr != nullptr) r = *reinterpret_cast<const u32x4_t*>(rr + k);
  };
  load_piece(c_begin + 8 * lane);
  float rstd = 0.f, rstd_lo = 0.f;
  if (live) {
    // eight short fp32 sums per lane, joined in fp64; the root in fp64, kept
    // as the sum of two floats (h * root is then rounded once to fp32)
    float ss[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) ss[e] = 0.f;
    auto add = [&](auto with_residual, const u32x4_t& xa, const u32x4_t& ra) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          float v = to_f32<DT>((uint16_t)(xa[q] >> (16 * h)));
          if constexpr (decltype(with_residual)::value)
            v = to_f32<DT>(from_f32<DT>(v + to_f32<DT>((uint16_t)(ra[q] >> (16 * h)))));
          ss[2 * q + h] = fmaf(v, v, ss[2 * q + h]);
        }
    };
    auto add_row = [&](auto with_residual) {
      if constexpr (BATCH == 1) {
        add(with_residual, a, r);
      } else {
        for (int k0 = 8 * lane; k0 < K; k0 += 512 * BATCH) {
          u32x4_t xa[BATCH], ra[BATCH];
#pragma unroll
          for (int i = 0; i < BATCH; ++i) {
            const bool in = k0 + 512 * i < K;
            xa[i] = in ? *reinterpret_cast<const u32x4_t*>(xr + k0 + 512 * i) : zero;
            ra[i] = decltype(with_residual)::value && in ? *reinterpret_cast<const u32x4_t*>(rr + k0 + 512 * i) : zero;
          }
#pragma unroll
          for (int i = 0; i < BATCH; ++i) add(with_residual, xa[i], ra[i]);
        }
      }
    };
    if (rr != nullptr)
      add_row(std::true_type{});
    else
      add_row(std::false_type{});
#pragma unroll
    for (int e = 4; e >= 1; e >>= 1)
#pragma unroll
      for (int i = 0; i < e; ++i) ss[i] += ss[i + e];
    double sum = (double)ss[0];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) sum += __shfl_xor(sum, o, 64);
    const double root = 1.0 / sqrt(sum / (double)K + (double)eps);
    rstd = (float)root;
    rstd_lo = (float)(root - (double)rstd);
  }
  int buf = 0;
  for (int c0 = c_begin; c0 < c_end; c0 += kProducerCols, buf ^= 1) {
    const int k = c0 + 8 * lane;
    float av[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) av[e] = __int_as_float(0x7fc00000);  // NaN: no row
    if (live && k < K) {
      u32x4_t out, hsum;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        uint32_t o2 = 0, h2 = 0;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          uint16_t hb = (uint16_t)(a[q] >> (16 * h));
          if (rr != nullptr) hb = from_f32<DT>(to_f32<DT>(hb) + to_f32<DT>((uint16_t)(r[q] >> (16 * h))));
          const float v = to_f32<DT>(hb);
          float n32 = fmaf(v, rstd, v * rstd_lo);
          asm("" : "+v"(n32));  // the fp32 value is rounded to DT, as vLLM does (no v_fma_mixlo_f16)
          const uint16_t nrm = from_f32<DT>(n32);
          const uint16_t yb = from_f32<DT>(to_f32<DT>(nrm) * to_f32<DT>((uint16_t)(wv[q] >> (16 * h))));
          av[2 * q + h] = fabsf(to_f32<DT>(yb));
          o2 |= (uint32_t)yb << (16 * h);
          h2 |= (uint32_t)hb << (16 * h);
        }
        out[q] = o2;
        hsum[q] = h2;
      }
      *reinterpret_cast<u32x4_t*>(y + (int64_t)m * K + k) = out;
      if (rr != nullptr) *reinterpret_cast<u32x4_t*>(residual_out + (int64_t)m * K + k) = hsum;
    }
    if (c0 + kProducerCols < c_end) load_piece(k + kProducerCols);
    store_chunk_maxima(s_abs[buf], av, sigma_chunks, c0, K);
  }
}

// Block = kSigmaChunkRows rows x 512 columns of y [M][F], RW rows per wave;
// gate_up rows hold [g (F values) | u (F values)], ld elements apart.  Every
// load of a thread is issued before the first is used (rows past the batch
// repeat its last row and are not counted); under a test per row they were
// waited for one by one.  One row per wave where the grid leaves the GPU short
// of waves (32 rows x 14336: 5.9 -> 4.3 us), four where it does not: there
// one row per wave costs 5-8 % (2048 rows x 28672: 83 against 77 us), as its
// blocks of 16 waves meet at the barrier.
template <typename DT, int RW>
__global__ __launch_bounds__(64 * kSigmaChunkRows / RW) void silu_mul_sigma_kernel(
    const uint16_t* __restrict__ gu, int64_t ld, uint16_t* __restrict__ y, float* __restrict__ sigma_chunks, int M,
    int F) {
  constexpr int R = kSigmaChunkRows, NW = R / RW;
  __shared__ float s_max[NW][kProducerCols];
  const int tid = threadIdx.x;
  const int r0 = blockIdx.y * R;
  const int k = blockIdx.x * kProducerCols + 8 * (tid & 63);
  const int rb = tid >> 6;
  float mx[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) mx[e] = __int_as_float(0x7fc00000);  // NaN: no row seen yet
  if (k < F) {
    u32x4_t g[RW], u[RW];
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      const uint16_t* row = gu + (int64_t)min(r0 + rb + NW * i, M - 1) * ld + k;
      g[i] = *reinterpret_cast<const u32x4_t*>(row);
      u[i] = *reinterpret_cast<const u32x4_t*>(row + F);
    }
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      const int m = r0 + rb + NW * i;
      if (m >= M) break;
      u32x4_t out;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        uint32_t o2 = 0;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const float gv = to_f32<DT>((uint16_t)(g[i][q] >> (16 * h)));
          const uint16_t act = from_f32<DT>(gv / (1.f + expf(-gv)));
          const uint16_t yb = from_f32<DT>(to_f32<DT>(act) * to_f32<DT>((uint16_t)(u[i][q] >> (16 * h))));
          mx[2 * q + h] = fmaxf(mx[2 * q + h], fabsf(to_f32<DT>(yb)));
          o2 |= (uint32_t)yb << (16 * h);
        }
        out[q] = o2;
      }
      *reinterpret_cast<u32x4_t*>(y + (int64_t)m * F + k) = out;
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) s_max[rb][8 * (tid & 63) + e] = mx[e];
  __syncthreads();
  for (int cc = tid; cc < kProducerCols; cc += 64 * NW) {
    const int kk = blockIdx.x * kProducerCols + cc;
    if (kk >= F) break;
    float v = s_max[0][cc];
#pragma unroll
    for (int w = 1; w < NW; ++w) v = fmaxf(v, s_max[w][cc]);
    sigma_chunks[(int64_t)blockIdx.y * F + kk] = v;
  }
}

int launch_rmsnorm_sigma(const uint16_t* x, int64_t ldx, const uint16_t* residual, uint16_t* residual_out,
                         const uint16_t* weight, float eps, uint16_t* y, float* sigma_chunks, int M, int K, int dtype,
                         hipStream_t st) {
  const int pieces = producer_pieces(M, K);
  const dim3 grid((K + pieces * kProducerCols - 1) / (pieces * kProducerCols),
                  (M + kSigmaChunkRows - 1) / kSigmaChunkRows);
  auto choose = [K](auto one, auto two, auto eight) {
    return K <= kProducerCols ? one : (K <= 2 * kProducerCols ? two : eight);
  };
  auto kernel = choose(rmsnorm_sigma_kernel<F16, 1>, rmsnorm_sigma_kernel<F16, 2>, rmsnorm_sigma_kernel<F16, 8>);
  if (dtype == GRINQH_DTYPE_BF16)
    kernel = choose(rmsnorm_sigma_kernel<BF16, 1>, rmsnorm_sigma_kernel<BF16, 2>, rmsnorm_sigma_kernel<BF16, 8>);
  hipLaunchKernelGGL(kernel, grid, dim3(kProducerThreads), 0, st, x, ldx, residual, residual_out, weight, eps, y,
                     sigma_chunks, M, K, pieces);
  return hipGetLastError() == hipSuccess ? GRINQH_OK : GRINQH_ERR_HIP;
}

int launch_silu_mul_sigma(const uint16_t* gu, int64_t ld, uint16_t* y, float* sigma_chunks, int M, int F, int dtype,
                          hipStream_t st) {
  const dim3 grid((F + kProducerCols - 1) / kProducerCols, (M + kSigmaChunkRows - 1) / kSigmaChunkRows);
  const bool few = (int64_t)grid.x * grid.y <= 2 * kTargetBlocks;  // at most two blocks of 16 waves per CU
  const dim3 block(64 * kSigmaChunkRows / (few ? 1 : 4));
  if (dtype == GRINQH_DTYPE_BF16) {
    auto kernel = few ? silu_mul_sigma_kernel<BF16, 1> : silu_mul_sigma_kernel<BF16, 4>;
    hipLaunchKernelGGL(kernel, grid, block, 0, st, gu, ld, y, sigma_chunks, M, F);
  } else {
    auto kernel = few ? silu_mul_sigma_kernel<F16, 1> : silu_mul_sigma_kernel<F16, 4>;
    hipLaunchKernelGGL(kernel, grid, block, 0, st, gu, ld, y, sigma_chunks, M, F);
  }
  return hipGetLastError() == hipSuccess ? GRINQH_OK : GRINQH_ERR_HIP;
}

}  // namespace grinqh
