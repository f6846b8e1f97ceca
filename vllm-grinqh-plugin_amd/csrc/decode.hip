// Decode-regime GRINQH product (M <= 64 per launch): graded or dense
// y = x * W_eff on v_mfma_f32_16x16x32_{f16,bf16}, HBM-bound.
//
// Replaces the reference's Triton GEMVs grinqh_gemv_uint32_packed
// (grinqh/kernel.py:39-167, one row) and grinqh_gemv_uint32_packed_batch_union
// (:170-360, batch union), and the dense branch of grinqh_gemm_or_gemv for
// small batches (:663-680, semantics of :561-587).
//
// Work decomposition
//   block   = (column block, K range), one-dimensional grid renumbered per XCD
//   column block: 16 or 32 plane-word columns (CG groups of 16): 256 or 512
//             logical columns (16 column tiles r, columns r*NW + w0 + c)
//   K range = `tiles_per_split` 32-row tiles (split-K)
//   waves   = 8 (two per SIMD): CG column groups x JG groups of output dwords
//             j x KW K sub-ranges; the CG * JG waves of a sub-range share its
//             tiles
//
// What bounds it: at small shapes the launch, the prologue and the split-K
// completion (about 10 us in all); in the loop no single unit: the phases of a
// tile (wait for its words, read them from LDS, unpack, multiply) follow one
// another with two waves per SIMD.  Counters, gate_up: graded 47 rows 41 us,
// VALU busy 39 % per SIMD, MFMA 14 %, waves waiting for memory or a dependency
// 34 % and to issue 25 % of their time; dense 16 rows 28 us, 30 %, 5 %, 41 %,
// 17 %, where the plane traffic (4.3 TB/s) is near what a copy reaches (5.1).
//
// The plane words come through LDS by direct buffer-to-LDS loads because of the
// traffic: with every wave loading its own tiles into registers, the two waves
// that share a tile requested it twice, and a stream of the same requests
// without arithmetic reached 2.1 TB/s (gate_up, one MI355X); each tile requested
// once through 16-byte LDS loads reaches 3.4 TB/s with 16 word columns per
// block, 4.6 with 32, 5.4 with 64 (longer runs of each plane line per block).
// The registers this frees took bf16 above 16 rows from four waves per block to
// eight.  Measured, product with its reduction: gate_up 16 rows dense 59.6 ->
// 36.2 us, 64 rows 66.9 -> 58.8, in bf16 104.5 -> 56; Llama-3-70B gate_up 16
// rows 178 -> 128.  Up to 16 rows, where a tile or its K range is small, waves
// load their own words all the same (plan_decode).
//
// Phase 1 (whole block): reduce the batch statistic of the block's rows from x
// (unless given), grade every row (sigma = max_m |x|: zone bits, midpoint
// bias), load the scales into LDS.
//
// Phase 2 (per wave): each wave of a K sub-range loads a share of the tiles'
// plane words and x straight into LDS, one or two tiles ahead; a (row, plane)
// the grading does not need has an offset past the buffer end, which leaves
// zeros without a memory access.  A handshake through LDS flags per tile says
// that all shares have arrived; then lane (c = lane & 15, q = lane >> 4) reads
// the 8 x Z words of its 8 rows (or has loaded them itself, two tiles ahead).
// Code bytes are rebuilt branch-free:
// G_z = rot(D_z, 2z), H_j = field merge of the G_z, V_j = rot(H_j, -2j); then
// turned into the MFMA B operand in one of two ways:
//   - code bytes (5-16 rows, and bf16): fp16 B = u as the subnormal u*2^-24
//     (one v_perm per register), bf16 B = u; the offset 128 and the midpoint
//     bias beta are removed by one extra MFMA per tile whose B operand is the
//     per-row value beta*2^sh - 128 (a "correction column" shared by all 16
//     columns), and per scale group y += s[g][n] * 2^-sh * (C[m][n] + Cv[m])
//     in fp32, as grinqh/kernel.py:148-158 applies scales;
//   - the scaled weight (17-64 rows in fp16): B = RNE(w_eff * s) in fp16,
//     accumulated straight into y (no per-group sums, no correction column).
//
// Split-K partials are reduced deterministically: the K sub-ranges of a block
// through LDS in fixed order; the K ranges of the grid either by the range
// that finishes last (small reductions: in range order) or by a second kernel
// (in strided lane sums joined by a fixed butterfly), both in fp32 before the
// output cast and bias, in an order that does not depend on timing.
#include <type_traits>

#include "grinqh_common.h"
#include "grinqh_launch.h"
#include "splitk_complete.h"

namespace grinqh {

// 17-64 rows in fp16 ("scaled" path) multiply the scaled weight RNE(w * s),
// built in registers as the prefill builds it in LDS, and accumulate the
// output directly: no per-group partial sums, no correction column, no group
// epilogue.  The registers this frees let a wave cover two output dwords of all
// 64 rows (128 sums per lane); in bf16 a wave covers two dwords of 32 rows or
// one of 64.  The weight is rounded once to fp16, as in the reference's dense
// path (grinqh/kernel.py:586).
template <typename DT, int MT>
constexpr bool decode_scaled() { return MT >= 2 && DT::id == F16::id; }

constexpr int kDecodeWaves = 8;
// K rows a block can hold (scales, grades)
constexpr int decode_rows_per_block(int cg) { return cg == 2 ? 1024 : 2048; }
// groups of output dwords among a block's waves (4 / this dwords per wave)
template <typename DT, int MT>
constexpr int decode_dword_groups() { return !decode_scaled<DT, MT>() && MT == 4 ? 4 : 2; }

// CG: groups of 16 word columns per block.  GB: words per lane and load into
// LDS: 4 (plane rows 16-byte aligned) or 1; or 0, up to 16 rows: each wave loads
// the words of its own tiles into registers, and x is staged whole (plan_decode
// says where)
template <typename DT, int MT, int Z, bool DENSE, int GB, int CG>
__global__ __launch_bounds__(64 * kDecodeWaves, 1) void decode_kernel(DecodeParams p) {
  constexpr bool SC = decode_scaled<DT, MT>();
  constexpr int NWV = kDecodeWaves;
  constexpr int NT = 64 * NWV;         // threads per block
  constexpr int WB = 16 * CG;          // plane-word columns per block
  constexpr int JG = decode_dword_groups<DT, MT>();
  constexpr int NJ = 4 / JG;           // output dwords j per wave
  constexpr int SG = CG * JG;          // waves per K sub-range
  constexpr int KW = NWV / SG;         // K sub-ranges per block
  constexpr bool DIRECT = GB == 0;
  static_assert(!DIRECT || (MT == 1 && CG == 1), "x is staged for 16 rows");
  constexpr int SH = 8 - 2 * Z;
  constexpr int RMAX = decode_rows_per_block(CG);
  static_assert(RMAX / 8 <= NT, "one statistic chunk per thread");
  constexpr int SC_GROUPS = RMAX / 32 + 1;  // scale groups a K range can touch (group size >= 32)
  constexpr int SPT = CG == 2 ? 3 : 2;      // 16-byte scale chunks a thread keeps in flight

  // Plane words and x of each K sub-range's tiles come into LDS by direct
  // buffer-to-LDS loads, PF tiles ahead, each wave of the sub-range loading a
  // share, in PF + 1 slots (one per tile of the unrolled loop) that are
  // separate LDS arrays, so that the compiler's wait for one slot's loads does
  // not also wait for the others'.  A plane slot holds, per sub-range,
  // [row in octet e][zone z][octet q][word column]: lane (c, q) reads its 8 x Z
  // words at one offset plus constants, without bank conflicts (with 32 word
  // columns the two halves are swapped for odd q).
  constexpr int PF = (MT == 4 && SC ? 1 : 2);
  constexpr int GL = DIRECT ? 1 : GB;                // words per lane and load
  constexpr int TILE = 32 * Z * WB * 4;              // bytes of one sub-range's tile
  constexpr int IPT = TILE / (64 * GL * 4);          // loads per tile
  constexpr int IPW = (IPT + SG - 1) / SG;           // at most per wave
  constexpr int XPW = (MT + SG - 1) / SG;            // x fragments per wave, at most
  constexpr int RED_SLOT = NJ * 4 * 64 * 16;         // one wave's sums of an m-tile
  constexpr int RED_SLOTS = (KW - 1) * SG;
  constexpr int RED_ARRAYS = PF + 1;
  constexpr int RED_PER = (RED_SLOTS + RED_ARRAYS - 1) / RED_ARRAYS;
  constexpr int PL_BYTES = DIRECT ? 16 : KW * TILE > RED_PER * RED_SLOT ? KW * TILE : RED_PER * RED_SLOT;
  constexpr int XR_BYTES = DIRECT ? 16 : KW * MT * 1024;
  // DIRECT: x of the whole K range, fragments of 1 KiB per tile (lane l's 16
  // bytes at byte 16 l), and, graded, each (row, plane)'s byte offset, bit 31 set
  // where the row does not need it
  constexpr int ZS = Z == 3 ? 4 : Z;
  constexpr int XS_BYTES = DIRECT ? RMAX / 32 * 1024 : 16;
  static_assert(!DIRECT || RED_SLOTS * RED_SLOT <= XS_BYTES, "the reduction reuses the staged x");
  __shared__ __align__(16) unsigned char s_xs[XS_BYTES];
  __shared__ __align__(16) uint32_t s_off[DIRECT && !DENSE ? RMAX * ZS : 4];
  constexpr int SIG_BYTES = MT > 1 && !DENSE ? NT * 8 * 4 : 0;  // at most NT / U slices of U chunks of 8 rows
  __shared__ __align__(16) unsigned char s_pl0[PL_BYTES > SIG_BYTES ? PL_BYTES : SIG_BYTES];
  __shared__ __align__(16) unsigned char s_pl1[PL_BYTES];
  __shared__ __align__(16) unsigned char s_pl2[PF == 2 ? PL_BYTES : 16];
  __shared__ __align__(16) unsigned char s_xr0[XR_BYTES];
  __shared__ __align__(16) unsigned char s_xr1[XR_BYTES];
  __shared__ __align__(16) unsigned char s_xr2[PF == 2 ? XR_BYTES : 16];
  __shared__ __align__(16) uint16_t s_bv[DENSE ? 8 : RMAX];  // row -> correction-column value, or -c_row
  __shared__ __align__(16) uint8_t s_zb[DENSE ? 16 : RMAX];  // row -> zone bits (low half) and their complement
  __shared__ __align__(16) uint16_t s_scale[SC_GROUPS * 16 * WB];  // (group, tile, column) scales
  __shared__ uint32_t s_smax;  // graded scaled path: largest |scale| (fp16 bits) above the overflow limit
  __shared__ int s_flag[NWV];  // the last tile whose share wave w has in LDS
  __shared__ int s_late;       // a wave gave up waiting for a share
  // graded, 17-64 rows, no statistic given: max |x[m][k]| per slice of the batch rows (an
  // entry that is NaN in every row gives 0; every output of such a batch is NaN)
  float* s_sig = reinterpret_cast<float*>(s_pl0);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform
  const int jg = wave % JG, cg = (wave / JG) % CG, kw = wave / SG;
  const int sw = wave % SG;  // this wave among those of its K sub-range
  if (lane == 0) s_flag[wave] = -(1 << 30);  // read by the others only after the next barrier
  if (tid == 0) s_late = DIRECT ? 0 : p.expired;          // written by others only after the next barrier
  const int c = lane & 15, q = lane >> 4;
  // logical block = (column block, K range), column blocks fastest, ranges of
  // consecutive logical blocks per XCD (adjacent column blocks share lines)
  const int col_blocks = (p.NW + WB - 1) / WB;
  const int lb = xcd_chunked(blockIdx.x, gridDim.x);
  const int w0 = (lb % col_blocks) * WB;
  const int split = lb / col_blocks;
  const int ntiles_total = p.K >> 5;
  const int tile0 = split * p.tiles_per_split;
  const int tile1 = min(tile0 + p.tiles_per_split, ntiles_total);
  const int nt = tile1 - tile0;
  const int R = nt * 32;
  const int row0 = tile0 * 32;
  const int g_first = row0 / p.gs;
  const int n_groups = (row0 + R - 1) / p.gs - g_first + 1;

  // Graded scaled path: RNE(w * s) overflows fp16 where |w| * |s| > 65504
  // (|w| <= 2^(2Z-1)), which the reference's fp32 products do not.  A block
  // whose scales reach past kScaleLimit multiplies them by 2^-e in LDS and its
  // sums by 2^e (both exact, except for scales that become subnormal).
  constexpr bool GUARD = SC && !DENSE;
  constexpr uint32_t kScaleLimit = 0x7BFFu - ((uint32_t)(2 * Z - 1) << 10);  // 65504 / 2^(2Z-1), fp16 bits
  uint32_t smax = 0;  // largest |scale| bits this thread staged
  if (GUARD && threadIdx.x == 0) s_smax = 0;
  const bool own_sigma = !DENSE && p.sigma == nullptr;  // block-uniform
  // (more than 16 rows) batch rows are dealt to this many threads per K chunk,
  // two or more rows each: fewer slices to take the maximum of
  const int sig_slices = min(NT / (R >> 3), (p.M + 1) >> 1);

  // Grading a row: zone bits, correction-column value and zone-0 flip.  Rows
  // with zone 0 active are consumed in offset binary (zone 0's digits flipped,
  // u = int8(U & mask) + 128, and the column value removes the 128); other rows
  // have bit 7 clear and need no flip:
  //   w_eff * 2^sh = u + beta * 2^sh - (zone 0 active ? 128 : 0).
  // A row with no active zone therefore contributes exact zeros.  Dense, every
  // row has the same constants.
  auto row_value = [&](uint32_t bits, int beta) -> uint16_t {
    if constexpr (SC)  // -c_row of the scaled weight (u >> sh) - c_row, an exact fp16 integer
      return f32_to_f16_bits(-(float)(1024 + ((bits & 1u) ? (128 >> SH) : 0) - beta));
    else
      return BOperand<DT>::correction(beta * (1 << SH) - ((bits & 1u) ? 128 : 0));
  };
  auto grade_row = [&](int rr, float s) {
    const uint32_t bits = zone_bits<Z>(s, p.thr.t);
    s_bv[rr] = row_value(bits, midpoint_bias<Z>(bits));
    s_zb[rr] = (uint8_t)(bits | ((bits ^ 15u) << 4));
    if constexpr (DIRECT) {
      const uint32_t row_off = (uint32_t)(row0 + rr) * (uint32_t)(Z * p.NW) * 4u;
#pragma unroll
      for (int z = 0; z < Z; ++z)
        s_off[rr * ZS + z] = ((bits >> z) & 1u) ? row_off + (uint32_t)(z * p.NW) * 4u : 0x80000000u;
    }
  };

  // ---- phase 1a: reduce the block's statistic from x (and stage x for direct
  // loads) and load the scales.
  // The scales are stored to LDS only once the first tiles' loads are issued,
  // so their memory round trip overlaps those loads; they are loaded after
  // every x load, so that waiting for x does not wait for them.  Out-of-range
  // buffer offsets read 0: nothing past the end of x or the scale array is
  // touched.
  const bool vec_scales = (p.NW % 8) == 0 && (reinterpret_cast<uintptr_t>(p.scale) & 15u) == 0;
  u32x4_t sv[SPT];
  {
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(p.x), (short)0, (int)((uint64_t)p.M * p.ldx * 2u), 0x00020000);
    const uint32_t sbytes = (uint32_t)((uint64_t)((p.K + p.gs - 1) / p.gs) * p.N * 2u);
    const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(p.scale), (short)0, (int)sbytes, 0x00020000);
    // the block's statistic above 16 rows: thread t takes K chunk u0 = t % U (8
    // rows of K) for batch rows t / U, t / U + S, ... (U = R / 8 <= NT chunks, S
    // slices), 8 loads at a time, and leaves its maxima in LDS; whoever grades a
    // row takes the maximum over the slices
    if (MT > 1 && own_sigma) {
      const int U = R >> 3, S = sig_slices;
      const int u0 = tid % U, sl = tid / U;
      if (sl < S) {
        float mx[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) mx[e] = 0.f;
        for (int m0 = sl; m0 < p.M; m0 += 8 * S) {
          u32x4_t v[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const int m = m0 + i * S;
            const uint32_t off = m < p.M ? (uint32_t)(((int64_t)m * p.ldx + row0 + 8 * u0) * 2) : 0x80000000u;
            v[i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(xr, (int)off, 0, 0));
          }
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            if (i == 2 && m0 - sl + 2 * S >= p.M) break;  // block-uniform: no rows in the rest
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              mx[2 * e] = fmaxf(mx[2 * e], fabsf(to_f32<DT>((uint16_t)(v[i][e] & 0xFFFFu))));
              mx[2 * e + 1] = fmaxf(mx[2 * e + 1], fabsf(to_f32<DT>((uint16_t)(v[i][e] >> 16))));
            }
          }
        }
        f32x4_t* dst = reinterpret_cast<f32x4_t*>(&s_sig[sl * R + 8 * u0]);
        dst[0] = f32x4_t{mx[0], mx[1], mx[2], mx[3]};
        dst[1] = f32x4_t{mx[4], mx[5], mx[6], mx[7]};
      }
    }
    if constexpr (DIRECT) {
      for (int t = wave; t < nt; t += NWV) {  // rows past the batch read 0
        const uint32_t off = c < p.M ? (uint32_t)(((int64_t)c * p.ldx + row0 + t * 32 + 8 * q) * 2) : 0x80000000u;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            xr, (__attribute__((address_space(3))) void*)(s_xs + t * 1024), 16, (int)off, 0, 0, 0);
      }
      asm volatile("" ::: "memory");  // no load below moves above these: the wait for x counts on it
    }
    auto load_scales = [&]() {
#pragma unroll
      for (int k = 0; k < SPT; ++k) {
        const int h = tid + NT * k;  // (group, tile, half) chunk
        const int gl = h / (32 * CG), r = (h / (2 * CG)) & 15, hf = h % (2 * CG);
        const uint32_t off =
            (gl < n_groups && vec_scales)
                ? (uint32_t)(((int64_t)(g_first + gl) * p.N + (int64_t)r * p.NW + w0 + 8 * hf) * 2)
                : 0x80000000u;
        sv[k] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(sr, (int)off, 0, 0));
      }
    };
    // Up to 16 rows a thread takes two K rows (four where the K range is longer
    // than two per thread) of every batch row, all loads in flight, and grades
    // them from registers: no slices in LDS, one barrier less (batch rows past
    // the last repeat it; a NaN is ignored as fmaxf does).  16 rows graded:
    // down 19.3 -> 18.3 us, gate_up 30.2 -> 29.5.
    auto grade_rows = [&](auto words) {
      constexpr int W = decltype(words)::value;  // two K rows each
      const int rr = 2 * W * tid;
      uint32_t v[16][W];
#pragma unroll
      for (int m = 0; m < 16; ++m) {
        const int row_off = (int)(((int64_t)min(m, p.M - 1) * p.ldx + row0) * 2);
        const int off = rr < R ? rr * 2 : (int)0x80000000u;
        if constexpr (W == 1) {
          v[m][0] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(xr, off, row_off, 0);
        } else {
          const u32x2_t u = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(xr, off, row_off, 0));
          v[m][0] = u[0];
          v[m][1] = u[1];
        }
      }
      load_scales();
      if (rr >= R) return;
#pragma unroll
      for (int w = 0; w < W; ++w) {
        float lo = 0.f, hi = 0.f;
#pragma unroll
        for (int m = 0; m < 16; ++m) {
          lo = fmaxf(lo, fabsf(to_f32<DT>((uint16_t)(v[m][w] & 0xFFFFu))));
          hi = fmaxf(hi, fabsf(to_f32<DT>((uint16_t)(v[m][w] >> 16))));
        }
        grade_row(rr + 2 * w, lo);
        grade_row(rr + 2 * w + 1, hi);
      }
    };
    if (MT > 1 || !own_sigma)
      load_scales();
    else if (R <= 2 * NT)
      grade_rows(std::integral_constant<int, 1>{});
    else
      grade_rows(std::integral_constant<int, 2>{});
    // more groups than those (short groups, long K ranges): stored at once
    for (int h = tid + NT * SPT; h < n_groups * 32 * CG && vec_scales; h += NT) {
      const int gl = h / (32 * CG), r = (h / (2 * CG)) & 15, hf = h % (2 * CG);
      const uint32_t off = (uint32_t)(((int64_t)(g_first + gl) * p.N + (int64_t)r * p.NW + w0 + 8 * hf) * 2);
      const u32x4_t v = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(sr, (int)off, 0, 0));
      *reinterpret_cast<u32x4_t*>(&s_scale[8 * h]) = v;
      if constexpr (GUARD) {
#pragma unroll
        for (int e = 0; e < 4; ++e) smax = max(smax, max(v[e] & 0x7FFFu, (v[e] >> 16) & 0x7FFFu));
      }
    }
  }
  // (direct: this wave's part of x has arrived, the scales loaded after it may
  // still be on their way)
  if constexpr (DIRECT) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(SPT) : "memory");
  __syncthreads();

  // ---- phase 1b (graded, unless graded above): grade each row.
  if constexpr (!DENSE) {
    // (the loop that reads the caller's statistic from global memory is kept
    // apart, so that the other has no global load and the scale loads stay in
    // flight through it)
    if (MT == 1 && own_sigma) {
      // graded from registers
    } else if (own_sigma) {  // this block's share of the batch statistic
      for (int rr = tid; rr < R; rr += NT) {
        float sg = 0.f;
        for (int s0 = 0; s0 < sig_slices; s0 += 8) {  // eight reads in flight (past the last slice: that one again)
          float v[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) v[i] = s_sig[min(s0 + i, sig_slices - 1) * R + rr];
#pragma unroll
          for (int i = 0; i < 8; ++i) sg = fmaxf(sg, v[i]);
        }
        grade_row(rr, sg);
      }
    } else {  // the batch statistic given by the caller
      for (int rr = tid; rr < R; rr += NT) grade_row(rr, precomputed_sigma(p, row0 + rr));
    }
    if (MT > 1 || !own_sigma) __syncthreads();
  }

  int up_exp = 0;  // the block's sums are scaled by 2^up_exp at the end
  // The scales into LDS, once the first tiles' plane loads are issued; then
  // the overflow guard.  The barriers carry no memory fence, so they do not
  // wait for those plane loads, only for the LDS accesses before them.  One
  // staging path per block: where the 16-byte loads were not issued their
  // zero fill would race with the element-wise stores to the same LDS words.
  auto stage_scales = [&]() {
    if (vec_scales) {
#pragma unroll
      for (int k = 0; k < SPT; ++k) {
        const int h = tid + NT * k;
        if (h < SC_GROUPS * 32 * CG) *reinterpret_cast<u32x4_t*>(&s_scale[8 * h]) = sv[k];
        if constexpr (GUARD) {
#pragma unroll
          for (int e = 0; e < 4; ++e) smax = max(smax, max(sv[k][e] & 0x7FFFu, (sv[k][e] >> 16) & 0x7FFFu));
        }
      }
    } else {  // column count not a multiple of 128: element-wise scale staging
      for (int idx = tid; idx < n_groups * 16 * WB; idx += NT) {
        const int gl = idx / (16 * WB), col = idx % (16 * WB);
        const int wcol = min(w0 + col % WB, p.NW - 1);
        s_scale[idx] = p.scale[(int64_t)(g_first + gl) * p.N + (int64_t)(col / WB) * p.NW + wcol];
        if constexpr (GUARD) smax = max(smax, (uint32_t)s_scale[idx] & 0x7FFFu);
      }
    }
    if (GUARD && smax > kScaleLimit) atomicMax(&s_smax, smax);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if constexpr (GUARD) {
      const uint32_t hm = s_smax;  // block-uniform
      if (hm > kScaleLimit) {
        up_exp = (int)(hm >> 10) - (int)(kScaleLimit >> 10);
        const float down = __builtin_ldexpf(1.f, -up_exp);
        for (int idx = tid; idx < n_groups * 16 * WB; idx += NT)
          s_scale[idx] = from_f32<DT>(to_f32<DT>(s_scale[idx]) * down);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      }
    }
  };

  // ---- phase 2: main loop over this wave's tiles
  f32x4_t Y[MT][NJ][4];
  f32x4_t C[MT][NJ][4];
  f32x4_t Cv[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int jj = 0; jj < NJ; ++jj)
#pragma unroll
      for (int b = 0; b < 4; ++b) Y[mt][jj][b] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // Lanes past the last word column read the last valid column instead (their
  // outputs are never stored), so every address below is in bounds.
  const int cw = 16 * cg + c;  // this lane's word column in the block
  const bool col_ok = (w0 + cw) < p.NW;
  const int wc = col_ok ? (w0 + cw) : (p.NW - 1);
  const float post = BOperand<DT>::kUnit / (float)(1 << SH);
  const int t_begin = (nt * kw) / KW, t_end = (nt * (kw + 1)) / KW;
  const int tiles_per_group = p.gs >> 5;

  // Loads past the end of the sub-range go through a descriptor of size 0, and
  // a (row, plane) the grading does not need has offset bit 31 set, past the
  // buffer end: both leave zeros in LDS without a memory access.  Lanes past
  // the last word column load the last valid words (never stored).
  const uint32_t row_bytes = (uint32_t)(Z * p.NW) * 4u;
  const int plane_bytes = (int)((uint64_t)p.K * row_bytes);
  const __amdgpu_buffer_rsrc_t prsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(p.planes), (short)0, plane_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t prsrc_none =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(p.planes), (short)0, 0, 0x00020000);
  const __amdgpu_buffer_rsrc_t xsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(p.x), (short)0, (int)((uint64_t)p.M * p.ldx * 2u), 0x00020000);
  const __amdgpu_buffer_rsrc_t xsrc_none =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.x), (short)0, 0, 0x00020000);
  // This lane's byte offset in a tile for each of the wave's loads, and the
  // bit of its (row, zone) in the lane's zone word: a lane's loads are all of
  // one octet lq and, where they divide evenly among the waves, of RW of its
  // rows, so one LDS read per tile covers them (a byte read and four VALU per
  // load before: gate_up at N = 28688, 8 rows graded, 37.7 -> 35.9 us).
  // Uneven (6 bits, four waves), the last waves' shares end early: the loads
  // they do not issue repeat the tile's last piece here.
  constexpr int G = WB / GL;  // pieces per (e, z, q)
  constexpr bool EVEN = IPT % SG == 0;
  constexpr int RW = EVEN ? 8 / SG : 8;
  constexpr int LAST = IPT * 64 - 1;
  static_assert(64 % (4 * G) == 0 && LAST / (4 * G) / Z < 8, "loads of one octet, rows of a tile");
  typedef typename std::conditional<RW == 2, uint16_t, typename std::conditional<RW == 4, uint32_t, uint64_t>::type>::type
      zones_t;
  const int lq = lane % (4 * G) / G, e0 = EVEN ? RW * sw : 0;
  uint32_t loff[IPW];
  int lbit[IPW];
#pragma unroll
  for (int i = 0; i < IPW; ++i) {
    const int pair = EVEN ? i * (64 / (4 * G)) + lane / (4 * G) : min((sw * IPW + i) * 64 + lane, LAST) / (4 * G);
    const int word = ((lane % G) * GL) ^ (CG == 2 ? 16 * (lq & 1) : 0);
    const int row = 8 * lq + e0 + pair / Z, z = pair % Z;
    loff[i] = (uint32_t)row * row_bytes + (uint32_t)(z * p.NW + min(w0 + word, p.NW - GL)) * 4u;
    lbit[i] = 8 * (pair / Z) + 4 + z;
  }
  typedef __attribute__((address_space(3))) void* lds_t;
  // this wave's share of tile t (plane words, and x[16*mt + c][rows 8q .. 8q+7]
  // as fragments of 1 KiB, lane l's 16 bytes at byte 16 l; rows m >= M read 0)
  auto read_zones = [&](int t) -> zones_t {  // (graded) of the rows this lane loads
    if constexpr (DENSE) return 0;
    const int tt = t < t_end ? t : t_begin;
    return *reinterpret_cast<const zones_t*>(&s_zb[tt * 32 + 8 * lq + e0]);
  };
  auto load_tile = [&](int t, unsigned char* pl, unsigned char* xr, zones_t zn) {
    const bool live = t < t_end;
    const int tt = live ? t : t_begin;
    const __amdgpu_buffer_rsrc_t xs = live ? xsrc : xsrc_none;
#pragma unroll
    for (int h = 0; h < XPW; ++h) {
      const int mt = XPW * sw + h;
      if (MT % SG != 0 && mt >= MT) break;  // wave-uniform
      const int m = 16 * mt + c;
      const uint32_t off = m < p.M ? (uint32_t)(((int64_t)m * p.ldx + row0 + tt * 32 + 8 * q) * 2) : 0x80000000u;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xs, (lds_t)(xr + (kw * MT + mt) * 1024), 16, (int)off, 0, 0, 0);
    }
    const __amdgpu_buffer_rsrc_t rs = live ? prsrc : prsrc_none;
    const int sbase = (int)((uint32_t)(row0 + tt * 32) * row_bytes);
#pragma unroll
    for (int i = 0; i < IPW; ++i) {
      const int gi = sw * IPW + i;
      if (IPT % SG != 0 && gi >= IPT) break;  // wave-uniform
      uint32_t off = loff[i];
      if constexpr (!DENSE) off |= (uint32_t)(zn >> lbit[i]) << 31;
      const lds_t dst = (lds_t)(pl + kw * TILE + gi * 64 * GL * 4);
      if constexpr (GB == 4)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, dst, 16, (int)off, sbase, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, dst, 4, (int)off, sbase, 0, 0);
    }
  };
  // DIRECT: the words of tile t that this lane multiplies (zeros past the range
  // and where the grading needs none)
  struct Tile {
    uint32_t D[8][Z];
  };
  auto load_words = [&](int t, Tile& T) {
    const bool live = t < t_end;
    const int tt = live ? t : t_begin;
    const __amdgpu_buffer_rsrc_t rs = live ? prsrc : prsrc_none;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      typedef uint32_t offs_t __attribute__((ext_vector_type(ZS)));
      offs_t o = {};
      if constexpr (!DENSE) o = *reinterpret_cast<const offs_t*>(&s_off[(tt * 32 + 8 * q + e) * ZS]);
#pragma unroll
      for (int z = 0; z < Z; ++z) {
        uint32_t off = (uint32_t)wc * 4u, base = 0;
        if constexpr (DENSE) {
          off += (uint32_t)(8 * q) * row_bytes;
          base = (uint32_t)(row0 + tt * 32 + e) * row_bytes + (uint32_t)(z * p.NW) * 4u;  // wave-uniform
        } else {
          off += o[z];
        }
        T.D[e][z] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs, (int)off, (int)base, 0);
      }
    }
  };
  // the LDS words this lane reads of a tile
  const int dpos = kw * TILE + (q * WB + ((16 * cg) ^ (CG == 2 ? 16 * (q & 1) : 0)) + c) * 4;

  // position of the current tile in its scale group and the group's index in
  // the staged scales, advanced per tile (no divisions in the loop)
  int gpos = (tile0 + t_begin) % tiles_per_group;
  int gloc = (tile0 + t_begin) / tiles_per_group - g_first;
  uint32_t s2[NJ][4];  // scaled path: (s, s) of the current group's columns
  const uint16_t dense_value = row_value((1u << Z) - 1u, 0);
  int polls = 0;  // of all this wave's waits, four at a time
  // one tile from its words and x: unpack, MFMA, group epilogue
  auto multiply = [&](int t, const u32x4_t (&A)[MT], uint32_t (&D)[8][Z]) __attribute__((always_inline)) {
    const bool first_of_group = (t == t_begin) || (gpos == 0);
    const bool last_of_group = (t + 1 == t_end) || (gpos + 1 == tiles_per_group);
    const int sb = t * 32 + 8 * q;

    // Rebuild the code bytes (offset binary) and turn them into B operands.
    u32x4_t bv;
    uint32_t xm[8];
    if constexpr (DENSE) {
      const uint32_t v = (uint32_t)dense_value * 0x00010001u;
      bv = u32x4_t{v, v, v, v};
#pragma unroll
      for (int e = 0; e < 8; ++e) xm[e] = 0xAAAAAAAAu;
    } else {
      bv = *reinterpret_cast<const u32x4_t*>(&s_bv[sb]);
      const u32x2_t zb = *reinterpret_cast<const u32x2_t*>(&s_zb[sb]);
#pragma unroll
      for (int e = 0; e < 8; ++e)  // zone 0's flip: bit 0 of the row's byte, spread
        xm[e] = (uint32_t)((int32_t)(zb[e >> 2] << (31 - 8 * (e & 3))) >> 31) & 0xAAAAAAAAu;
    }
    prepare_planes<Z>(D, xm);
    if constexpr (SC) {
      // B = RNE(w * s) with s2 = (s, s) of this lane's columns for the group
      // and bv = (-c_row, -c_row') per row pair; the output accumulates directly.
      if (first_of_group) {
        const uint16_t* srow = &s_scale[(gloc * 16 + 4 * jg * NJ) * WB + cw];
#pragma unroll
        for (int jj = 0; jj < NJ; ++jj)
#pragma unroll
          for (int b = 0; b < 4; ++b) s2[jj][b] = (uint32_t)srow[(4 * jj + b) * WB] * 0x00010001u;
      }
#pragma unroll
      for (int jj = 0; jj < NJ; ++jj) {
        uint32_t V[8];
        code_dwords<Z>(D, jg * NJ + jj, V);
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          u32x4_t B;
#pragma unroll
          for (int pp = 0; pp < 4; ++pp) B[pp] = Dequant<F16, SH>::pair(V[2 * pp], V[2 * pp + 1], b, bv[pp], s2[jj][b]);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) Y[mt][jj][b] = mfma16x16x32<DT>(A[mt], B, Y[mt][jj][b]);
        }
      }
    }
    if constexpr (!SC) {
      if (first_of_group) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          Cv[mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int jj = 0; jj < NJ; ++jj)
#pragma unroll
            for (int b = 0; b < 4; ++b) C[mt][jj][b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
      }
#pragma unroll
      for (int jj = 0; jj < NJ; ++jj) {
        uint32_t V[8];
        code_dwords<Z>(D, jg * NJ + jj, V);
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          u32x4_t B;
#pragma unroll
          for (int pp = 0; pp < 4; ++pp) B[pp] = BOperand<DT>::pair(V[2 * pp], V[2 * pp + 1], b);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) C[mt][jj][b] = mfma16x16x32<DT>(A[mt], B, C[mt][jj][b]);
        }
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) Cv[mt] = mfma16x16x32<DT>(A[mt], bv, Cv[mt]);
    }

    if (!SC && last_of_group) {  // y += s[g][n] * 2^-sh * (C + Cv), scales from LDS
      const uint16_t* srow = &s_scale[(gloc * 16 + 4 * jg * NJ) * WB + cw];
#pragma unroll
      for (int jj = 0; jj < NJ; ++jj)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const float sc = to_f32<DT>(srow[(4 * jj + b) * WB]) * post;
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int e = 0; e < 4; ++e) Y[mt][jj][b][e] = fmaf(sc, C[mt][jj][b][e] + Cv[mt][e], Y[mt][jj][b][e]);
        }
    }
    if (gpos + 1 == tiles_per_group) {
      gpos = 0;
      ++gloc;
    } else {
      ++gpos;
    }
  };
  // one tile through LDS: handshake, loads of tile t + PF, then the tile
  auto step = [&](int t, const unsigned char* pcur, const unsigned char* xcur, unsigned char* pnext,
                  unsigned char* xnext) __attribute__((always_inline)) {
    // own share of tile t: wait until at most the loads issued after it are in
    // flight (every wave's share of them, at least).  Then the handshake:
    // publish it, and wait until every other wave of the K sub-range has
    // published its share, which also means it has read the slots of earlier
    // tiles, the one the next loads overwrite among them.  Every wave
    // publishes before it waits, so every wait ends.  It is bounded all the
    // same: a wave whose waits have used up their polls goes on with whatever the
    // slot holds, all in bounds, and the block's outputs become NaN.
    const zones_t zn = read_zones(t + PF);
    constexpr int LATER = (PF - 1) * ((IPT % SG == 0 ? IPW : 0) + (MT % SG == 0 ? XPW : 0));
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LATER) : "memory");
    if (lane == 0) __hip_atomic_store(&s_flag[wave], t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
#pragma unroll
    for (int pj = 0; pj < SG; ++pj) {
      if (pj == sw) continue;
      auto waiting = [&]() {
        return __builtin_amdgcn_readfirstlane(__hip_atomic_load(&s_flag[kw * SG + pj], __ATOMIC_RELAXED,
                                                                __HIP_MEMORY_SCOPE_WORKGROUP)) < t;
      };
      while (waiting() && waiting() && waiting() && waiting() && polls < kTilePolls) ++polls;
    }
    asm volatile("" ::: "memory");
    load_tile(t + PF, pnext, xnext, zn);
    __builtin_amdgcn_sched_barrier(0);

    u32x4_t A[MT];  // x[16*mt + c][rows 8q .. 8q+7 of the tile]
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      A[mt] = *reinterpret_cast<const u32x4_t*>(xcur + (kw * MT + mt) * 1024 + lane * 16);
    uint32_t D[8][Z];
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int z = 0; z < Z; ++z)
        D[e][z] = *reinterpret_cast<const uint32_t*>(pcur + dpos + (e * Z + z) * 16 * WB);
    multiply(t, A, D);
  };

  {
    int t = t_begin;
    if constexpr (DIRECT) {
      // three tile buffers: tiles t + 1 and t + 2 are in flight while tile t is
      // unpacked
      auto own_step = [&](int t1, Tile& cur, Tile& next, bool more) __attribute__((always_inline)) {
        if (more) load_words(t1 + 2, next);
        __builtin_amdgcn_sched_barrier(0);
        const u32x4_t A[1] = {*reinterpret_cast<const u32x4_t*>(s_xs + t1 * 1024 + lane * 16)};
        multiply(t1, A, cur.D);
      };
      Tile TA, TB, TC;
      load_words(t_begin, TA);
      load_words(t_begin + 1, TB);
      stage_scales();
      for (; t + 3 <= t_end; t += 3) {
        own_step(t, TA, TC, true);
        own_step(t + 1, TB, TA, true);
        own_step(t + 2, TC, TB, true);
      }
      // at most two tiles left, already loaded into TA and TB
      if (t < t_end) own_step(t, TA, TC, false);
      if (t + 1 < t_end) own_step(t + 1, TB, TA, false);
    } else if constexpr (PF == 2) {
      load_tile(t_begin, s_pl0, s_xr0, read_zones(t_begin));
      load_tile(t_begin + 1, s_pl1, s_xr1, read_zones(t_begin + 1));
      stage_scales();
      if constexpr (MT == 1) {
        for (; t + 3 <= t_end; t += 3) {
          step(t, s_pl0, s_xr0, s_pl2, s_xr2);
          step(t + 1, s_pl1, s_xr1, s_pl0, s_xr0);
          step(t + 2, s_pl2, s_xr2, s_pl1, s_xr1);
        }
        if (t < t_end) step(t, s_pl0, s_xr0, s_pl2, s_xr2);
        if (t + 1 < t_end) step(t + 1, s_pl1, s_xr1, s_pl0, s_xr0);
      } else {  // (one copy per slot: 1-2 % faster here, 2-4 % slower at 5-16 rows)
        for (; t < t_end; t += 3) {
          step(t, s_pl0, s_xr0, s_pl2, s_xr2);
          if (t + 1 >= t_end) break;
          step(t + 1, s_pl1, s_xr1, s_pl0, s_xr0);
          if (t + 2 >= t_end) break;
          step(t + 2, s_pl2, s_xr2, s_pl1, s_xr1);
        }
      }
    } else {
      load_tile(t_begin, s_pl0, s_xr0, read_zones(t_begin));
      stage_scales();
      for (; t < t_end; t += 2) {
        step(t, s_pl0, s_xr0, s_pl1, s_xr1);
        if (t + 1 >= t_end) break;
        step(t + 1, s_pl1, s_xr1, s_pl0, s_xr0);
      }
    }
  }
  if (polls >= kTilePolls) s_late = 1;  // read after the reduction's barriers
  // the slots are reused below: none of this wave's loads may still be on its
  // way to them (loads past the range leave zeros)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  if (GUARD && up_exp > 0) {
    const float up = __builtin_ldexpf(1.f, up_exp);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int jj = 0; jj < NJ; ++jj)
#pragma unroll
        for (int b = 0; b < 4; ++b) Y[mt][jj][b] *= up;
  }

  // ---- phase 3: reduce the K sub-ranges of this block, one m-tile per round.
  // The sums of m-tile mt are added by the waves of K sub-range mt % KW (its
  // owner), in fixed order kw = 0, 1, ..., KW-1, and those waves write that
  // m-tile's outputs, so that the block's stores are spread over its waves:
  // at 64 rows each wave stores 32 values per lane instead of two waves
  // storing 128, which is more agent-scope stores than one wave keeps in
  // flight (it then waits for them to reach memory).  The other sub-ranges
  // leave their sums in the staging area, free now, one slot per wave.
  auto owns = [&](int mt) { return kw == mt % KW; };  // wave-uniform
  if (KW > 1) {
    auto red_slot = [&](int i) -> f32x4_t* {  // wave slots are spread over the plane slots (direct: in the staged x)
      if constexpr (DIRECT) return reinterpret_cast<f32x4_t*>(s_xs + i * RED_SLOT);
      unsigned char* base = i < RED_PER ? s_pl0 : (PF == 1 || i < 2 * RED_PER) ? s_pl1 : s_pl2;
      return reinterpret_cast<f32x4_t*>(base + (i % RED_PER) * RED_SLOT);
    };
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int own = mt % KW;
      __syncthreads();
      if (kw != own) {
        f32x4_t* slot = red_slot((kw < own ? kw : kw - 1) * SG + sw);
#pragma unroll
        for (int jj = 0; jj < NJ; ++jj)
#pragma unroll
          for (int b = 0; b < 4; ++b) slot[(jj * 4 + b) * 64 + lane] = Y[mt][jj][b];
      }
      __syncthreads();
      if (kw == own) {
#pragma unroll
        for (int jj = 0; jj < NJ; ++jj)
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            auto part = [&](int k2) -> f32x4_t {  // sub-range k2's sums
              if (k2 == own) return Y[mt][jj][b];
              return red_slot((k2 < own ? k2 : k2 - 1) * SG + sw)[(jj * 4 + b) * 64 + lane];
            };
            f32x4_t acc = part(0);
#pragma unroll
            for (int k2 = 1; k2 < KW; ++k2) acc += part(k2);
            Y[mt][jj][b] = acc;
          }
      }
    }
  }

  // the scaled path multiplies w_eff * s directly: graded rows with a
  // non-finite activation become NaN, as in the reference
  if constexpr (SC && !DENSE) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      if (!owns(mt)) continue;
#pragma unroll
      for (int jj = 0; jj < NJ; ++jj)
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
          for (int e = 0; e < 4; ++e) Y[mt][jj][b][e] = graded_nonfinite_to_nan(Y[mt][jj][b][e]);
    }
  }

  // A wave gave up waiting, so a tile may have been multiplied before it was
  // complete: the block's outputs (or partial sums) are overwritten by NaN.
  // Apart from the stores of the sums, whose registers a branch around them
  // would spill.
  static_assert(KW > 1, "the reduction's barriers precede this read");
  const bool late = !DIRECT && s_late != 0;  // block-uniform
  auto poison = [&]() {
    __builtin_amdgcn_s_waitcnt(0);  // the stores of the sums
#pragma unroll 1
    for (int i = 0; i < MT * NJ * 16; ++i) {
      const int mt = i / (NJ * 16), m = 16 * mt + 4 * q + (i & 3);
      const int64_t n = (int64_t)(4 * jg * NJ + (i / 4) % (4 * NJ)) * p.NW + wc;
      if (kw != mt % KW || m >= p.M || !col_ok) continue;
      if (p.splits == 1)
        p.y[(int64_t)m * p.N + n] = from_f32<DT>(__int_as_float(0x7fc00000));
      else
        store_partial(&p.partial[((int64_t)split * p.M + m) * p.N + n], __int_as_float(0x7fc00000));
    }
  };

  // ---- phase 4: output (direct, or split-K partials + last-block reduction)
  // Output (m, n) of this lane: m = 16*mt + 4*q + e, n = (4*(jg*NJ+jj)+b)*NW + w0 + c.
  auto col_of = [&](int jj, int b) -> int64_t { return (int64_t)(4 * (jg * NJ + jj) + b) * p.NW + wc; };
  if (p.splits == 1) {
    if (col_ok) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        if (!owns(mt)) continue;
#pragma unroll
        for (int jj = 0; jj < NJ; ++jj)
#pragma unroll
          for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int m = 16 * mt + 4 * q + e;
              if (m < p.M) p.y[(int64_t)m * p.N + col_of(jj, b)] = finish_output<DT>(Y[mt][jj][b][e], p.bias,
                                                                                  (int)col_of(jj, b));
            }
      }
    }
    if (late) poison();
    return;
  }

  // Split-K: this K range's partial sums go to partial[split][m][n]; the
  // range that finishes last (or the reduce kernel that follows on the
  // stream) adds the ranges in fixed order.  Agent-scope (sc1) stores: the
  // last range may read them from another XCD, and before the reduce kernel
  // they stream out during the kernel instead of being written back from L2
  // at its end.  With a slab of partial sums below 2 GiB they are raw buffer
  // stores without branches: the row part of an offset (past the slab for
  // rows m >= M and lanes past the last word column, whose stores the range
  // check drops) in the vector offset, the column tile's part in the scalar
  // offset.
  if ((int64_t)p.M * p.N * 4 < ((int64_t)1 << 31)) {
    const __amdgpu_buffer_rsrc_t prs =
        __builtin_amdgcn_make_buffer_rsrc(p.partial + (int64_t)split * p.M * p.N, (short)0,
                                          (int)((uint32_t)p.M * (uint32_t)p.N * 4u), 0x00020000);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      if (!owns(mt)) continue;
      uint32_t roff[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = 16 * mt + 4 * q + e;
        roff[e] = (m < p.M && col_ok) ? ((uint32_t)m * (uint32_t)p.N + (uint32_t)wc) * 4u : 0x80000000u;
      }
#pragma unroll
      for (int jj = 0; jj < NJ; ++jj)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const uint32_t coff = (uint32_t)(4 * (jg * NJ + jj) + b) * (uint32_t)p.NW * 4u;  // wave-uniform
#pragma unroll
          for (int e = 0; e < 4; ++e)
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(Y[mt][jj][b][e]), prs, (int)roff[e], (int)coff,
                                                  kCpolSc1);
        }
    }
  } else if (col_ok) {
    float* part = p.partial + (int64_t)split * p.M * p.N;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      if (!owns(mt)) continue;
#pragma unroll
      for (int jj = 0; jj < NJ; ++jj)
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int m = 16 * mt + 4 * q + e;
            if (m < p.M) store_partial(&part[(int64_t)m * p.N + col_of(jj, b)], Y[mt][jj][b][e]);
          }
    }
  }
  if (late) poison();
  if (p.counters != nullptr) splitk_complete<DT, 1024 * MT * CG / NT, NT>(p, lb % col_blocks, w0, WB);
}

// y[m][n] = cast(sum_{s=0..splits-1} partial[s][m][n]) (+ bias), four
// consecutive columns per chunk.  TPC lanes of one wave share a chunk: lane
// `sub` adds ranges sub, sub + TPC, ... in increasing order (all its loads in
// flight at once), then the TPC sums are combined by a fixed butterfly, so the
// result is the same on every run.
template <typename DT, int TPC>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ partial, int splits, int M,
                                                            int N, const uint16_t* __restrict__ bias,
                                                            uint16_t* __restrict__ y) {
  constexpr int BATCH = 16;
  const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t i = g / TPC;  // 4-column chunk
  const int sub = (int)(g % TPC);
  const int64_t total = (int64_t)M * N / 4;
  const bool live = i < total;
  const f32x4_t* src = reinterpret_cast<const f32x4_t*>(partial) + (live ? i : 0);
  f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int s0 = sub; s0 < splits; s0 += TPC * BATCH) {
    f32x4_t v[BATCH];
#pragma unroll
    for (int k = 0; k < BATCH; ++k) {
      const int s = s0 + k * TPC;
      v[k] = (live && s < splits) ? __builtin_nontemporal_load(src + (int64_t)s * total) : f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int k = 0; k < BATCH; ++k) acc += v[k];
  }
#pragma unroll
  for (int o = TPC / 2; o >= 1; o >>= 1)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] += __shfl_xor(acc[e], o, 64);
  if (!live || sub != 0) return;
  const int n = (int)((i * 4) % N);
  uint16_t o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = finish_output<DT>(acc[e], bias, n + e);
  *reinterpret_cast<u32x2_t*>(y + i * 4) = u32x2_t{(uint32_t)o[0] | ((uint32_t)o[1] << 16),
                                                   (uint32_t)o[2] | ((uint32_t)o[3] << 16)};
}

// sigma_k = max_m |x[m][k]| over the whole batch (NaN ignored unless all NaN,
// as fmaxf does), computed once for kernels that grade from it.  A block
// covers 32 columns; its 8 row groups take every 8th row with 8 loads in
// flight each, and the 8 partial maxima are combined through LDS.  GZ = 0
// writes sigma; GZ = Z writes each row's grade word (grade_word) instead.
template <typename DT, int GZ>
__global__ __launch_bounds__(256) void sigma_kernel(const uint16_t* __restrict__ x, int64_t ldx, int M, int K,
                                                    float* __restrict__ sigma, uint32_t* __restrict__ grades,
                                                    GradeThresholds thr) {
  constexpr int COLS = 32, GROUPS = 256 / COLS, BATCH = 8;
  __shared__ float s_part[GROUPS][COLS];
  const int kk = threadIdx.x % COLS, mg = threadIdx.x / COLS;
  const int k = blockIdx.x * COLS + kk;
  const int kc = min(k, K - 1);  // columns past the end read a valid one and are not stored
  float s = __int_as_float(0x7fc00000);  // NaN: no row seen yet
  for (int m0 = mg; m0 < M; m0 += GROUPS * BATCH) {
    uint16_t v[BATCH];
#pragma unroll
    for (int i = 0; i < BATCH; ++i) {
      const int m = min(m0 + GROUPS * i, M - 1);  // rows past the end repeat the last row
      v[i] = x[(int64_t)m * ldx + kc];
    }
#pragma unroll
    for (int i = 0; i < BATCH; ++i) s = fmaxf(s, fabsf(to_f32<DT>(v[i])));
  }
  s_part[mg][kk] = s;
  __syncthreads();
  if (mg == 0 && k < K) {
#pragma unroll
    for (int g = 1; g < GROUPS; ++g) s = fmaxf(s, s_part[g][kk]);
    if constexpr (GZ == 0)
      sigma[k] = s;
    else
      grades[k] = grade_word<DT, GZ>(s, thr.t);
  }
}

DecodePlan plan_decode(int64_t M, int64_t K, int64_t N, int max_bits, bool dense, bool wide) {
  DecodePlan pl{};
  pl.mt = M <= 16 ? 1 : (M <= 32 ? 2 : 4);
  const int64_t NW = N / 16, T = K / 32;
  const int64_t bytes_per_split = M * N * (int64_t)sizeof(float);
  int64_t splits = 1;
  auto choose = [&](int cg) {
    pl.cg = cg;
    pl.col_blocks = (int)((NW + 16 * cg - 1) / (16 * cg));
    // K sub-ranges per block; at 17-32 rows half of them, so that short K
    // ranges still fill the GPU (1024 x 2560 at 17 rows: 12.0 -> 10.6 us)
    const int kw = pl.mt == 2 ? 2 : 4 / cg;
    const int64_t tiles_max = decode_rows_per_block(cg) / 32;
    const int64_t min_splits = (T + tiles_max - 1) / tiles_max;
    // one block per CU, all blocks resident at once: the per-block set-up
    // (staging, grading) is paid once per CU rather than once per round
    const int64_t want = kTargetBlocks / pl.col_blocks > 0 ? kTargetBlocks / pl.col_blocks : 1;
    int64_t max_splits = T / (2 * kw);
    if (max_splits < 1) max_splits = 1;
    splits = want < max_splits ? want : max_splits;
    if (splits < min_splits) splits = min_splits;
    if (splits > 1 && bytes_per_split > 0) {
      int64_t cap = (int64_t)kMaxPartialBytes / bytes_per_split;
      if (cap < min_splits) cap = min_splits;
      if (splits > cap) splits = cap;
    }
  };
  // Dense batches of up to 32 rows are bound by the plane traffic, which
  // blocks of 32 word columns read in whole 128-byte lines, for twice the K
  // ranges and so twice the partial sums.  6 and 8 bits: taken where those stay
  // below 0.3 of the plane bytes (16 / 32 columns, us: 16 rows gate_up 46 / 36,
  // down 25.8 / 23.0, Llama-3-70B gate_up 147 / 126, 24 rows gate_up 49 / 42;
  // above the line qkv 16.4 / 16.9, o_proj 14.1 / 15.5).  4 bits: up to 16 rows
  // and below 0.2 (gate_up 28.7 / 26.6; down, at 0.29, 17.0 / 18.1; 24 rows
  // gate_up 30.2 / 35.1, Llama-3-70B down 55.4 / 65.8).  2 bits: never (gate_up
  // 21.2 / 24.7).  Graded batches read fewer planes and are bound by their
  // unpacking (gate_up 29.9 / 33.5).
  choose(1);
  const int64_t percent = max_bits >= 6 ? 30 : (max_bits == 4 && pl.mt == 1) ? 20 : 0;
  if (wide && dense && pl.mt <= 2 && percent > 0) {
    choose(2);
    if (splits * 16 * pl.mt * 4 * 100 > percent * K * max_bits / 8) choose(1);
  }
  if (splits < 1) splits = 1;
  int64_t tps = (T + splits - 1) / splits;
  if (tps < 1) tps = 1;
  splits = (T + tps - 1) / tps;
  if (splits < 1) splits = 1;
  pl.splits = (int)splits;
  pl.tiles_per_split = (int)tps;
  pl.workspace = splits > 1 ? (size_t)(splits * bytes_per_split) : 0;
  // Up to 16 rows, waves that load their own words (twice the requests, but no
  // handshake per tile and no LDS round trip) are faster than shared tiles
  // where a tile or a wave's share of the K range is small, and, graded, where
  // the shared tiles come by 4-byte loads.  16 rows, fp16, shared / direct us:
  //   2 bits: down 14.3 / 13.4 dense, 15.2 / 14.0 graded; 4096 x 28688 24.1 /
  //     22.5 and 25.9 / 24.3; but dense gate_up (2048 rows a block) 21.2 / 22.6
  //   graded, rows not 16-byte aligned: 2080 x 6160 13.8 / 12.6, 4096 x 28688
  //     36.1 / 33.6
  //   graded, short K ranges: o_proj (256 rows a block) 12.1 / 11.7, qkv (416)
  //     13.7 / 13.7, in 4 bits 12.7 / 12.4; longer ones down (896) 18.4 / 19.1,
  //     gate_up (2048) 29.2 / 35.5
  pl.load_words = wide ? 4 : 1;
  const bool direct = dense ? max_bits == 2 && (!wide || tps <= 32) : max_bits == 2 || !wide || tps <= 16;
  if (pl.mt == 1 && direct) pl.load_words = 0;
  return pl;
}

template <typename DT, int MT, int Z>
static void launch_decode_t(const DecodeParams& p, const DecodePlan& pl, bool dense, hipStream_t st) {
  const dim3 grid(pl.col_blocks * pl.splits), block(64 * kDecodeWaves);
  // (which of the forms exist: plan_decode)
  auto kernel = decode_kernel<DT, MT, Z, true, 4, 1>;
  if constexpr (MT == 1) {
    if (!dense) kernel = decode_kernel<DT, MT, Z, false, 0, 1>;
    if constexpr (Z == 1) {
      if (dense && pl.load_words == 0) kernel = decode_kernel<DT, MT, Z, true, 0, 1>;
    } else {
      if (!dense && pl.load_words == 4) kernel = decode_kernel<DT, MT, Z, false, 4, 1>;
      if (dense && pl.load_words == 1) kernel = decode_kernel<DT, MT, Z, true, 1, 1>;
    }
  } else {
    if (!dense) kernel = decode_kernel<DT, MT, Z, false, 4, 1>;
    if (pl.load_words == 1) kernel = dense ? decode_kernel<DT, MT, Z, true, 1, 1> : decode_kernel<DT, MT, Z, false, 1, 1>;
  }
  if constexpr (MT == 1 ? Z >= 2 : MT == 2 && Z >= 3)
    if (pl.cg == 2) kernel = decode_kernel<DT, MT, Z, true, 4, 2>;  // (dense only)
  launch_main_kernel(kernel, grid, block, st, p);
}

template <typename DT, int MT>
static int launch_decode_mt(const DecodeParams& p, const DecodePlan& pl, int Z, bool dense, hipStream_t st) {
  switch (Z) {
    case 1: launch_decode_t<DT, MT, 1>(p, pl, dense, st); break;
    case 2: launch_decode_t<DT, MT, 2>(p, pl, dense, st); break;
    case 3: launch_decode_t<DT, MT, 3>(p, pl, dense, st); break;
    case 4: launch_decode_t<DT, MT, 4>(p, pl, dense, st); break;
    default: return GRINQH_ERR_INVALID;
  }
  return GRINQH_OK;
}

template <typename DT>
static int launch_decode_dt(const DecodeParams& p, const DecodePlan& pl, int Z, bool dense, hipStream_t st) {
  switch (pl.mt) {
    case 1: return launch_decode_mt<DT, 1>(p, pl, Z, dense, st);
    case 2: return launch_decode_mt<DT, 2>(p, pl, Z, dense, st);
    case 4: return launch_decode_mt<DT, 4>(p, pl, Z, dense, st);
    default: return GRINQH_ERR_INVALID;
  }
}

int launch_decode(const DecodeParams& p, const DecodePlan& pl, int max_bits, int dtype, bool dense,
                  hipStream_t st) {
  const int Z = max_bits / 2;
  const int rc = dtype == GRINQH_DTYPE_BF16 ? launch_decode_dt<BF16>(p, pl, Z, dense, st)
                                            : launch_decode_dt<F16>(p, pl, Z, dense, st);
  if (rc != GRINQH_OK) return rc;
  return hipGetLastError() == hipSuccess ? GRINQH_OK : GRINQH_ERR_HIP;
}

template <typename DT, int TPC>
static void launch_reduce_t(const DecodeParams& p, int splits, hipStream_t st) {
  const int64_t chunks = (int64_t)p.M * p.N / 4;
  const dim3 grid((unsigned)((chunks * TPC + 255) / 256));
  hipLaunchKernelGGL((splitk_reduce_kernel<DT, TPC>), grid, dim3(256), 0, st, p.partial, splits, p.M, p.N, p.bias,
                     p.y);
}

template <typename DT>
static void launch_reduce_dt(const DecodeParams& p, int splits, hipStream_t st) {
  // lanes per 4-column chunk: one lane adds up to 16 ranges with all its
  // loads in flight (qkv, o_proj and down at 16 and 64 rows: 3-6 % faster
  // products than four lanes and a butterfly); 64 ranges and more take 16
  // lanes (four lanes of 16 loads each were 5-14 % slower there)
  if (splits >= 64)
    launch_reduce_t<DT, 16>(p, splits, st);
  else if (splits > 16)
    launch_reduce_t<DT, 4>(p, splits, st);
  else
    launch_reduce_t<DT, 1>(p, splits, st);
}

int launch_splitk_reduce(const DecodeParams& p, int splits, int dtype, hipStream_t st) {
  if (dtype == GRINQH_DTYPE_BF16)
    launch_reduce_dt<BF16>(p, splits, st);
  else
    launch_reduce_dt<F16>(p, splits, st);
  return hipGetLastError() == hipSuccess ? GRINQH_OK : GRINQH_ERR_HIP;
}

int launch_sigma(const uint16_t* x, int64_t ldx, int M, int K, int dtype, float* sigma, hipStream_t st) {
  if (K == 0) return GRINQH_OK;
  const dim3 grid((K + 31) / 32);
  const GradeThresholds none{};
  if (dtype == GRINQH_DTYPE_BF16)
    hipLaunchKernelGGL((sigma_kernel<BF16, 0>), grid, dim3(256), 0, st, x, ldx, M, K, sigma, nullptr, none);
  else
    hipLaunchKernelGGL((sigma_kernel<F16, 0>), grid, dim3(256), 0, st, x, ldx, M, K, sigma, nullptr, none);
  return hipGetLastError() == hipSuccess ? GRINQH_OK : GRINQH_ERR_HIP;
}

template <typename DT>
static void launch_grade_words_dt(const uint16_t* x, int64_t ldx, int M, int K, int Z, const GradeThresholds& thr,
                                  uint32_t* grades, hipStream_t st) {
  const dim3 grid((K + 31) / 32);
  switch (Z) {
    case 1: hipLaunchKernelGGL((sigma_kernel<DT, 1>), grid, dim3(256), 0, st, x, ldx, M, K, nullptr, grades, thr); break;
    case 2: hipLaunchKernelGGL((sigma_kernel<DT, 2>), grid, dim3(256), 0, st, x, ldx, M, K, nullptr, grades, thr); break;
    case 3: hipLaunchKernelGGL((sigma_kernel<DT, 3>), grid, dim3(256), 0, st, x, ldx, M, K, nullptr, grades, thr); break;
    default: hipLaunchKernelGGL((sigma_kernel<DT, 4>), grid, dim3(256), 0, st, x, ldx, M, K, nullptr, grades, thr); break;
  }
}

int launch_grade_words(const uint16_t* x, int64_t ldx, int M, int K, int dtype, int max_bits,
                       const GradeThresholds& thr, uint32_t* grades, hipStream_t st) {
  if (K == 0) return GRINQH_OK;
  if (max_bits < 2 || max_bits > 8 || (max_bits & 1)) return GRINQH_ERR_INVALID;
  if (dtype == GRINQH_DTYPE_BF16)
    launch_grade_words_dt<BF16>(x, ldx, M, K, max_bits / 2, thr, grades, st);
  else
    launch_grade_words_dt<F16>(x, ldx, M, K, max_bits / 2, thr, grades, st);
  return hipGetLastError() == hipSuccess ? GRINQH_OK : GRINQH_ERR_HIP;
}

}  // namespace grinqh
