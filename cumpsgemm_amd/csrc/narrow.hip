// Real products whose result is a few rows or columns wide: a large matrix
// applied to a few vectors.  Bound by one reading of the large operand.
//
// The tiled kernels stage both operands through LDS with a barrier per K-step,
// which keeps one step's 32 KB per CU in flight at best.  Here nothing is shared
// inside the K loop: a workgroup owns 32 rows of the large operand, its waves
// take every 8th (16th) 32-wide K-step, load both operands straight into the
// registers of v_mfma_f32_16x16x32 fragments and never wait for one another until
// their sums meet in LDS.  A wave waits for a step's loads before it multiplies;
// what covers them is the CU's other waves.  Neighbouring waves read neighbouring
// 128-byte pieces of the same rows.  Every wave splits the narrow operand for
// itself (it comes from L2), which is cheap while that is no larger than the
// piece of the large operand beside it: kNarrowMax.
// 8192 x 16 x 8192 TN, operands not in a cache: 71.6 -> 63.4 us (4.2 TB/s).
//
// Fragments: lane l supplies row l % 16 of a 16-row block and eight of the step's
// 32 K-values.  Which eight is free as long as both operands agree: 4g .. 4g + 3
// and 16 + 4g .. (g = l / 16), so that the four lanes of a row read 64 contiguous
// bytes with each of two 16-byte loads.  A row-contiguous large operand is read
// as pairs of rows (2 (l % 16), + 1), 8 bytes a lane, 128 contiguous bytes a line.
#include "narrow.hpp"
#include <atomic>

namespace cumpsgemm_amd {
namespace {

// floats between the narrow side's rows of the sums in LDS (written without bank conflicts for a K-contiguous large
// operand; row pairs meet two to a bank)
constexpr int kRowStride = 36;

__device__ inline int k_of(const int g, const int j) { return (j < 4 ? 0 : 12) + 4 * g + j; }

// NB blocks of 16 rows of an operand.  PAIR: row-contiguous, lanes hold row pairs.
template <bool KC, int NB, bool PAIR> struct NarrowOperand {
  static_assert(!PAIR || (!KC && NB == 2), "row pairs");
  f8_t v[NB];

  __device__ static inline int row_of(const int b, const int lane) {
    return PAIR ? 2 * (lane & 15) + b : b * 16 + (lane & 15);
  }
  // byte offsets of this lane's rows from the tile's first element; a row past
  // the end reads the last one again (its products are not stored)
  __device__ static inline void offsets(uint32_t (&row_off)[NB], const uint32_t ld, const int rows, const int lane) {
#pragma unroll
    for (int b = 0; b < NB; b++) {
      const int r = row_of(b, lane);
      row_off[b] = (uint32_t)(r < rows ? r : rows - 1) * (KC ? ld : 1u) * 4u;
    }
  }
  __device__ inline void load(const float *base, const uint32_t (&row_off)[NB], const uint32_t ld, const int lane) {
    const uint32_t g = (uint32_t)lane >> 4;
    if constexpr (KC) {
      typedef float f4u_t __attribute__((ext_vector_type(4), aligned(4)));
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const char *p = reinterpret_cast<const char *>(base) + (row_off[b] + g * 16u);
        const f4u_t lo = *reinterpret_cast<const f4u_t *>(p), hi = *reinterpret_cast<const f4u_t *>(p + 64);
#pragma unroll
        for (int j = 0; j < 4; j++) {
          v[b][j] = lo[j];
          v[b][4 + j] = hi[j];
        }
      }
    } else {
      const __amdgpu_buffer_rsrc_t rsrc =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base), 0, 0xffffffff, 0x00020000);
      const uint32_t line = ld * 4u;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const uint32_t at = (j < 4 ? j : 12 + j) * line; // (uniform)
        if constexpr (PAIR) {
          typedef unsigned int u2_t __attribute__((ext_vector_type(2)));
          // (taken apart as a 64-bit integer: the elements of the vector result are mis-narrowed by this toolchain)
          const uint64_t w = __builtin_bit_cast(
              uint64_t, (u2_t)__builtin_amdgcn_raw_buffer_load_b64(rsrc, row_off[0] + 4u * g * line, at, 0));
          v[0][j] = __uint_as_float((uint32_t)w);
          v[1][j] = __uint_as_float((uint32_t)(w >> 32));
        } else {
#pragma unroll
          for (int b = 0; b < NB; b++)
            v[b][j] = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, row_off[b] + 4u * g * line, at, 0));
        }
      }
    }
  }
  // the partial K-step at the end: a K-value past it is read from the step's
  // first one and replaced by zero
  __device__ inline void load_tail(const float *base, const uint32_t (&row_off)[NB], const uint32_t ld, const int k_left,
                                   const int lane) {
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base), 0, 0xffffffff, 0x00020000);
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const int k = k_of(lane >> 4, j);
        const bool in = k < k_left;
        const uint32_t off = row_off[b] + (in ? (uint32_t)k : 0u) * (KC ? 4u : ld * 4u);
        const float t = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, off, 0, 0));
        v[b][j] = in ? t : 0.0f;
      }
  }
};

template <Prec P, bool BIG_KC, bool SMALL_KC, int FB>
__global__ __launch_bounds__(1024) void narrow_kernel(const NarrowArgs args) {
  using PT = prec_traits<P>;
  constexpr int NP = PT::NP, WB = 2;
  static_assert(WB * 16 == (int)kNarrowRows && FB * 16 <= (int)kNarrowMax, "tile");
  using Big = NarrowOperand<BIG_KC, WB, !BIG_KC>;
  using Small = NarrowOperand<SMALL_KC, FB, false>;
  extern __shared__ __attribute__((aligned(16))) float sums[]; // [wave][FB * 16][kRowStride]

  const int tid = threadIdx.x, lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
  uint32_t tile, zero;
  map_tile(blockIdx.x, gridDim.x, 1, tile, zero); // (neighbouring rows on one XCD)
  const uint32_t own = tile * kNarrowRows; // first row this workgroup stores
  // (the last tile ends at the last row: it shares rows with the one before it)
  const uint32_t row0 = own + kNarrowRows > args.wide ? args.wide - kNarrowRows : own;

  const uint32_t whole = args.k / 32, tail = args.k % 32;
  const uint32_t first = blockIdx.z * args.steps_per_chunk;
  const uint32_t last = first + args.steps_per_chunk < whole ? first + args.steps_per_chunk : whole;
  const float *const big = args.big + (uint64_t)row0 * (BIG_KC ? args.ld_big : 1);
  const float *const small = args.small;
  const uint64_t big_step = BIG_KC ? 32 : 32 * args.ld_big, small_step = SMALL_KC ? 32 : 32 * args.ld_small;
  const uint32_t ldb = (uint32_t)args.ld_big, lds = (uint32_t)args.ld_small;

  uint32_t big_off[WB], small_off[FB];
  Big::offsets(big_off, ldb, (int)kNarrowRows, lane);
  Small::offsets(small_off, lds, (int)args.few, lane);

  f4v_t acc[PT::NACC][FB][WB];
#pragma unroll
  for (int s = 0; s < PT::NACC; s++)
#pragma unroll
    for (int f = 0; f < FB; f++)
#pragma unroll
      for (int b = 0; b < WB; b++) acc[s][f][b] = f4v_t{0.0f, 0.0f, 0.0f, 0.0f};

  struct Step {
    Big big;
    Small small;
  };
  auto load = [&](Step &x, const uint32_t step) {
    x.big.load(big + step * big_step, big_off, ldb, lane);
    x.small.load(small + step * small_step, small_off, lds, lane);
  };
  auto multiply = [&](const Step &x) {
    u4_t bp[WB][NP], sp[FB][NP];
#pragma unroll
    for (int b = 0; b < WB; b++) splitter<P>::run(x.big.v[b], bp[b]);
#pragma unroll
    for (int f = 0; f < FB; f++) splitter<P>::run(x.small.v[f], sp[f]);
#pragma unroll
    for (int t = 0; t < PT::NPROD; t++)
#pragma unroll
      for (int f = 0; f < FB; f++)
#pragma unroll
        for (int b = 0; b < WB; b++)
          acc[PT::ACC[t]][f][b] =
              mfma_block<PT::IS_BF16>(sp[f][PT::PB[t]], bp[b][PT::PA[t]], acc[PT::ACC[t]][f][b]);
  };

  // the partial step goes to the last chunk, to the wave whose turn it is there
  if (tail != 0 && blockIdx.z == gridDim.z - 1 && wave == (last - first) % waves) {
    Step x;
    x.big.load_tail(big + whole * big_step, big_off, ldb, (int)tail, lane);
    x.small.load_tail(small + whole * small_step, small_off, lds, (int)tail, lane);
    multiply(x);
  }
  uint32_t step = first + wave;
  if (step < last) {
    // (past its last step a wave reads that step once more, to no use, instead of branching around the loads.  The
    // compiler moves a set's loads behind the multiplication of the other: held in front of it, with the steps in pairs
    // and barriers to the scheduler, 8192 x 16 x 8192 TN takes 59 instead of 63 us and 16384 x 16 x 8192 NN 117 instead
    // of 108, and short K on many rows 5 - 15 % longer for the registers)
    auto next = [&](const uint32_t s) { return s + waves < last ? s + waves : s; };
    Step x, y;
    load(x, step);
    while (true) {
      load(y, next(step));
      multiply(x);
      step += waves;
      if (step >= last) break;
      load(x, next(step));
      multiply(y);
      step += waves;
      if (step >= last) break;
    }
  }

  // sums of the waves: MFMA row (-> narrow side) 4 (l / 16) + v, MFMA column (-> wide side) l % 16
  float *const mine = sums + wave * (FB * 16 * kRowStride);
#pragma unroll
  for (int f = 0; f < FB; f++)
#pragma unroll
    for (int b = 0; b < WB; b++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        float x = acc[0][f][b][v];
        if constexpr (PT::NACC == 2) x += acc[1][f][b][v] * PT::CORR_SCALE;
        mine[(f * 16 + 4 * (lane >> 4) + v) * kRowStride + Big::row_of(b, lane)] = x;
      }
  __syncthreads();
  for (uint32_t e = tid; e < FB * 16 * kNarrowRows; e += blockDim.x) {
    // (consecutive threads along C's columns)
    const uint32_t w = args.few_is_n ? e % kNarrowRows : e / (FB * 16);
    const uint32_t f = args.few_is_n ? e / kNarrowRows : e % (FB * 16);
    if (f >= args.few || row0 + w < own) continue;
    float x = 0.0f;
    for (uint32_t i = 0; i < waves; i++) x += sums[(i * FB * 16 + f) * kRowStride + w];
    const uint64_t row = row0 + w;
    float *const cp = args.c + (args.few_is_n ? f * args.ldc + row : row * args.ldc + f);
    if (args.atomic_out) atomicAdd(cp, x * args.alpha);
    else if (args.beta == 0.0f) *cp = x * args.alpha;
    else *cp = x * args.alpha + args.beta * *cp;
  }
}

template <Prec P, bool BIG_KC, bool SMALL_KC, int FB>
void launch_one(const NarrowArgs &args, uint32_t waves, uint32_t chunks, hipStream_t stream) {
  const uint32_t lds = waves * FB * 16 * kRowStride * 4;
  if (lds > 64 * 1024) { // (allowed once per kernel and device)
    static std::atomic<bool> done[64] = {};
    int dev = 0;
    (void)hipGetDevice(&dev);
    if (dev < 0 || dev >= 64 || !done[dev].load(std::memory_order_acquire)) {
      (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&narrow_kernel<P, BIG_KC, SMALL_KC, FB>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, 16 * FB * 16 * kRowStride * 4);
      if (dev >= 0 && dev < 64) done[dev].store(true, std::memory_order_release);
    }
  }
  const dim3 grid((args.wide + kNarrowRows - 1) / kNarrowRows, 1, chunks);
  hipLaunchKernelGGL((narrow_kernel<P, BIG_KC, SMALL_KC, FB>), grid, dim3(waves * 64), lds, stream, args);
}

template <Prec P> void launch_prec(const NarrowArgs &args, bool big_kc, bool small_kc, uint32_t waves, uint32_t chunks,
                                   hipStream_t stream) {
  auto pick = [&](auto fb) {
    constexpr int FB = decltype(fb)::value;
    if (big_kc) {
      if (small_kc) launch_one<P, true, true, FB>(args, waves, chunks, stream);
      else launch_one<P, true, false, FB>(args, waves, chunks, stream);
    } else {
      if (small_kc) launch_one<P, false, true, FB>(args, waves, chunks, stream);
      else launch_one<P, false, false, FB>(args, waves, chunks, stream);
    }
  };
  if (args.few <= 16) pick(std::integral_constant<int, 1>{});
  else pick(std::integral_constant<int, 2>{});
}
} // namespace

bool narrow_offsets_fit(uint64_t ld_big, uint64_t ld_small) {
  // 32 rows, or 32 lines, of each operand
  const uint64_t limit = 0x7fffffffull / (33 * 4);
  return ld_big < limit && ld_small < limit;
}

void launch_narrow(const NarrowArgs &args, Prec p, bool big_kc, bool small_kc, uint32_t waves, uint32_t chunks,
                   hipStream_t stream) {
  if (p == Prec::BF16X3) launch_prec<Prec::BF16X3>(args, big_kc, small_kc, waves, chunks, stream);
  else launch_prec<Prec::FP16TCEC>(args, big_kc, small_kc, waves, chunks, stream);
}
} // namespace cumpsgemm_amd
