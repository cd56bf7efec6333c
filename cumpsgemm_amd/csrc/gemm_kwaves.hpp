// Small products: one workgroup per tile of C, the waves of a workgroup share out
// K instead of the tile.
//
// What bounds a product of a few hundred rows and columns is not arithmetic but
// round trips: a workgroup of the tiled kernels passes a barrier per 32-wide
// K-step and its loads run one step ahead of it (1024^3: 32 steps of 0.4 us).
// Here wave w takes K-steps w, w + W, w + 2 W ... and computes the whole tile over
// them, on its own: it loads its 32 K-values of the tile's rows, splits them,
// passes them through a piece of LDS that no other wave touches -- LDS operations
// of one wave happen in order, so there is no barrier in the K loop -- and
// multiplies.  The sums of the waves meet in LDS at the end.  Every element of the
// tile's operands is loaded once and split once, as in the tiled kernels.
//
// One K-step of a wave is multiplied beside the splitting of the next and the
// loads of the one after that, piece by piece (a wave issues its MFMAs and vector
// instructions one after the other, and MFMAs issued in a row keep the vector
// unit from the SIMD's other waves).  All loads are 16 bytes a lane, of a
// row-contiguous operand too: a quarter of the load instructions.
//
// Two waves to a SIMD where the registers allow it (not bf16x3) and a CU gets two workgroups,
// or one of eight waves (otherwise: kwaves_rule.hpp, the forms for one workgroup on a CU): a wave alone issues a
// vector instruction every 5 clocks and a conversion every 8, two of them together twice
// as many, and MFMAs of one run beside splitting of the other.  On a 64 x 64 (complex
// 32 x 32) tile that is two workgroups of four waves on a CU; complex products of no more
// tiles than CUs take one of eight.  us, one workgroup of four waves per CU -> so: real
// FP16TCEC 1152^3 NN 25.4 -> 20.3 (tiled 24.4), 1408^3 30.5 -> 26.8, 1531 x 1021 x 777 TT
// 22.7 -> 18.8 (tiled 19.6); FP16TC 1152^3 17.5 -> 15.0; complex FP16TCEC 512^3 NN 8.5 -> 7.6,
// 640^3 16.6 -> 12.9, 900 x 300 x 900 22.9 -> 17.5, 512 x 512 x 2048 22.0 -> 20.8.
//
// FP16TCEC, us, tiled -> here (calls of a graph; a loop of single calls takes 4 at least):
// 512^3 NN 9.9 -> 4.7, NT 10.1 -> 4.6, 1024^3 NN 16.0 -> 12.9, NT 21.2 -> 12.2, TN 13.6 -> 12.8;
// complex 256^3 NN 13.2 -> 5.5, NT 13.6 -> 5.4, 512^3 NN 14.9 -> 7.8, NT 16.9 -> 7.7.
// Larger products are bound by what a small tile reads (2048^3 NN 58 -> 74): see kwaves_rule.hpp.
#pragma once
#include "gemm_kernel.hpp"

namespace cumpsgemm_amd {

// W waves; OCC waves per SIMD that the register allocator must leave room for.
template <Prec P_, bool CPLX_, bool A_KC_, bool B_KC_, int BM_, int BN_, int W_, int OCC_, bool SCALED_ = false>
struct KWavesCfg {
  static constexpr Prec P = P_;
  static constexpr bool CPLX = CPLX_, A_KC = A_KC_, B_KC = B_KC_, SCALED = SCALED_;
  static constexpr int BM = BM_, BN = BN_, W = W_, OCC = OCC_;
  static constexpr int NT = W * 64;
  static constexpr bool TWO_PER_SIMD = OCC == 2;
  static constexpr int TM = BM / 32, TN = BN / 32;
  static constexpr int NP = prec_traits<P>::NP, NC = CPLX ? 2 : 1;
  // LDS: planes of 64-byte rows (32 K-values), 16 bytes of padding after every fourth row
  static constexpr int A_PLANE = BM * 68, B_PLANE = BN * 68;
  static constexpr int WAVE_BYTES = (A_PLANE + B_PLANE) * NP * NC;
  // sums of a wave: columns of C, 16 bytes of padding after each
  static constexpr int COL = BM * NC + 4; // floats
  static constexpr int SUM_BYTES = W * BN * COL * 4;
  static constexpr int LDS_BYTES = W * WAVE_BYTES > SUM_BYTES ? W * WAVE_BYTES : SUM_BYTES;
  // floats of a column that a thread adds up at a time, and how many such units a thread has
  static constexpr int UNIT = BM * BN * NC / NT < 4 ? BM * BN * NC / NT : 4, OWN = BM * BN * NC / NT / UNIT;
  static_assert(UNIT % NC == 0 && UNIT * OWN * NT == BM * BN * NC && LDS_BYTES <= 160 * 1024, "");
};

// Byte offset of (row, 16-byte chunk) in a plane.  16 bytes of padding after every
// fourth row instead of a swizzle: a lane of a row-contiguous operand writes one
// chunk of four consecutive rows, lanes l and l + 1 the same chunk of rows four
// apart; that, the 8-byte writes of a K-contiguous operand (8 rows x 64 bytes) and
// the fragment reads (32 rows, two chunks) all spread evenly over the banks (real
// 512^3: no conflicts; the sums of 64 x 64 tiles add 256 cycles a workgroup).  A complex
// row-contiguous operand writes rows two apart, which meet in pairs: 512^3 NT 5.6e5
// conflict cycles in all, 2200 a workgroup, NN 3.0e5, TN 3e4.
__device__ constexpr int kwave_lds(const int row, const int chunk) { return row * 64 + (row >> 2) * 16 + chunk * 16; }

// K-value at position j of 16-byte chunk c of an LDS row (complex: the order in
// which eight lanes, 16 bytes each, read 128 contiguous bytes of a row twice).
template <bool CPLX> __device__ constexpr int kwave_k_of(const int c, const int j) {
  if constexpr (!CPLX) return 8 * c + j;
  return 4 * c + (j >> 2) * 2 + (j & 1) + ((j & 2) ? 16 : 0);
}

// 32 K-values of ROWS rows of an operand, as one wave loads and splits them.
//   KC:  eight lanes to a row, eight rows a load; a piece is 4 K-values of a row.
//   !KC: row-contiguous; a load holds EPL rows of each of 64 / LPL K-lines, a lane
//        keeps KPL lines of the same EPL rows; a piece is 8 (4) K-values of a row.
template <Prec P, bool CPLX, bool KC, int ROWS, bool SCALED> struct WaveOperand {
  static constexpr int NC = CPLX ? 2 : 1, NP = prec_traits<P>::NP, PLANE = ROWS * 68;
  static constexpr int EPL = 4 / NC, LPL = ROWS / EPL, KPL = ROWS * 32 * NC / 4 / 64;
  static constexpr int LOADS = KC ? ROWS / 8 * NC : KPL;
  static constexpr int KV = KC || KPL == 4 ? 4 : 8;           // K-values of a piece
  static constexpr int PIECES = KC ? ROWS / 8 : EPL * KPL / KV; // (row-contiguous: EPL rows of one chunk, then the next)
  static constexpr int WEIGHT = KV * NC;
  static_assert(KV == 4 || KV == 8, "half or whole chunk");
  typedef float f4u_t __attribute__((ext_vector_type(4)));
  f4u_t v[LOADS];
  uint32_t off[KC ? PIECES : 1];

  __device__ static inline int row_of(const int i, const int lane) { return KC ? 8 * i + (lane >> 3) : (lane % LPL) * EPL + i % EPL; }
  // first position along K (of 32) of a lane's piece i
  __device__ static inline int pos_of(const int i, const int lane) { return KC ? (lane & 7) * 4 : lane / LPL * KPL + i / EPL * KV; }
  // K-value of a lane's position j from there
  __device__ static inline int k_of(const int i, const int lane, const int j) {
    const int at = pos_of(i, lane) + j;
    return kwave_k_of<CPLX>(at >> 3, at & 7);
  }
  __device__ inline void offsets(const uint32_t ld, const int rows, const int lane) {
    const uint32_t k0 = (uint32_t)k_of(0, lane, 0);
    if constexpr (KC) {
#pragma unroll
      for (int i = 0; i < PIECES; i++) {
        const int row = row_of(i, lane);
        off[i] = ((uint32_t)(row < rows ? row : rows - 1) * ld + k0) * (uint32_t)(NC * 4);
      }
    } else {
      off[0] = (k0 * ld + (uint32_t)row_of(0, lane)) * (uint32_t)(NC * 4);
    }
  }
  __device__ static inline f4u_t load16(const __amdgpu_buffer_rsrc_t rsrc, const uint32_t off, const uint32_t at) {
    // (taken apart as integers: the elements of a vector result are mis-narrowed by this toolchain)
    const unsigned __int128 w =
        __builtin_bit_cast(unsigned __int128, (u4_t)__builtin_amdgcn_raw_buffer_load_b128(rsrc, off, at, 0));
    return f4u_t{__uint_as_float((uint32_t)w), __uint_as_float((uint32_t)(w >> 32)), __uint_as_float((uint32_t)(w >> 64)),
                 __uint_as_float((uint32_t)(w >> 96))};
  }
  // load number I of a whole K-step.  (A row-contiguous tile lies inside the matrix:
  // the host sees to it; rows of a K-contiguous one past the edge re-read the last.)
  template <int I> __device__ inline void load(const float *base, const uint32_t ld) {
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base), 0, 0xffffffff, 0x00020000);
    if constexpr (KC) {
      v[I] = load16(rsrc, off[I / NC], (I % NC) * 128);
    } else {
      const uint32_t line = __builtin_amdgcn_readfirstlane(ld * (uint32_t)(NC * 4));
      v[I] = load16(rsrc, off[0], (uint32_t)kwave_k_of<CPLX>(I >> 3, I & 7) * line);
    }
  }
  // zero for a lane's K-values before `from` (the partial K-step loaded as the last 32 K-values of the matrix)
  __device__ inline void drop_before(const int from, const int lane) {
    if constexpr (KC) {
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const bool in = k_of(0, lane, j) >= from; // (the same for every piece)
#pragma unroll
        for (int i = 0; i < PIECES; i++)
#pragma unroll
          for (int q = 0; q < NC; q++) {
            f4u_t &x = v[i * NC + j * NC / 4];
            x[(j * NC + q) % 4] = in ? x[(j * NC + q) % 4] : 0.0f;
          }
      }
    } else {
#pragma unroll
      for (int i = 0; i < KPL; i++) {
        const bool in = k_of(0, lane, i) >= from;
#pragma unroll
        for (int e = 0; e < 4; e++) v[i][e] = in ? v[i][e] : 0.0f;
      }
    }
  }
  // the partial K-step at the end (k_left < 32 K-values): a K-value past it is read from the step's first and replaced by zero
  __device__ inline void load_tail(const float *base, const uint32_t ld, const int rows, const int k_left, const int lane) {
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base), 0, 0xffffffff, 0x00020000);
    if constexpr (KC) {
#pragma unroll
      for (int i = 0; i < PIECES; i++) {
        const int row = row_of(i, lane);
        const uint32_t row_off = (uint32_t)(row < rows ? row : rows - 1) * ld * (uint32_t)(NC * 4);
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const int k = k_of(i, lane, j);
          const bool in = k < k_left;
#pragma unroll
          for (int q = 0; q < NC; q++) {
            const float t = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, row_off + (uint32_t)((in ? k : 0) * NC + q) * 4u, 0, 0));
            v[i * NC + j * NC / 4][(j * NC + q) % 4] = in ? t : 0.0f;
          }
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < KPL; i++) {
        const int k = k_of(0, lane, i);
        const bool in = k < k_left;
        const f4u_t t = load16(rsrc, ((uint32_t)(in ? k : 0) * ld + (uint32_t)row_of(0, lane)) * (uint32_t)(NC * 4), 0);
#pragma unroll
        for (int e = 0; e < 4; e++) v[i][e] = in ? t[e] : 0.0f;
      }
    }
  }
  // K-value j, component c of piece I
  template <int I> __device__ inline float value(const int j, const int c) const {
    if constexpr (KC) return v[I * NC + j * NC / 4][(j * NC + c) % 4];
    else return v[I / EPL * KV + j][I % EPL * NC + c];
  }
  // registers (loads) that nothing needs any more once piece i is stored, pieces in order
  static constexpr int first_freed(const int i) { return KC ? i * NC : i / EPL * KV; }
  static constexpr int freed(const int i) { return KC ? NC : i % EPL == EPL - 1 ? KV : 0; }
  // split piece I and write it to LDS, planes [component][term][row][chunk]
  template <int I> __device__ inline void store(char *lds_op, const int lane, const float s, const float s2048) const {
    const int pos = pos_of(I, lane), at = kwave_lds(row_of(I, lane), pos >> 3) + (pos & 7) * 2;
#pragma unroll
    for (int c = 0; c < NC; c++) {
      u4_t out[NP];
#pragma unroll
      for (int q = 0; q < KV / 2; q++) {
        uint32_t terms[NP];
        split_pair<P, SCALED>(value<I>(2 * q, c), value<I>(2 * q + 1, c), s, s2048, terms);
#pragma unroll
        for (int p = 0; p < NP; p++) out[p][q] = terms[p];
      }
#pragma unroll
      for (int p = 0; p < NP; p++) {
        char *const to = lds_op + (c * NP + p) * PLANE + at;
        if constexpr (KV == 4) {
          typedef uint32_t u2v_t __attribute__((ext_vector_type(2)));
          *reinterpret_cast<u2v_t *>(to) = u2v_t{out[p][0], out[p][1]};
        } else {
          *reinterpret_cast<u4_t *>(to) = out[p];
        }
      }
    }
  }
};

template <int LO, int HI, class F> __device__ inline void static_for(F &&f) {
  if constexpr (LO < HI) {
    f(std::integral_constant<int, LO>{});
    static_for<LO + 1, HI>(f);
  }
}

// The product (called by the kernels at the end of this file).
template <class Cfg> __device__ inline void kwaves_product(const GemmArgs &args) {
  constexpr Prec P = Cfg::P;
  using PT = prec_traits<P>;
  constexpr bool CPLX = Cfg::CPLX;
  constexpr int BM = Cfg::BM, BN = Cfg::BN, TM = Cfg::TM, TN = Cfg::TN, NP = Cfg::NP, NC = Cfg::NC, W = Cfg::W;

  float coef_a = 1.0f, coef_b = 1.0f, coef_c = 1.0f;
  if constexpr (Cfg::SCALED) {
    const int sflag = *args.scale_flag;
    const float ma = __uint_as_float(*args.scale_max_a), mb = __uint_as_float(*args.scale_max_b);
    if ((sflag & 0x40) && ma != 0.0f) {
      coef_a = 16384.0f / ma;
      coef_c *= ma / 16384.0f;
    }
    if ((sflag & 0x20) && mb != 0.0f) {
      coef_b = 16384.0f / mb;
      coef_c *= mb / 16384.0f;
    }
    auto uniform = [](float x) {
      return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(x)));
    };
    coef_a = uniform(coef_a);
    coef_b = uniform(coef_b);
    coef_c = uniform(coef_c);
  }
  const float coef_a2048 = coef_a * 2048.0f, coef_b2048 = coef_b * 2048.0f;
  const float alpha_re = args.alpha_re * coef_c, alpha_im = args.alpha_im * coef_c;

  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  uint32_t tile_m, tile_n, tile_b;
  map_tile_batched(blockIdx.x, args.tiles_m, args.tiles_n, args.batch, tile_m, tile_n, tile_b);
  const uint32_t m0 = tile_m * BM, n0 = tile_n * BN;
  const uint32_t ml0 = (args.m >= (uint32_t)BM && m0 + BM > args.m) ? args.m - BM : m0;
  const uint32_t nl0 = (args.n >= (uint32_t)BN && n0 + BN > args.n) ? args.n - BN : n0;
  const uint64_t lda = args.lda, ldb = args.ldb;
  const float *const a = reinterpret_cast<const float *>(args.a) + tile_b * args.stride_a * NC;
  const float *const b = reinterpret_cast<const float *>(args.b) + tile_b * args.stride_b * NC;
  float *const c = reinterpret_cast<float *>(args.c) + tile_b * args.stride_c * NC;
  const float *const a_tile = a + (Cfg::A_KC ? ml0 * lda : ml0) * NC;
  const float *const b_tile = b + (Cfg::B_KC ? nl0 * ldb : nl0) * NC;
  const uint64_t a_kstep = (Cfg::A_KC ? 32 : 32 * lda) * NC, b_kstep = (Cfg::B_KC ? 32 : 32 * ldb) * NC;

  WaveOperand<P, CPLX, Cfg::A_KC, BM, Cfg::SCALED> oa;
  WaveOperand<P, CPLX, Cfg::B_KC, BN, Cfg::SCALED> ob;
  const int rows_a = (int)((args.m - ml0 < (uint32_t)BM) ? args.m - ml0 : BM);
  const int rows_b = (int)((args.n - nl0 < (uint32_t)BN) ? args.n - nl0 : BN);
  oa.offsets((uint32_t)lda, rows_a, lane);
  ob.offsets((uint32_t)ldb, rows_b, lane);

  // accumulators: MFMA rows run along M, MFMA columns along N
  constexpr int NSET = CPLX ? 4 : 1;
  f16v_t acc[NSET][PT::NACC][TN][TM];
#pragma unroll
  for (int q = 0; q < NSET; q++)
#pragma unroll
    for (int s = 0; s < PT::NACC; s++)
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int v = 0; v < 16; v++) acc[q][s][j][i][v] = 0.0f;

  char *const sa = lds + wave * Cfg::WAVE_BYTES, *const sb = sa + Cfg::A_PLANE * NP * NC;
  const int frag_at = kwave_lds(lane & 31, lane >> 5);
  struct Frags {
    u4_t a[NC][NP][TM], b[NC][NP][TN];
  };
  auto frag_load = [&](Frags &f, const int h) {
#pragma unroll
    for (int q = 0; q < NC; q++)
#pragma unroll
      for (int p = 0; p < NP; p++) {
#pragma unroll
        for (int i = 0; i < TM; i++)
          f.a[q][p][i] = *reinterpret_cast<const u4_t *>(sa + (q * NP + p) * Cfg::A_PLANE + frag_at + h * 32 + i * 32 * 68);
#pragma unroll
        for (int j = 0; j < TN; j++)
          f.b[q][p][j] = *reinterpret_cast<const u4_t *>(sb + (q * NP + p) * Cfg::B_PLANE + frag_at + h * 32 + j * 32 * 68);
      }
  };
  // MFMA number X of a K-step: 16-wide K-slice, product, block of the tile (complex: real product)
  constexpr int HALF_MFMAS = PT::NPROD * TM * TN * NSET, STEP_MFMAS = 2 * HALF_MFMAS;
  auto mma = [&](const Frags &f0, const Frags &f1, auto x_tag) {
    constexpr int X = decltype(x_tag)::value, r = X % HALF_MFMAS;
    constexpr int q = r % NSET, i = r / NSET % TM, j = r / NSET / TM % TN, t = r / NSET / TM / TN;
    constexpr int s = PT::ACC[t], pa = PT::PA[t], pb = PT::PB[t];
    constexpr int ca = CPLX && (q == 1 || q == 3) ? 1 : 0, cb = CPLX && (q == 1 || q == 2) ? 1 : 0;
    const Frags &f = X < HALF_MFMAS ? f0 : f1;
    acc[q][s][j][i] = mfma_block<PT::IS_BF16>(f.a[ca][pa][i], f.b[cb][pb][j], acc[q][s][j][i]);
  };

  const int whole = (int)(args.k / 32), tail = (int)(args.k % 32);
  const int mine = whole > wave ? (whole - wave + W - 1) / W : 0;
  const bool has_tail = tail != 0 && whole % W == wave;
  const int steps = mine + (has_tail ? 1 : 0);
  const float *ap = a_tile + wave * a_kstep, *bp = b_tile + wave * b_kstep;
  constexpr int PA = decltype(oa)::PIECES, PB = decltype(ob)::PIECES;
  constexpr int WA = decltype(oa)::WEIGHT, WB = decltype(ob)::WEIGHT, WSUM = PA * WA + PB * WB;
  auto store_piece = [&](auto i_tag) {
    constexpr int I = decltype(i_tag)::value;
    if constexpr (I < PA) oa.template store<I>(sa, lane, coef_a, coef_a2048);
    else ob.template store<I - PA>(sb, lane, coef_b, coef_b2048);
  };
  // the loads into the registers that storing piece I has freed
  auto load_after = [&](auto i_tag) {
    constexpr int I = decltype(i_tag)::value;
    auto of = [&](auto &o, const float *base, const uint64_t ld, auto j_tag) {
      using O = std::remove_reference_t<decltype(o)>;
      constexpr int J = decltype(j_tag)::value;
      constexpr int first = O::first_freed(J), count = O::freed(J);
      static_for<first, first + count>([&](auto l) { o.template load<decltype(l)::value>(base, (uint32_t)ld); });
    };
    if constexpr (I < PA) of(oa, ap, lda, i_tag);
    else of(ob, bp, ldb, std::integral_constant<int, I - PA>{});
  };
  auto advance = [&]() {
    ap += a_kstep * W;
    bp += b_kstep * W;
  };
  if (steps > 0) {
    if (W > 1 && has_tail && whole > 0) {
      // The last 32 K-values without those of the step before: loads of 16 bytes, where load_tail reads a K-contiguous
      // operand value by value.  (us, load_tail -> so: real 500^3 NN 5.57 -> 5.33, TN 5.34 -> 5.10, complex TN 8.64 ->
      // 8.29.  Not with one wave to a tile: many small matrices are bound by the bytes they read, and the step before is
      // not on the chip yet.  128 x 128 x 100 x 1000 NT 32 -> 38.)
      const uint64_t back = 32 - tail;
      const float *const ap0 = ap, *const bp0 = bp;
      ap = a_tile + whole * a_kstep - back * (Cfg::A_KC ? 1 : lda) * NC;
      bp = b_tile + whole * b_kstep - back * (Cfg::B_KC ? 1 : ldb) * NC;
      static_for<0, PA + PB>(load_after);
      oa.drop_before((int)back, lane);
      ob.drop_before((int)back, lane);
      ap = ap0;
      bp = bp0;
    } else if (has_tail) {
      oa.load_tail(a_tile + whole * a_kstep, (uint32_t)lda, rows_a, tail, lane);
      ob.load_tail(b_tile + whole * b_kstep, (uint32_t)ldb, rows_b, tail, lane);
    } else {
      static_for<0, PA + PB>(load_after);
      advance();
    }
    static_for<0, PA + PB>(store_piece);
    if (steps > 1) {
      static_for<0, PA + PB>(load_after);
      advance();
    }
    if constexpr (Cfg::TWO_PER_SIMD) {
      // One set of fragments: 128 accumulator registers, 64 of loads in flight and
      // 32 of fragments leave room for a second wave on the SIMD.  The first half of
      // a step's MFMAs run beside the other wave's splitting, the second half beside
      // this wave's.
      Frags f;
      auto step = [&](auto stage_tag, auto load_tag) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
        frag_load(f, 0);
        static_for<0, HALF_MFMAS>([&](auto x) { mma(f, f, x); });
        __builtin_amdgcn_sched_barrier(0);
        frag_load(f, 1);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
        static_for<0, PA + PB>([&](auto i_tag) {
          constexpr int I = decltype(i_tag)::value;
          constexpr int w0 = I < PA ? I * WA : PA * WA + (I - PA) * WB, w1 = w0 + (I < PA ? WA : WB);
          static_for<HALF_MFMAS + HALF_MFMAS * w0 / WSUM, HALF_MFMAS + HALF_MFMAS * w1 / WSUM>(
              [&](auto x) { mma(f, f, x); });
          if constexpr (decltype(stage_tag)::value) store_piece(i_tag);
          if constexpr (decltype(load_tag)::value) load_after(i_tag);
          __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (decltype(load_tag)::value) advance();
      };
      int t = 0;
      for (; t + 2 < steps; t++) step(std::true_type{}, std::true_type{});
      if (t + 1 < steps) step(std::true_type{}, std::false_type{});
      step(std::false_type{}, std::false_type{});
    } else {
      Frags f0, f1;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
      frag_load(f0, 0);
      // one K-step beside the staging of the next
      constexpr int LAST = STEP_MFMAS / 6, BESIDE = STEP_MFMAS - LAST;
      auto step = [&](auto load_tag) {
        frag_load(f1, 1);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
        static_for<0, PA + PB>([&](auto i_tag) {
          constexpr int I = decltype(i_tag)::value;
          constexpr int w0 = I < PA ? I * WA : PA * WA + (I - PA) * WB, w1 = w0 + (I < PA ? WA : WB);
          static_for<BESIDE * w0 / WSUM, BESIDE * w1 / WSUM>([&](auto x) { mma(f0, f1, x); });
          store_piece(i_tag);
          if constexpr (decltype(load_tag)::value) load_after(i_tag);
          __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (decltype(load_tag)::value) advance();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
        frag_load(f0, 0);
        static_for<BESIDE, STEP_MFMAS>([&](auto x) { mma(f0, f1, x); });
      };
      int t = 0;
      for (; t + 2 < steps; t++) step(std::true_type{});
      if (t + 1 < steps) step(std::false_type{});
      frag_load(f1, 1);
      static_for<0, STEP_MFMAS>([&](auto x) { mma(f0, f1, x); });
    }
  }

  // ---- sums of the waves ------------------------------------------------------
  // Each wave writes its sums to LDS, columns of C; thread t then adds up 16 bytes
  // of a column at a time.
  constexpr int COL = Cfg::COL, OWN = Cfg::OWN, U = Cfg::UNIT, UPC = BM * NC / U; // units per column
  const bool beta_zero = (args.beta_re == 0.0f) && (!CPLX || args.beta_im == 0.0f);
  const bool full = ml0 == m0 && nl0 == n0 && rows_a == BM && rows_b == BN;
  typedef float unit_t __attribute__((ext_vector_type(U), aligned(4)));
  const int t0 = threadIdx.x;
  auto unit_m = [&](const int x) { return (t0 + x * Cfg::NT) % UPC * (U / NC); };
  auto unit_n = [&](const int x) { return (t0 + x * Cfg::NT) / UPC; };
  auto place = [&](const int x) { return c + ((uint64_t)(nl0 + unit_n(x)) * args.ldc + (ml0 + unit_m(x))) * NC; };
  auto inside = [&](const int x, const int e) { // element e (of U / NC) of unit x
    const uint32_t mm = ml0 + unit_m(x) + e, nn = nl0 + unit_n(x);
    return mm < args.m && nn < args.n && mm >= m0 && nn >= n0;
  };
  unit_t old[OWN];
  if (!beta_zero) {
#pragma unroll
    for (int x = 0; x < OWN; x++) {
      const float *const p = place(x);
      if (full) {
        old[x] = *reinterpret_cast<const unit_t *>(p);
      } else {
#pragma unroll
        for (int e = 0; e < U; e++) old[x][e] = inside(x, e / NC) ? p[e] : 0.0f;
      }
    }
  }
  float *const red = reinterpret_cast<float *>(lds);
  __syncthreads(); // (every wave is done with its planes)
  const float sgn_a = args.conj_a ? -1.0f : 1.0f, sgn_b = args.conj_b ? -1.0f : 1.0f, sgn_ab = sgn_a * sgn_b;
#pragma unroll
  for (int j = 0; j < TN; j++)
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int g = 0; g < 4; g++) {
        // rows 32 i + 8 g + 4 (l / 32) .. + 3 of column 32 j + l % 32
        float *const to = red + (wave * BN + j * 32 + (lane & 31)) * COL + (i * 32 + g * 8 + 4 * (lane >> 5)) * NC;
        f4v_t out[NC];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          float p[NSET];
#pragma unroll
          for (int q = 0; q < NSET; q++) {
            p[q] = acc[q][0][j][i][4 * g + e];
            if constexpr (PT::NACC == 2) p[q] += acc[q][1][j][i][4 * g + e] * PT::CORR_SCALE;
          }
          if constexpr (!CPLX) {
            out[0][e] = p[0];
          } else {
            // re = ar*br - sa*sb*ai*bi, im = sb*ar*bi + sa*ai*br, sa (sb) = -1 when op(A) (op(B)) conjugates
            out[e >> 1][(e & 1) * 2] = p[0] - sgn_ab * p[1];
            out[e >> 1][(e & 1) * 2 + 1] = sgn_b * p[2] + sgn_a * p[3];
          }
        }
#pragma unroll
        for (int q = 0; q < NC; q++) reinterpret_cast<f4v_t *>(to)[q] = out[q];
      }
  typedef float sum_t __attribute__((ext_vector_type(U)));
  __syncthreads();
#pragma unroll
  for (int x = 0; x < OWN; x++) {
    float sum[U] = {};
#pragma unroll
    for (int w = 0; w < W; w++) {
      const sum_t y = *reinterpret_cast<const sum_t *>(red + (w * BN + unit_n(x)) * COL + unit_m(x) * NC);
#pragma unroll
      for (int e = 0; e < U; e++) sum[e] += y[e];
    }
    unit_t out;
#pragma unroll
    for (int e = 0; e < U; e += NC) {
      if constexpr (!CPLX) {
        out[e] = sum[e] * alpha_re;
      } else {
        out[e] = sum[e] * alpha_re - sum[e + 1] * alpha_im;
        out[e + 1] = sum[e + 1] * alpha_re + sum[e] * alpha_im;
      }
    }
    float *const p = place(x);
    if (!beta_zero) {
#pragma unroll
      for (int e = 0; e < U; e += NC) {
        if constexpr (!CPLX) {
          out[e] += args.beta_re * old[x][e];
        } else {
          out[e] += args.beta_re * old[x][e] - args.beta_im * old[x][e + 1];
          out[e + 1] += args.beta_im * old[x][e] + args.beta_re * old[x][e + 1];
        }
      }
    }
    if (full) {
      *reinterpret_cast<unit_t *>(p) = out;
    } else {
#pragma unroll
      for (int e = 0; e < U; e++)
        if (inside(x, e / NC)) p[e] = out[e];
    }
  }
}

__device__ inline bool kwaves_accepts(const int flag, const uint32_t mask) { return ((1u << (flag & 31)) & mask) != 0; }

template <class Cfg>
__global__ __launch_bounds__(Cfg::NT)
__attribute__((amdgpu_waves_per_eu(Cfg::OCC, Cfg::OCC))) void kwaves_gemm_tcec_kernel(const GemmArgs args) {
  if (args.launch_flag != nullptr && !kwaves_accepts(*args.launch_flag, args.flag_accept_mask)) return;
  kwaves_product<Cfg>(args);
}

// Both of AUTO's candidates, on the same tile: the launch flag says which product a
// workgroup computes, instead of a launch each of which one finds nothing to do.  What
// bounds a call this small is the boundaries between its kernels: statistics, decision
// and one product instead of two.  us, whole calls, decided for FP16TCEC / bf16x3: 64^3
// 8.9 -> 7.3 / 10.7 -> 8.8, 512^3 NN 15.5 -> 13.9 / 21.4 -> 19.5, 1200^3 NN 41.4 -> 37.2 /
// 58.8 -> 54.2; complex 128^3 12.3 -> 11.0 / 16.6 -> 14.5, 512^3 18.9 -> 17.6 / 27.0 -> 25.0.
template <class CfgA, class CfgB>
__global__ __launch_bounds__(CfgA::NT)
__attribute__((amdgpu_waves_per_eu(CfgA::OCC < CfgB::OCC ? CfgA::OCC : CfgB::OCC, CfgA::OCC < CfgB::OCC ? CfgA::OCC : CfgB::OCC)))
void kwaves_either_gemm_tcec_kernel(const GemmArgs args, const uint32_t accept_a, const uint32_t accept_b) {
  static_assert(CfgA::NT == CfgB::NT && CfgA::BM == CfgB::BM && CfgA::BN == CfgB::BN, "one grid for both");
  const int flag = *args.launch_flag;
  if (kwaves_accepts(flag, accept_a)) kwaves_product<CfgA>(args);
  else if (kwaves_accepts(flag, accept_b)) kwaves_product<CfgB>(args);
}
} // namespace cumpsgemm_amd
