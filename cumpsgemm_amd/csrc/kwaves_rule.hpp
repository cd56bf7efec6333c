// Which products the small-product kernel (gemm_kwaves.hpp) takes and with which
// tile.  Host arithmetic on sizes and layouts alone.
#pragma once
#include <cstdint>
#include <initializer_list>

namespace cumpsgemm_amd {

constexpr int kKWavesForms = 5; // tiles per precision, real or complex
constexpr int kKWavesAlone = 4; // the form for one workgroup on a CU
constexpr int kKWavesFourWaves = 2; // real: the tile of the eight-wave form with four
constexpr unsigned kKWavesModuleId = 6; // what used_kernel_module_id reports (0 - 4 are the tile classes, 5 the narrow kernel)

// Tile and waves of a form, workgroups that a CU holds at once, and the time of a
// tile in us: `fill` for prologue, sums and write-out, `step` per K-step of a wave,
// longer by `beside` for every other workgroup on the CU; `once` is paid by the first
// round alone.  bm == 0: no such form.
struct KWavesForm {
  int bm, bn, waves, resident;
  double fill, step, beside, once;
};
// ... and what the plan of the tiled kernels takes: us = tiled0 + tiled_per_step *
// cost, the plan's cost in K-steps of a 256 x 128 tile, + tiled_split if K is split.
//
// All of it fitted on 188 products (84 real, m and n 64 - 4096, K 64 - 8192, 60 real
// batches of up to 1024 matrices of 32 - 640, 44 complex; four layouts, padded, with
// and without C), each timed with every form and tiled, in every precision; the forms
// with two waves to a SIMD on 640 others, the first and the last form again on 3200 (without
// `once` a short K of 257 - 512 tiles went to 64 x 64 that is faster on 32 x 32 or tiled,
// bf16x2 512 x 2254 x 128 NN 6.1 us, 64 x 64 7.5; with it in every round batches went back to
// the tiled kernels, 320^3 x 116 bf16x2 NT 47 us, tiled 86).  On 3900 other products, of which
// the rule takes 2937: time over the tiled time, geometric mean (the fastest side by hindsight),
//               real         real batches  complex      complex batches
//   FP16TCEC    0.65 (0.63)  0.69 (0.67)   0.53 (0.52)  0.57 (0.57)
//   bf16x3      0.61 (0.60)  0.67 (0.65)   0.47 (0.47)  0.62 (0.62)
//   FP16TC      0.60 (0.59)  0.67 (0.66)   0.46 (0.46)  0.51 (0.51)
//   bf16x2      0.69 (0.67)  0.68 (0.65)   0.57 (0.55)  0.61 (0.60)
// 2.7 % are slower than tiled by 5 %, 1.5 % by 10 %, the worst takes 1.31 times as long; 400 AUTO
// calls 0.77 real, 0.71 complex, none slower by 2 %.
// Forms of one wave to a SIMD, which has the registers for two sets of fragments or for a 64 x 32 complex tile, are the
// faster ones where a CU has no second workgroup anyway.  2100 real and 1500 complex products, geometric mean: real
// FP16TCEC, against two waves on a SIMD, up to K = 256 1.04, 512 0.99, 1024 0.97, 2048 0.96, 4096 0.94 (FP16TC and
// bf16x2 1.00, 0.98: left out); complex against the faster of its other two, where those are two to a CU: K <= 256
// 1.2 - 1.3, 1024 FP16TC 0.93, others 1.06 - 1.09, beyond 2048 0.83 and 0.94 - 0.95.
// (Tried beside these and left out: 64 x 64 with eight waves at two to a SIMD, up to
// 10 % faster than four where K >= 2048 and 256 tiles or fewer, 0 - 4 % else, no better
// over the 640; 64 x 32 and 32 x 64 with four and eight waves, 64 x 64 with one and two,
// within 1 %; 128 x 64 spills.  Complex with one or two waves: batches are faster tiled.)
struct KWavesModel {
  KWavesForm form[kKWavesForms];
  double tiled0, tiled_per_step, tiled_split;
};
// `prec`: 0 FP16TCEC, 1 FP16TC, 2 bf16x3, 3 bf16x2
inline const KWavesModel &kwaves_model(int prec, bool cplx) {
  static const KWavesModel real[4] = {
      {{{64, 64, 4, 2, 3.11, 1.07, 0.72, 0.5}, {32, 32, 8, 2, 1.13, 0.88, 0.71}, {32, 32, 4, 4, 1.08, 0.50, 0.74}, {32, 32, 1, 16, 2.4, 0.37, 0.22}, {64, 64, 4, 1, 3.6, 0.93, 0.0}}, 4.1, 1.63, -2.1},
      {{{64, 64, 4, 2, 2.10, 0.67, 1.25, 1.0}, {32, 32, 8, 2, 0.98, 0.87, 0.55}, {32, 32, 4, 4, 1.00, 0.47, 0.67}, {32, 32, 1, 16, 2.4, 0.23, 0.37}}, 4.8, 1.27, 0.9},
      {{{64, 64, 4, 1, 3.6, 1.65, 0.0}, {32, 32, 8, 1, 1.62, 1.17, 0.0}, {32, 32, 4, 3, 1.29, 0.76, 0.55}, {32, 32, 1, 12, 2.2, 0.68, 0.17}}, 2.5, 2.29, -2.4},
      {{{64, 64, 4, 2, 2.78, 0.94, 0.93, 0.97}, {32, 32, 8, 2, 1.12, 0.87, 0.78}, {32, 32, 4, 4, 1.09, 0.50, 0.73}, {32, 32, 1, 16, 2.5, 0.39, 0.21}}, 4.0, 1.61, -1.6}};
  static const KWavesModel complex[4] = {
      {{{32, 32, 4, 2, 1.50, 1.02, 0.94}, {32, 32, 8, 1, 1.15, 1.77, 0.0}, {}, {}, {64, 32, 4, 1, 3.7, 1.75, 0.0}}, 2.8, 2.05, -5.4},
      {{{32, 32, 4, 2, 1.09, 0.51, 1.72}, {32, 32, 8, 1, 0.74, 1.28, 0.0}, {}, {}, {64, 32, 4, 1, 2.5, 1.12, 0.0}}, 3.6, 1.50, -3.4},
      {{{32, 32, 4, 1, 2.3, 1.71, 0.0}, {}, {}, {}}, 0.9, 3.83, -14.3},
      {{{32, 32, 4, 2, 1.55, 0.97, 1.06}, {32, 32, 8, 1, 0.99, 1.85, 0.0}, {}, {}, {64, 32, 4, 1, 3.8, 1.80, 0.0}}, 3.1, 2.09, -6.1}};
  return (cplx ? complex : real)[prec];
}

struct KWavesProblem {
  bool cplx, a_kc, b_kc; // operand stored K-contiguous
  uint64_t m, n, k, batch, lda, ldb;
};

inline uint64_t kwaves_tiles(const KWavesForm &f, const KWavesProblem &p) {
  return (p.m + f.bm - 1) / f.bm * ((p.n + f.bn - 1) / f.bn) * p.batch;
}

inline double kwaves_time(const KWavesForm &f, const KWavesProblem &p, unsigned cus) {
  const uint64_t steps = ((p.k + 31) / 32 + f.waves - 1) / f.waves;
  const uint64_t tiles = kwaves_tiles(f, p), per_cu = (tiles + cus - 1) / cus;
  const uint64_t rounds = per_cu <= (uint64_t)f.resident ? 1 : (per_cu + f.resident - 1) / f.resident;
  const double beside = (double)((per_cu < (uint64_t)f.resident ? per_cu : (uint64_t)f.resident) - 1);
  // Workgroups of one wave hardly run in rounds: as one ends the next begins.  Half way between whole rounds and none, on
  // 350 drawn batches against whole ones: 11 take 0.55 - 0.96 of the time (416^3 x 35 bf16x2 TN 64 -> 35 us, 262^3 x 152
  // FP16TCEC NT 88 -> 69, 128 x 36 x 102 x 870 bf16x3 NN 41 -> 30), 4 are slower by 3 - 5 %; with no rounds at all two of
  // 150 by 10 - 13 % (256^3 x 77 FP16TCEC TT 18.5 -> 21.0).
  double in_rounds = (double)rounds;
  if (f.waves == 1 && rounds > 1) in_rounds = 0.5 * ((double)tiles / ((double)cus * f.resident) + in_rounds);
  return 2.2 + f.once + in_rounds * (f.fill + (double)steps * f.step * (1.0 + f.beside * beside));
}

// Whether a form can serve the product at all.
inline bool kwaves_can_serve(const KWavesForm &f, const KWavesProblem &p) {
  if (f.bm == 0 || p.k == 0) return false;
  // a row-contiguous operand is read 16 bytes a lane: its tile must lie inside the matrix
  if ((!p.a_kc && p.m < (uint64_t)f.bm) || (!p.b_kc && p.n < (uint64_t)f.bn)) return false;
  // byte offsets inside a tile's K-step are 31 bits
  auto fits = [&](bool kc, uint64_t rows, uint64_t ld) {
    return ld < 0x80000000ull && ((kc ? rows : 32) * ld + (kc ? 32 : rows)) * (p.cplx ? 8 : 4) < 0x7fffffffull;
  };
  if (!fits(p.a_kc, (uint64_t)f.bm, p.lda) || !fits(p.b_kc, (uint64_t)f.bn, p.ldb)) return false;
  // threads of a launch along one axis (sizes below 2^31, at most 65535 matrices: see run_gemm)
  if ((p.m + f.bm - 1) / f.bm * ((p.n + f.bn - 1) / f.bn) >= (1ull << 32)) return false;
  return kwaves_tiles(f, p) * (uint64_t)f.waves * 64 < (1ull << 32);
}

// The form that serves the product, or -1: the tiled kernels do.  `tiled_steps`,
// `tiled_split`: the tiled plan's cost as above, whether it splits K.  `asked`: -1, or
// 0 never, 1 ... this form wherever it can.
inline int choose_kwaves_form(int prec, const KWavesProblem &p, unsigned cus, double tiled_steps, bool tiled_split,
                              int asked) {
  if (asked == 0) return -1;
  const KWavesModel &model = kwaves_model(prec, p.cplx);
  // (complex tiles take 6 % longer per step with two row-contiguous operands, 7 % less with none)
  const double layout = !p.cplx ? 1.0 : p.a_kc && p.b_kc ? 0.93 : !p.a_kc && !p.b_kc ? 1.06 : 1.0;
  const double tiled = model.tiled0 + layout * model.tiled_per_step * tiled_steps + (tiled_split ? model.tiled_split : 0.0);
  // Both sides are estimates, within 10 - 30 % of the times: with 1.0 here the number of products that get more than
  // 3 % slower doubles and the mean stays; with 0.8 (long ones 0.7) a third of the losses is left, and the mean of 10000
  // real products (drawn for the forms of one wave to a SIMD) goes from 0.643 to 0.660 of the tiled time.  Long ones have
  // less to gain: 0.8.  (Complex ones: 0.95; 3 of 240 slower by 5 %, with 1.0 for short ones 5.)
  double best_time = (p.cplx ? 0.95 : tiled > 30.0 ? 0.8 : 0.9) * tiled;
  int best = -1;
  for (int i = 0; i < kKWavesForms; i++) {
    const KWavesForm &f = model.form[i];
    // (a small product's call is bound by the host: what rules a form out without a division comes first)
    if (i == kKWavesAlone && asked < 0 && !p.cplx && p.k <= 512) continue;
    if (!kwaves_can_serve(f, p)) continue;
    if (asked > 0) {
      if (asked == i + 1) return i;
      continue;
    }
    // More than a short K, and more than two rounds of workgroups: bound by what a tile this small reads, which the fit
    // misses.  With more than 1024 tiles of 64 x 64, 70 products take 1.05 - 1.13 of the tiled time (5256 x 805 x 545 FP16TCEC
    // NT 35.7 us, tiled 34.1; 2216 x 1984 x 3200 TN 126, 113).
    const uint64_t per_cu = (kwaves_tiles(f, p) + cus - 1) / cus;
    if (per_cu > 2ull * f.resident && p.k > 512) continue;
    if (i == kKWavesAlone && per_cu > 1) continue;
    // (complex, more than one round of tiles: the fit is up to 10 % short.  FP16TC 1000^3 NN 23.2 us tiled, 26.1 here.)
    const bool rounds = p.cplx && per_cu > (uint64_t)f.resident;
    const double t = kwaves_time(f, p, cus) * (rounds ? 1.1 : 1.0);
    if (t < best_time) {
      best = i;
      best_time = t;
    }
  }
  if (asked < 0 && !p.cplx && p.batch == 1 && best == 0 && model.form[0].resident == 2 && p.k > 512 && (p.a_kc || p.b_kc) &&
      (kwaves_tiles(model.form[0], p) + cus - 1) / cus == 3) {
    // Three tiles of 64 x 64 on a CU that holds two: a round for the third, and where the estimates still send them here
    // that of the tiled kernels is too dear.  16 drawn products, 513 - 600 tiles: 1.12 of the tiled time, 0.90 - 1.41
    // (3392 x 591 x 2932 FP16TCEC TT 106 us, tiled 76).  Not with two row-contiguous operands (7: 0.91), nor with four
    // tiles (47: 0.84), nor batches, whose tiled estimate has not that fault (160 x 288 x 640 x 47 FP16TC NN 31 us, tiled 49).
    best = -1;
  }
  if (asked < 0 && p.cplx && best >= 0 && model.form[best].waves == 8 &&
      kwaves_tiles(model.form[best], p) > (uint64_t)cus * model.form[best].resident) {
    // Complex tiles with eight waves as well: beyond one round the fit makes them too cheap.  670 products of more tiles
    // than CUs: 1.16 - 1.3 times the faster of the other two forms.  Of 23 sent to them four waves take 0.74 - 0.89 of
    // that, and 0.82 of the tiled time, two of them 1.05 and 1.12 (us, eight / four waves / tiled: FP16TC 1088 x 512 x 480 TN
    // 13.5, 10.8, 11.3; 768 x 768 x 203 NN 11.0, 8.5, 11.0; bf16x2 960 x 576 x 448 NN 18.3, 16.1, 14.4).
    best = 0;
  }
  if (asked < 0 && !p.cplx && best >= 0 && model.form[best].waves == 8) {
    // Eight waves on a tile pay while all workgroups are on the chip at once: the fit makes their second round too cheap.
    // 36 of 10000 drawn products were sent to one.  The 32 up to K = 512 take 0.72 - 1.01 of the time with four waves on
    // the same tile (2560 x 586 x 224 FP16TC NN, us: 9.1, four waves 6.8, tiled 6.7; 231^3 x 22 NT 11.4, 8.9, 11.1).
    // Beyond, the tiled kernels are faster where they split K (736 x 1349 x 8128 NN 147, four waves 157, tiled 88), but
    // not where AUTO keeps them from it (2763 x 347 x 5808 NN 122, tiled 148).
    const uint64_t per_cu = (kwaves_tiles(model.form[best], p) + cus - 1) / cus;
    if (per_cu > (uint64_t)model.form[best].resident) {
      if (p.k <= 512) best = kKWavesFourWaves;
      else if (tiled_split) best = -1;
    } else if (per_cu > 1 && p.k >= 2560 && tiled_split && !p.a_kc && !p.b_kc) {
      // Two of them on a CU read a long K of two row-contiguous operands slower than the fit has it: 20 of 17000 drawn
      // products, 19 of them 1.05 - 1.63 times as long as with K split (1090 x 256 x 3360 FP16TC 34.0 us, tiled 22.3;
      // FP16TCEC 528 x 528 x 2880 24.3, 22.3).  K 2048 - 2559: 8 of 18 longer, 7 shorter; other layouts level.
      best = -1;
    }
  }
  return best;
}

// AUTO's candidates (bf16x3, FP16TCEC) where both go to this kernel with the forms given: which of the two forms one
// launch takes for both, or -1: a launch each.  Apart, a call pays for the launch that finds nothing to do (1.7 us in a
// graph, 3 - 5 in a loop of calls); together they hold as many workgroups on a CU as the larger of them, which must
// cost neither more than that (complex 640^3, 400 tiles: FP16TCEC runs two to a CU apart, 26.5 us a call, and one
// together, 27.3).
inline int choose_kwaves_either_form(const KWavesProblem &p, unsigned cus, int form_bf16, int form_fp16) {
  constexpr double LAUNCH = 1.7;
  if (!p.cplx && form_fp16 == kKWavesAlone) form_fp16 = 0; // (the same tile and waves; 1 - 6 % of the product for a launch)
  if (form_bf16 < 0 || form_fp16 < 0) return -1;
  const KWavesModel &ma = kwaves_model(2, p.cplx), &mb = kwaves_model(0, p.cplx);
  const double apart_a = kwaves_time(ma.form[form_bf16], p, cus), apart_b = kwaves_time(mb.form[form_fp16], p, cus);
  double best_time = apart_a + apart_b + 2 * LAUNCH;
  int best = -1;
  for (const int i : {form_fp16, form_bf16}) {
    KWavesForm a = ma.form[i], b = mb.form[i];
    if (a.bm == 0 || b.bm == 0 || a.waves != b.waves || !kwaves_can_serve(a, p)) continue;
    a.resident = b.resident = a.resident < b.resident ? a.resident : b.resident;
    if (a.waves == 8 && (kwaves_tiles(a, p) + cus - 1) / cus > (uint64_t)a.resident) continue; // (one round only, as above)
    const double ta = kwaves_time(a, p, cus), tb = kwaves_time(b, p, cus);
    if (ta < apart_a + LAUNCH && tb < apart_b + LAUNCH && ta + tb < best_time) {
      best = i;
      best_time = ta + tb;
    }
  }
  return best;
}
} // namespace cumpsgemm_amd
