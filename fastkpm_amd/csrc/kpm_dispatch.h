// kpm_dispatch.h -- host-side table of kernel instantiations.
//
// One KSet holds the host stubs of every kernel for one (storage type S,
// real/complex, block size B, lanes per group L, packets per lane KQ).  The
// instantiations live in four translation units (kpm_inst_{d,f}{c,r}.hip) that
// compile in parallel; kpm_capi.hip looks sets up by runtime parameters.
#pragma once
#include <hip/hip_runtime.h>

namespace fkd {

template <typename S>
struct RSource;

template <class S>
struct KSet {
  void (*mom)(const int*, const int*, const S*, const S*, const S*, S*, int, int, int, double,
              double, double*, int, RSource<S>) = nullptr;
  // mom without the early load of the own rows (step_fn; 8-row blocks on a wave)
  void (*mom_late)(const int*, const int*, const S*, const S*, const S*, S*, int, int, int,
                   double, double, double*, int, RSource<S>) = nullptr;
  // mom for patterns bound by one long row (step_fn; real FP64 4-row blocks)
  void (*mom_long)(const int*, const int*, const S*, const S*, const S*, S*, int, int, int,
                   double, double, double*, int, RSource<S>) = nullptr;
  void (*xi)(const int*, const int*, const S*, const S*, const S*, S*, double*, int, int, int,
             double, double, double, double, int, int) = nullptr;
  // xi with its column passes side by side (blocks of 4 and 8)
  void (*xi_apart)(const int*, const int*, const S*, const S*, const S*, S*, double*, int, int, int,
                   double, double, double, double, int, int) = nullptr;
  void (*ad_fused)(const int*, const int*, const S*, const S*, const S*, const S*, const S*, S*,
                   S*, double*, int, int, int, double, double, double, double, double,
                   double, int) = nullptr;
  void (*ad_plain)(const int*, const int*, const S*, const S*, const S*, const S*, const S*, S*,
                   S*, double*, int, int, int, double, double, double, double, double,
                   double, int) = nullptr;
  // backward steps reading alpha_{m-1} from the forward table (D fused on H's
  // pattern, or not)
  void (*ad_stored)(const int*, const int*, const S*, const S*, const S*, const S*, const S*,
                    const S*, S*, double*, int, int, int, double, double, double, double, double,
                    double, int) = nullptr;
  void (*ad_stored_plain)(const int*, const int*, const S*, const S*, const S*, const S*,
                          const S*, const S*, S*, double*, int, int, int, double, double, double,
                          double, double, double, int) = nullptr;
  void (*outer_ss)(const int*, const int*, const S*, const S*, double*, int, int, int,
                   double) = nullptr;
  void (*outer_sd)(const int*, const int*, const S*, const double*, double*, int, int, int,
                   double) = nullptr;
  void (*outer_ds)(const int*, const int*, const double*, const S*, double*, int, int, int,
                   double) = nullptr;
  // matrix-core kernels (complex 8x8 blocks only; null otherwise), same
  // signatures as mom / ad_fused / ad_plain
  void (*mfma_mom)(const int*, const int*, const S*, const S*, const S*, S*, int, int, int, double,
                   double, double*, int, RSource<S>) = nullptr;
  void (*mfma_ad_fused)(const int*, const int*, const S*, const S*, const S*, const S*, const S*,
                        S*, S*, double*, int, int, int, double, double, double, double, double,
                        double, int) = nullptr;
  void (*mfma_ad_plain)(const int*, const int*, const S*, const S*, const S*, const S*, const S*,
                        S*, S*, double*, int, int, int, double, double, double, double, double,
                        double, int) = nullptr;
  // row-resident matrix-core variants (rows of at most 8 blocks, vectors
  // under 4 GiB): forward step, fused autodiff step
  void (*mfma_mom_rr)(const int*, const int*, const S*, const S*, const S*, S*, int, int, int,
                      double, double, double*, int, RSource<S>) = nullptr;
  void (*mfma_ad_rr)(const int*, const int*, const S*, const S*, const S*, const S*, const S*,
                     S*, S*, double*, int, int, int, double, double, double, double, double,
                     double, int) = nullptr;
  // the same for rows of at most 7 blocks (no padding slot)
  void (*mfma_mom_rr7)(const int*, const int*, const S*, const S*, const S*, S*, int, int, int,
                       double, double, double*, int, RSource<S>) = nullptr;
  void (*mfma_ad_rr7)(const int*, const int*, const S*, const S*, const S*, const S*, const S*,
                      S*, S*, double*, int, int, int, double, double, double, double, double,
                      double, int) = nullptr;
  // FP32 only: the row-resident forward and autodiff steps on pairs of column
  // tiles (the padded width a multiple of 16 packets), 8 and 7 block slots
  void (*mfma_mom_rr2)(const int*, const int*, const S*, const S*, const S*, S*, int, int, int,
                       double, double, double*, int, RSource<S>) = nullptr;
  void (*mfma_mom_rr2_7)(const int*, const int*, const S*, const S*, const S*, S*, int, int, int,
                         double, double, double*, int, RSource<S>) = nullptr;
  void (*mfma_ad_rr2)(const int*, const int*, const S*, const S*, const S*, const S*, const S*,
                      S*, S*, double*, int, int, int, double, double, double, double, double,
                      double, int) = nullptr;
  void (*mfma_ad_rr2_7)(const int*, const int*, const S*, const S*, const S*, const S*, const S*,
                        S*, S*, double*, int, int, int, double, double, double, double, double,
                        double, int) = nullptr;
  // the backward steps reading alpha_{m-1} from the forward table (signature of
  // ad_stored): general (D fused on H's pattern, or not), row-resident for
  // rows of at most 8 and 7 blocks, FP32 on pairs of column tiles
  void (*mfma_ads[6])(const int*, const int*, const S*, const S*, const S*, const S*, const S*,
                      const S*, S*, double*, int, int, int, double, double, double, double, double,
                      double, int) = {};
  // outer_ss on the matrix cores (padded width a multiple of 8 packets)
  void (*mfma_outer)(const int*, const int*, const S*, const S*, double*, int, int, int,
                     double) = nullptr;
  int B = 0, L = 0, KQ = 0;
};

// The forward step of a geometry on nb block rows; long_row: one long row sets its time.
// Such a row takes two real 4x4 FP64 blocks a batch instead of one (moments of M = 40, us,
// one / two, rows of 5 blocks and one of 65, S = 24: 2000 rows 630 / 534, 9000 716 / 592,
// 30000 889 / 656; one of 25: 287 / 265, 350 / 310; complex and smaller blocks lost up to
// 17 % by it at 25).  With 8-row blocks on a wave a row, the early load of the own rows
// costs one of four waves a SIMD: it pays while every row's wave is resident either way,
// two on each of 1024 SIMDs.  Moments of M = 64 with and without, real FP64 x 8 x 128
// (us): 32x32 369 / 431, 10^3 584 / 629, 45x45 627 / 627; 46x46 717 / 698, 16^3 1419 / 1099,
// 20^3 2303 / 2057.
constexpr int kEarlyRows = 2048;
template <class S>
auto step_fn(const KSet<S>& ks, int nb, bool long_row) {
  if (long_row && ks.mom_long != nullptr) return ks.mom_long;
  return nb > kEarlyRows && ks.mom_late != nullptr ? ks.mom_late : ks.mom;
}

// Entries of mfma_ads.
enum MfmaAds { ADS_FUSED = 0, ADS_PLAIN = 1, ADS_RR = 2, ADS_RR7 = 3, ADS_RR2 = 4, ADS_RR2_7 = 5 };

// Geometries compiled for each block size (lanes per group, packets per lane).
struct GeomChoice {
  int L, KQ;
};
// Block sizes with compiled kernels.
inline bool block_supported(int b) { return b == 1 || b == 2 || b == 4 || b == 8; }
// List of (L, KQ) compiled for block size b; returns the count.
int geometries_for_block(int b, GeomChoice* out, int cap);

bool find_kset_dc(int B, int L, int KQ, KSet<double>* out);  // double, complex
bool find_kset_dr(int B, int L, int KQ, KSet<double>* out);  // double, real
bool find_kset_fc(int B, int L, int KQ, KSet<float>* out);   // float, complex
bool find_kset_fr(int B, int L, int KQ, KSet<float>* out);   // float, real

}  // namespace fkd

// The list of compiled (B, L, KQ) geometries.  B = 1, 2 take up to 4 packets
// per lane; B = 4 up to 2; B = 8 one (its accumulators are 8x larger).  One
// packet per lane keeps the register count (and so the occupancy) of the
// fused autodiff step low at a given pass width; four packets over eight
// lanes gives it longer loads per lane (the FP32 autodiff step at S = 64).
// For 2x2 blocks, two packets over a whole wave carry 128 FP64 columns in one
// pass with the row wave-uniform (scalar row offsets, indices and H) at 3
// waves per SIMD in the autodiff step, where 32 lanes x 4 packets hold 2 (the
// tuner takes it for C3's FP64 forward step, with the lattice row order).
#define FKD_FOR_EACH_GEOMETRY(X)                                                       \
  X(1, 4, 1) X(1, 4, 2) X(1, 8, 2) X(1, 8, 4) X(1, 16, 1) X(1, 16, 2) X(1, 16, 4)      \
  X(1, 32, 1) X(1, 32, 4) X(1, 64, 1) X(1, 64, 4)                                      \
  X(2, 4, 1) X(2, 4, 2) X(2, 8, 2) X(2, 8, 4) X(2, 16, 1) X(2, 16, 2) X(2, 16, 4)      \
  X(2, 32, 1) X(2, 32, 4) X(2, 64, 1) X(2, 64, 2) X(2, 64, 4)                          \
  X(4, 4, 1) X(4, 4, 2) X(4, 8, 2) X(4, 16, 1) X(4, 16, 2) X(4, 32, 1) X(4, 32, 2)     \
  X(4, 64, 1) X(4, 64, 2)                                                              \
  X(8, 4, 1) X(8, 8, 1) X(8, 16, 1) X(8, 32, 1) X(8, 64, 1)
