// kpm_resident.h -- whole-recursion kernels for small lattices.
//
// The probe columns of the recursions are independent, so where one column of
// the vector fits the LDS twice a workgroup runs a whole recursion on its own
// column: two LDS buffers hold the vectors of the current and the previous
// order, a step ends with one workgroup barrier, and nothing is launched or
// synchronised between steps.  A thread owns RPT block rows; the first DREG
// blocks of each stay in its registers for the whole recursion, further
// blocks are read from the L2 every step (packed so that consecutive threads
// read consecutive 16-byte packets).
//
// Every vector is also written, column by column, to a table in HBM
// ([order][column][orbital row]); what needs sums over columns or orders runs
// afterwards on the whole chip: the moment dots (k_res_dots), D as one sum
// over all orders and columns (k_res_outer, no read-modify-write per step),
// the table sums of stoch_matrix (k_table_sums).
//
// A row's products and the axpby are the operations of the step kernels in
// kpm_kernels.h, in FP32 in the same order, so that the vectors are bitwise
// theirs (FP64 takes the diagonal block first); the dots and D accumulate in FP64.
#pragma once
#include "kpm_kernels.h"

namespace fkd {

constexpr int RES_T = 512;  // most threads of a workgroup (256 VGPRs each)

// Geometry of one (type, block size, block rows per thread).
template <typename S, bool CX, int B, int RPT>
struct ResGeo {
  static constexpr int HS = CX ? 2 : 1;
  static constexpr int NV = B * HS;      // scalars of one block row in one column
  static constexpr int NH = B * B * HS;  // scalars of one H block
  static constexpr int BYTES = NV * (int)sizeof(S);
  static constexpr int HB = NH * (int)sizeof(S);
  static constexpr int PB = HB < 16 ? HB : 16;  // bytes of one packet of an H block
  static constexpr int PN = PB / (int)sizeof(S);
  static constexpr int PK = HB / PB;            // packets of an H block
  // Blocks of each row kept in registers by a kernel that holds VL values per
  // orbital row across the products: what VL vectors and about 44 VGPRs of
  // addresses and temporaries (52 where other blocks are streamed) leave of
  // 256 (a few instances spill up to 48 bytes; six VGPRs less for ST lost more:
  // 45x45 x 2 FP64 forward step 2.4 -> 3.1 us).  Loading the streamed blocks one ahead cost the
  // registers of two blocks and lost: 45x42 x 2 FP32 forward step 1.9 -> 2.7 us.
  template <int VL, bool ST>
  static constexpr int dreg() {
    constexpr int d = ((ST ? 204 : 212) - VL * RPT * (BYTES / 4)) / (RPT * (HB / 4 + 1));
    return d < 0 ? 0 : d > 16 ? 16 : d;
  }
};
constexpr int RES_VL_FWD = 2, RES_VL_XI = 2, RES_VL_BWD = 5;
// Two more vectors with RES_OWN.
constexpr int res_vl(int vl, int mode) { return mode == 2 ? vl + 2 : vl; }
// FP64 with streamed blocks keeps the registers of one more vector free: 9^3 x 2
// (two rows a thread) streamed two blocks of seven slower than three.
template <typename S, bool ST>
constexpr int RES_VL_BWD_LA = ST && sizeof(S) == 8 ? 3 : 2;

// N scalars at p (16-byte packets where the size allows; a smaller element is
// one access).
template <typename S, int N>
__device__ __forceinline__ void ldn(const S* p, S (&v)[N]) {
  constexpr int B = N * (int)sizeof(S);
  constexpr int W = (B % 16 == 0 ? 16 : B) / (int)sizeof(S);
  typedef S V __attribute__((ext_vector_type(W)));
  if constexpr (W == 1) {
    v[0] = p[0];
  } else {
#pragma unroll
    for (int c = 0; c < N / W; c++) {
      const V t = *reinterpret_cast<const V*>(p + c * W);
#pragma unroll
      for (int e = 0; e < W; e++) v[c * W + e] = t[e];
    }
  }
}

template <typename S, int N>
__device__ __forceinline__ void stn(S* p, const S (&v)[N]) {
  constexpr int B = N * (int)sizeof(S);
  constexpr int W = (B % 16 == 0 ? 16 : B) / (int)sizeof(S);
  typedef S V __attribute__((ext_vector_type(W)));
  if constexpr (W == 1) {
    p[0] = v[0];
  } else {
#pragma unroll
    for (int c = 0; c < N / W; c++) {
      V t;
#pragma unroll
      for (int e = 0; e < W; e++) t[e] = v[c * W + e];
      *reinterpret_cast<V*>(p + c * W) = t;
    }
  }
}

// H as the resident kernels read it: block d of the row owned by thread slot
// i (i < nt) as PK packets at (d * PK + k) * nt + i, and the LDS byte offset
// of its column block (FP64: block 0 is the diagonal one); rows with fewer blocks,
// and slots past the last row, are filled with zero blocks on the zero vector
// block nb.
template <typename S>
struct ResH {
  const S* val;
  const int* off;
  int nb, nt, deg;
};

// LDS bytes of one vector buffer: nb block rows and the zero block.
template <int BYTES>
__host__ __device__ constexpr int res_buf_bytes(int nb) {
  return ((nb + 1) * BYTES + 15) / 16 * 16;
}

template <typename S, bool CX, int B>
__global__ __launch_bounds__(WG) void k_res_pack_H(const int* __restrict__ rp,
                                                   const int* __restrict__ ci,
                                                   const S* __restrict__ hv, int nb, int nt, int deg,
                                                   S* __restrict__ val, int* __restrict__ off) {
  using GE = ResGeo<S, CX, B, 1>;
  const int n = nt * deg;
  for (int w = blockIdx.x * WG + threadIdx.x; w < n; w += gridDim.x * WG) {
    const int d = w / nt, i = w % nt;
    int p = i < nb ? rp[i] + d : 0;
    const bool live = i < nb && p < rp[i + 1];
    if (sizeof(S) == 8 && live) {  // FP64: the diagonal block first, then the others in order
      int pd = rp[i];
      while (ci[pd] != i) pd++;  // every row has one (set_H requires it)
      if (p <= pd) p = d == 0 ? pd : p - 1;
    }
    off[w] = (live ? ci[p] : nb) * GE::BYTES;
#pragma unroll
    for (int k = 0; k < GE::PK; k++)
#pragma unroll
      for (int e = 0; e < GE::PN; e++)
        val[((size_t)(d * GE::PK + k) * nt + i) * GE::PN + e] =
            live ? hv[(size_t)p * GE::NH + k * GE::PN + e] : S(0);
  }
}

// What a kernel does with the blocks and vectors its registers do not have to
// hold.  RES_ST: blocks past DREG are streamed.  RES_OWN (FP64, every block in
// registers): the thread's own rows of the last two vectors stay in registers
// too, so the diagonal block and the recursion's second term read no LDS: five
// accesses of a vector element instead of seven on a 2-D lattice (M = 128: 16x16 x 2
// moments 54.5 -> 50.5 us, autodiff_matrix 125 -> 119).
enum ResMode { RES_REG = 0, RES_ST = 1, RES_OWN = 2 };

// The registers a thread keeps of H.
template <typename S, bool CX, int B, int RPT, int VL, int MODE>
struct ResRegs {
  static constexpr bool ST = MODE == RES_ST, OWN = MODE == RES_OWN;
  using GE = ResGeo<S, CX, B, RPT>;
  static constexpr int DREG = GE::template dreg<VL, ST>();
  static constexpr int DA = DREG > 0 ? DREG : 1;
  S h[RPT][DA][GE::NH];
  int off[RPT][DA];

  static __device__ __forceinline__ void block(const ResH<S>& H, int d, int i, S (&v)[GE::NH]) {
#pragma unroll
    for (int k = 0; k < GE::PK; k++) {
      S t[GE::PN];
      ldn<S, GE::PN>(H.val + ((size_t)(d * GE::PK + k) * H.nt + i) * GE::PN, t);
#pragma unroll
      for (int e = 0; e < GE::PN; e++) v[k * GE::PN + e] = t[e];
    }
  }

  __device__ __forceinline__ void load(const ResH<S>& H) {
#pragma unroll
    for (int d = 0; d < DREG; d++)
#pragma unroll
      for (int k = 0; k < RPT; k++) {
        const int i = k * blockDim.x + threadIdx.x;
        if (d < H.deg) {
          block(H, d, i, h[k][d]);
          off[k][d] = H.off[d * H.nt + i];
        } else {
#pragma unroll
          for (int e = 0; e < GE::NH; e++) h[k][d][e] = S(0);
          off[k][d] = H.nb * GE::BYTES;
        }
      }
  }

  static __device__ __forceinline__ void mac(S (&acc)[GE::NV], const S (&hh)[GE::NH],
                                             const S (&x)[GE::NV]) {
    constexpr int HS = GE::HS;
#pragma unroll
    for (int bj = 0; bj < B; bj++)
#pragma unroll
      for (int bi = 0; bi < B; bi++) {
        const int e = (bj * B + bi) * HS;
        cmac<CX, HS>(&acc[bi * HS], hh[e], CX ? hh[e + HS - 1] : S(0), &x[bj * HS]);
      }
  }

  template <int D0>
  __device__ __forceinline__ void group(int deg, const char* xb, const S (*own)[GE::NV],
                                        S (&acc)[RPT][GE::NV]) const {
    if constexpr (D0 < DREG) {
      constexpr int D1 = D0 + (D0 == 0 ? 5 : 2) < DREG ? D0 + (D0 == 0 ? 5 : 2) : DREG;
      if (D0 < deg) {
#pragma unroll
        for (int k = 0; k < RPT; k++) {
          S x[D1 - D0][GE::NV];
#pragma unroll
          for (int d = D0; d < D1; d++)
            if (!OWN || d > 0)
              ldn<S, GE::NV>(reinterpret_cast<const S*>(xb + off[k][d]), x[d - D0]);
#pragma unroll
          for (int d = D0; d < D1; d++) {
            if constexpr (OWN) {
              if (d == 0) {
                mac(acc[k], h[k][0], own[k]);
                continue;
              }
            }
            mac(acc[k], h[k][d], x[d - D0]);
          }
        }
        group<D1>(deg, xb, own, acc);
      }
    }
  }

  // acc[k] = (Hs x) of the thread's rows, x in LDS at xb (its own rows, with OWN,
  // in `own`)
  __device__ __forceinline__ void mul(const ResH<S>& H, const char* xb, const S (*own)[GE::NV],
                                      S (&acc)[RPT][GE::NV]) const {
#pragma unroll
    for (int k = 0; k < RPT; k++)
#pragma unroll
      for (int e = 0; e < GE::NV; e++) acc[k][e] = S(0);
    // whole groups without a branch, so that a group's LDS reads are in flight
    // together: five blocks (a 2-D lattice row), then pairs; blocks past the
    // row's end are zero on the zero vector block
    group<0>(H.deg, xb, own, acc);
    if constexpr (ST) {
      for (int d = DREG; d < H.deg; d++) {
#pragma unroll
        for (int k = 0; k < RPT; k++) {
          const int i = k * blockDim.x + threadIdx.x;
          S hh[GE::NH], x[GE::NV];
          block(H, d, i, hh);
          ldn<S, GE::NV>(reinterpret_cast<const S*>(xb + H.off[d * H.nt + i]), x);
          mac(acc[k], hh, x);
        }
      }
    }
  }
};

// Column s of the packed R (N x sp, row-major), one thread's block rows.
template <typename S, bool CX, int B, int RPT>
__device__ __forceinline__ void res_load_R(const S* __restrict__ R, int sp, int nb, int s,
                                           S (&r)[RPT][B * (CX ? 2 : 1)]) {
  constexpr int HS = CX ? 2 : 1;
#pragma unroll
  for (int k = 0; k < RPT; k++) {
    const int i = k * blockDim.x + threadIdx.x;
#pragma unroll
    for (int bi = 0; bi < B; bi++)
#pragma unroll
      for (int c = 0; c < HS; c++)
        r[k][bi * HS + c] = i < nb ? R[((size_t)(B * i + bi) * sp + s) * HS + c] : S(0);
  }
}

// The thread's own block rows of the vector at yb (clamped past the last row).
template <typename S, int RPT, int NV>
__device__ __forceinline__ void res_own(const char* yb, int nb, S (&y)[RPT][NV]) {
#pragma unroll
  for (int k = 0; k < RPT; k++) {
    const int i = min((int)(k * blockDim.x + threadIdx.x), nb - 1);
    ldn<S, NV>(reinterpret_cast<const S*>(yb + i * NV * (int)sizeof(S)), y[k]);
  }
}

template <typename S, int B, int RPT, int NV>
__device__ __forceinline__ void res_zero_block(char* lds, int nb, int bufb) {
  if (threadIdx.x < 2 * NV)
    reinterpret_cast<S*>(lds + (threadIdx.x / NV) * bufb + nb * NV * (int)sizeof(S))[threadIdx.x % NV] =
        S(0);
}

// Forward recursion alpha_0 = R, alpha_1 = Hs R, alpha_{m+1} = 2 Hs alpha_m -
// alpha_{m-1} (engine_cpu.cpp:63-84) of column blockIdx.x: slots 0 .. nsteps of
// the table.  Bound: LDS reads (nb * deg * B elements a step at 128 B per
// clock) plus the barrier while H fits the registers, the L2 stream of the
// remaining blocks otherwise.  A step of the launched kernels took 4.5 us of
// launch and latency at these sizes; here 0.56 us at 16x16 x 2 FP64, 0.50 us
// at 32x32 x 1, 1.3 us at 45x42 x 2 FP32 (5.2 us before).
template <typename S, bool CX, int B, int RPT, int MODE>
__global__ __launch_bounds__(RES_T) void k_res_forward(ResH<S> H, const S* __restrict__ R, int sp,
                                                       S* __restrict__ tab, size_t slot,
                                                       int nsteps) {
  using GE = ResGeo<S, CX, B, RPT>;
  constexpr int NV = GE::NV;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int bufb = res_buf_bytes<GE::BYTES>(H.nb);
  const size_t col = (size_t)blockIdx.x * H.nb * NV;
  constexpr bool OWN = MODE == RES_OWN;
  ResRegs<S, CX, B, RPT, res_vl(RES_VL_FWD, MODE), MODE> G;
  G.load(H);
  S x1[OWN ? RPT : 1][NV], x0[OWN ? RPT : 1][NV];  // OWN: rows of alpha_m, alpha_{m-1}
  {
    S r[RPT][NV];
    res_load_R<S, CX, B, RPT>(R, sp, H.nb, blockIdx.x, r);
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      const int i = k * blockDim.x + threadIdx.x;
      if constexpr (OWN)
#pragma unroll
        for (int e = 0; e < NV; e++) {
          x1[k][e] = r[k][e];
          x0[k][e] = S(0);
        }
      if (i < H.nb) {
        stn<S, NV>(reinterpret_cast<S*>(lds + i * GE::BYTES), r[k]);
        stn<S, NV>(tab + col + (size_t)i * NV, r[k]);
      }
    }
  }
  res_zero_block<S, B, RPT, NV>(lds, H.nb, bufb);
  __syncthreads();
  for (int m = 0; m < nsteps; m++) {
    const char* xb = lds + (m & 1) * bufb;
    char* yb = lds + ((m & 1) ^ 1) * bufb;  // holds alpha_{m-1}
    S acc[RPT][NV];
    G.mul(H, xb, x1, acc);
    S* out = tab + (size_t)(m + 1) * slot + col;
    S y[RPT][NV];
    if constexpr (!OWN) res_own<S, RPT, NV>(yb, H.nb, y);
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      const int i = k * blockDim.x + threadIdx.x;
#pragma unroll
      for (int e = 0; e < NV; e++) {
        if constexpr (OWN) y[k][e] = x0[k][e];
        y[k][e] = m > 0 ? fma(S(2), acc[k][e], -y[k][e]) : acc[k][e];
        if constexpr (OWN) {
          x0[k][e] = x1[k][e];
          x1[k][e] = y[k][e];
        }
      }
      if (i < H.nb) {
        stn<S, NV>(reinterpret_cast<S*>(yb + i * GE::BYTES), y[k]);
        stn<S, NV>(out + (size_t)i * NV, y[k]);
      }
    }
    __syncthreads();
  }
}

// Backward recursion of autodiff_matrix (engine_cpu.cpp:278-294) of column
// blockIdx.x from the forward table:
//   beta_m = 2 Hs beta_{m+1} - beta_{m+2} + 4 c_{2m} alpha_m
//            + 2 c_{2m+1} alpha_{m+1} + 2 c_{2m-1} alpha_{m-1} (m > 1)
// into slots m = M2-1 .. 1 of btab, with beta_{M2} = sb alpha_{M2-1} kept
// virtual (the first step scales its product).  The thread's rows of alpha_m and
// alpha_{m+1} stay in registers, or (LA) in two more LDS buffers, which leaves
// the registers of three vectors to blocks of H (45x42 x 2 FP32: all of it, 2.7 ->
// 2.4 us a step).
template <typename S, bool CX, int B, int RPT, int MODE, bool LA>
__global__ __launch_bounds__(RES_T) void k_res_backward(ResH<S> H, const S* __restrict__ tab,
                                                        S* __restrict__ btab, size_t slot, int M2,
                                                        const double* __restrict__ c, double sb) {
  using GE = ResGeo<S, CX, B, RPT>;
  constexpr int NV = GE::NV;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int bufb = res_buf_bytes<GE::BYTES>(H.nb);
  const size_t col = (size_t)blockIdx.x * H.nb * NV;
  constexpr bool OWN = MODE == RES_OWN;
  ResRegs<S, CX, B, RPT, LA ? RES_VL_BWD_LA<S, MODE == RES_ST> : res_vl(RES_VL_BWD, MODE), MODE> G;
  G.load(H);
  S b1[OWN ? RPT : 1][NV], b2o[OWN ? RPT : 1][NV];  // OWN: rows of beta_{m+1}, beta_{m+2}
  S ai[LA ? 1 : RPT][NV], a1[LA ? 1 : RPT][NV];
#pragma unroll
  for (int k = 0; k < RPT; k++) {
    const int i = min((int)(k * blockDim.x + threadIdx.x), H.nb - 1);
    S(&t)[NV] = ai[LA ? 0 : k], (&t1)[NV] = a1[LA ? 0 : k];
    ldn<S, NV>(tab + (size_t)(M2 - 1) * slot + col + (size_t)i * NV, t);
    ldn<S, NV>(tab + (size_t)M2 * slot + col + (size_t)i * NV, t1);
    // clamped rows: the same value
    stn<S, NV>(reinterpret_cast<S*>(lds + i * GE::BYTES), t);
    if constexpr (OWN)
#pragma unroll
      for (int e = 0; e < NV; e++) {
        b1[k][e] = t[e];
        b2o[k][e] = S(0);
      }
    if constexpr (LA) {
      stn<S, NV>(reinterpret_cast<S*>(lds + 2 * bufb + i * GE::BYTES), t);
      stn<S, NV>(reinterpret_cast<S*>(lds + 3 * bufb + i * GE::BYTES), t1);
    }
  }
  res_zero_block<S, B, RPT, NV>(lds, H.nb, bufb);
  __syncthreads();
  int q = 0;
  for (int m = M2 - 1; m >= 1; m--, q ^= 1) {
    const bool first = m == M2 - 1, second = m == M2 - 2;
    const S ab2 = (S)(2.0 * (first ? sb : 1.0)), asb2 = (S)(second ? sb : 0.0);
    const S ac4 = (S)(4 * c[2 * m]), ac2 = (S)(2 * c[2 * m + 1]);
    const S aw = (S)(m > 1 ? 2 * c[2 * m - 1] : 0.0);
    S an[RPT][NV];
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      const int i = min((int)(k * blockDim.x + threadIdx.x), H.nb - 1);
      ldn<S, NV>(tab + (size_t)(m - 1) * slot + col + (size_t)i * NV, an[k]);
    }
    const char* xb = lds + q * bufb;
    char* yb = lds + (q ^ 1) * bufb;  // holds beta_{m+2}
    const char* ab = lds + (2 + q) * bufb;      // LA: alpha_m
    char* a1b = lds + (2 + (q ^ 1)) * bufb;     // LA: alpha_{m+1}, then alpha_{m-1}
    S acc[RPT][NV];
    G.mul(H, xb, b1, acc);
    S* out = btab + (size_t)m * slot + col;
    S y[RPT][NV];
    if constexpr (!OWN) res_own<S, RPT, NV>(yb, H.nb, y);
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      const int i = k * blockDim.x + threadIdx.x;
      S(&t)[NV] = ai[LA ? 0 : k], (&t1)[NV] = a1[LA ? 0 : k];
      if constexpr (LA) {
        const int o = min(i, H.nb - 1) * GE::BYTES;
        ldn<S, NV>(reinterpret_cast<const S*>(ab + o), t);
        ldn<S, NV>(reinterpret_cast<const S*>(a1b + o), t1);
      }
#pragma unroll
      for (int e = 0; e < NV; e++) {
        if constexpr (OWN) y[k][e] = b2o[k][e];
        const S b2 = first || second ? asb2 * t1[e] : y[k][e];
        S v = fma(ab2, acc[k][e], -b2);
        v = fma(ac4, t[e], v);
        v = fma(ac2, t1[e], v);
        y[k][e] = fma(aw, an[k][e], v);
        if constexpr (OWN) {
          b2o[k][e] = b1[k][e];
          b1[k][e] = y[k][e];
        }
        if constexpr (!LA) {
          t1[e] = t[e];
          t[e] = an[k][e];
        }
      }
      if (i < H.nb) {
        stn<S, NV>(reinterpret_cast<S*>(yb + i * GE::BYTES), y[k]);
        stn<S, NV>(out + (size_t)i * NV, y[k]);
        if constexpr (LA) stn<S, NV>(reinterpret_cast<S*>(a1b + i * GE::BYTES), an[k]);
      }
    }
    __syncthreads();
  }
}

// xi = sum_{m<M} c_m T_m(Hs) R of column blockIdx.x, by the Clenshaw
// recurrence from R (u null; b_{M-1} = c_{M-1} R virtual), or as
// v + 2 T_K(Hs) u from the table sums u, v (K = M steps).  `r0` is slot 0 of the
// output layout (column by column), where R is also written when u is null.
template <typename S, bool CX, int B, int RPT, int MODE>
__global__ __launch_bounds__(RES_T) void k_res_xi(ResH<S> H, const S* __restrict__ R, int sp,
                                                  const S* __restrict__ u, const S* __restrict__ v,
                                                  const double* __restrict__ c, int M,
                                                  S* __restrict__ r0, S* __restrict__ xi) {
  using GE = ResGeo<S, CX, B, RPT>;
  constexpr int NV = GE::NV;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int bufb = res_buf_bytes<GE::BYTES>(H.nb);
  const size_t col = (size_t)blockIdx.x * H.nb * NV;
  constexpr bool OWN = MODE == RES_OWN;
  ResRegs<S, CX, B, RPT, res_vl(RES_VL_XI, MODE), MODE> G;
  G.load(H);
  S x1[OWN ? RPT : 1][NV], x0[OWN ? RPT : 1][NV];  // OWN: rows of the last two vectors
  const bool cl = u == nullptr;
  {
    S x[RPT][NV];
    if (cl) res_load_R<S, CX, B, RPT>(R, sp, H.nb, blockIdx.x, x);
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      const int i = k * blockDim.x + threadIdx.x;
      if constexpr (OWN)
#pragma unroll
        for (int e = 0; e < NV; e++) x1[k][e] = x0[k][e] = S(0);
      if (i >= H.nb) continue;
      if (cl)
        stn<S, NV>(r0 + col + (size_t)i * NV, x[k]);
      else
        ldn<S, NV>(u + col + (size_t)i * NV, x[k]);
      if constexpr (OWN)
#pragma unroll
        for (int e = 0; e < NV; e++) x1[k][e] = x[k][e];
      stn<S, NV>(reinterpret_cast<S*>(lds + i * GE::BYTES), x[k]);
    }
  }
  const S* src = (cl ? r0 : v) + col;  // the source: R, or v added by the last step
  res_zero_block<S, B, RPT, NV>(lds, H.nb, bufb);
  __syncthreads();
  const int n = cl ? M - 1 : M;  // steps
  for (int t = 0; t < n; t++) {
    const bool last = t == n - 1;
    // y = cx Hs x + cz z + cr r
    double cx, cz, cr;
    if (cl) {
      const double cm = c[M - 1];
      cx = (last ? 1.0 : 2.0) * (t == 0 ? cm : 1.0);
      cz = t == 0 ? 0.0 : t == 1 ? -cm : -1.0;
      cr = c[M - 2 - t];
    } else {
      cx = (t == 0 ? 1.0 : 2.0) * (last ? 2.0 : 1.0);
      cz = t == 0 ? 0.0 : last ? -2.0 : -1.0;
      cr = last ? 1.0 : 0.0;
    }
    const S acx = (S)cx, acz = (S)cz, acr = (S)cr;
    const char* xb = lds + (t & 1) * bufb;
    char* yb = lds + ((t & 1) ^ 1) * bufb;
    S acc[RPT][NV];
    G.mul(H, xb, x1, acc);
    S y[RPT][NV];
    if constexpr (!OWN) res_own<S, RPT, NV>(yb, H.nb, y);
#pragma unroll
    for (int k = 0; k < RPT; k++)
#pragma unroll
      for (int e = 0; e < NV; e++) {
        if constexpr (OWN) y[k][e] = x0[k][e];
        y[k][e] = t > 0 ? fma(acx, acc[k][e], acz * y[k][e]) : acx * acc[k][e];
      }
    if (cr != 0.0) {
      S r[RPT][NV];  // written by this thread, or by an earlier kernel
#pragma unroll
      for (int k = 0; k < RPT; k++)
        ldn<S, NV>(src + (size_t)min((int)(k * blockDim.x + threadIdx.x), H.nb - 1) * NV, r[k]);
#pragma unroll
      for (int k = 0; k < RPT; k++)
#pragma unroll
        for (int e = 0; e < NV; e++) y[k][e] = fma(acr, r[k][e], y[k][e]);
    }
    if constexpr (OWN)
#pragma unroll
      for (int k = 0; k < RPT; k++)
#pragma unroll
        for (int e = 0; e < NV; e++) {
          x0[k][e] = x1[k][e];
          x1[k][e] = y[k][e];
        }
#pragma unroll
    for (int k = 0; k < RPT; k++) {
      const int i = k * blockDim.x + threadIdx.x;
      if (i >= H.nb) continue;
      if (last)
        stn<S, NV>(xi + col + (size_t)i * NV, y[k]);
      else
        stn<S, NV>(reinterpret_cast<S*>(yb + i * GE::BYTES), y[k]);
    }
    __syncthreads();
  }
}

#ifdef FKD_RES_SHARED
// Moment dots of the table: partial (m, y) = the sums over slice y of |alpha_m|^2
// and Re<alpha_{m+1}, alpha_m> for m = blockIdx.x, in FP64; cnt scalars a slot.
// One streaming pass (the second operand is the next workgroups' first).
template <typename S>
__global__ __launch_bounds__(WG) void k_res_dots(const S* __restrict__ tab, size_t slot, size_t cnt,
                                                 double* __restrict__ partial) {
  constexpr int NS = Vec16<S>::N;
  const S* a = tab + (size_t)blockIdx.x * slot;
  const S* b = a + slot;
  const size_t np = cnt / NS;
  double dmm = 0.0, dm1 = 0.0;
  for (size_t q = (size_t)blockIdx.y * WG + threadIdx.x; q < np; q += (size_t)gridDim.y * WG) {
    double x[NS], y[NS];
    ldv<S, NS>(a + q * NS, x);
    ldv<S, NS>(b + q * NS, y);
#pragma unroll
    for (int e = 0; e < NS; e++) {
      dmm = fma(x[e], x[e], dmm);
      dm1 = fma(y[e], x[e], dm1);
    }
  }
  if (blockIdx.y == 0 && threadIdx.x < cnt - np * NS) {  // scalars past the last packet
    const double x = (double)a[np * NS + threadIdx.x], y = (double)b[np * NS + threadIdx.x];
    dmm = fma(x, x, dmm);
    dm1 = fma(y, x, dm1);
  }
  wg_sum2(dmm, dm1, partial + 2 * ((size_t)blockIdx.x * gridDim.y + blockIdx.y));
}

// The terms of a D sum over the tables, term t = (a, b, f): D_p += f sum_s a_i b_j^+.
//   autodiff (M2 + 1 terms, one when M2 = 1): diag R R^+, alpha_0 beta_1^+,
//     2 alpha_m beta_{m+1}^+ (m = 1 .. M2-2), 2 sb alpha_{M2-1} alpha_{M2-1}^+
//   stoch (M2 = 0, two terms): (R xi^+ + xi R^+) / 2, tab = R, btab = xi
template <typename S>
struct ResTerms {
  const S* tab;
  const S* btab;
  size_t slot;
  int M2;
  double diag, sb;
  __device__ __forceinline__ void get(int t, const S*& a, const S*& b, double& f) const {
    if (M2 == 0) {
      a = t == 0 ? tab : btab;
      b = t == 0 ? btab : tab;
      f = 0.5;
    } else if (t == 0) {
      a = b = tab;
      f = diag;
    } else if (t == M2) {
      a = b = tab + (size_t)(M2 - 1) * slot;
      f = 2 * sb;
    } else {
      a = tab + (size_t)(t - 1) * slot;
      b = btab + (size_t)t * slot;
      f = t == 1 ? 1.0 : 2.0;
    }
  }
};

// Partial sums of D over slice blockIdx.y of the (term, column) pairs, one
// thread per D block: 2B loads per B^2 complex products, L1-bound; FP64 sums.
template <typename S, bool CX, int B>
__global__ __launch_bounds__(WG) void k_res_outer(const int* __restrict__ drp,
                                                  const int* __restrict__ dci, int nb, int nnzb,
                                                  ResTerms<S> T, int nterm, int ncol, int per,
                                                  double* __restrict__ part) {
  using GE = ResGeo<S, CX, B, 1>;
  constexpr int NV = GE::NV, NH = GE::NH, HS = GE::HS;
  const int p = blockIdx.x * WG + threadIdx.x;
  if (p >= nnzb) return;
  int lo = 0, hi = nb;  // the block row holding p
  while (hi - lo > 1) {
    const int mid = (lo + hi) / 2;
    if (drp[mid] <= p) lo = mid; else hi = mid;
  }
  const size_t oi = (size_t)lo * NV, oj = (size_t)dci[p] * NV, cs = (size_t)nb * NV;
  double acc[NH];
#pragma unroll
  for (int e = 0; e < NH; e++) acc[e] = 0.0;
  int q = blockIdx.y * per;
  const int q1 = min(q + per, nterm * ncol);
  while (q < q1) {
    const int t = q / ncol, s0 = q % ncol, s1 = min(ncol, s0 + q1 - q);
    const S *A, *Bp;
    double f;
    T.get(t, A, Bp, f);
    A += s0 * cs + oi;
    Bp += s0 * cs + oj;
#pragma unroll 4
    for (int s = s0; s < s1; s++, A += cs, Bp += cs) {
      S a[NV], b[NV];
      ldn<S, NV>(A, a);
      ldn<S, NV>(Bp, b);
#pragma unroll
      for (int bi = 0; bi < B; bi++) {
        const double ar = f * (double)a[bi * HS];
        const double ai = CX ? f * (double)a[bi * HS + HS - 1] : 0.0;
#pragma unroll
        for (int bj = 0; bj < B; bj++) {
          double* d = acc + (bj * B + bi) * HS;
          const double br = (double)b[bj * HS];
          d[0] = fma(ar, br, d[0]);
          if constexpr (CX) {
            const double bim = (double)b[bj * HS + 1];
            d[0] = fma(ai, bim, d[0]);
            d[1] = fma(ai, br, d[1]);
            d[1] = fma(-ar, bim, d[1]);
          }
        }
      }
    }
    q += s1 - s0;
  }
  double* o = part + ((size_t)blockIdx.y * nnzb + p) * NH;
#pragma unroll
  for (int e = 0; e < NH; e++) o[e] = acc[e];
}

// A slot of the table (column by column, n elements each, s of them) as a vector of
// the step kernels: n rows of sp elements, zero from column s on.  32 x 32 tiles
// through LDS, both sides in runs of 32 elements; two vectors a call.
constexpr int RES_TILE = 32;
template <typename S, bool CX>
__global__ __launch_bounds__(WG) void k_res_to_rows(const S* __restrict__ src, int n, int s,
                                                    int sp, S* __restrict__ dst) {
  struct E {
    S v[CX ? 2 : 1];
  };
  __shared__ E t[RES_TILE][RES_TILE + 1];
  const int r0 = blockIdx.x * RES_TILE, c0 = blockIdx.y * RES_TILE;
  const int x = threadIdx.x % RES_TILE, y = threadIdx.x / RES_TILE;
#pragma unroll
  for (int k = y; k < RES_TILE; k += WG / RES_TILE) {
    E e{};
    if (r0 + x < n && c0 + k < s)
      e = reinterpret_cast<const E*>(src)[(size_t)(c0 + k) * n + r0 + x];
    t[k][x] = e;
  }
  __syncthreads();
#pragma unroll
  for (int k = y; k < RES_TILE; k += WG / RES_TILE)
    if (r0 + k < n && c0 + x < sp)
      reinterpret_cast<E*>(dst)[(size_t)(r0 + k) * sp + c0 + x] = t[x][k];
}

// n doubles from pinned host memory (the coefficients of a call).
__global__ __launch_bounds__(WG) void k_res_coef(const double* __restrict__ src,
                                                 double* __restrict__ dst, int n) {
  const int k = blockIdx.x * WG + threadIdx.x;
  if (k < n) dst[k] = src[k];
}
#endif  // FKD_RES_SHARED

// Entry points of one (storage type, real/complex, block size, rows per
// thread); first index: ResMode; every block of a row in registers (rows of at
// most dreg_* blocks) except with RES_ST.
template <class S>
struct ResSet {
  void (*pack)(const int*, const int*, const S*, int, int, int, S*, int*) = nullptr;
  void (*fwd[3])(ResH<S>, const S*, int, S*, size_t, int) = {};
  // second index 1: own rows of alpha in LDS (four buffers instead of two)
  void (*bwd[3][2])(ResH<S>, const S*, S*, size_t, int, const double*, double) = {};
  void (*xi[3])(ResH<S>, const S*, int, const S*, const S*, const double*, int, S*, S*) = {};
  int dreg_fwd[3] = {}, dreg_bwd[3][2] = {}, dreg_xi[3] = {};  // 0: no such kernel
  int elem_bytes = 0;   // one block row of one column
  int block_bytes = 0;  // one H block
};

// Block rows per thread compiled for block size b: 1, 2, .. res_max_rpt(b)
// (at most 4096 orbital rows); block sizes 1, 2, 4.
constexpr int res_max_rpt(int b) { return b == 1 ? 8 : b == 2 ? 4 : b == 4 ? 2 : 0; }

bool find_res_dc(int B, int RPT, ResSet<double>* out);
bool find_res_dr(int B, int RPT, ResSet<double>* out);
bool find_res_fc(int B, int RPT, ResSet<float>* out);
bool find_res_fr(int B, int RPT, ResSet<float>* out);

}  // namespace fkd
