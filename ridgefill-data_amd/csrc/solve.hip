// The ridge solve of the closed-form fit on gfx950, all in fp64 (code/kva/ridge.py:80-105: RidgeFit solves
// W(lam) = (C + lam s I)^-1 Cxy with s = mean(diag C), by one eigendecomposition of C; this computes the same
// closed form through the inverse of C + lam s I).
//
//   k_dgemm       C = alpha op(A) op(B) + beta Ci, row-major fp64, v_mfma_f64_16x16x4f64. A workgroup of 4 wave64s
//                 computes a T x T tile (128, 64 or 32) over K in BK-deep blocks; each wave a T/2 x T/2 quarter of
//                 16 x 16 MFMA tiles (lane l feeds A[l % 16][l / 16] and B[l / 16][l % 16] and holds
//                 D[l / 16 + 4 i][l % 16] in its register pair i: the fp64 output's rows interleave, unlike the
//                 fp32 16x16x4 variant's 4 (l / 16) + i). Blocks are double-buffered in LDS (72 KB at T 128, BK 16,
//                 so two workgroups share a CU and fill each other's barrier and LDS-latency gaps), the next block
//                 loaded into registers while the current one is multiplied. LDS rows of BK + 2 doubles (k
//                 contiguous) or T + 16 (k-major), so the fragment reads of each half-wave fall in distinct
//                 banks. The k order of the sums is that of one pass over K in steps of 4.
//   k_spd_inv128  the inverse of a 128 x 128 symmetric positive definite block, one workgroup (below).
//   the inverse   of an n x n SPD matrix (n a multiple of 128, its lower triangle) by block recursion on
//                 [A11 .; A21 A22]: X11 = A11^-1, T = A21 X11, S = A22 - T A21^T (the Schur complement, SPD),
//                 X22 = S^-1, X21 = -X22 T, X11 -= T^T X21, X12 = X21^T. Symmetric results are computed on their
//                 lower tiles only; the product that forms X21 stores X12 too. d 4096, three lambdas: 6.7 ms of
//                 kernels for the inverses (18.6 with 64 x 64 leaves, every product in full and separate copies and
//                 transposes), one lambda 4.0 (15.2), d 1024 0.65 (2.9).
//   k_gemv_rows   out = init + alpha v M, rows summed by 4 waves in order (the bias's vector products).
//   rf_ridge_solve  per lambda: A = C + lam s I padded to a multiple of 128 with an identity block, X = A^-1,
//                 W = X[:d, :d] Cxy (k_dgemm, or k_solve_wt's W^T; the dominant 2 d^2 R flops, 26.4 ms for four
//                 targets of 4096 and three lambdas, 79 % of the fp64 MFMA peak), bias = mean_y - (mean_x X) Cxy
//                 (= mean_y - mean_x W; one pass over Cxy for every lambda). Up to 8 lambdas go together:
//                 every launch of the recursion carries all of them in its grid.
#include <algorithm>

#include "rf_common.h"

namespace rf {
namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

// C = alpha op(A) op(B) + beta Ci for each matrix of a batch (blockIdx.y, element strides s*).
struct DgemmArgs {
  const double* A;        // [M, K], or with AT [K, M]
  int64_t lda;
  const double* B;        // [K, N], or with BT [N, K]
  int64_t ldb;
  double* C;
  int64_t ldc;
  int M, N, K;
  double alpha, beta;
  int64_t sa, sb, sc;
  const double* Ci;       // read when beta != 0 (may be C itself)
  int64_t ldci, sci;
  double* Ct;             // if given: C^T is stored there too (with lower: its tiles above the diagonal)
  int64_t ldct, sct;
  int lower;              // M == N: only the tiles on and below the diagonal are computed
};

// A T x T tile per workgroup, K in BK-deep blocks. Requires K and N even (with AT also M), even strides and
// 16-byte aligned operands (checked by the host callers). Loads past M, N or K read a clamped in-bounds address
// and are replaced by zeros (no divergent branches in the loop).
// T and BK: the solve's large products take 128 and 16 (two workgroups per CU); the inverse's take the largest
// tile that still gives the batch about a workgroup per CU, with deeper K blocks for the smaller tiles, whose
// time is the chain of loads, barriers and MFMAs of one workgroup (64 x 64 x 64 took 21 us in a 128 x 128 tile
// with 16-deep blocks, most of it waiting).
// store(row, col, value) takes the elements inside M x N; ROWS_FAST: the order of the tiles in flight.
template <int T, int BK, bool AT, bool BT, bool ROWS_FAST, class Store>
__device__ __forceinline__ void dgemm(const DgemmArgs& a, Store store) {
  constexpr int MT = T / 32;                      // 16 x 16 MFMA tiles per wave and dimension
  constexpr int RST = BK + 2, CST = T + 16;       // LDS row strides in doubles: [T][BK] and [BK][T] images
  constexpr int LD = T * BK / 512;                // double2 loads per thread, block and operand
  constexpr int AS = AT ? BK * CST : T * RST, BS = BT ? T * RST : BK * CST;
  __shared__ __align__(16) double As[2][AS];
  __shared__ __align__(16) double Bs[2][BS];
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6), wm = w >> 1, wn = w & 1;
  int tm, tn;
  if (a.lower) {
    tm = static_cast<int>((sqrtf(8.f * static_cast<float>(blockIdx.x) + 1.f) - 1.f) * 0.5f);
    while (tm * (tm + 1) / 2 > static_cast<int>(blockIdx.x)) --tm;
    while ((tm + 1) * (tm + 2) / 2 <= static_cast<int>(blockIdx.x)) ++tm;
    tn = static_cast<int>(blockIdx.x) - tm * (tm + 1) / 2;
  } else {                                        // the fast direction's blocks share the other's panel
    const int per = ((ROWS_FAST ? a.M : a.N) + T - 1) / T, q = blockIdx.x / per, r = blockIdx.x - q * per;
    tm = ROWS_FAST ? r : q;
    tn = ROWS_FAST ? q : r;
  }
  const int m0 = tm * T, n0 = tn * T;
  const int64_t z = blockIdx.y;
  const double* __restrict__ Ag = a.A + z * a.sa;
  const double* __restrict__ Bg = a.B + z * a.sb;
  double2 ra[LD], rb[LD];
  unsigned ok = 0;
  // chunk j = t + 256 i of a [T][BK] image: row j / (BK / 2), k pair j % (BK / 2); of a [BK][T] image: k row
  // j / (T / 2), column pair j % (T / 2). The zero masks are applied when the block is written to LDS, after
  // the multiply that hides the loads.
  auto load_one = [&](const double* __restrict__ g, int64_t ld, int r0, int R, int k0, bool kmajor, int j, bool& in) {
    const int r = kmajor ? r0 + 2 * (j % (T / 2)) : r0 + j / (BK / 2);
    const int k = kmajor ? k0 + j / (T / 2) : k0 + 2 * (j % (BK / 2));
    in = r < R && k < a.K;
    const int rc = kmajor ? min(r, R - 2) : min(r, R - 1), kc = kmajor ? min(k, a.K - 1) : min(k, a.K - 2);
    return *reinterpret_cast<const double2*>(kmajor ? g + static_cast<int64_t>(kc) * ld + rc
                                                    : g + static_cast<int64_t>(rc) * ld + kc);
  };
  auto gload = [&](int k0) {
    ok = 0;
#pragma unroll
    for (int i = 0; i < LD; ++i) {
      bool in;
      ra[i] = load_one(Ag, a.lda, m0, a.M, k0, AT, t + 256 * i, in);
      ok |= in ? 1u << i : 0u;
      rb[i] = load_one(Bg, a.ldb, n0, a.N, k0, !BT, t + 256 * i, in);
      ok |= in ? 1u << (LD + i) : 0u;
    }
  };
  auto put = [&](double* s, bool kmajor, int j, bool in, const double2& v) {
    const int at = kmajor ? j / (T / 2) * CST + 2 * (j % (T / 2)) : j / (BK / 2) * RST + 2 * (j % (BK / 2));
    *reinterpret_cast<double2*>(s + at) = double2{in ? v.x : 0.0, in ? v.y : 0.0};
  };
  auto swrite = [&](int s) {
#pragma unroll
    for (int i = 0; i < LD; ++i) {
      put(As[s], AT, t + 256 * i, (ok >> i) & 1, ra[i]);
      put(Bs[s], !BT, t + 256 * i, (ok >> (LD + i)) & 1, rb[i]);
    }
  };
  f64x4 acc[MT][MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < MT; ++nt) acc[mt][nt] = f64x4{0.0, 0.0, 0.0, 0.0};
  const int nkb = (a.K + BK - 1) / BK;
  gload(0);
  swrite(0);
  __syncthreads();
  const int lr = lane & 15, lk = lane >> 4;
  const int ma = wm * (T / 2) + lr, nb = wn * (T / 2) + lr;
  for (int kb = 0; kb < nkb; ++kb) {
    const int s = kb & 1;
    if (kb + 1 < nkb) gload((kb + 1) * BK);
    const double* as = AT ? As[s] + lk * CST + ma : As[s] + ma * RST + lk;
    const double* bs = BT ? Bs[s] + nb * RST + lk : Bs[s] + lk * CST + nb;
#pragma unroll
    for (int kk = 0; kk < BK / 4; ++kk) {
      double af[MT], bf[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) af[mt] = AT ? as[kk * 4 * CST + mt * 16] : as[mt * 16 * RST + kk * 4];
#pragma unroll
      for (int nt = 0; nt < MT; ++nt) bf[nt] = BT ? bs[nt * 16 * RST + kk * 4] : bs[kk * 4 * CST + nt * 16];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < MT; ++nt)
          acc[mt][nt] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[mt], bf[nt], acc[mt][nt], 0, 0, 0);
    }
    if (kb + 1 < nkb) swrite(s ^ 1);                // stage s ^ 1 was last read before the previous barrier
    __syncthreads();
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < MT; ++nt) {
      const int col = n0 + nb + nt * 16;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = m0 + wm * (T / 2) + mt * 16 + lk + 4 * i;
        if (row < a.M && col < a.N) store(row, col, a.alpha * acc[mt][nt][i], tm != tn);
      }
    }
}

template <int T, int BK, bool AT, bool BT>
__global__ __launch_bounds__(256, T == 32 ? 1 : 2) void k_dgemm(DgemmArgs a) {
  const int64_t z = blockIdx.y;
  double* C = a.C + z * a.sc;
  const double* Ci = a.Ci + z * a.sci;
  double* Ct = a.Ct ? a.Ct + z * a.sct : nullptr;
  dgemm<T, BK, AT, BT, true>(a, [&](int64_t row, int64_t col, double v, bool off_diagonal) {
    if (a.beta != 0.0) v += a.beta * Ci[row * a.ldci + col];
    C[row * a.ldc + col] = v;
    if (Ct && (off_diagonal || !a.lower)) Ct[col * a.ldct + row] = v;
  });
}

// The weights in F.linear layout, W^T = Cxy^T X (X symmetric), rounded to fp32 where they are formed: row j width + r
// of the product is output r of target j. A pass that transposed and rounded fp64 weights afterwards took 1.2 ms for
// four targets and three lambdas at d 4096, beside writing and keeping them in fp64 (1.6 GB).
constexpr int WT_TARGETS = 64;
struct WtOut {
  float* p[WT_TARGETS];     // per target: [lambda][width][d]
  int width;
};
__global__ __launch_bounds__(256, 2) void k_solve_wt(DgemmArgs a, WtOut o) {
  const int64_t z = blockIdx.y, d = a.N;
  dgemm<128, 16, true, false, false>(a, [&](int row, int col, double v, bool) {
    const int j = row / o.width, r = row - j * o.width;
    o.p[j][(z * o.width + r) * d + col] = static_cast<float>(v);
  });
}

// A double of the lane in row position n of this lane's 16-lane row (DPP row_newbcast).
template <int n>
__device__ __forceinline__ double row_bcast(double v) {
  const int2 u = __builtin_bit_cast(int2, v);
  return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_update_dpp(0, u.x, 0x150 + n, 0xf, 0xf, true),
                                              __builtin_amdgcn_update_dpp(0, u.y, 0x150 + n, 0xf, 0xf, true)));
}

// One elimination step KK of a wave's 16 x 16 inverse: lane (r = l % 16, g = l / 16) holds row r, columns 4 g ..
// 4 g + 3. p = M[KK][KK]; row KK /= p (M[KK][KK] = 1 / p); every other row: M[r][j] -= M[r][KK] / p M[KK][j],
// M[r][KK] = -M[r][KK] / p.
template <int KK>
__device__ __forceinline__ void inv16_step(double (&m)[4], int r, int g) {
  constexpr int GK = KK / 4, EK = KK & 3;
  const double rinv = 1.0 / __shfl(m[EK], GK * 16 + KK, 64);
  const double f = __shfl(m[EK], GK * 16 + r, 64) * rinv;       // M[r][KK] / p
  const bool own = r == KK;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const double prow = row_bcast<KK>(m[e]);
    const double v = own ? prow * rinv : m[e] - f * prow;
    m[e] = (e == EK && g == GK) ? (own ? rinv : -f) : v;
  }
}

constexpr int LEAF = 128;

// X = A^-1 for a 128 x 128 SPD block (its lower triangle is read), one workgroup of 4 wave64s per matrix: blocked
// Gauss-Jordan without pivoting (stable for SPD matrices) in 16-wide block steps. The matrix stays in registers as
// MFMA accumulators, wave w holding block rows 2 w and 2 w + 1. Step k, with P = M[k][k]^-1, R the block row k and
// C the block column k before the step (both published in LDS, double-buffered, one barrier per step):
//   G_i = C_i P;  M[i][j] -= G_i R_j (i, j != k);  M[i][k] = -G_i;  M[k][j] = P R_j;  M[k][k] = P.
// Every wave forms P itself (inv16_step, lane = row and column group) rather than wait for one that does. P is
// symmetric up to rounding, so a lane's P[l % 16][4 s + l / 16] serves as A and as B operand of k-step s;
// G_i^T = P C_i^T comes out of the MFMA in the A operand's order, so no product passes through LDS.
// Bound by its chain: 8 steps of 16 dependent eliminations and 72 MFMAs a wave. It replaces two 64 x 64 leaves of
// 64 elimination steps each (37 us a launch) and the seven launches that joined them (about 20 us a product).
__global__ __launch_bounds__(256, 1) void k_spd_inv128(const double* __restrict__ A, int64_t lda,
                                                       double* __restrict__ X, int64_t ldx, int64_t sa, int64_t sx) {
  constexpr int NB = LEAF / 16, RS = LEAF + 16, CS = 18;
  __shared__ __align__(16) double Rp[2][16 * RS];       // block row k: [16][128]
  __shared__ __align__(16) double Cp[2][LEAF * CS];     // block column k: [128][16]
  A += static_cast<int64_t>(blockIdx.x) * sa;
  X += static_cast<int64_t>(blockIdx.x) * sx;
  const int t = threadIdx.x, lane = t & 63, lr = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  f64x4 m[2][NB];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 16 * (2 * w + a) + g + 4 * i, col = 16 * j + lr;
        m[a][j][i] = A[static_cast<int64_t>(max(row, col)) * lda + min(row, col)];
      }
#pragma unroll
  for (int k = 0; k < NB; ++k) {
    double* rp = Rp[k & 1];
    double* cp = Cp[k & 1];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int i = 0; i < 4; ++i) cp[(16 * (2 * w + a) + g + 4 * i) * CS + lr] = m[a][k][i];
    if (w == k / 2) {
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) rp[(g + 4 * i) * RS + 16 * j + lr] = m[k & 1][j][i];
    }
    __syncthreads();
    double p[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) p[e] = rp[lr * RS + 16 * k + 4 * g + e];
    inv16_step<0>(p, lr, g);  inv16_step<1>(p, lr, g);  inv16_step<2>(p, lr, g);  inv16_step<3>(p, lr, g);
    inv16_step<4>(p, lr, g);  inv16_step<5>(p, lr, g);  inv16_step<6>(p, lr, g);  inv16_step<7>(p, lr, g);
    inv16_step<8>(p, lr, g);  inv16_step<9>(p, lr, g);  inv16_step<10>(p, lr, g); inv16_step<11>(p, lr, g);
    inv16_step<12>(p, lr, g); inv16_step<13>(p, lr, g); inv16_step<14>(p, lr, g); inv16_step<15>(p, lr, g);
    // the operand order of k-step s: P[lr][4 s + g], from lane (lr, group s), element g
    double pf[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      double v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = __shfl(p[e], s * 16 + lr, 64);
      pf[s] = g < 2 ? (g == 0 ? v[0] : v[1]) : (g == 2 ? v[2] : v[3]);
    }
    double ng[2][4];                                    // -G_i[lr][4 s + g]
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      f64x4 gt = f64x4{0.0, 0.0, 0.0, 0.0}, gn = gt;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const double c = cp[(16 * (2 * w + a) + lr) * CS + 4 * s + g];
        gt = __builtin_amdgcn_mfma_f64_16x16x4f64(pf[s], c, gt, 0, 0, 0);
        gn = __builtin_amdgcn_mfma_f64_16x16x4f64(c, pf[s], gn, 0, 0, 0);
      }
      const bool own = 2 * w + a == k;                  // wave-uniform
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        ng[a][i] = own ? pf[i] : -gt[i];
        m[a][k][i] = own ? pf[i] : -gn[i];
      }
      if (own) {
#pragma unroll
        for (int j = 0; j < NB; ++j)
          if (j != k) m[a][j] = f64x4{0.0, 0.0, 0.0, 0.0};
      }
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      if (j == k) continue;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const double b = rp[(4 * s + g) * RS + 16 * j + lr];
#pragma unroll
        for (int a = 0; a < 2; ++a) m[a][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ng[a][s], b, m[a][j], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        X[static_cast<int64_t>(16 * (2 * w + a) + g + 4 * i) * ldx + 16 * j + lr] = m[a][j][i];
}

// out_l[c] = init[c] + alpha sum_r v_l[r] M_l[r][c] for the batch's NL vectors v_l (sv apart) and matrices M_l
// (sm apart; sm 0: one matrix for all, read once), c < cols, r < rows. Block: 128 columns (a double2 per
// lane), its 4 waves summing row quarters in row order; the quarters are added in order (fixed bits).
template <int NL>
__global__ __launch_bounds__(256) void k_gemv_rows(const double* __restrict__ v, int64_t sv,
                                                   const double* __restrict__ M, int64_t ldm, int64_t sm, int rows,
                                                   int cols, const double* __restrict__ init, double alpha,
                                                   double* __restrict__ out, int64_t so) {
  __shared__ double2 part[4][NL][64];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int c = blockIdx.x * 128 + 2 * lane;
  const int l0 = NL == 1 ? blockIdx.y : 0;              // NL > 1: the shared matrix, every vector at once
  const double* __restrict__ Ml = M + static_cast<int64_t>(l0) * sm;
  const int per = (rows + 3) / 4, r0 = w * per, r1 = min(rows, r0 + per);
  double2 acc[NL];
#pragma unroll
  for (int l = 0; l < NL; ++l) acc[l] = double2{0.0, 0.0};
  if (c < cols) {
    const double* __restrict__ p = Ml + c;
    int r = r0;
    for (; r + 8 <= r1; r += 8) {
      double2 x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = *reinterpret_cast<const double2*>(p + static_cast<int64_t>(r + u) * ldm);
#pragma unroll
      for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int l = 0; l < NL; ++l) {
          const double s = v[(l0 + l) * sv + r + u];
          acc[l].x += s * x[u].x;
          acc[l].y += s * x[u].y;
        }
    }
    for (; r < r1; ++r) {
      const double2 x = *reinterpret_cast<const double2*>(p + static_cast<int64_t>(r) * ldm);
#pragma unroll
      for (int l = 0; l < NL; ++l) {
        const double s = v[(l0 + l) * sv + r];
        acc[l].x += s * x.x;
        acc[l].y += s * x.y;
      }
    }
  }
#pragma unroll
  for (int l = 0; l < NL; ++l) part[w][l][lane] = acc[l];
  __syncthreads();
  if (w == 0 && c < cols) {
#pragma unroll
    for (int l = 0; l < NL; ++l) {
      double2 s = part[0][l][lane];
#pragma unroll
      for (int i = 1; i < 4; ++i) {
        s.x += part[i][l][lane].x;
        s.y += part[i][l][lane].y;
      }
      double2 o = init ? *reinterpret_cast<const double2*>(init + c) : double2{0.0, 0.0};
      o.x += alpha * s.x;
      o.y += alpha * s.y;
      *reinterpret_cast<double2*>(out + (l0 + l) * so + c) = o;
    }
  }
}

// dst[i][j] = src[i][j] + (i == j ? shift : 0) for i, j < n_src, and the identity on the padding up to n.
struct Shifts {
  double v[8];
};

__global__ __launch_bounds__(256) void k_dshift(const double* __restrict__ src, int64_t lds, int n_src,
                                                double* __restrict__ dst, int64_t ldd, int n, int64_t sd, Shifts sh) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const double shift = sh.v[blockIdx.y];
  dst += static_cast<int64_t>(blockIdx.y) * sd;
  if (idx >= static_cast<int64_t>(n) * n) return;
  const int i = static_cast<int>(idx / n), j = static_cast<int>(idx % n);
  double v;
  if (i < n_src && j < n_src) v = src[static_cast<int64_t>(i) * lds + j] + (i == j ? shift : 0.0);
  else v = (i == j) ? 1.0 : 0.0;
  dst[static_cast<int64_t>(i) * ldd + j] = v;
}

// Launches on one stream for a batch of `nb` matrices laid out at fixed element strides (the lambdas of one
// solve): every matrix argument is the batch's first matrix and its stride.
struct Solver {
  hipStream_t stream;
  const char* fn;
  int nb;
  int rc = RF_OK;

  bool ok() {
    if (rc == RF_OK) rc = check_launch(fn);
    return rc == RF_OK;
  }
  // One k_dgemm per product: 128 x 128 tiles where they give the batch 192 workgroups or more, else 64 x 64, else
  // 32 x 32. us per product of edge m (M = N = K = m) over three matrices, as 128 x 128 tiles -> as chosen here:
  // m 128 21 -> 6, 256 47 -> 8 (32 x 32), 512 89 -> 32 (64 x 64), 1024 179 (128 x 128), 2048 990.
  template <bool AT, bool BT>
  void gemm(const DgemmArgs& a) {
    if (rc != RF_OK || a.M <= 0 || a.N <= 0) return;
    auto tiles = [&](int T) {
      const int64_t tm = (a.M + T - 1) / T, tn = (a.N + T - 1) / T;
      return a.lower ? tm * (tm + 1) / 2 : tm * tn;
    };
    auto grid = [&](int T) { return dim3(static_cast<unsigned>(tiles(T)), nb); };
    if (tiles(128) * nb >= 192)
      hipLaunchKernelGGL((k_dgemm<128, 16, AT, BT>), grid(128), dim3(256), 0, stream, a);
    else if (tiles(64) * nb >= 192)
      hipLaunchKernelGGL((k_dgemm<64, 32, AT, BT>), grid(64), dim3(256), 0, stream, a);
    else
      hipLaunchKernelGGL((k_dgemm<32, 64, AT, BT>), grid(32), dim3(256), 0, stream, a);
    ok();
  }
  // X = A^-1 for each matrix of the batch (n x n SPD, n a multiple of 128, its lower triangle read; matrices sa / sx
  // apart); work: each matrix's own work_doubles(n) doubles, sw apart.
  void inverse(const double* A, int64_t lda, int64_t sa, double* X, int64_t ldx, int64_t sx, int n, double* work,
               int64_t sw) {
    if (rc != RF_OK) return;
    if (n == LEAF) {
      hipLaunchKernelGGL(k_spd_inv128, dim3(nb), dim3(256), 0, stream, A, lda, X, ldx, sa, sx);
      ok();
      return;
    }
    const int h = LEAF * ((n + 2 * LEAF - 1) / (2 * LEAF)), h2 = n - h;
    const double* A21 = A + static_cast<int64_t>(h) * lda;
    const double* A22 = A21 + h;
    double* X12 = X + h;
    double* X21 = X + static_cast<int64_t>(h) * ldx;
    double* X22 = X21 + h;
    double* T = work;                                   // [h2, h]
    double* S = work + static_cast<int64_t>(h2) * h;    // [h2, h2], its lower tiles
    double* deeper = S + static_cast<int64_t>(h2) * h2;
    inverse(A, lda, sa, X, ldx, sx, h, work, sw);       // X11 (T and S are not live yet)
    // T = A21 X11
    gemm<false, false>({A21, lda, X, ldx, T, h, h2, h, h, 1.0, 0.0, sa, sx, sw, T, h, sw, nullptr, 0, 0, 0});
    // S = A22 - T A21^T
    gemm<false, true>({T, h, A21, lda, S, h2, h2, h2, h, -1.0, 1.0, sw, sa, sw, A22, lda, sa, nullptr, 0, 0, 1});
    inverse(S, h2, sw, X22, ldx, sx, h2, deeper, sw);   // X22 = S^-1
    // X21 = -X22 T, and X12 = X21^T
    gemm<false, false>({X22, ldx, T, h, X21, ldx, h2, h, h2, -1.0, 0.0, sx, sw, sx, X21, ldx, sx, X12, ldx, sx, 0});
    // X11 -= T^T X21, symmetric
    gemm<true, false>({T, h, X21, ldx, X, ldx, h, h, h2, -1.0, 1.0, sw, sx, sx, X, ldx, sx, X, ldx, sx, 1});
  }
};

// doubles of work the recursion needs for n (T and S at this level, then the deeper levels)
int64_t work_doubles(int n) {
  if (n <= LEAF) return 0;
  const int64_t h = LEAF * ((n + 2 * LEAF - 1) / (2 * LEAF)), h2 = n - h;
  return std::max(work_doubles(static_cast<int>(h)), h2 * h + h2 * h2 + work_doubles(static_cast<int>(h2)));
}

int64_t padded(int64_t d) { return (d + LEAF - 1) / LEAF * LEAF; }

constexpr int MAX_LAMBDAS = 8;           // lambdas solved together (one batch of inverses)

size_t solve_workspace(int64_t d, int nlam) {
  const int64_t n = padded(d);
  const int nb = std::max(1, std::min(nlam, MAX_LAMBDAS));
  return static_cast<size_t>(nb) * (2 * n * n + work_doubles(static_cast<int>(n)) + n) * sizeof(double) + 256;
}

// out_l = init + alpha v_l M for l < nb with one matrix M shared by the batch (read once).
void gemv_shared(int nb, const double* v, int64_t sv, const double* M, int64_t ldm, int rows, int cols,
                 const double* init, double alpha, double* out, int64_t so, hipStream_t stream) {
  const dim3 grid((cols + 127) / 128), block(256);
  switch (nb) {
#define RF_GEMV(NL) \
  case NL: hipLaunchKernelGGL(k_gemv_rows<NL>, grid, block, 0, stream, v, sv, M, ldm, 0, rows, cols, init, alpha, out, so); break;
    RF_GEMV(1) RF_GEMV(2) RF_GEMV(3) RF_GEMV(4) RF_GEMV(5) RF_GEMV(6) RF_GEMV(7) RF_GEMV(8)
#undef RF_GEMV
    default: break;
  }
}

}  // namespace
}  // namespace rf

using namespace rf;

extern "C" int rf_ridge_solve_workspace_bytes(int64_t d, int nlam, size_t* bytes) {
  if (d <= 0 || d > 65536 || nlam <= 0 || !bytes)
    return fail(RF_EINVAL_ARG, "rf_ridge_solve_workspace_bytes: d %lld, nlam %d", (long long)d, nlam);
  *bytes = solve_workspace(d, nlam);
  return RF_OK;
}

// Shared by the two entry points: fp64 weights into w, or (wt) fp32 ones in F.linear layout per target.
static int ridge_solve(const char* fn, const double* cxx, int64_t ldc, int64_t d, const double* cxy, int64_t ldb,
                       int64_t R, const double* mean_x, const double* mean_y, const double* lams, int nlam, double scale,
                       double* w, int64_t ldw, int64_t w_stride, float* const* wt, int64_t width, double* bias,
                       int64_t bias_stride, void* workspace, size_t ws_bytes, hipStream_t stream) {
  if (!cxx || !cxy || !lams || (!w && !wt) || !workspace) return fail(RF_EINVAL_ARG, "%s: null pointer", fn);
  if (bias && (!mean_x || !mean_y)) return fail(RF_EINVAL_ARG, "%s: the bias needs mean_x and mean_y", fn);
  if (d <= 0 || d > 65536 || R <= 0 || R > (1ll << 30) || R % 2 || d % 2 || ldc < d || ldb < R || ldb % 2 ||
      ldw < R || ldw % 2 || nlam <= 0 || (nlam > 1 && w_stride < d * ldw) || (bias && nlam > 1 && bias_stride < R))
    return fail(RF_EINVAL_SHAPE, "%s: d %lld, R %lld (even), ldc %lld, ldb %lld, ldw %lld (even, >= R), nlam %d, "
                "w_stride %lld, bias_stride %lld", fn, (long long)d, (long long)R, (long long)ldc, (long long)ldb,
                (long long)ldw, nlam, (long long)w_stride, (long long)bias_stride);
  if (!aligned16(cxy) || (w && !aligned16(w)) || !aligned16(workspace) || (mean_x && !aligned16(mean_x)) ||
      (bias && (!aligned16(bias) || !aligned16(mean_y) || (nlam > 1 && bias_stride % 2))))
    return fail(RF_EINVAL_SHAPE, "%s: cxy, w, mean_x, mean_y, bias and the workspace must be 16-byte aligned "
                "(bias_stride even)", fn);
  if (ws_bytes < solve_workspace(d, nlam))
    return fail(RF_EINVAL_ARG, "%s: workspace %zu bytes, needs %zu (rf_ridge_solve_workspace_bytes)", fn, ws_bytes,
                solve_workspace(d, nlam));
  for (int l = 0; l < nlam; ++l)
    if (!(lams[l] > 0.0) || !(scale > 0.0))
      return fail(RF_EINVAL_ARG, "%s: lambda %g, scale %g (both must be positive)", fn, lams[l], scale);
  const int n = static_cast<int>(padded(d));
  const int64_t nn = static_cast<int64_t>(n) * n, nw = work_doubles(n);
  double* A = static_cast<double*>(workspace);
  for (int l0 = 0; l0 < nlam; l0 += MAX_LAMBDAS) {        // up to MAX_LAMBDAS inverses as one batch
    const int nb = std::min(MAX_LAMBDAS, nlam - l0);
    double* X = A + nb * nn;
    double* work = X + nb * nn;
    Solver s{stream, fn, nb};
    Shifts sh{};
    for (int l = 0; l < nb; ++l) sh.v[l] = lams[l0 + l] * scale;
    hipLaunchKernelGGL(k_dshift, dim3(static_cast<unsigned>((nn + 255) / 256), nb), dim3(256), 0, stream, cxx, ldc,
                       static_cast<int>(d), A, static_cast<int64_t>(n), n, nn, sh);
    if (!s.ok()) return s.rc;
    s.inverse(A, n, nn, X, n, nn, n, work, nw);
    const int di = static_cast<int>(d), ri = static_cast<int>(R);
    if (w) {
      double* wl = w + l0 * w_stride;
      s.gemm<false, false>({X, n, cxy, ldb, wl, ldw, di, ri, di, 1.0, 0.0, nn, 0, w_stride, wl, ldw, w_stride, nullptr, 0,
                            0, 0});
    } else {
      for (int64_t j = 0; j < R / width && s.rc == RF_OK; j += WT_TARGETS) {
        const int nt = static_cast<int>(std::min<int64_t>(WT_TARGETS, R / width - j));
        WtOut o{};
        o.width = static_cast<int>(width);
        for (int i = 0; i < nt; ++i) o.p[i] = wt[j + i] + static_cast<int64_t>(l0) * width * d;
        const int m = static_cast<int>(nt * width);
        const DgemmArgs g{cxy + j * width, ldb, X, n, nullptr, 0, m, di, di, 1.0, 0.0, 0, nn, 0, nullptr, 0, 0, nullptr,
                          0, 0, 0};
        hipLaunchKernelGGL(k_solve_wt, dim3(static_cast<unsigned>(((m + 127) / 128) * ((di + 127) / 128)), nb), dim3(256),
                           0, stream, g, o);
        s.ok();
      }
    }
    if (bias && s.rc == RF_OK) {                       // mean_y - mean_x W = mean_y - (mean_x X) Cxy
      double* u = work + nb * nw;
      hipLaunchKernelGGL(k_gemv_rows<1>, dim3(static_cast<unsigned>((d + 127) / 128), nb), dim3(256), 0, stream,
                         mean_x, 0, X, static_cast<int64_t>(n), nn, static_cast<int>(d), static_cast<int>(d), nullptr,
                         1.0, u, static_cast<int64_t>(n));
      if (!s.ok()) return s.rc;
      gemv_shared(nb, u, n, cxy, ldb, static_cast<int>(d), static_cast<int>(R), mean_y, -1.0,
                  bias + l0 * bias_stride, bias_stride, stream);
      if (!s.ok()) return s.rc;
    }
    if (s.rc != RF_OK) return s.rc;
  }
  return RF_OK;
}

extern "C" int rf_ridge_solve(const double* cxx, int64_t ldc, int64_t d, const double* cxy, int64_t ldb, int64_t R,
                              const double* mean_x, const double* mean_y, const double* lams, int nlam, double scale,
                              double* w, int64_t ldw, int64_t w_stride, double* bias, int64_t bias_stride,
                              void* workspace, size_t ws_bytes, hipStream_t stream) {
  if (!w) return fail(RF_EINVAL_ARG, "rf_ridge_solve: null pointer");
  return ridge_solve("rf_ridge_solve", cxx, ldc, d, cxy, ldb, R, mean_x, mean_y, lams, nlam, scale, w, ldw, w_stride,
                     nullptr, R, bias, bias_stride, workspace, ws_bytes, stream);
}

extern "C" int rf_ridge_solve_wt(const double* cxx, int64_t ldc, int64_t d, const double* cxy, int64_t ldb, int targets,
                                 int64_t width, const double* mean_x, const double* mean_y, const double* lams, int nlam,
                                 double scale, float* const* wt, double* bias, int64_t bias_stride, void* workspace,
                                 size_t ws_bytes, hipStream_t stream) {
  const char* fn = "rf_ridge_solve_wt";
  if (!wt) return fail(RF_EINVAL_ARG, "%s: null pointer", fn);
  if (targets <= 0 || width <= 0 || width % 2 || width > (1ll << 24) || width * targets > (1ll << 30))
    return fail(RF_EINVAL_SHAPE, "%s: %d targets of width %lld (even)", fn, targets, (long long)width);
  for (int j = 0; j < targets; ++j)
    if (!wt[j]) return fail(RF_EINVAL_ARG, "%s: null pointer for target %d", fn, j);
  const int64_t R = width * targets;
  return ridge_solve(fn, cxx, ldc, d, cxy, ldb, R, mean_x, mean_y, lams, nlam, scale, nullptr, R, d * R, wt, width, bias,
                     bias_stride, workspace, ws_bytes, stream);
}
