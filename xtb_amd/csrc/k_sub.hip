// Density of a closed-shell molecule with an orbital gap without a full
// diagonalisation: between the first and the last SCC iteration only the
// density is needed, and with every occupation 0 or 2 it depends on the
// occupied subspace alone, not on the orbitals inside it.
//
// C keeps the orbitals of the molecule's last full diagonalisation (o
// occupied, v virtual columns).  In that basis the Fock matrix A = C^T H C of
// a later iteration is close to diagonal, and its occupied subspace is the
// span of Y = [I; X] with the v x o matrix X that solves
//
//     R(X) = A_vo + A_vv X - X (A_oo + A_ov X) = 0.
//
// X starts from the previous iteration's and takes X -= R / D, D = a_vv - a_oo
// (element-wise, the diagonals) until max |R| is as small as the off-diagonal
// elements of a finished diagonalisation (jac_tol max(max |A_ii|, 1)).  A
// step is two products of 2 N v o and 2 v o^2 flops.  max |R| falls by 20 to
// 30 times per step for alkanes (gap 11 eV), by 10 for 32 waters (8 eV) and
// by 2.5 for 700 waters (4 eV); where it falls by less than 6 times, the step
// becomes one of the second-order Richardson iteration,
// X' = X_old + w (X - R / D - X_old), with w for the contraction seen (21 ->
// 13 steps for 700 waters).  The density is
// P = 2 (C Y) (I + X^T X)^-1 (C Y)^T with the inverse from the product
// (I - M)(I + M^2)(I + M^4)(I + M^8), M = X^T X, whose neglected part M^16 is
// bounded below 1e-16.
//
// Why a converged X is the occupied subspace: the plain step is X -> X - D^-1
// T X with T the (symmetrisable) map Z -> A'_vv Z - Z A'_oo of the decoupled
// blocks.  It contracts by rho < 1 only if D^-1 T has its spectrum in
// [1 - rho, 1 + rho] (and the second-order one only if that lies above 0), so
// T is positive definite and every virtual eigenvalue lies above every
// occupied one by at least (1 - rho) min D.  The path is left unless that is
// at least kSubGapKt kT, rho being the contraction seen over the last steps
// (sub_rate during the steps, sub_gap_kept at convergence): the Fermi
// occupations of the frontier orbitals are then within e^-26 = 5e-12 of 1 and
// 0, the size of the density error that the tolerance of R admits, and far
// below the 1e-9 from which entropy counts.
// The occupations handed back are those of the last diagonalisation.
#pragma once
#include "device_util.h"
#include "engine.h"

namespace xtbamd {

constexpr int kSubSteps = 24;        // steps per SCC iteration at most
// a molecule that gave up gets a fresh basis from its full diagonalisation,
// which is closer to the next iterations' orbitals (700 waters: given up on
// the first basis, 8 to 10 steps on the second); after a second time it
// stays with full diagonalisations
constexpr int kSubTries = 2;
constexpr double kSubGapKt = 52.0;   // smallest gap in units of kT
constexpr double kSubRhoMax = 0.8;   // largest contraction of a plain step
constexpr double kSubRhoMin = 0.15;  // smallest contraction that takes the second-order step
constexpr double kSubDrop = 1e-17;   // a factor I + E of the inverse with o max |E| below this is left out
constexpr double kSubInvMax = 1e-8;  // largest o max |M^8|: the next factor is its square
// per-molecule integers (kSubInts each)
constexpr int kSubPhase = 0;   // 0 full diagonalisation, 1 iterating, 2 converged, 3 given up, 4 density formed
constexpr int kSubPar = 1;     // which of the two X buffers holds X
constexpr int kSubX = 2;       // X belongs to the current C
constexpr int kSubOff = 3;     // attempts given up in this run
constexpr int kSubPend = 4;    // stopped without orbital energies: one diagonalisation to come
constexpr int kSubFresh = 5;   // X starts from the first-order guess
constexpr int kSubNext = 6;    // steps taken in this SCC iteration
constexpr int kSubMay = 7;     // may take the path in the next SCC iteration
constexpr int kSubInts = 8;
// residual maxima: one per step, then those of E_2 = M^4 and E_3 = M^8
constexpr int kSubRes = kSubSteps + 2;

// product kinds (the 64 x 64 tiles of a launch name theirs)
constexpr int kSubSym = 16;   // the tile is one of a symmetric result
enum SubOp { kSubB = 0, kSubR, kSubM, kSubCY, kSubE1, kSubZ2, kSubE, kSubZ, kSubCYZ, kSubP };

__device__ __forceinline__ int sub_occ(const MolDesc& md) { return md.nel / 2; }

// per-molecule doubles: tolerance of max |R|, the contraction allowed and the
// contraction seen, then the factor w of each step
constexpr int kSubTol = 0, kSubLim = 1, kSubRho = 2, kSubW = 3, kSubDbls = kSubW + kSubSteps;

// the contraction of a plain step that explains max |R| falling by r per step
// of the second-order iteration with factor w (r > sqrt(w - 1))
__device__ __forceinline__ double sub_mu(double r, double w) { return (r * r + w - 1.0) / (w * r); }

// step s is not needed: an earlier one converged (a step that did not run
// leaves its maximum at 0)
__device__ __forceinline__ bool sub_step_done(const unsigned long long* __restrict__ res,
                                              const double* __restrict__ sd, int s) {
  return s > 0 && __longlong_as_double((long long)res[s - 1]) <= sd[kSubTol];
}

// the full diagonalisation takes the molecule over
__device__ __forceinline__ void sub_give_up(int* si, MolState* st) {
  si[kSubPhase] = 3;
  si[kSubOff] += 1;
  si[kSubX] = 0;
  si[kSubPend] = 0;
  st->diag = 1;
}

// max |R| fell too slowly over the three steps before step s >= 5
__device__ __forceinline__ bool sub_slow(const unsigned long long* __restrict__ res, const double* __restrict__ sd,
                                         int s) {
  auto at = [&](int k) { return __longlong_as_double((long long)res[k]); };
  const double wl = sd[kSubW + s - 1], r = cbrt(at(s - 1) / at(s - 4));
  return !(r * r <= wl - 1.0 || sub_mu(r, wl) <= sd[kSubLim]);
}

// A molecule that converged with t residuals did so at a contraction that
// keeps the gap: of the last three steps, of the first one or two (which are
// plain) where there are fewer, of the SCC iteration before where X needed
// one step only
__device__ __forceinline__ bool sub_gap_kept(const unsigned long long* __restrict__ res,
                                             const double* __restrict__ sd, int t) {
  if (t >= 5) return !sub_slow(res, sd, t);
  if (t < 2) return sd[kSubRho] <= sd[kSubLim];
  const double r = __longlong_as_double((long long)res[min(t - 1, 2)]) / __longlong_as_double((long long)res[0]);
  return (t == 2 ? r : sqrt(r)) <= sd[kSubLim];
}

// one thread: the factor w of step s, or the end where max |R| is a NaN or
// falls too slowly (the mean of three steps: it may rise for one when w sets in)
__device__ __forceinline__ void sub_rate(const unsigned long long* __restrict__ res, double* sd, int* si,
                                         MolState* st, int s) {
  auto at = [&](int k) { return __longlong_as_double((long long)res[k]); };
  double rho = sd[kSubRho], w = 1.0;
  if (s > 0) {
    const double wl = sd[kSubW + s - 1];
    if (!(at(s - 1) < 1e300) || (s >= 5 && sub_slow(res, sd, s))) {
      sub_give_up(si, st);
      return;
    }
    const double r = s >= 4 ? cbrt(at(s - 1) / at(s - 4)) : 0.0;
    if (r * r > 1.1 * (wl - 1.0)) rho = fmax(rho, fmin(kSubRhoMax, sub_mu(r, wl)));
    sd[kSubRho] = rho;
    // the plain step is better as long as max |R| falls faster than the
    // second-order iteration's sqrt(w - 1)
    rho = fmin(rho, 0.95 * sd[kSubLim]);   // so that the optimal rate is not taken for a contraction over the limit
    if (s > 1 && rho >= kSubRhoMin) {
      const double wo = 2.0 / (1.0 + sqrt(1.0 - rho * rho)), r1 = at(s - 1) / at(s - 2);
      if (wl != 1.0 || r1 * r1 > wo - 1.0) w = wo;
    }
  }
  sd[kSubW + s] = w;
}

// E_k (k = 2, 3) is left out of the inverse
__device__ __forceinline__ bool sub_dropped(const unsigned long long* __restrict__ res, int o, int k) {
  return (double)o * __longlong_as_double((long long)res[kSubSteps + k - 2]) < kSubDrop;
}

// one workgroup per molecule: which path its SCC iteration takes.  MolState's
// diag = 1: full diagonalisation.
__global__ void __launch_bounds__(256) k_sub_begin(const MolDesc* __restrict__ desc, MolState* state,
                                                   const double* __restrict__ A, double* diag, int* sub,
                                                   unsigned long long* res, double* dbl, double jac_tol,
                                                   double min_gap, int allow) {
  __shared__ double sh[4];
  const int m = blockIdx.x;
  const MolDesc md = desc[m];
  MolState& st = state[m];
  int* si = sub + m * kSubInts;
  const int active = st.active, first = st.iter == 0;
  const int o = sub_occ(md), N = md.nao;
  const bool able = allow && active && !first && si[kSubMay];
  __syncthreads();
  bool on = false;
  double top = -1e300, low = -1e300, big = 0.0;   // max occupied, -min virtual
  if (able) {
    const double* Am = A + md.m0;
    for (int i = threadIdx.x; i < N; i += blockDim.x) {
      const double d = Am[(long long)i * N + i];
      diag[md.o0 + i] = d;
      if (i < o) top = fmax(top, d);
      else low = fmax(low, -d);
      big = fmax(big, fabs(d));
    }
    top = block_max<256>(top, sh);
    low = block_max<256>(low, sh);
    big = block_max<256>(big, sh);
    // the contraction that still guarantees the gap, with room for a rate
    on = (1.0 - kSubRhoMin) * (-low - top) >= min_gap;
    for (int s = threadIdx.x; s < kSubRes; s += blockDim.x) res[(long long)m * kSubRes + s] = 0ull;
  }
  if (threadIdx.x == 0) {
    if (first && active) si[kSubOff] = 0;
    if (active) {
      si[kSubPend] = 0;
      si[kSubFresh] = on && !si[kSubX];
      if (!on || si[kSubFresh]) si[kSubPar] = 0;
      si[kSubX] = on;
    }
    si[kSubPhase] = on ? 1 : 0;
    si[kSubNext] = 0;
    st.diag = active && !on ? 1 : 0;
    if (on) {
      double* sd = dbl + (long long)m * kSubDbls;
      sd[kSubTol] = jac_tol * fmax(big, 1.0);
      sd[kSubLim] = fmin(kSubRhoMax, 1.0 - min_gap / (-low - top));
      sd[kSubRho] = si[kSubFresh] ? 0.0 : 0.9 * sd[kSubRho];
    }
  }
}

// X = -A_vo / D of the molecules without one
__global__ void __launch_bounds__(256) k_sub_start(const MolDesc* __restrict__ desc, const double* __restrict__ A,
                                                   const double* __restrict__ diag, const int* __restrict__ sub,
                                                   double* X, int sub_wg) {
  const int m = blockIdx.y;
  const MolDesc md = desc[m];
  if (md.nao <= sub_wg || sub[m * kSubInts + kSubPhase] != 1 || !sub[m * kSubInts + kSubFresh]) return;
  const int N = md.nao, o = sub_occ(md), v = N - o;
  const double* Am = A + md.m0;
  const double* d = diag + md.o0;
  for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < (long long)v * o;
       t += (long long)gridDim.x * blockDim.x) {
    const int i = (int)(t / o), j = (int)(t % o);
    const double x = -Am[(long long)(o + i) * N + j] / (d[o + i] - d[j]);
    X[md.m0 + t] = x;
    X[md.m0 + 2LL * v * o + (long long)j * v + i] = x;
  }
}

// Buffers of the products (each N x N per molecule at m0): X holds X and its
// transpose twice (4 v o <= N^2: X of parity 0 and 1, then X^T of both); G,
// T, W, H, P are scratch (their own contents are dead between the Fock
// transform and the density).
struct SubBufs {
  const double *A, *C, *diag;
  double *X, *G, *T, *W, *H, *P;
};

// One wave's 32 x 32 block (row0, col0) of one product of a molecule
// (wave_mm).  Every operand but C is kept so that the product runs down its
// rows: A, the powers of M and the partial products Z are symmetric, X is
// kept with its transpose, C Y and C Y Z are formed transposed (o x N).
// Symmetric results (M, E_k = M^(2^k), Z_k, P) are formed on the upper blocks
// and mirrored.  Z_2 = (I - M)(I + E_1), Z_(k+1) = Z_k (I + E_k).
// par: the parity of X; ws: the factor w of the step (kSubR); level: k of E_k
// and Z_k; e2, e3: E_2, E_3 take part.  big: maximum (bit pattern) of |R|, |E|.
// Buffers: M, E_3 in G, E_1, Z_3 in P, E_2 in H, Z_2, Z_4 in W, (C Y)^T in T.
struct SubShape {
  int rows, cols;
};
__device__ __forceinline__ SubShape sub_shape(int op, int N, int o) {
  const int v = N - o;
  switch (op) {
    case kSubB: return {N, o};
    case kSubR: return {v, o};
    case kSubCY:
    case kSubCYZ: return {o, N};
    case kSubP: return {N, N};
    default: return {o, o};
  }
}

template <bool RMINOR>
__device__ __forceinline__ void sub_block(int op, int level, bool sym, const MolDesc& md, const SubBufs& bf, int par,
                                          double ws, bool e2, bool e3, int row0, int col0, unsigned long long& big) {
  const int N = md.nao, o = sub_occ(md), v = N - o;
  const long long vo = (long long)v * o;
  double* Xm = bf.X + md.m0;
  const double* X = Xm + par * vo;
  double* G = bf.G + md.m0;
  double* T = bf.T + md.m0;
  double* W = bf.W + md.m0;
  double* H = bf.H + md.m0;
  double* P = bf.P + md.m0;
  // result (M x Nc) = L^T R with L (K x M), R (K x Nc), or R (Nc x K) for C
  const double *Lp, *Rp;
  int ldl = o, ldr = o, M = o, Nc = o, K = o;
  switch (op) {
    case kSubB: Lp = bf.A + md.m0 + (long long)o * N; ldl = N; Rp = X; M = N; K = v; break;
    case kSubR: Lp = X + 2 * vo; ldl = v; Rp = G; M = v; break;
    case kSubM: Lp = X; Rp = X; K = v; break;
    case kSubCY: Lp = X; Rp = bf.C + md.m0 + o; ldr = N; Nc = N; K = v; break;
    case kSubE1: Lp = G; Rp = G; break;
    case kSubZ2: Lp = G; Rp = P; break;
    case kSubE:
      if (level == 3 && !e2) return;
      Lp = Rp = level == 2 ? P : H;
      break;
    case kSubZ:
      if (level == 3 ? !e2 : !e3) return;
      Lp = level == 3 ? W : P;
      Rp = level == 3 ? H : G;
      break;
    case kSubCYZ: Lp = e2 && !e3 ? P : W; Rp = T; ldr = N; Nc = N; break;
    default: Lp = G; ldl = N; Rp = T; ldr = N; M = Nc = N; break;
  }
  if (row0 >= M || col0 >= Nc || (sym && row0 > col0)) return;
  const int lane = threadIdx.x & 63, i16 = lane & 15, k4 = lane >> 4;
  v4d acc[2][2];
  wave_mm<RMINOR>(Lp, ldl, M, Rp, ldr, Nc, K, row0, col0, acc);
  // maxima on the bit patterns: a NaN counts as the largest value
  auto see = [&](double x) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(fabs(x));
    big = big > b ? big : b;
  };
  const double* dg = bf.diag + md.o0;
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int gj = col0 + 16 * c + i16;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int gi = row0 + 16 * r + k4 + 4 * i;
        if (gi >= M || gj >= Nc) continue;
        if (sym && gi > gj) continue;
        const long long e = (long long)gi * Nc + gj, et = (long long)gj * Nc + gi;
        const double x = acc[r][c][i];
        switch (op) {
          case kSubB: G[e] = bf.A[md.m0 + (long long)gi * N + gj] + x; break;
          case kSubR: {
            const double rr = G[(long long)(o + gi) * o + gj] - x;
            double* xn = Xm + (par ^ 1) * vo;   // holds the X before this one
            double x1 = X[e] - rr / (dg[o + gi] - dg[gj]);
            if (ws != 1.0) {
              const double x0 = xn[e];
              x1 = x0 + ws * (x1 - x0);
            }
            xn[e] = x1;
            xn[2 * vo + (long long)gj * v + gi] = x1;
            see(rr);
            break;
          }
          case kSubM: G[e] = x; G[et] = x; break;
          case kSubCY: T[e] = bf.C[md.m0 + (long long)gj * N + gi] + x; break;
          case kSubE1: P[e] = x; P[et] = x; break;
          case kSubZ2: {
            const double z = ((gi == gj ? 1.0 : 0.0) - G[e]) + (P[e] - x);
            W[e] = z;
            W[et] = z;
            break;
          }
          case kSubE: {
            double* E = level == 2 ? H : G;
            E[e] = x;
            E[et] = x;
            see(x);
            break;
          }
          case kSubZ: {
            double* Z = level == 3 ? P : W;
            const double z = (level == 3 ? W : P)[e] + x;
            Z[e] = z;
            Z[et] = z;
            break;
          }
          case kSubCYZ: G[e] = x; break;
          default: P[e] = 2.0 * x; P[et] = 2.0 * x; break;
        }
      }
    }
}

// A 64 x 64 tile of a product per workgroup, a wave per quarter; tiles
// (molecule, row tile, column tile, kind).  For the molecules above sub_wg.
template <bool RMINOR>
__global__ void __launch_bounds__(256) k_sub_gemm(const int4* __restrict__ tiles, const MolDesc* __restrict__ desc,
                                                  SubBufs bf, MolState* state, int* sub, unsigned long long* res,
                                                  double* dbl, int step, int level) {
  const int4 tl = tiles[blockIdx.x];
  const int m = tl.x, op = tl.w & 15;
  // (the last launch of the list of Z and E tiles forms Z_4 only: there is no
  // E_4, and no residual slot for its maximum)
  if (m < 0 || (op == kSubE && level > 3)) return;
  int* si = sub + m * kSubInts;
  if (si[kSubPhase] != (op <= kSubR ? 1 : 2)) return;
  unsigned long long* rs = res + (long long)m * kSubRes;
  double* sd = dbl + (long long)m * kSubDbls;
  const MolDesc md = desc[m];
  int par = si[kSubPar];
  if (op <= kSubR) {
    if (sub_step_done(rs, sd, step)) return;
    par = (par + step) & 1;
    // the first tile's workgroup sets the factor of this step for the second
    // product's launch, or gives the molecule up
    if (op == kSubB && tl.y == 0 && tl.z == 0 && threadIdx.x == 0) sub_rate(rs, sd, si, state + m, step);
  }
  const bool e2 = !sub_dropped(rs, sub_occ(md), 2), e3 = e2 && !sub_dropped(rs, sub_occ(md), 3);
  const int w = threadIdx.x >> 6;
  unsigned long long big = 0ull;
  sub_block<RMINOR>(op, level, (tl.w & kSubSym) != 0, md, bf, par, op == kSubR && step > 0 ? sd[kSubW + step] : 1.0,
                    e2, e3, tl.y * kTile + 32 * (w >> 1), tl.z * kTile + 32 * (w & 1), big);
  if (op == kSubR || op == kSubE) {
#pragma unroll
    for (int sft = 32; sft > 0; sft >>= 1) {
      const unsigned long long ob = __shfl_xor(big, sft, 64);
      big = big > ob ? big : ob;
    }
    // (most waves of a large molecule find a larger maximum there already)
    unsigned long long* to = op == kSubR ? &rs[step] : &rs[kSubSteps + level - 2];
    if ((threadIdx.x & 63) == 0 && big > __atomic_load_n(to, __ATOMIC_RELAXED)) atomicMax(to, big);
  }
}

// The whole of an SCC iteration's subspace path of one molecule in one
// workgroup (its waves share out the 32 x 32 blocks of a product): up to
// sub_wg orbitals a product is shorter than a launch, and a batch has a
// molecule for every compute unit.  One call site of the product (two with the
// row-minor C Y) in a loop over the sequence of kinds.  sub_wg_threads: a wave
// per block of the launch's largest molecule.  With 8 waves for every size the
// one that works is the first of each workgroup, and those of all workgroups
// of a compute unit share a SIMD (ms a run of 1000 molecules, with a
// diagonalisation in every iteration, 8 waves, now: 6 AOs 2.6, 4.3, 2.9; 24
// AOs 6.6, 7.8, 5.8; 60 AOs 18.5, 18.7, 16.5; one molecule unchanged).
inline int sub_wg_threads(int max_nao) { return max_nao <= 32 ? 64 : max_nao <= 64 ? 256 : 512; }
__global__ void __launch_bounds__(512) k_sub_wg(const int* __restrict__ list, const MolDesc* __restrict__ desc,
                                                SubBufs bf, MolState* state, int* sub, unsigned long long* res,
                                                double* dbl) {
  __shared__ unsigned long long top;
  __shared__ int phase, more;
  const int m = list[blockIdx.x];
  int* si = sub + m * kSubInts;
  if (si[kSubPhase] != 1) return;
  unsigned long long* rs = res + (long long)m * kSubRes;
  double* sd = dbl + (long long)m * kSubDbls;
  const MolDesc md = desc[m];
  const int N = md.nao, o = sub_occ(md), v = N - o;
  const int tid = threadIdx.x, w = tid >> 6, nw = blockDim.x >> 6;
  const int par0 = si[kSubPar];
  if (si[kSubFresh]) {
    const double* Am = bf.A + md.m0;
    const double* d = bf.diag + md.o0;
    double* X = bf.X + md.m0;
    for (int t = tid; t < v * o; t += blockDim.x) {
      const int i = t / o, j = t % o;
      const double x = -Am[(long long)(o + i) * N + j] / (d[o + i] - d[j]);
      X[t] = x;
      X[2LL * v * o + (long long)j * v + i] = x;
    }
  }
  // thread 0 decides between the two barriers after each product, when no wave
  // reads the shared words
  if (tid == 0) {
    top = 0ull;
    sub_rate(rs, sd, si, state + m, 0);
  }
  int op = kSubB, step = 0, level = 0;
  bool e2 = false, e3 = false;
  __syncthreads();
  for (;;) {
    const int par = (par0 + step) & 1;
    const bool sym = op == kSubM || op == kSubE1 || op == kSubZ2 || op == kSubE || op == kSubZ || op == kSubP;
    const SubShape sh = sub_shape(op, N, o);
    const int nr = (sh.rows + 31) / 32, nc = (sh.cols + 31) / 32;
    const double ws = op == kSubR && step > 0 ? sd[kSubW + step] : 1.0;
    unsigned long long big = 0ull;
    if (op == kSubCY) {
      for (int t = w; t < nr * nc; t += nw)
        sub_block<true>(op, level, sym, md, bf, par, ws, e2, e3, 32 * (t / nc), 32 * (t % nc), big);
    } else {
      // (the two kinds that share a launch run one after the other here)
      for (int t = w; t < nr * nc; t += nw)
        sub_block<false>(op, level, sym, md, bf, par, ws, e2, e3, 32 * (t / nc), 32 * (t % nc), big);
    }
    if (op == kSubR || op == kSubE) {
#pragma unroll
      for (int sft = 32; sft > 0; sft >>= 1) {
        const unsigned long long ob = __shfl_xor(big, sft, 64);
        big = big > ob ? big : ob;
      }
      if ((tid & 63) == 0) atomicMax(&top, big);
    }
    __syncthreads();
    if (tid == 0) {
      more = 1;
      if (op == kSubR) {
        rs[step] = top;
        if (sub_step_done(rs, sd, step + 1)) {
          more = 0;
          if (!sub_gap_kept(rs, sd, step + 1)) sub_give_up(si, state + m);
        } else if (step + 1 >= kSubSteps) sub_give_up(si, state + m);
        else sub_rate(rs, sd, si, state + m, step + 1);
      } else if (op == kSubE) {
        rs[kSubSteps + level - 2] = top;
        if (level == 3 && !((double)o * __longlong_as_double((long long)top) <= kSubInvMax)) sub_give_up(si, state + m);
      }
      top = 0ull;
      phase = si[kSubPhase];
    }
    __syncthreads();
    if (phase != 1) return;   // given up
    // the next product
    if (op == kSubB) op = kSubR;
    else if (op == kSubR) {
      ++step;
      op = more ? kSubB : kSubM;
    } else if (op == kSubM) op = kSubCY;
    else if (op == kSubCY) op = kSubE1;
    else if (op == kSubE1) op = kSubZ2;
    else if (op == kSubZ2) {
      op = kSubE;
      level = 2;
    } else if (op == kSubE) {
      if (level == 2) e2 = !sub_dropped(rs, o, 2);
      else e3 = e2 && !sub_dropped(rs, o, 3);
      // E_2, Z_3, E_3, Z_4
      if (level == 2 && e2) {
        op = kSubZ;
        level = 3;
      } else if (level == 3 && e3) {
        op = kSubZ;
        level = 4;
      } else {
        op = kSubCYZ;
      }
    } else if (op == kSubZ) {
      op = level == 3 ? kSubE : kSubCYZ;
    } else if (op == kSubCYZ) op = kSubP;
    else break;
  }
  if (tid == 0) {
    si[kSubPar] = (par0 + step) & 1;
    si[kSubNext] = step;
    si[kSubPend] = 1;
    si[kSubPhase] = 4;
  }
}

// after the steps [0, nstep): converged molecules to phase 2, given up ones
// to phase 3 with a full diagonalisation; densities formed before to phase 4
__global__ void k_sub_outcome(MolState* state, int nmol, int* sub, const unsigned long long* __restrict__ res,
                              const double* __restrict__ dbl, const MolDesc* __restrict__ desc, int sub_wg,
                              int nstep) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= nmol || desc[m].nao <= sub_wg) return;
  int* si = sub + m * kSubInts;
  if (si[kSubPhase] == 2) si[kSubPhase] = 4;
  if (si[kSubPhase] != 1) return;
  const unsigned long long* rs = res + (long long)m * kSubRes;
  const double* sd = dbl + (long long)m * kSubDbls;
  int t = 0;
  while (t < nstep && !sub_step_done(rs, sd, t)) ++t;
  si[kSubNext] = t;
  if (sub_step_done(rs, sd, t)) {
    if (!sub_gap_kept(rs, sd, t)) {
      sub_give_up(si, state + m);
      return;
    }
    si[kSubPhase] = 2;
    si[kSubPar] = (si[kSubPar] + t) & 1;
    si[kSubPend] = 1;
  } else if (t >= kSubSteps) {
    sub_give_up(si, state + m);
  }
}

// after the powers of M: a molecule whose inverse would need another factor
// (X too large) takes the full diagonalisation instead.
// cnt[0]: still iterating, cnt[1]: full diagonalisations, cnt[2]: most steps
// (of the molecules above sub_wg)
__global__ void __launch_bounds__(256) k_sub_check(const MolDesc* __restrict__ desc, MolState* state, int nmol,
                                                   int* sub, const unsigned long long* __restrict__ res, int sub_wg,
                                                   int* cnt) {
  __shared__ double sh[4];
  double run = 0.0, full = 0.0, most = 0.0;
  for (int m = threadIdx.x; m < nmol; m += blockDim.x) {
    int* si = sub + m * kSubInts;
    if (si[kSubPhase] == 2) {
      const double e3 = __longlong_as_double((long long)res[(long long)m * kSubRes + kSubSteps + 1]);
      if (!(sub_occ(desc[m]) * e3 <= kSubInvMax)) {
        sub_give_up(si, state + m);
      }
    }
    if (si[kSubPhase] == 1) run += 1.0;
    if (si[kSubPhase] != 0 && desc[m].nao > sub_wg) most = fmax(most, (double)si[kSubNext]);
    full += state[m].diag ? 1.0 : 0.0;
  }
  run = block_sum<256>(run, sh);
  full = block_sum<256>(full, sh);
  most = block_max<256>(most, sh);
  if (threadIdx.x == 0) {
    cnt[0] = (int)run;
    cnt[1] = (int)full;
    cnt[2] = (int)most;
  }
}

// after an SCC iteration, cnt[0]: molecules still iterating, cnt[1]: those of
// them that may take the path in the next one (kSubMay; closed shells with
// occupied and virtual orbitals, on the path now or with a gap of the last
// orbitals that k_sub_begin would ask of the diagonal: below it the iteration
// would queue the path's launches and wait for their counts for nothing, 8.9
// instead of 8.2 ms for a polyene of 20 carbons, gap 1.45 eV)
__global__ void __launch_bounds__(256) k_sub_next(const MolDesc* __restrict__ desc, const MolState* __restrict__ state,
                                                  int nmol, int* sub, const double* __restrict__ emo, double min_gap,
                                                  int* cnt) {
  __shared__ double sh[4];
  double run = 0.0, may = 0.0;
  for (int m = threadIdx.x; m < nmol; m += blockDim.x) {
    const MolDesc& md = desc[m];
    int* si = sub + m * kSubInts;
    const int o = sub_occ(md);
    bool on = state[m].active && si[kSubOff] < kSubTries && md.nopen == 0 && (md.nel & 1) == 0 && md.n > 1 && o >= 1 &&
              o < md.nao;
    if (on && si[kSubPhase] != 2 && si[kSubPhase] != 4) {
      const double* e = emo + md.o0;
      on = (1.0 - kSubRhoMin) * (e[o] - e[o - 1]) >= min_gap;
    }
    si[kSubMay] = on ? 1 : 0;
    run += state[m].active ? 1.0 : 0.0;
    may += on ? 1.0 : 0.0;
  }
  run = block_sum<256>(run, sh);
  may = block_sum<256>(may, sh);
  if (threadIdx.x == 0) {
    cnt[0] = (int)run;
    cnt[1] = (int)may;
  }
}

// molecules that stopped iterating without orbital energies: diag = 1
__global__ void __launch_bounds__(256) k_sub_pending(MolState* state, int nmol, int* sub, int* cnt) {
  __shared__ double sh[4];
  double c = 0.0;
  for (int m = threadIdx.x; m < nmol; m += blockDim.x) {
    int* si = sub + m * kSubInts;
    const bool p = !state[m].active && !state[m].failed && si[kSubPend];
    state[m].diag = p ? 1 : 0;
    if (p) {
      si[kSubPend] = 0;
      si[kSubX] = 0;
      c += 1.0;
    }
  }
  c = block_sum<256>(c, sh);
  if (threadIdx.x == 0) cnt[0] = (int)c;
}

// ---------------------------------------------------------------------------
// The last diagonalisation of a molecule on the subspace path: with X known,
//
//     U = [ Qo  -(X Qo)^T ]      Qo = (I + X^T X)^(-1/2)
//         [ X Qo     Qv   ]      Qv = (I + X X^T)^(-1/2)   (X Qo = Qv X)
//
// is orthogonal and U^T A U falls into an occupied and a virtual block (what
// couples them is R, below the tolerance of a finished diagonalisation), so
// two problems of about half the size are left: half the rounds per sweep
// and a quarter of the elements per round each.
// The inverse square roots start from I - M / 2 + 3 M^2 / 8 (error 5 M^3 / 16)
// and take one step Q <- Q (3 I - Q^2 (I + M)) / 2 (error e -> 3 e^2 / 4), a
// second one where M^6 is not below rounding.  The error after the second is
// not looked at: the path admits o max |M^8| up to 1e-8, so ||M|| up to 0.1,
// whose start of 3e-4 leaves 7e-8 after the first step and 4e-15 after the
// second, the size of the rounding of the rotation's products.
constexpr int kRotVirt = 8;   // a kind + kRotVirt: the same for the virtual block (not kRotU)
enum RotOp { kRotM = 0, kRotQ1, kRotS, kRotG, kRotQ, kRotU };
constexpr double kRotOne = 1e-10;   // o max |M^4| up to which one step is enough

__device__ __forceinline__ bool rot_two(const unsigned long long* __restrict__ res, int o) {
  return !((double)o * __longlong_as_double((long long)res[kSubSteps]) < kRotOne);
}

// M in G, the Q of level 0 in W and of level 1 in H (both blocks in one N x N
// buffer: o x o, then v x v); U replaces M in G
__global__ void __launch_bounds__(256) k_rot_gemm(const int4* __restrict__ tiles, const MolDesc* __restrict__ desc,
                                                  SubBufs bf, const MolState* __restrict__ state,
                                                  const int* __restrict__ sub,
                                                  const unsigned long long* __restrict__ res, int level) {
  const int4 tl = tiles[blockIdx.x];
  const int m = tl.x, op = tl.w & 7;
  if (m < 0 || !state[m].diag) return;
  const bool virt = (tl.w & kRotVirt) != 0, sym = (tl.w & kSubSym) != 0;
  const MolDesc md = desc[m];
  const int N = md.nao, o = sub_occ(md), v = N - o;
  const bool two = rot_two(res + (long long)m * kSubRes, o);
  if (level > 0 && !two) return;
  const long long vo = (long long)v * o, off = md.m0 + (virt ? (long long)o * o : 0);
  const double* X = bf.X + md.m0 + sub[m * kSubInts + kSubPar] * vo;
  double* Mb = bf.G + off;
  double* T = bf.T + off;
  double* cur = (level & 1 ? bf.H : bf.W) + off;
  double* oth = (level & 1 ? bf.W : bf.H) + off;
  const int nb = virt ? v : o;
  const double *Lp = cur, *Rp = cur;
  int ldl = nb, M = nb, K = nb;
  switch (op) {
    case kRotM: Lp = Rp = virt ? X + 2 * vo : X; K = N - nb; break;
    case kRotQ1: Lp = Rp = Mb; break;
    case kRotS: break;
    case kRotG: Lp = oth; Rp = Mb; break;
    case kRotQ: Rp = T; break;
    default: Lp = X + 2 * vo; ldl = v; M = v; Rp = (two ? bf.W : bf.H) + md.m0; break;
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, i16 = lane & 15, k4 = lane >> 4;
  const int row0 = tl.y * kTile + 32 * (w >> 1), col0 = tl.z * kTile + 32 * (w & 1);
  if (row0 >= M || col0 >= nb || (sym && row0 > col0)) return;
  v4d acc[2][2];
  wave_mm<false>(Lp, ldl, M, Rp, nb, nb, K, row0, col0, acc);
  double* U = bf.G + md.m0;
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int gj = col0 + 16 * c + i16;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int gi = row0 + 16 * r + k4 + 4 * i;
        if (gi >= M || gj >= nb || (sym && gi > gj)) continue;
        const long long e = (long long)gi * nb + gj, et = (long long)gj * nb + gi;
        const double x = acc[r][c][i], one = gi == gj ? 1.0 : 0.0;
        switch (op) {
          case kRotM: Mb[e] = x; Mb[et] = x; break;
          case kRotQ1: {
            const double y = one - 0.5 * Mb[e] + 0.375 * x;
            cur[e] = y;
            cur[et] = y;
            break;
          }
          case kRotS: oth[e] = x; oth[et] = x; break;
          case kRotG: {
            const double y = 1.5 * one - 0.5 * (oth[e] + x);
            T[e] = y;
            T[et] = y;
            break;
          }
          case kRotQ: oth[e] = x; oth[et] = x; break;
          default:
            U[(long long)(o + gi) * N + gj] = x;
            U[(long long)gj * N + o + gi] = -x;
            break;
        }
      }
    }
}

// the diagonal blocks of U
__global__ void __launch_bounds__(256) k_rot_diag(const MolDesc* __restrict__ desc, const MolState* __restrict__ state,
                                                  const unsigned long long* __restrict__ res,
                                                  const double* __restrict__ W, const double* __restrict__ H,
                                                  double* U) {
  const int m = blockIdx.y;
  if (!state[m].diag) return;
  const MolDesc md = desc[m];
  const int N = md.nao, o = sub_occ(md), v = N - o;
  const double* Q = (rot_two(res + (long long)m * kSubRes, o) ? W : H) + md.m0;
  const long long oo = (long long)o * o, all = oo + (long long)v * v;
  for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < all; t += (long long)gridDim.x * blockDim.x) {
    const long long u = t < oo ? t : t - oo;
    const int nb = t < oo ? o : v, r0 = t < oo ? 0 : o;
    U[md.m0 + (r0 + u / nb) * N + r0 + u % nb] = Q[t];
  }
}

}  // namespace xtbamd
