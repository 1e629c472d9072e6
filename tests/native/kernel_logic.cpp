// Host runs of the bookkeeping of single kernels (one lane, see
// hip/hip_runtime.h beside this file).  kernel_logic CHECK: exit status 0 if
// the check holds.
#include <hip/hip_runtime.h>
#include <sys/mman.h>
#include <unistd.h>

#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>

#include "k_linalg.hip"
#include "k_sub.hip"

using namespace xtbamd;
namespace xtbamd {
thread_local double lds[1];   // the dynamic LDS of a kernel that is not run here
}

// an array whose end is the end of a readable page: a read behind it faults
template <class T>
T* guarded(size_t n) {
  const size_t page = (size_t)sysconf(_SC_PAGESIZE), bytes = n * sizeof(T), room = (bytes + page - 1) / page * page;
  char* p = (char*)mmap(nullptr, room + page, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
  if (p == MAP_FAILED || mprotect(p + room, page, PROT_NONE) != 0) std::abort();
  return (T*)(p + room - bytes);
}

static int failures = 0;
#define EXPECT(c)                                                     \
  do {                                                                \
    if (!(c)) {                                                       \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c);             \
      ++failures;                                                     \
    }                                                                 \
  } while (0)

// one closed-shell molecule of N orbitals, o of them occupied, on the subspace path
struct One {
  MolDesc md;
  MolState st;
  int* si = guarded<int>(kSubInts);
  unsigned long long* res = guarded<unsigned long long>(kSubRes);
  double* sd = guarded<double>(kSubDbls);
  std::vector<double> A, C, ev, X, G, T, W, H, P;
  One(int N, int o) {
    std::memset(&md, 0, sizeof(md));
    std::memset(&st, 0, sizeof(st));
    md.n = 2;
    md.nao = N;
    md.nel = 2 * o;
    st.active = 1;
    for (auto* v : {&A, &C, &X, &G, &T, &W, &H, &P}) v->assign((size_t)N * N, 0.0);
    for (int i = 0; i < N; ++i) ev.push_back(i < o ? -10.0 : 5.0);
  }
  SubBufs bufs() { return SubBufs{A.data(), C.data(), ev.data(), X.data(), G.data(), T.data(), W.data(), H.data(), P.data()}; }
};

// every product launch of an iteration stays inside the molecule's residuals
// and factors, those of the last molecule of the batch too
static void sub_products() {
  One m(80, 30);
  const int steps[] = {0, 1, kSubSteps - 1};
  const int dens[][2] = {{kSubM, 0}, {kSubCY, 0}, {kSubE1, 0}, {kSubZ2, 2}, {kSubE, 2}, {kSubZ, 3},
                         {kSubE, 3}, {kSubZ, 4},  {kSubE, 4},  {kSubCYZ, 0}, {kSubP, 0}};
  for (int s : steps)
    for (int op : {(int)kSubB, (int)kSubR}) {
      m.si[kSubPhase] = 1;
      m.sd[kSubTol] = -1.0;
      int4 tile{0, 0, 0, op};
      k_sub_gemm<false>(&tile, &m.md, m.bufs(), &m.st, m.si, m.res, m.sd, s, 0);
    }
  for (auto& d : dens) {
    m.si[kSubPhase] = 2;
    m.res[kSubSteps] = m.res[kSubSteps + 1] = (unsigned long long)__double_as_longlong(1e-3);
    std::printf("product %d level %d\n", d[0], d[1]);
    std::fflush(stdout);
    int4 tile{0, 0, 0, d[0] == kSubCY || d[0] == kSubCYZ ? d[0] : d[0] | kSubSym};
    if (d[0] == kSubCY)
      k_sub_gemm<true>(&tile, &m.md, m.bufs(), &m.st, m.si, m.res, m.sd, 0, d[1]);
    else
      k_sub_gemm<false>(&tile, &m.md, m.bufs(), &m.st, m.si, m.res, m.sd, 0, d[1]);
  }
}

// a lane's count and marks take every problem of the lane that k_jac_small
// does not solve, whatever its size; a problem that left the rounds
// unfinished fails its molecule
static void jacobi_unfinished() {
  const int n = 5;
  JacobiProb pr[n];
  MolState st[n];
  std::memset(pr, 0, sizeof(pr));
  std::memset(st, 0, sizeof(st));
  int state[n * kJacState] = {}, active = -1;
  double scale[n];
  unsigned long long off[2 * n] = {};
  const int dim[n] = {48, 80, 48, 20, 0}, small[n] = {0, 0, 0, 1, 1};
  for (int p = 0; p < n; ++p) {
    pr[p].dim = dim[p];
    pr[p].small = small[p];
    pr[p].mol = p;
    pr[p].nb = (dim[p] + 15) / 16;
    pr[p].nbp = pr[p].nb + (pr[p].nb & 1);
    pr[p].rounds = std::max(1, pr[p].nbp - 1);
    pr[p].maxsw = 40;
    scale[p] = 1.0;
    st[p].active = st[p].diag = 1;
    off[p] = (unsigned long long)__double_as_longlong(p == 2 ? 1e-15 : 1.0);
  }
  pr[1].group = 1;
  state[3 * kJacState] = 1;   // k_jac_small's
  k_jac_count(pr, n, state, 0, &active);
  EXPECT(active == 2);
  k_jac_count(pr, n, state, 1, &active);
  EXPECT(active == 1);
  k_jac_mark(pr, n, scale, state, off, 0, &active, 1e-12, -1);
  EXPECT(active == 2 && state[2 * kJacState] == 1 && state[0] == 0);
  state[1 * kJacState] = state[1 * kJacState + 1] = 1;   // given up
  for (unsigned p = 0; p < n + 1; ++p) {
    blockIdx.x = p;
    k_jac_fold(pr, n, state, st, 3);
  }
  blockIdx.x = 0;
  EXPECT(st[0].failed == 3 && st[0].active == 0);   // unfinished
  EXPECT(st[1].failed == 3 && st[1].active == 0);
  for (int p = 2; p < n; ++p) EXPECT(st[p].failed == 0 && st[p].active == 1);
}

// a molecule that converges within few steps is held to the contraction that
// its gap allows, too
static void sub_contraction() {
  // residuals, allowed contraction, carried one, factor of the later steps; stays on the path
  struct {
    std::vector<double> r;
    double lim, rho, w;
    bool stays;
  } cases[] = {
      {{2e-11}, 0.3, 0.0, 1.0, true},
      {{2e-11}, 0.3, 0.5, 1.0, false},
      {{1e-9, 2e-11}, 0.3, 0.2, 1.0, true},
      {{1e-9, 2e-11}, 0.01, 0.0, 1.0, false},
      {{6e-11, 2.5e-11}, 0.3, 0.0, 1.0, false},
      {{1e-10, 7e-11, 4.9e-11, 2.9e-11}, 0.3, 0.0, 1.0, false},
      {{1e-10, 7e-11, 4.9e-11, 2.9e-11}, 0.8, 0.0, 1.0, true},
      {{1e-3, 1e-4, 1e-5, 1e-6, 1e-7, 1e-11}, 0.3, 0.0, 1.0, true},
      {{1e-9, 1e-10, 6e-11, 5e-11, 4e-11, 2.9e-11}, 0.3, 0.0, 1.0, false},
      // second-order steps: falling by sqrt(w - 1) is their optimum
      {{1e-9, 4e-10, 2e-10, 9e-11, 5e-11, 2.5e-11}, 0.8, 0.6, 1.2, true},
  };
  for (auto& c : cases) {
    One m(80, 30);
    const int t = (int)c.r.size();
    m.si[kSubPhase] = 1;
    m.sd[kSubTol] = 3e-11;
    m.sd[kSubLim] = c.lim;
    m.sd[kSubRho] = c.rho;
    for (int s = 0; s < t; ++s) {
      m.res[s] = (unsigned long long)__double_as_longlong(c.r[s]);
      m.sd[kSubW + s] = s > 1 ? c.w : 1.0;
    }
    k_sub_outcome(&m.st, 1, m.si, m.res, m.sd, &m.md, 64, kSubSteps);
    std::printf("%d steps, limit %g: phase %d\n", t, c.lim, m.si[kSubPhase]);
    EXPECT(m.si[kSubNext] == t);
    EXPECT(m.si[kSubPhase] == (c.stays ? 2 : 3));
    EXPECT(m.st.diag == (c.stays ? 0 : 1) && m.si[kSubOff] == (c.stays ? 0 : 1));
  }
}

// who may take the path in the next iteration: not the molecules that gave up,
// open shells, filled bases and gaps far below the bound
static void sub_next() {
  struct {
    int active, off, nopen, nel, nao, phase;
    double gap;
    bool may;
  } cases[] = {{1, 0, 0, 8, 6, 0, 4.0, true},  {1, 0, 0, 8, 6, 0, 1.0, false}, {1, 0, 0, 8, 6, 2, 1.0, true},
               {1, 0, 0, 8, 6, 4, 1.0, true},  {1, 1, 0, 8, 6, 3, 4.0, true},  {1, 2, 0, 8, 6, 3, 4.0, false},
               {0, 0, 0, 8, 6, 4, 4.0, false}, {1, 0, 1, 7, 6, 0, 4.0, false}, {1, 0, 0, 12, 6, 0, 4.0, false}};
  for (auto& c : cases) {
    MolDesc md;
    MolState st;
    std::memset(&md, 0, sizeof(md));
    std::memset(&st, 0, sizeof(st));
    md.n = 3;
    md.nao = c.nao;
    md.nel = c.nel;
    md.nopen = c.nopen;
    st.active = c.active;
    int* si = guarded<int>(kSubInts);
    int* cnt = guarded<int>(2);
    double* e = guarded<double>(c.nao);
    si[kSubOff] = c.off;
    si[kSubPhase] = c.phase;
    for (int i = 0; i < c.nao; ++i) e[i] = i < c.nel / 2 ? -12.0 : -12.0 + c.gap;
    k_sub_next(&md, &st, 1, si, e, 1.344, cnt);
    EXPECT(cnt[0] == c.active && cnt[1] == (c.may ? 1 : 0) && si[kSubMay] == cnt[1]);
  }
}

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "sub_products") sub_products();
  else if (what == "jacobi_unfinished") jacobi_unfinished();
  else if (what == "sub_contraction") sub_contraction();
  else if (what == "sub_next") sub_next();
  else return 2;
  return failures ? 1 : 0;
}
