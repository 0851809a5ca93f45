// Line kernels of the assembly compiled for the host, one thread per lane:
// every element record, table, equation number and matrix position that they
// touch lies in an array of exactly its size (address sanitizer), and the sums
// equal direct quadrature over the elements.
//
//   main P NG NC fp32 rhs accum nel1 nel2 nel3 nseg fix gval
//   main long
//
// with CONFIG defined as CASE(P, NG, NC) for the degree, points and components
// to build.
// fix: 0 none, 1 all faces, 2 the face u = 0, 3 at random.  accum: 0 own rows,
// 1 shared rows found by search, 2 shared rows with positions, 3 a work list
// of one-patch items (scalar, FP32 without and FP64 with right-hand side).
#include "lines.hpp"

#include <sys/mman.h>

#include <barrier>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <memory>
#include <random>
#include <thread>
#include <vector>

using namespace ifem;

thread_local HostDim threadIdx, blockIdx;

// ---- a workgroup of threads -----------------------------------------------------
static std::unique_ptr<std::barrier<>> group_barrier;
static std::vector<std::unique_ptr<std::barrier<>>> wave_barrier;
static bool votes[16][64];
static double lanes[16][64];

void host_barrier() { group_barrier->arrive_and_wait(); }

bool host_wave_votes(bool vote, unsigned long long* mask)
{
  const int w = threadIdx.x >> 6;
  votes[w][threadIdx.x & 63] = vote;
  wave_barrier[w]->arrive_and_wait();
  for (int l = 0; l < 64; l++)
    if (votes[w][l]) *mask |= 1ull << l;
  wave_barrier[w]->arrive_and_wait();
  return vote;
}

double host_wave_swap(double v, int from)
{
  const int w = threadIdx.x >> 6;
  lanes[w][threadIdx.x & 63] = v;
  wave_barrier[w]->arrive_and_wait();
  const double r = lanes[w][from];
  wave_barrier[w]->arrive_and_wait();
  return r;
}

template <typename F>
static void launch(int threads, int blocks, F kernel)
{
  group_barrier = std::make_unique<std::barrier<>>(threads);
  wave_barrier.clear();
  for (int w = 0; w < threads / 64; w++) wave_barrier.push_back(std::make_unique<std::barrier<>>(64));
  std::vector<std::thread> th;
  for (int t = 0; t < threads; t++)
    th.emplace_back([=] {
      for (int b = 0; b < blocks; b++) {
        threadIdx.x = t;
        blockIdx.x = b;
        kernel();
        group_barrier->arrive_and_wait();
      }
    });
  for (std::thread& t : th) t.join();
}

// ---- a system with random tables and records --------------------------------------
static std::mt19937_64 engine(7);
static double uniform() { return std::uniform_real_distribution<double>(-1.0, 1.0)(engine); }

struct System {
  int P, NG, NC, n[3], nel[3];
  std::vector<double> N[3], D[3], geo, gval;
  std::vector<int> eq, ci;
  std::vector<int64_t> rp;
  int neq = 0;

  int node(int i, int j, int k) const { return i + n[0] * (j + n[1] * k); }
  bool inside(int i, int j, int k) const
  {
    return i >= 0 && j >= 0 && k >= 0 && i < n[0] && j < n[1] && k < n[2];
  }
  int records() const { return NC == 1 ? GeoRec<1>::N : GeoRec<3>::N; }

  System(int p, int ng, int nc, const int* ne, int fix, int first_free = 0) : P(p), NG(ng), NC(nc)
  {
    for (int d = 0; d < 3; d++) {
      nel[d] = ne[d];
      n[d] = ne[d] + P;
      N[d].resize((size_t)nel[d] * NG * (P + 1));
      D[d].resize(N[d].size());
      for (double& v : N[d]) v = uniform();
      for (double& v : D[d]) v = uniform();
    }
    geo.resize((size_t)nel[0] * nel[1] * nel[2] * records() * NG * NG * NG);
    for (double& v : geo) v = uniform();
    eq.resize((size_t)n[0] * n[1] * n[2] * NC);
    gval.resize(eq.size());
    for (size_t q = 0; q < eq.size(); q++) {
      const int nd = (int)(q / NC), i = nd % n[0], j = (nd / n[0]) % n[1], k = nd / (n[0] * n[1]);
      bool fixed = i < first_free;
      if (fix == 1) fixed |= i == 0 || i == n[0] - 1 || j == 0 || j == n[1] - 1 || k == 0 || k == n[2] - 1;
      if (fix == 2) fixed |= i == 0;
      if (fix == 3) fixed |= uniform() > 0.7;
      eq[q] = fixed ? -1 : neq++;
      gval[q] = fixed ? uniform() : 0.0;
    }
    rp.assign(neq + 1, 0);
    each_row([&](int r, int i, int j, int k) {
      each_neighbour(i, j, k, [&](int nb) {
        for (int c = 0; c < NC; c++)
          if (eq[nb * NC + c] >= 0) ci.push_back(eq[nb * NC + c]);
      });
      rp[r + 1] = (int64_t)ci.size();
    });
  }
  template <typename F>
  void each_row(F f) const
  {
    for (size_t q = 0; q < eq.size(); q++) {
      const int nd = (int)(q / NC);
      if (eq[q] >= 0) f(eq[q], nd % n[0], (nd / n[0]) % n[1], nd / (n[0] * n[1]));
    }
  }
  template <typename F>
  void each_neighbour(int i, int j, int k, F f) const
  {
    for (int dk = -P; dk <= P; dk++)
      for (int dj = -P; dj <= P; dj++)
        for (int di = -P; di <= P; di++)
          if (inside(i + di, j + dj, k + dk)) f(node(i + di, j + dj, k + dk));
  }

  AsmArgs args() const
  {
    AsmArgs a{};
    a.n1 = n[0], a.n2 = n[1], a.n3 = n[2];
    a.nel1 = nel[0], a.nel2 = nel[1], a.nel3 = nel[2];
    a.tabN1 = N[0].data(), a.tabN2 = N[1].data(), a.tabN3 = N[2].data();
    a.tabD1 = D[0].data(), a.tabD2 = D[1].data(), a.tabD3 = D[2].data();
    a.gp_geo = const_cast<double*>(geo.data());
    a.lam = 0.7, a.mu = 0.4;
    a.body[0] = 0.3, a.body[1] = -1.1, a.body[2] = 0.6;
    a.ncomp = NC, a.ng = NG;
    a.eq = eq.data();
    a.rowptr = rp.data();
    a.colind = ci.data();
    return a;
  }

  // K and b by direct quadrature, element by element
  void reference(std::vector<double>& K, std::vector<double>& b, bool rhs, bool prescribed) const
  {
    const int P1 = P + 1, nen = P1 * P1 * P1, gp3 = NG * NG * NG;
    K.assign(ci.size(), 0.0);
    b.assign(neq, 0.0);
    std::vector<double> g(3 * nen), val(nen);
    for (int e = 0; e < nel[0] * nel[1] * nel[2]; e++) {
      const int e1 = e % nel[0], e2 = (e / nel[0]) % nel[1], e3 = e / (nel[0] * nel[1]);
      const double* R = geo.data() + (size_t)e * records() * gp3;
      std::vector<double> Ke((size_t)nen * NC * nen * NC, 0.0), fe((size_t)nen * NC, 0.0);
      for (int q = 0; q < gp3; q++) {
        const int at1 = (e1 * NG + q % NG) * P1, at2 = (e2 * NG + (q / NG) % NG) * P1,
                  at3 = (e3 * NG + q / (NG * NG)) * P1;
        auto rec = [&](int c) { return R[c * gp3 + q]; };
        for (int x = 0; x < nen; x++) {
          const int x1 = at1 + x % P1, x2 = at2 + (x / P1) % P1, x3 = at3 + x / (P1 * P1);
          const double d[3] = {D[0][x1] * N[1][x2] * N[2][x3], N[0][x1] * D[1][x2] * N[2][x3],
                               N[0][x1] * N[1][x2] * D[2][x3]};
          val[x] = N[0][x1] * N[1][x2] * N[2][x3];
          for (int i = 0; i < 3; i++)
            g[3 * x + i] = NC == 1 ? d[i] : d[0] * rec(i) + d[1] * rec(3 + i) + d[2] * rec(6 + i);
        }
        for (int x = 0; x < nen; x++) {
          for (int i = 0; rhs && i < NC; i++) {
            const double body[3] = {0.3, -1.1, 0.6};
            fe[x * NC + i] += NC == 1 ? rec(6) * val[x] : rec(9) * val[x] * body[i];
          }
          for (int y = 0; y < nen; y++) {
            const double *u = &g[3 * x], *v = &g[3 * y];
            if (NC == 1) {
              Ke[x * nen + y] += u[0] * (rec(0) * v[0] + rec(1) * v[1] + rec(2) * v[2]) +
                                 u[1] * (rec(1) * v[0] + rec(3) * v[1] + rec(4) * v[2]) +
                                 u[2] * (rec(2) * v[0] + rec(4) * v[1] + rec(5) * v[2]);
              continue;
            }
            const double dot = u[0] * v[0] + u[1] * v[1] + u[2] * v[2];
            for (int i = 0; i < 3; i++)
              for (int j = 0; j < 3; j++)
                Ke[(size_t)(x * 3 + i) * nen * 3 + y * 3 + j] +=
                    rec(9) * (0.7 * u[i] * v[j] + 0.4 * u[j] * v[i] + (i == j ? 0.4 * dot : 0.0));
          }
        }
      }
      auto dof = [&](int z) {
        const int x = z / NC;
        return node(e1 + x % P1, e2 + (x / P1) % P1, e3 + x / (P1 * P1)) * NC + z % NC;
      };
      for (int x = 0; x < nen * NC; x++) {
        const int r = eq[dof(x)];
        if (r < 0) continue;
        b[r] += fe[x];
        for (int y = 0; y < nen * NC; y++) {
          const double v = Ke[(size_t)x * nen * NC + y];
          const int c = eq[dof(y)];
          if (c < 0) {
            if (prescribed) b[r] -= v * gval[dof(y)];
            continue;
          }
          int64_t at = rp[r];
          while (ci[at] != c) at++;
          K[at] += v;
        }
      }
    }
  }
};

static double difference(const std::vector<double>& a, const std::vector<double>& ref, double base)
{
  double d = 0.0, m = 1e-300;
  for (size_t q = 0; q < ref.size(); q++) {
    const double e = std::fabs(a[q] - base - ref[q]);
    d = e <= 1e300 ? std::fmax(d, e) : 1e300; // not a number: not written
    m = std::fmax(m, std::fabs(ref[q]));
  }
  return d / m;
}

template <int P, int NG, int NC, typename T, bool RHS>
static int run(int accum, const int* nel, int nseg, int fix, bool prescribed)
{
  using C = LineCfg<P, NG, NC>;
  System s(P, NG, NC, nel, fix);
  constexpr bool F32 = sizeof(T) == 4;
  const bool shared = accum == 1 || accum == 2;
  const double base = shared ? 1.0 : NAN, zero = shared ? 1.0 : 0.0;
  std::vector<double> K, b, val(F32 ? 0 : s.ci.size(), base), rhs(F32 ? 0 : s.neq, base);
  std::vector<float> val32(F32 ? s.ci.size() : 0, (float)base);
  s.reference(K, b, RHS, prescribed && !F32);
  AsmArgs a = s.args();
  a.val64 = F32 ? nullptr : val.data();
  a.val32 = F32 ? val32.data() : nullptr;
  a.rhs = F32 ? nullptr : rhs.data();
  a.gval = prescribed && !F32 ? s.gval.data() : nullptr;
  a.accum = shared;
  std::vector<int64_t> pptr(s.eq.size() + 1, 0), pmap;
  if (accum == 2) {
    for (size_t q = 0; q < s.eq.size(); q++) {
      if (s.eq[q] >= 0)
        for (int64_t z = s.rp[s.eq[q]]; z < s.rp[s.eq[q] + 1]; z++) pmap.push_back(z);
      pptr[q + 1] = (int64_t)pmap.size();
    }
    a.pmap = pmap.data();
    a.pptr = pptr.data();
  }
  const AsmArgs* ap = &a;
  const int ngj = (a.n2 + C::NL - 1) / C::NL, total = ngj * a.n3 * nseg;
  const int blocks = (total + 7) / 8 * 8;
  if (accum == 3) {
    if constexpr (NC == 1 && NG == P + 1 && F32 != RHS) {
      std::vector<LineItem> items;
      for (int g = 0; g < total; g++) {
        const int seg = g % nseg, jg = (g / nseg) % ngj, k = g / (nseg * ngj);
        const int j0 = a.n2 * jg / ngj, j1 = a.n2 * (jg + 1) / ngj;
        items.push_back({0, j0, j1 - j0, k, a.n1 * seg / nseg, a.n1 * (seg + 1) / nseg});
      }
      int queue = 0;
      const LineItem* it = items.data();
      const int n = (int)items.size();
      launch(C::TH, 1, [=, &queue] { k_lines_batch<P, T, RHS, false>(ap, it, n, &queue); });
    } else {
      return 2;
    }
  } else if (shared) {
    launch(C::TH, blocks, [=] { k_lines<P, NG, NC, T, RHS, true, false>(ap, ngj, nseg, total); });
  } else {
    launch(C::TH, blocks, [=] { k_lines<P, NG, NC, T, RHS, false, false>(ap, ngj, nseg, total); });
  }
  if (F32) val.assign(val32.begin(), val32.end());
  const double eK = difference(val, K, zero), eb = F32 || !(RHS || prescribed) ? 0.0 : difference(rhs, b, zero);
  const bool ok = eK <= (F32 ? 1e-5 : 1e-12) && eb <= 1e-12;
  std::printf("neq %d K %.1e b %.1e %s\n", s.neq, eK, eb, ok ? "ok" : "WRONG");
  return !ok;
}

template <int P, int NG, int NC>
static int choose(bool fp32, bool rhs, int accum, const int* nel, int nseg, int fix, bool prescribed)
{
  if (fp32) return run<P, NG, NC, float, false>(accum, nel, nseg, fix, prescribed);
  return rhs ? run<P, NG, NC, double, true>(accum, nel, nseg, fix, prescribed)
             : run<P, NG, NC, double, false>(accum, nel, nseg, fix, prescribed);
}

// ---- a line so long that a group's records span more than 2^31 values ---------------
// The last rows of a patch of 4,000,000 x 11 x 1 elements in untouched virtual
// memory, where only the records of the last elements are set, against a short
// patch with the same records, tables and free functions: the same bits.
template <typename T>
static T* untouched(size_t count)
{
  void* p = mmap(nullptr, sizeof(T) * count, PROT_READ | PROT_WRITE,
                 MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (p == MAP_FAILED) {
    std::printf("no address space\n");
    std::exit(3);
  }
  return static_cast<T*>(p);
}

static int long_line()
{
  constexpr int P = 1, NG = 2, P1 = 2;
  using C = LineCfg<P, NG, 1>;
  constexpr int R = GeoRec<1>::N * NG * NG * NG;
  constexpr int ne[3] = {6, 11, 1}, L = 4000000, shift = L - ne[0];
  System s(P, NG, 1, ne, 0, 4); // free: the last three columns
  AsmArgs a = s.args();
  std::vector<double> val(s.ci.size(), NAN), rhs(s.neq, NAN), lval(val), lrhs(rhs);
  a.val64 = val.data();
  a.rhs = rhs.data();
  AsmArgs b = a;
  b.nel1 = L;
  b.n1 = L + P;
  b.val64 = lval.data();
  b.rhs = lrhs.data();
  double *tN = untouched<double>((size_t)L * NG * P1), *tD = untouched<double>((size_t)L * NG * P1);
  for (size_t q = 0; q < s.N[0].size(); q++) {
    tN[(size_t)shift * NG * P1 + q] = s.N[0][q];
    tD[(size_t)shift * NG * P1 + q] = s.D[0][q];
  }
  b.tabN1 = tN;
  b.tabD1 = tD;
  double* geo = untouched<double>((size_t)L * ne[1] * ne[2] * R);
  for (int e2 = 0; e2 < ne[1]; e2++)
    for (int q = 0; q < ne[0] * R; q++)
      geo[((size_t)L * e2 + shift) * R + q] = s.geo[(size_t)ne[0] * e2 * R + q];
  b.gp_geo = geo;
  int* eq = untouched<int>((size_t)b.n1 * b.n2 * b.n3);
  for (int k = 0; k < b.n3; k++)
    for (int j = 0; j < b.n2; j++)
      for (int i = -4; i < s.n[0]; i++)
        eq[(size_t)(i + shift) + (size_t)b.n1 * (j + (size_t)b.n2 * k)] = i < 0 ? -1 : s.eq[s.node(i, j, k)];
  b.eq = eq;
  using Sh = LineShared<P, NG, 1, double, true>;
  static Sh sh;
  static_assert(C::NL >= 12, "one group takes all lines of a plane");
  for (int k = 0; k < s.n[2]; k++) {
    const AsmArgs *pa = &a, *pb = &b;
    launch(C::TH, 1, [=] {
      line_group<P, NG, 1, double, true, false, C::wide(ne[0])>(*const_args(pa), 0, pa->n2, k, pa->n1 - 3, pa->n1, sh);
    });
    launch(C::TH, 1, [=] {
      line_group<P, NG, 1, double, true, false, C::wide(L)>(*const_args(pb), 0, pb->n2, k, pb->n1 - 3, pb->n1, sh);
    });
  }
  const bool ok = val == lval && rhs == lrhs;
  std::printf("neq %d long %s\n", s.neq, ok ? "ok" : "WRONG");
  return !ok;
}

int main(int argc, char** argv)
{
  if (argc == 2) return long_line();
  if (argc != 13) return 2;
  int v[12];
  for (int q = 0; q < 12; q++) v[q] = std::atoi(argv[q + 1]);
  const int key = v[0] * 100 + v[1] * 10 + v[2];
  switch (key) {
#define CASE(P, NG, NC)                                                                            \
  case P * 100 + NG * 10 + NC:                                                                     \
    return choose<P, NG, NC>(v[3] != 0, v[4] != 0, v[5], v + 6, v[9], v[10], v[11] != 0);
    CONFIG
  }
  return 2;
}
