// Test driver for csrc/patch_tables.cpp (built by tests/test_patch_tables.py with g++, no GPU):
// colored sweeps run from the records, the patches of a color in random order and every
// access checked against its array, must give the sweep in which all patches of a color read
// the state from before the color.  Prints OK or FAIL.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>
#include "patch_tables.hpp"
#include "pmg_problem.h"
using namespace pmg;

extern "C" int pmg_color_cells(int, int, const int *, const int *, int, int *, int *, int *);
extern "C" int pmg_sequential_schedule(int, const int *, const int *, int, int, const int *, const int *, const int *,
                                       const int *, const int *, const int *, int *, int *, int *);

static int bad = 0;
#define CHECK(x) do { if (!(x)) { if (bad++ < 5) printf("line %d: %s\n", __LINE__, #x); } } while (0)

struct Sys {   // the level and its state: velocity (3 per dof), pressure
  const pmg_level_desc *d;
  std::vector<int> ug, pg;
};

static void row_vel(const pmg_level_desc &d, int r, const std::vector<double> &u, const std::vector<double> &p, double *s) {
  for (int k = d.a_rowptr[r]; k < d.a_rowptr[r + 1]; ++k)
    for (int c = 0; c < 3; ++c) s[c] += d.a[0][k] * u[3 * d.a_kcol[k] + c];
  if (r < d.n_active)
    for (int k = d.bt_rowptr[r]; k < d.bt_rowptr[r + 1]; ++k)
      for (int c = 0; c < 3; ++c) s[c] += d.bt[c][k] * p[d.bt_kcol[k]];
}

// the sweep from its definition: residuals of all patches of a color, then the updates
static void plain(const Sys &S, int nc, const int *ptr, const int *order, std::vector<double> &u, std::vector<double> &p) {
  const pmg_level_desc &d = *S.d;
  for (int k = 0; k < nc; ++k) {
    const std::vector<double> u0 = u, p0 = p;
    for (int q = ptr[k]; q < ptr[k + 1]; ++q) {
      const int *U = &S.ug[27 * size_t(order[q])], *P = &S.pg[4 * size_t(order[q])];
      for (int j = 0; j < 27; ++j) {
        double s[3] = {0, 0, 0};
        row_vel(d, U[j], u0, p0, s);
        for (int c = 0; c < 3; ++c) u[3 * U[j] + c] = u0[3 * U[j] + c] + 0.3 * (1.0 - s[c]);
      }
      for (int j = 0; j < 4; ++j) {
        double s = 0;
        for (int e = d.b_rowptr[P[j]]; e < d.b_rowptr[P[j] + 1]; ++e)
          for (int c = 0; c < 3; ++c) s += d.b[c][e] * u0[3 * d.b_kcol[e] + c];
        p[P[j]] = p0[P[j]] + 0.3 * (1.0 - s);
      }
    }
  }
}

// the sweep from the records
static void records(const Sys &S, const PatchTables &T, int nc, const int *ptr, std::vector<double> &ub,
                    std::vector<double> &p, std::mt19937 &rng, bool fp64) {
  const pmg_level_desc &d = *S.d;
  const long nb = long(T.n_buffers) * d.n_udof;
  const int words = fp64 ? (T.grid ? PatchShape64<true>::words : PatchShape64<false>::words)
                         : T.grid ? PatchShape<true>::words : PatchShape<false>::words;
  const int p_own = fp64 ? (T.grid ? PatchShape64<true>::own : PatchShape64<false>::own)
                         : T.grid ? PatchShape<true>::own : PatchShape<false>::own;
  for (int k = 0; k < nc; ++k) {
    std::vector<int> at;
    for (int q = ptr[k]; q < ptr[k + 1]; ++q) at.push_back(q);
    std::shuffle(at.begin(), at.end(), rng);
    for (int q : at) {
      const int *rc = &T.rec[size_t(q) * T.stride];
      const int nh = rc[PR_HEAD + 1], nr = rc[PR_HEAD + 2];
      CHECK(rc[PR_HEAD] >= 0 && rc[PR_HEAD] < T.n_patterns && nh > 0 && nh <= PT_HALO && PR_HALO + nh <= T.stride);
      CHECK(nr >= 0 && nr <= PT_RUNS);
      const uint32_t *pat = &T.pat[size_t(rc[PR_HEAD]) * words];
      std::vector<double> hv(3 * nh), hp(4 * nr), r(85, NAN);
      for (int i = 0; i < nh; ++i) {
        CHECK(rc[PR_HALO + i] >= 0 && rc[PR_HALO + i] < nb);
        for (int c = 0; c < 3; ++c) hv[3 * i + c] = ub[3 * long(rc[PR_HALO + i]) + c];
      }
      for (int i = 0; i < 4 * nr; ++i) {
        CHECK(rc[PR_RUN + i / 4] >= 0 && rc[PR_RUN + i / 4] + i % 4 < d.n_pdof);
        hp[i] = p[rc[PR_RUN + i / 4] + i % 4];
      }
      // places of a quad's A (B) rows without an entry read the zero behind the halo
      for (int qd = 0; qd < 8; ++qd) {
        const int off = fp64 ? (T.grid ? PatchShape64<true>::off_a(qd) : PatchShape64<false>::off_a(qd))
                             : 64 * (T.grid ? PatchShape<true>::off_a(qd) : PatchShape<false>::off_a(qd));
        const int len = fp64 ? 128 * (T.grid ? PatchShape64<true>::a(qd) : PatchShape64<false>::a(qd))
                             : 64 * (((T.grid ? PatchShape<true>::a(qd) : PatchShape<false>::a(qd)) + 1) / 2);
        int entries = 0, used = 0;
        for (int e = 4 * qd; e < 4 * qd + 4; ++e) entries += rc[PR_DESC + 4 * e + 2] & 255;
        for (int w = off; w < off + len; ++w)
          used += ((pat[w] & 0xffffu) != unsigned(PT_ZERO)) + ((pat[w] >> 16) != unsigned(PT_ZERO));
        CHECK(used == entries);
      }
      for (int e = 0; e < 32; ++e) {
        const int *dc = rc + PR_DESC + 4 * e, qd = e / 4;
        const int n = dc[2] & 255, m = (dc[2] >> 8) & 255, row = (dc[2] >> 16) & 255;
        const int sa = fp64 ? 4 * (T.grid ? PatchShape64<true>::a(qd) : PatchShape64<false>::a(qd))
                            : T.grid ? PatchShape<true>::a(qd) : PatchShape<false>::a(qd);
        const int sb = fp64 ? (qd == 1 ? 0 : 4) : T.grid ? PatchShape<true>::bt(qd) : PatchShape<false>::bt(qd);
        const int off_a = fp64 ? (T.grid ? PatchShape64<true>::off_a(qd) : PatchShape64<false>::off_a(qd))
                               : 64 * (T.grid ? PatchShape<true>::off_a(qd) : PatchShape<false>::off_a(qd));
        const int off_bt = fp64 ? (T.grid ? PatchShape64<true>::off_bt(qd) : PatchShape64<false>::off_bt(qd))
                                : 64 * (T.grid ? PatchShape<true>::off_bt(qd) : PatchShape<false>::off_bt(qd));
        CHECK((n + 15) / 16 <= sa && (m + 15) / 16 <= sb);
        // position of entry j of a row of len entries: in FP64 the kernel's lane reads the four
        // entries from the start of its window on
        auto pos = [&](int off, int j, int len) {
          size_t w;
          int half;
          if (fp64) {
            const int lane = j % 64 / 4, jb = j / 4 * 4, ld = len >= 4 ? std::min(jb, len - 4) : 0, u = j - ld;
            CHECK(u >= 0 && u < 4 && ld + u >= jb);
            w = size_t(off) + 2 * (64 * (j / 64) + (e % 4) * 16 + lane) + u / 2;
            half = u & 1;
          } else {
            w = size_t(off) + 64 * (j / 32) + (e % 4) * 16 + j % 16;
            half = (j / 16) & 1;
          }
          CHECK(w < size_t(p_own));
          return int((pat[w] >> (16 * half)) & 0xffffu);
        };
        if (row == PT_NOROW) {
          CHECK(n == 0 && m == 0);
          continue;
        }
        if (qd == 1) {
          CHECK(row >= 27 && row < 31 && dc[0] + n <= d.b_nnz && dc[3] >= 0 && dc[3] < d.n_pdof);
          double s = 0;
          for (int j = 0; j < n; ++j) {
            CHECK(pos(off_a, j, n) < nh);
            for (int c = 0; c < 3; ++c) s += d.b[c][dc[0] + j] * hv[3 * pos(off_a, j, n) + c];
          }
          r[81 + row - 27] = 1.0 - s;
          continue;
        }
        CHECK(row < 27 && dc[0] + n <= d.a_nnz && dc[1] + m <= d.bt_nnz && dc[3] >= 0 && dc[3] < d.n_udof);
        double s[3] = {0, 0, 0};
        for (int j = 0; j < n; ++j) {
          CHECK(pos(off_a, j, n) < nh);
          for (int c = 0; c < 3; ++c) s[c] += d.a[0][dc[0] + j] * hv[3 * pos(off_a, j, n) + c];
        }
        for (int j = 0; j < m; ++j) {
          CHECK(pos(off_bt, j, m) < 4 * nr);
          for (int c = 0; c < 3; ++c) s[c] += d.bt[c][dc[1] + j] * hp[pos(off_bt, j, m)];
        }
        for (int c = 0; c < 3; ++c) r[27 * c + row] = 1.0 - s[c];
      }
      for (int j = 0; j < 27; ++j) {
        const int own = (pat[p_own + j / 2] >> (16 * (j & 1))) & 0xffffu, out = rc[PR_OUT + j];
        CHECK(own < nh && out >= 0 && out < nb && out % d.n_udof == rc[PR_DOFS + j]);
        for (int c = 0; c < 3; ++c) ub[3 * long(out) + c] = hv[3 * own + c] + 0.3 * r[27 * c + j];
      }
      for (int j = 0; j < 4; ++j) {
        CHECK(rc[PR_DOFS + 27 + j] >= 0 && rc[PR_DOFS + 27 + j] < d.n_pdof);
        p[rc[PR_DOFS + 27 + j]] += 0.3 * r[81 + j];
      }
    }
  }
}

// the A rows of edge dofs (75 entries) with up to 30 more, at dofs of several cells in the halos of
// all cells of the dof: the general record shape with halos as before; how many rows have more
static int longer_rows(pmg_level_desc &d, const std::vector<int> &ug, std::vector<int> &ptr, std::vector<int> &col,
                       std::vector<double> &val) {
  std::vector<std::vector<int>> cells(d.n_udof), halo(d.n_cells);
  for (int c = 0; c < d.n_cells; ++c) {
    for (int j = 0; j < 27; ++j) {
      const int r = ug[27 * size_t(c) + j];
      cells[r].push_back(c);
      halo[c].insert(halo[c].end(), d.a_kcol + d.a_rowptr[r], d.a_kcol + d.a_rowptr[r + 1]);
    }
    std::sort(halo[c].begin(), halo[c].end());
    halo[c].erase(std::unique(halo[c].begin(), halo[c].end()), halo[c].end());
  }
  int longer = 0;
  ptr.assign(1, 0);
  for (int r = 0; r < d.n_udof; ++r) {
    const int k0 = d.a_rowptr[r], n = d.a_rowptr[r + 1] - k0;
    std::vector<std::pair<int, double>> row;
    for (int k = k0; k < k0 + n; ++k) row.push_back({d.a_kcol[k], d.a[0][k]});
    if (n == 75 && r < d.n_active) {
      int more = 0;
      for (int g : halo[cells[r][0]]) {
        bool in = more < 30 && cells[g].size() > 1 && !std::count(d.a_kcol + k0, d.a_kcol + k0 + n, g);
        for (int c : cells[r]) in = in && std::binary_search(halo[c].begin(), halo[c].end(), g);
        if (in) row.push_back({g, 1e-3 * ++more});
      }
      longer += more > 5;
      std::sort(row.begin(), row.end());
    }
    for (auto &e : row) {
      col.push_back(e.first);
      val.push_back(e.second);
    }
    ptr.push_back(int(col.size()));
  }
  d.a_rowptr = ptr.data();
  d.a_kcol = col.data();
  d.a[0] = val.data();
  d.a_nnz = ptr.back();
  return longer;
}

static void run(const char *name, pmgp_problem *prob, int level, int mode, bool fp64) {
  pmg_level_desc d;
  pmgp_level_desc(prob, level, &d);
  Sys S{&d, {}, {}};
  std::vector<int> ub(d.n_cells);
  for (int c = 0; c < d.n_cells; ++c) {
    ub[c] = 27 * c;
    for (int j = 0; j < 27; ++j) S.ug.push_back(d.u_global[d.u_begin[c] + j]);
    for (int j = 0; j < 4; ++j) S.pg.push_back(d.p_global[d.p_begin[c] + j]);
  }
  std::vector<int> lptr, lcol;
  std::vector<double> lval;
  const int longer = mode == 5 ? longer_rows(d, S.ug, lptr, lcol, lval) : 0;
  std::vector<int> ptr(d.n_cells + 1), order(d.n_cells);
  int nc = 0;
  if (mode == 1)   // the level sets of the Gauss-Seidel order
    pmg_sequential_schedule(d.n_cells, S.ug.data(), S.pg.data(), d.n_udof, d.n_pdof, d.a_rowptr, d.a_kcol, d.bt_rowptr,
                            d.bt_kcol, d.b_rowptr, d.b_kcol, &nc, ptr.data(), order.data());
  else
    pmg_color_cells(d.n_cells, 27, ub.data(), S.ug.data(), d.n_udof, &nc, ptr.data(), order.data());
  std::mt19937 rng(11);
  if (mode == 2 || mode == 4) {   // a corner cell (dofs of 3 and 7 updates), a third of the cells in no color
    std::vector<int> p2(1, 0), o2;
    for (int k = 0; k < nc; ++k) {
      for (int q = ptr[k]; q < ptr[k + 1]; ++q)
        if (mode == 2 ? order[q] != 0 : rng() % 3) o2.push_back(order[q]);
      p2.push_back(int(o2.size()));
    }
    std::copy(p2.begin(), p2.end(), ptr.begin());
    std::copy(o2.begin(), o2.end(), order.begin());
  }
  if (mode == 3) {   // two cells of one color that share dofs: refused
    ptr[1] += 1;
    std::sort(order.begin(), order.begin() + ptr[1]);
  }
  PatchTables T;
  build_patch_tables(&d, S.ug, S.pg, nc, ptr.data(), order.data(), fp64, T);
  if (mode == 3) {
    CHECK(!T.ok);
    return;
  }
  // in mode 4 a patch may read what another of its color updates in place: then it is refused
  CHECK(T.ok || mode == 4);
  if (!T.ok) return;
  CHECK(T.grid || longer > 0);
  std::normal_distribution<double> N01;
  std::vector<double> u(3 * size_t(d.n_udof)), p(d.n_pdof);
  for (auto &v : u) v = N01(rng);
  for (auto &v : p) v = N01(rng);
  std::vector<double> b(3 * size_t(d.n_udof) * T.n_buffers, NAN), q = p;
  std::copy(u.begin(), u.end(), b.begin());
  for (int sweep = 0; sweep < 2; ++sweep) {
    plain(S, nc, ptr.data(), order.data(), u, p);
    records(S, T, nc, ptr.data(), b, q, rng, fp64);
  }
  double err = 0, nrm = 0;
  for (size_t i = 0; i < u.size(); ++i) { const double e = std::fabs(u[i] - b[i]); CHECK(e == e); err = std::max(err, e); nrm = std::max(nrm, std::fabs(u[i])); }
  for (size_t i = 0; i < p.size(); ++i) { const double e = std::fabs(p[i] - q[i]); CHECK(e == e); err = std::max(err, e); }
  printf("%s level %d mode %d: %d cells, %d colors, %d buffers, %d patterns%s, difference %.1e of %.1e\n", name, level,
         mode, d.n_cells, nc, T.n_buffers, T.n_patterns, T.grid ? "" : ", general", err, nrm);
  CHECK(err <= 1e-12 * nrm);
}

int main() {
  struct Spec { const char *name; int c[3], levels, faces; double perturb; } specs[] = {
      {"cube", {4, 4, 4}, 2, 63, 0.0}, {"open box", {2, 3, 5}, 2, 21, 0.1}, {"single cell wide", {1, 1, 6}, 1, 0, 0.0},
      {"channel", {6, 1, 1}, 2, 1 | 4 | 8 | 16 | 32, 0.0}, {"fine", {3, 3, 3}, 3, 63, 0.1}};
  for (const Spec &s : specs) {
    pmgp_config c;
    pmgp_config_default(&c);
    c.cx = s.c[0]; c.cy = s.c[1]; c.cz = s.c[2];
    c.n_levels = s.levels; c.nu = 0.1; c.dirichlet_faces = s.faces; c.perturb = s.perturb;
    c.conv_kind = PMGP_CONV_FOURIER; c.rhs_kind = PMGP_RHS_FOURIER;
    pmgp_problem *P = nullptr;
    if (pmgp_create(&c, &P)) { printf("create failed\n"); return 1; }
    for (int l = 0; l < s.levels; ++l)
      for (int mode = 0; mode < 12; ++mode) run(s.name, P, l, mode % 6, mode >= 6);
    pmgp_destroy(P);
  }
  printf(bad ? "FAIL %d\n" : "OK\n", bad);
  return bad != 0;
}
