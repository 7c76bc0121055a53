// patch_tables.cpp - builds the records of patch_tables.hpp (host code, once per level).
#include "patch_tables.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <deque>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>
#include <unordered_map>
#include <utility>

namespace pmg {

namespace {

constexpr int NU = 27, NP = 4;

// Which copy of the velocity holds a dof after its i-th of m updates in a sweep.  The new value
// goes to another copy than the old one, so that the patches of the same color still read the
// old one, and the last update ends in copy 0 again.  A dof of one cell only is updated in
// place (the caller checks that no other patch of the color reads it).
int copy_after(int i, int m) {
  if (m == 1 || i == 0 || i == m) return 0;
  if (m % 2 == 1 && i == m - 1) return 2;
  return i % 2;
}

struct Dofs {   // the colors that update a dof, ascending
  std::vector<int> ptr, col, cell;
};

bool color_lists(int n_dof, int per_cell, const std::vector<int> &glob, int n_colors, const int *ptr,
                 const int *order, Dofs &out) {
  out.ptr.assign(n_dof + 1, 0);
  for (int q = 0; q < ptr[n_colors]; ++q)
    for (int j = 0; j < per_cell; ++j) out.ptr[glob[size_t(order[q]) * per_cell + j] + 1]++;
  for (int i = 0; i < n_dof; ++i) out.ptr[i + 1] += out.ptr[i];
  out.col.resize(out.ptr[n_dof]);
  out.cell.resize(out.ptr[n_dof]);
  std::vector<int> at(out.ptr.begin(), out.ptr.end() - 1);
  for (int k = 0; k < n_colors; ++k)
    for (int q = ptr[k]; q < ptr[k + 1]; ++q)
      for (int j = 0; j < per_cell; ++j) {
        const int g = glob[size_t(order[q]) * per_cell + j];
        // two cells of one color (or one cell twice) on a dof: the updates would not be ordered
        if (at[g] > out.ptr[g] && out.col[at[g] - 1] == k) return false;
        out.col[at[g]] = k;
        out.cell[at[g]++] = order[q];
      }
  return true;
}

// hash of a pattern -> its words and its number
using Patterns = std::unordered_multimap<uint64_t, std::pair<const std::vector<uint32_t> *, int>>;

struct Scratch {
  std::vector<int> mark, pmark;   // dof -> place in the halo (valid where stamp matches)
  std::vector<int> stamp, pstamp;
  std::vector<int> halo, runs;
  std::vector<uint32_t> pat;      // the pattern of the cell in work
  Patterns seen;                  // those this thread has met
};

uint64_t pattern_hash(const std::vector<uint32_t> &w) {
  uint64_t h = w.size();
  for (size_t i = 0; i + 1 < w.size(); i += 2) {
    h = (h ^ (w[i] | uint64_t(w[i + 1]) << 32)) * 0x9e3779b97f4a7c15ull;
    h ^= h >> 32;
  }
  return h;
}

}  // namespace

void build_patch_tables(const pmg_level_desc *d, const std::vector<int> &ug, const std::vector<int> &pg, int n_colors,
                        const int *ptr, const int *order, bool fp64, PatchTables &T) {
  T = PatchTables{};
  const int n_pos = ptr[n_colors];
  if (n_pos <= 0 || d->n_pdof % 4 != 0) return;
  for (int i = 0; i < d->n_udof; ++i)
    if (d->a_rowptr[i + 1] - d->a_rowptr[i] > PT_ROW || d->bt_rowptr[i + 1] - d->bt_rowptr[i] > PT_BT) return;
  for (int i = 0; i < d->n_pdof; ++i)
    if (d->b_rowptr[i + 1] - d->b_rowptr[i] > PT_BT) return;
  Dofs U, P;
  if (!color_lists(d->n_udof, NU, ug, n_colors, ptr, order, U)) return;
  if (!color_lists(d->n_pdof, NP, pg, n_colors, ptr, order, P)) return;
  for (int i = 0; i < d->n_pdof; ++i)
    if (P.ptr[i + 1] - P.ptr[i] > 1) return;   // pressures are updated in place
  for (int i = 0; i < d->n_udof; ++i) {
    const int m = U.ptr[i + 1] - U.ptr[i];
    if (m > 1) T.n_buffers = std::max(T.n_buffers, m % 2 ? 3 : 2);
  }
  if (long(T.n_buffers) * d->n_udof > 0x7fffffffL / 4) return;

  std::vector<int> color_of(n_pos);
  for (int k = 0; k < n_colors; ++k)
    for (int q = ptr[k]; q < ptr[k + 1]; ++q) color_of[q] = k;
  auto len_a = [&](int r) { return d->a_rowptr[r + 1] - d->a_rowptr[r]; };
  auto len_bt = [&](int r) { return r < d->n_active ? d->bt_rowptr[r + 1] - d->bt_rowptr[r] : 0; };
  // local rows by decreasing length into the velocity quads, heaviest wavefronts last filled
  static const int quad_order[7] = {0, 2, 4, 5, 6, 7, 3};
  auto row_places = [&](const int *u, int (&place)[NU]) {
    int key[NU];   // A length, BT length, the lower row first
    for (int j = 0; j < NU; ++j) key[j] = len_a(u[j]) << 16 | len_bt(u[j]) << 8 | (31 - j);
    std::sort(key, key + NU, [](int a, int b) { return a > b; });
    for (int k = 0; k < NU; ++k) place[31 - (key[k] & 31)] = quad_order[k / 4] * 4 + k % 4;
  };
  using G = PatchShape<true>;
  using R = PatchShape<false>;
  using G64 = PatchShape64<true>;
  using R64 = PatchShape64<false>;
  T.grid = true;
  for (int q = 0; q < n_pos && T.grid; ++q) {
    const int *u = &ug[size_t(order[q]) * NU];
    int place[NU];
    row_places(u, place);
    for (int j = 0; j < NU; ++j) {
      const int qd = place[j] / 4;
      T.grid = T.grid && len_a(u[j]) <= 16 * G::a(qd) && len_bt(u[j]) <= 16 * G::bt(qd);
    }
  }
  int off_a[8], off_bt[8], len_pat[8];   // words
  for (int qd = 0; qd < 8; ++qd) {
    len_pat[qd] = fp64 ? 128 * (T.grid ? G64::a(qd) : R64::a(qd)) : 64 * (((T.grid ? G::a(qd) : R::a(qd)) + 1) / 2);
    off_a[qd] = fp64 ? (T.grid ? G64::off_a(qd) : R64::off_a(qd)) : 64 * (T.grid ? G::off_a(qd) : R::off_a(qd));
    off_bt[qd] = fp64 ? (T.grid ? G64::off_bt(qd) : R64::off_bt(qd)) : 64 * (T.grid ? G::off_bt(qd) : R::off_bt(qd));
  }
  const int own = fp64 ? (T.grid ? G64::own : R64::own) : T.grid ? G::own : R::own;
  const int words = fp64 ? (T.grid ? G64::words : R64::words) : T.grid ? G::words : R::words;

  // records with a fixed largest halo, then packed to the level's own largest halo
  const int wide = PR_HALO + PT_HALO;
  std::unique_ptr<int[]> rec(new int[size_t(n_pos) * wide]);   // zeroed by the threads
  std::deque<std::vector<uint32_t>> known;   // the patterns in the order of arrival (their places stay)
  Patterns known_at;
  std::mutex known_mu;
  std::atomic<bool> ok{true};
  std::atomic<int> next{0};
  std::atomic<int> hmax{0};
  auto work_cells = [&] {
    Scratch W;
    W.mark.assign(d->n_udof, 0);
    W.stamp.assign(d->n_udof, -1);
    W.pmark.assign(d->n_pdof / 4, 0);
    W.pstamp.assign(d->n_pdof / 4, -1);
    for (;;) {
      const int q0 = next.fetch_add(64), q1 = std::min(n_pos, q0 + 64);
      if (q0 >= n_pos || !ok) return;
      for (int q = q0; q < q1 && ok; ++q) {
        const int cell = order[q], color = color_of[q];
        const int *u = &ug[size_t(cell) * NU], *p = &pg[size_t(cell) * NP];
        W.halo.clear();
        W.runs.clear();
        auto see = [&](int g) {
          if (W.stamp[g] != q) {
            W.stamp[g] = q;
            W.halo.push_back(g);
          }
        };
        for (int j = 0; j < NU; ++j) {
          see(u[j]);
          for (int k = d->a_rowptr[u[j]]; k < d->a_rowptr[u[j] + 1]; ++k) see(d->a_kcol[k]);
          if (u[j] < d->n_active)
            for (int k = d->bt_rowptr[u[j]]; k < d->bt_rowptr[u[j] + 1]; ++k) {
              const int g = d->bt_kcol[k] / 4;
              if (W.pstamp[g] != q) {
                W.pstamp[g] = q;
                W.runs.push_back(g);
              }
            }
        }
        for (int j = 0; j < NP; ++j)
          for (int k = d->b_rowptr[p[j]]; k < d->b_rowptr[p[j] + 1]; ++k) see(d->b_kcol[k]);
        const int nh = int(W.halo.size()), nr = int(W.runs.size());
        if (nh > PT_HALO || nr > PT_RUNS) {
          ok = false;
          return;
        }
        std::sort(W.halo.begin(), W.halo.end());
        std::sort(W.runs.begin(), W.runs.end());
        int h = hmax.load();
        while (nh > h && !hmax.compare_exchange_weak(h, nh)) {
        }
        int *rc = &rec[size_t(q) * wide];
        std::fill(rc, rc + wide, 0);
        for (int i = 0; i < nh; ++i) {
          const int g = W.halo[i];
          W.mark[g] = i;
          const int b = U.ptr[g], m = U.ptr[g + 1] - b;
          int k = 0;
          while (k < m && U.col[b + k] < color) ++k;
          // updated in place by another patch of this color: its old value would be lost
          if (m == 1 && U.col[b] == color && U.cell[b] != cell) ok = false;
          rc[PR_HALO + i] = copy_after(k, m) * d->n_udof + g;
        }
        for (int i = 0; i < nr; ++i) {
          const int g = W.runs[i];
          W.pmark[g] = i;
          rc[PR_RUN + i] = 4 * g;
          for (int j = 4 * g; j < 4 * g + 4; ++j)
            if (P.ptr[j + 1] > P.ptr[j] && P.col[P.ptr[j]] == color && P.cell[P.ptr[j]] != cell) ok = false;
        }
        for (int j = 0; j < NU; ++j) {
          const int b = U.ptr[u[j]], m = U.ptr[u[j] + 1] - b;
          int k = 0;
          while (k < m && U.col[b + k] < color) ++k;
          rc[PR_OUT + j] = copy_after(k + 1, m) * d->n_udof + u[j];
          rc[PR_DOFS + j] = u[j];
        }
        for (int j = 0; j < NP; ++j) rc[PR_DOFS + NU + j] = p[j];
        rc[PR_HEAD + 1] = nh;
        rc[PR_HEAD + 2] = nr;
        // rows and their column positions
        for (int e = 0; e < 32; ++e) rc[PR_DESC + 4 * e + 2] = PT_NOROW << 16;
        W.pat.assign(words, 0u);
        for (int qd = 0; qd < 8; ++qd)
          std::fill(W.pat.begin() + off_a[qd], W.pat.begin() + off_a[qd] + len_pat[qd], uint32_t(PT_ZERO) * 0x10001u);
        auto set = [&](size_t w, int half, int pos) {
          W.pat[w] = (W.pat[w] & ~(0xffffu << (16 * half))) | uint32_t(pos) << (16 * half);
        };
        auto put = [&](int off, int e, int j, int n, int pos) {   // entry j of n of the row at place e
          if (fp64) {
            // entry u of the lane's window, which starts at most n - 4 (row_window)
            const int lane = j % 64 / 4, jb = j / 4 * 4, first = n >= 4 ? std::min(jb, n - 4) : 0, u = j - first;
            set(size_t(off) + 2 * (64 * (j / 64) + (e % 4) * 16 + lane) + u / 2, u & 1, pos);
          } else {
            const int step = j / 16, lane = (e % 4) * 16 + j % 16;
            set(size_t(off) + 64 * (step / 2) + lane, step & 1, pos);
          }
        };
        auto desc = [&](int e, int k0, int q0b, int n, int m, int row, int g) {
          int *o = rc + PR_DESC + 4 * e;
          o[0] = k0;
          o[1] = q0b;
          o[2] = n | m << 8 | row << 16;
          o[3] = g;
        };
        int place[NU];
        row_places(u, place);
        for (int j = 0; j < NU; ++j) {
          const int e = place[j], qd = e / 4, g = u[j], k0 = d->a_rowptr[g], n = len_a(g), m = len_bt(g);
          const int q0b = d->bt_rowptr[g];
          desc(e, k0, q0b, n, m, j, g);
          for (int k = 0; k < n; ++k) put(off_a[qd], e, k, n, W.mark[d->a_kcol[k0 + k]]);
          for (int k = 0; k < m; ++k) {
            const int c = d->bt_kcol[q0b + k];
            put(off_bt[qd], e, k, m, 4 * W.pmark[c / 4] + c % 4);
          }
          set(size_t(own) + j / 2, j & 1, W.mark[g]);
        }
        for (int j = 0; j < NP; ++j) {
          const int e = 4 + j, k0 = d->b_rowptr[p[j]], n = d->b_rowptr[p[j] + 1] - k0;
          desc(e, k0, 0, n, 0, NU + j, p[j]);
          for (int k = 0; k < n; ++k) put(off_a[1], e, k, n, W.mark[d->b_kcol[k0 + k]]);
        }
        // a few hundred patterns among all cells: almost every one is found without the lock
        const uint64_t hash = pattern_hash(W.pat);
        auto find = [&](const Patterns &in) {
          for (auto [it, end] = in.equal_range(hash); it != end; ++it)
            if (*it->second.first == W.pat) return it->second;
          return std::pair<const std::vector<uint32_t> *, int>(nullptr, -1);
        };
        auto at = find(W.seen);
        if (!at.first) {
          std::lock_guard<std::mutex> lk(known_mu);
          at = find(known_at);
          if (!at.first) {
            known.push_back(W.pat);
            at = {&known.back(), int(known.size()) - 1};
            known_at.emplace(hash, at);
          }
          W.seen.emplace(hash, at);
        }
        rc[PR_HEAD] = at.second;
      }
    }
  };
  auto work = [&] {   // out of memory: the level keeps the two-launch form
    try {
      work_cells();
    } catch (const std::bad_alloc &) {
      ok = false;
    }
  };
  {
    const int nt = std::max(1, std::min({8, int(std::thread::hardware_concurrency()), (n_pos + 255) / 256}));
    std::vector<std::thread> th;
    try {
      th.reserve(nt);
      for (int i = 1; i < nt; ++i) th.emplace_back(work);
    } catch (const std::system_error &) {   // no more threads: this one does the rest
    }
    work();
    for (auto &t : th) t.join();
  }
  if (!ok) return;
  // the patterns in the order of their first cell, whatever order the threads met them in
  std::vector<int> number(known.size(), -1);
  T.pat.resize(known.size() * size_t(words));
  for (int q = 0; q < n_pos; ++q) {
    int &id = rec[size_t(q) * wide + PR_HEAD];
    if (number[id] < 0) {
      number[id] = T.n_patterns++;
      std::copy(known[id].begin(), known[id].end(), &T.pat[size_t(number[id]) * words]);
    }
    id = number[id];
  }
  T.stride = (PR_HALO + hmax + 15) / 16 * 16;   // at most wide
  for (int q = 1; q < n_pos; ++q) std::memmove(&rec[size_t(q) * T.stride], &rec[size_t(q) * wide], 4 * size_t(T.stride));
  T.rec = std::move(rec);
  T.ok = true;
}

}  // namespace pmg
