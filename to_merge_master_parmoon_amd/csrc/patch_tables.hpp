// patch_tables.hpp - the per-cell records of the fused colored Vanka step (k_patch.hip).
//
// One workgroup computes the local residual of one cell's patch and solves and applies it in
// the same launch.  For that it needs the patch's rows, the dofs they read (the halo) and,
// because patches of one color read dofs that other patches of the color update, the place
// where the value from before the color is kept.
#pragma once
#include <cstdint>
#include <memory>
#include <vector>

#include "pmg.h"

namespace pmg {

constexpr int PT_HALO = 384;    // most velocity dofs in a patch's halo (343 on a hexahedral grid)
constexpr int PT_ZERO = PT_HALO; // halo position that holds zero: what lanes past a row's end read
constexpr int PT_RUNS = 32;     // most runs of four pressure dofs in a halo (27 there)
constexpr int PT_ROW = 128;     // longest A row, 8 steps of 16 lanes
constexpr int PT_BT = 32;       // longest BT row and B row, 2 steps

// Record of one cell (ints, PatchTables::stride apart, in color order).  The 31 rows of a patch
// are dealt to 8 "quads" of four 16-lane groups: quad 2 w + s is the s-th row of the groups of
// wavefront w.  Quad 1 holds the four pressure rows, the others the velocity rows, longest first.
constexpr int PR_DESC = 0;      // 32 x {first A (B) entry, first BT entry, n | m << 8 | row << 16, global row}
constexpr int PR_HEAD = 128;    // pattern, velocity halo size, pressure runs, 0
constexpr int PR_OUT = 132;     // 27: where the new velocity goes (buffer * n_udof + dof)
constexpr int PR_DOFS = 160;    // 27 velocity and 4 pressure dofs of the patch
constexpr int PR_RUN = 192;     // first dof of every pressure run
constexpr int PR_HALO = 224;    // where every halo velocity is read (buffer * n_udof + dof)
constexpr int PT_NOROW = 255;   // row number of an empty place

// Steps of 16 entries of a quad's longest A (quad 1: B) row and BT row.  GRID: as on a
// hexahedral grid, 8 vertex rows of up to 125 A and 32 BT entries, 12 edge rows of up to 75 and
// 16, 7 face and cell rows of up to 45 and 8; else as many as a record takes.
//
// A pattern holds the positions of the rows' columns in the halo, shared by all cells whose rows
// have the same structure (a few hundred on a refined mesh): 32-bit words of two 16-bit
// positions, steps 2 p and 2 p + 1 of a lane at (off_a(quad) + p) * 64 + lane (off_bt for the
// BT row); then the patch's own 27 dofs.  Places without an entry hold PT_ZERO (A, B) or 0 (BT,
// whose values the kernels mask), so that no row is touched by a value it is not coupled to.
template <bool GRID>
struct PatchShape {
  static constexpr int a(int quad) { return quad == 1 ? 2 : !GRID ? 8 : quad == 0 || quad == 2 ? 8 : quad == 3 || quad == 7 ? 3 : 5; }
  static constexpr int bt(int quad) { return quad == 1 ? 0 : !GRID || quad == 0 || quad == 2 ? 2 : 1; }
  // first 64-word block of the quad's A positions and of its BT positions
  static constexpr int off_a(int quad) { return quad == 0 ? 0 : off_bt(quad - 1) + (bt(quad - 1) + 1) / 2; }
  static constexpr int off_bt(int quad) { return off_a(quad) + (a(quad) + 1) / 2; }
  static constexpr int own = 64 * (off_bt(7) + (bt(7) + 1) / 2);   // first word of the own dofs
  static constexpr int words = own + 16;                            // of a pattern (14 for the own dofs)
};

// The same for FP64 rows, whose lanes take four consecutive entries of every 64 (row_window): two
// words of two positions per lane and batch of 64, at off_a(quad) + 2 * (64 * batch + lane).
template <bool GRID>
struct PatchShape64 {
  static constexpr int a(int quad) { return quad == 1 || (GRID && (quad == 3 || quad == 7)) ? 1 : 2; }   // batches
  static constexpr int off_a(int quad) { return quad == 0 ? 0 : off_bt(quad - 1) + (quad == 2 ? 0 : 128); }
  static constexpr int off_bt(int quad) { return off_a(quad) + 128 * a(quad); }   // (none in quad 1)
  static constexpr int own = off_bt(7) + 128;
  static constexpr int words = own + 16;
};

struct PatchTables {
  bool ok = false;           // false: some patch does not fit, the two-launch form is used
  int stride = 0;            // ints per record
  int n_buffers = 1;         // copies of the velocity the step alternates between
  int n_patterns = 0;
  bool grid = false;         // the patterns have PatchShape*<true>, else <false>
  std::unique_ptr<int[]> rec;   // stride ints per color position
  std::vector<uint32_t> pat;
};

// ug / pg: 27 velocity and 4 pressure dofs of every cell; cells of color k are
// order[ptr[k] .. ptr[k + 1]); fp64: patterns of PatchShape64
void build_patch_tables(const pmg_level_desc *d, const std::vector<int> &ug, const std::vector<int> &pg, int n_colors,
                        const int *ptr, const int *order, bool fp64, PatchTables &out);

}  // namespace pmg
