// wx_common.h - shared constants and device data structures.
#pragma once

#include <cstdint>

namespace wx {

constexpr int NC = 16;             // cells per block edge (ncells_block)
constexpr int NG = 2;              // ghost layers (nghost)
constexpr int NB = NC + 2 * NG;    // 20: stored edge with ghosts
constexpr int NCELL = NB * NB * NB;
constexpr int NINT = NC * NC * NC; // 4096 interior cells
// The plain form stores a block's variable as its interior (i fastest), then
// its face ghosts as 12 planes of 16 x 16: rows of the interior and of a
// ghost plane fill whole 128-byte lines.  (In a 20^3 cube every row straddles
// two lines and a ghost of an x face is alone in its line: the writes of
// partial lines, shared between the chiplets' L2s, took most of the time.)
constexpr int NSTORE = NINT + 12 * NC * NC;
constexpr int MAXV = 8;

// source/constants.f90:52-104
enum { LEFT = 0, RIGHT, FRONT, BACK, BOTTOM, TOP };     // 0-based face index
enum { BC_REFLECTIVE = 1, BC_FREE_FLOW = 2, BC_PERIODIC = 3 };
enum { NEIGH_SAME = 1, NEIGH_COARSER = 2, NEIGH_FINER = 3, NEIGH_BOUNDARY = 4 };
enum { SOLVER_HLL1 = 2, SOLVER_HLL = 3, SOLVER_HLLC = 4, SOLVER_HLLE = 5, SOLVER_HLLD = 6 };

// Index checks of the CPU emulation of the kernels (the emulator build
// defines WX_EMU_CHECKS): a violated range aborts with its source line.
// Nothing in the GPU build.
#ifdef WX_EMU_CHECKS
void wx_emu_check_failed(const char *what, const char *file, int line);
#define WX_EMU_CHECK(c) ((c) ? (void)0 : wx_emu_check_failed(#c, __FILE__, __LINE__))
#else
#define WX_EMU_CHECK(c) ((void)0)
#endif

// Index of cell (i,j,k) in the plain form's arrays: the interior, or a face
// ghost (one coordinate in [-1, 0] or [17, 18]; reference bounds
// nxmin..nxmax).  Ghost planes: face x 2 + layer - 1, then the two transverse
// coordinates, the lower axis fastest.
__host__ __device__ constexpr inline int cid(int i, int j, int k) {
  const bool xg = i < 1 || i > NC, yg = j < 1 || j > NC, zg = k < 1 || k > NC;
  WX_EMU_CHECK(i >= -1 && i <= NC + 2 && j >= -1 && j <= NC + 2 && k >= -1 && k <= NC + 2);
  WX_EMU_CHECK((int)xg + (int)yg + (int)zg <= 1);
  const int gx = i < 1 ? -i : i - NC + 1, gy = 4 + (j < 1 ? -j : j - NC + 1), gz = 8 + (k < 1 ? -k : k - NC + 1);
  const int plane = xg ? gx : (yg ? gy : gz);
  const int row = zg ? j - 1 : k - 1, col = xg ? j - 1 : i - 1;
  return (xg || yg || zg) ? NINT + (plane * NC + row) * NC + col : ((k - 1) * NC + (j - 1)) * NC + (i - 1);
}

// One face of one block in the neighbour table.  For NEIGH_FINER the four
// sources are stored by transverse quadrant q = t1 + 2*t2 (t1, t2 the
// sibling coordinates of the source along the face's first and second
// transverse axes); for the other types only src[0] is used.  A periodic
// domain face is stored as NEIGH_SAME with the wrapped partner.
struct Face {
  int type;
  int src[4];
};

// Per-block record
struct BlockInfo {
  int level;       // 1-based
  int sib[3];      // siblingCoords (0/1), -1 at level 1
  int bid;         // reference block ID
  int coords[3];   // 1-based block coordinates at its level
  Face face[6];
};

}  // namespace wx
