// Layout of the neighbour-list workspace (dpk_nlist_build), shared by the
// kernels that reuse its cell list (the cell-blocked force kernel).
#pragma once

#include <cstddef>

namespace dpk {

struct NlistWs {
  int* cell_count;  // [ncells]
  int* cell_start;  // [ncells + 1] exclusive prefix
  int* cell_atoms;  // [natoms] atoms sorted by cell
  int* atom_cell;   // [natoms] global cell id of each atom
  int* atom_slot;   // [natoms] position of each atom inside its cell
  int* cell_tmp;    // [natoms] binning scratch (arrival order inside each cell)
};

inline size_t nlist_align256(size_t b) { return (b + 255) & ~size_t(255); }

inline size_t nlist_ws_bytes(int natoms, int ncells) {
  return nlist_align256(sizeof(int) * (size_t)ncells) +
         nlist_align256(sizeof(int) * ((size_t)ncells + 1)) +
         4 * nlist_align256(sizeof(int) * (size_t)natoms);
}

inline NlistWs nlist_ws(void* workspace, int natoms, int ncells) {
  char* ws = static_cast<char*>(workspace);
  NlistWs w;
  w.cell_count = reinterpret_cast<int*>(ws);
  ws += nlist_align256(sizeof(int) * (size_t)ncells);
  w.cell_start = reinterpret_cast<int*>(ws);
  ws += nlist_align256(sizeof(int) * ((size_t)ncells + 1));
  w.cell_atoms = reinterpret_cast<int*>(ws);
  ws += nlist_align256(sizeof(int) * (size_t)natoms);
  w.atom_cell = reinterpret_cast<int*>(ws);
  ws += nlist_align256(sizeof(int) * (size_t)natoms);
  w.atom_slot = reinterpret_cast<int*>(ws);
  ws += nlist_align256(sizeof(int) * (size_t)natoms);
  w.cell_tmp = reinterpret_cast<int*>(ws);
  return w;
}

// Workgroups that share a cell's centres (W wavefronts each): one where the
// cells alone fill the chip, more -- down to a centre a wavefront -- where a
// few cells hold all atoms (a small periodic box is one to eight cells).
// Search and forces of 81 water atoms in one cell: 132 and 82 us with one
// workgroup, 43 and 21 us with six and eleven; 5,324 Cu atoms in 64 cells: 128
// and 119 us, 53 and 102 us.
inline int cell_parts(int natoms, int ncells, int W, int ncu) {
  const int rounds = (natoms + ncells * W - 1) / (ncells * W), room = ncu / ncells;
  const int p = rounds < room ? rounds : room;
  return p > 1 ? p : 1;
}

}  // namespace dpk
