// The neighbourhood of a cell on the regular hexagonal lattice, as
// compile-time tables.
//
// Cells are numbered by offset: 0 the cell, 1..6 its neighbours W, SW, SE, E,
// NE, NW, 7..18 the second ring (7 + 2d: two steps along direction d, 8 + 2d:
// one step along d and one along d + 1).  Edge 3*i + K is edge K (W, SW, SE)
// owned by cell i, vertex 2*i + x corner x (upper left, lower left) owned by
// cell i.  hex_layout.cpp builds the record of 19 cell ids per cell and
// checks that the mesh's tables are these.
#pragma once

namespace omega_hip {
namespace hexl {

constexpr int kCells = 19, kEdges = 57, kVerts = 38;
constexpr int kRec = 20; // ints per record (16-byte aligned)

// axial coordinates of the directions W, SW, SE, E, NE, NW
constexpr int DQ[6] = {-1, 0, 1, 1, 0, -1};
constexpr int DR[6] = {0, -1, -1, 0, 1, 1};

constexpr int cell_q(int i) {
  if (i == 0) return 0;
  if (i < 7) return DQ[i - 1];
  const int d = (i - 7) / 2;
  return DQ[d] + DQ[(i - 7) % 2 ? (d + 1) % 6 : d];
}
constexpr int cell_r(int i) {
  if (i == 0) return 0;
  if (i < 7) return DR[i - 1];
  const int d = (i - 7) / 2;
  return DR[d] + DR[(i - 7) % 2 ? (d + 1) % 6 : d];
}
// cell at an offset, -1 outside the two rings
constexpr int cell_at(int q, int r) {
  for (int i = 0; i < kCells; ++i)
    if (cell_q(i) == q && cell_r(i) == r) return i;
  return -1;
}
constexpr int nbr(int i, int d) { return cell_at(cell_q(i) + DQ[d], cell_r(i) + DR[d]); }

// edge in direction d of cell i: its own for d < 3, otherwise edge d - 3 of
// the neighbour across it (-1 outside the rings)
constexpr int cell_edge(int i, int d) {
  if (d < 3) return 3 * i + d;
  const int n = nbr(i, d);
  return n < 0 ? -1 : 3 * n + d - 3;
}
// corner k of cell i: 0 upper left, 1 lower left (own), 2 bottom, 3 lower
// right, 4 upper right, 5 top
constexpr int corner(int i, int k) {
  if (k < 2) return 2 * i + k;
  const int n = nbr(i, k == 2 ? 2 : (k == 5 ? 4 : 3));
  return n < 0 ? -1 : 2 * n + (k == 2 || k == 4 ? 0 : 1);
}

struct Edge {
  int c[2], v[2]; // cells_on_edge, vertices_on_edge
};
constexpr Edge edge(int e) {
  const int i = e / 3, K = e % 3;
  return Edge{{nbr(i, K), i}, {corner(i, K + 1), corner(i, K)}};
}

// edges_on_vertex, cells_on_vertex and the edges' signs (+1 when the vertex
// is the edge's second)
struct Vert {
  int e[3], c[3];
  double s[3];
};
constexpr Vert vert(int w) {
  const int i = w / 2;
  const int W = nbr(i, 0), SW = nbr(i, 1), NW = nbr(i, 5);
  if (w % 2 == 0) return Vert{{3 * i, 3 * NW + 2, 3 * NW + 1}, {i, NW, W}, {1.0, 1.0, -1.0}};
  return Vert{{3 * i, 3 * W + 2, 3 * i + 1}, {W, SW, i}, {-1.0, -1.0, 1.0}};
}

// PV stencil of the owned edge K: edges_on_edge slot j, and its TRiSK weight
// in units of the mesh's smallest nonzero one.  Slots 0..4 run round the
// neighbour across the edge, 5..9 round the cell, each from the side after
// the edge.
constexpr int kMult[3][5] = {{2, 1, 0, 1, 2}, {2, -1, 0, 1, -2}, {-2, -1, 0, -1, -2}};
constexpr int pv_edge(int K, int j) {
  return j < 5 ? cell_edge(K + 1, (K + 3 + 1 + j) % 6) : cell_edge(0, (K + 1 + j - 5) % 6);
}
constexpr int pv_mult(int K, int j) { return kMult[K][j % 5]; }

// Edges a cell's Laplacian reads: those of the cell and of its first three
// neighbours.
struct Needs {
  bool lap[kEdges];
};
constexpr Needs make_needs() {
  Needs n{};
  for (int i = 0; i < 4; ++i)
    for (int d = 0; d < 6; ++d) n.lap[cell_edge(i, d)] = true;
  return n;
}
constexpr Needs kNeed = make_needs();

} // namespace hexl
} // namespace omega_hip
