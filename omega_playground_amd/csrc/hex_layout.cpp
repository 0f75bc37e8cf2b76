// Records for the pattern-specialised kernels on the regular hexagonal mesh.
//
// For every edge the record holds its ten edges-on-edge and the ten distinct
// vertices and cells they touch, in first-appearance order; every edge must
// reproduce the tables of hex_pattern.hpp exactly, every cell must own three
// edges (its local edges 0..2, in class order) and two vertices, and every
// cell edge must list the cell second for j < 3 and first for j >= 3.  Any
// mismatch leaves hex_ok false and the general kernels are used.
#include <algorithm>
#include <cmath>

#include "hex_lattice.hpp"
#include "hex_pattern.hpp"
#include "internal.hpp"

namespace omega_hip {

namespace {

// Ids numbered in first-appearance order against an expected numbering:
// expect(k, id) is true when id is the k-th distinct id, known or new; that
// the ids taken are distinct is checked once at the end.
template <int most> struct Appear {
  int id[most], n = 0;
  bool expect(int k, int x) {
    if (k < n) return id[k] == x;
    if (k > n || n == most) return false;
    id[n++] = x;
    return true;
  }
  bool distinct() const {
    for (int i = 1; i < n; ++i)
      for (int j = 0; j < i; ++j)
        if (id[i] == id[j]) return false;
    return true;
  }
};

} // namespace

bool build_hex_records(DeviceMesh &dm) {
  const HostMesh &m = dm.host;
  const int NC = m.ncells, NE = m.nedges, ME = m.max_edges;
  dm.hex_ok = false;
  dm.hexd_ok = false;
  if (ME < 6 || dm.me2 != hex::kSlots) return false;
  // cells_on_cell in device numbering, derived from the cell's edges
  dm.coc_h.assign((size_t)NC * 6, 0);
  for (int c = 0; c < NC; ++c) {
    if (dm.noc_h[c] != 6) return false;
    if (dm.eofs_h[c + 1] - dm.eofs_h[c] != 3 || dm.vofs_h[c + 1] - dm.vofs_h[c] != 2) return false;
    for (int j = 0; j < 6; ++j) {
      const int e = dm.eoc_h[(size_t)c * ME + j];
      if (j < 3 && e != dm.eofs_h[c] + j) return false;
      const int a0 = dm.coe_h[2 * (size_t)e], a1 = dm.coe_h[2 * (size_t)e + 1];
      const int other = hex::cell_is_second(j) ? a0 : a1;
      const int self = hex::cell_is_second(j) ? a1 : a0;
      if (self != c || other == c) return false;
      dm.coc_h[(size_t)c * 6 + j] = other;
    }
  }
  dm.hexrec_h.assign((size_t)NE * hex::kRecInts, 0);
  for (int c = 0; c < NC; ++c) {
    for (int k = 0; k < 3; ++k) {
      const int e = dm.eofs_h[c] + k;
      if (dm.noe_h[e] != hex::kSlots) return false;
      Appear<hex::kUniq> uv, uc;
      int *rec = &dm.hexrec_h[(size_t)e * hex::kRecInts];
      for (int j = 0; j < hex::kSlots; ++j) {
        const int ej = dm.eoe_h[(size_t)e * dm.me2 + j];
        rec[j] = ej;
        if (!uv.expect(hex::LV0[k][j], dm.voe_h[2 * (size_t)ej]) ||
            !uv.expect(hex::LV1[k][j], dm.voe_h[2 * (size_t)ej + 1]) ||
            !uc.expect(hex::LC0[k][j], dm.coe_h[2 * (size_t)ej]) ||
            !uc.expect(hex::LC1[k][j], dm.coe_h[2 * (size_t)ej + 1]))
          return false;
      }
      if (uv.n != hex::kUniq || uc.n != hex::kUniq || !uv.distinct() || !uc.distinct()) return false;
      for (int s = 0; s < 2; ++s) {
        if (uv.id[hex::OWNV[k][s]] != dm.voe_h[2 * (size_t)e + s]) return false;
        if (uc.id[hex::OWNC[k][s]] != dm.coe_h[2 * (size_t)e + s]) return false;
      }
      std::copy(uv.id, uv.id + hex::kUniq, rec + 10);
      std::copy(uc.id, uc.id + hex::kUniq, rec + 20);
    }
  }
  dm.hex_ok = true;
  // diagnostics rows: every cell's owned vertices must follow the hexd maps
  dm.hexd_ok = true;
  for (int c = 0; c < NC && dm.hexd_ok; ++c) {
    int E[8], Cl[7];
    for (int j = 0; j < 6; ++j) E[j] = dm.eoc_h[(size_t)c * ME + j];
    Cl[0] = c;
    for (int j = 0; j < 6; ++j) Cl[1 + j] = dm.coc_h[(size_t)c * 6 + j];
    const int v0 = dm.vofs_h[c];
    E[6] = dm.eov_h[3 * (size_t)v0 + 2];
    E[7] = dm.eov_h[3 * (size_t)(v0 + 1) + 1];
    for (int i = 0; i < 2 && dm.hexd_ok; ++i)
      for (int j = 0; j < 3; ++j) {
        const int v = v0 + i;
        if (dm.eov_h[3 * (size_t)v + j] != E[hexd::VE[i][j]] ||
            dm.cov_h[3 * (size_t)v + j] != Cl[hexd::VC[i][j]])
          dm.hexd_ok = false;
      }
  }
  // per-cell union stencil: every cell must reproduce the hexu tables
  dm.hexu_ok = false;
  dm.hexu_h.assign((size_t)NC * hexu::kRec, 0);
  for (int c = 0; c < NC; ++c) {
    Appear<hexu::kNE> ue;
    Appear<hexu::kNV> uv;
    Appear<hexu::kNC> uc;
    bool ok = true;
    for (int k = 0; k < 3; ++k) ok = ok && ue.expect(k, dm.eofs_h[c] + k);
    for (int k = 0; k < 3 && ok; ++k) {
      const size_t e = dm.eofs_h[c] + k;
      for (int j = 0; j < hex::kSlots; ++j) {
        const size_t ej = dm.eoe_h[e * dm.me2 + j];
        ok = ok && ue.expect(hexu::TE[k][j], (int)ej) && uv.expect(hexu::TV0[k][j], dm.voe_h[2 * ej]) &&
             uv.expect(hexu::TV1[k][j], dm.voe_h[2 * ej + 1]) &&
             uc.expect(hexu::TC0[k][j], dm.coe_h[2 * ej]) &&
             uc.expect(hexu::TC1[k][j], dm.coe_h[2 * ej + 1]);
      }
      for (int s = 0; s < 2; ++s)
        ok = ok && uv.expect(hexu::OV[k][s], dm.voe_h[2 * e + s]) &&
             uc.expect(hexu::OC[k][s], dm.coe_h[2 * e + s]);
    }
    for (int j = 0; j < 6 && ok; ++j) {
      const size_t e = dm.eoc_h[(size_t)c * ME + j];
      ok = ue.expect(hexu::CE[j], (int)e) && uc.expect(hexu::CC0[j], dm.coe_h[2 * e]) &&
           uc.expect(hexu::CC1[j], dm.coe_h[2 * e + 1]);
    }
    ok = ok && uc.expect(hexu::SELF, c) && ue.n == hexu::kNE && uv.n == hexu::kNV &&
         uc.n == hexu::kNC && ue.distinct() && uv.distinct() && uc.distinct();
    if (!ok) {
      dm.hexu_h.clear();
      return true;
    }
    int *rec = &dm.hexu_h[(size_t)c * hexu::kRec];
    std::copy(ue.id, ue.id + hexu::kNE, rec);
    std::copy(uv.id, uv.id + hexu::kNV, rec + hexu::kNE);
    std::copy(uc.id, uc.id + hexu::kNC, rec + hexu::kNE + hexu::kNV);
  }
  dm.hexu_ok = true;
  return true;
}

// Every table the one-launch stage kernels replace by lattice arithmetic is
// checked here: neighbours that step back and round a corner as on the
// lattice (then the cell at an offset does not depend on the path to it),
// edges, vertices and edges-on-edge at their lattice places, and one
// magnitude per coefficient kind with the signs and TRiSK multiples of
// hex_lattice.hpp, bit for bit.
void build_hex_stage(DeviceMesh &dm) {
  dm.stage_ok = false;
  dm.hexc_h.clear();
  const HostMesh &m = dm.host;
  const int NC = m.ncells, ME = m.max_edges;
  if (!dm.hex_ok || !dm.coef_uni || !dm.off32 || dm.me2 != hex::kSlots) return;
  // a cell's three edge rows are one 24-bit factor of the velocities' offsets
  if (3 * (size_t)m.nlayers * sizeof(double) >= size_t(1) << 24) return;
  namespace hl = hexl;
  HexCoef &q = dm.stage_coef;
  const double C = dm.cdiv_h[3], ke = dm.cke_h[0], R = dm.crv_h[0], th = dm.cth_h[0];
  const double w1 = dm.w_h[1];
  for (int j = 0; j < 6; ++j)
    if (dm.cdiv_h[j] != (j < 3 ? -C : C) || dm.cke_h[j] != ke) return;
  for (int x = 0; x < 2; ++x)
    for (int j = 0; j < 3; ++j)
      if (dm.crv_h[3 * x + j] != hl::vert(x).s[j] * R || dm.cth_h[3 * x + j] != th) return;
  for (int K = 0; K < 3; ++K)
    for (int j = 0; j < 10; ++j)
      if (dm.w_h[K * 10 + j] != hl::pv_mult(K, j) * w1) return;
  // products by powers of two must be exact: no tiny coefficients
  for (double x : {C, ke, R, th, w1})
    if (!(std::fabs(x) > 1e-200 && std::fabs(x) < 1e200)) return;
  const int *coc = dm.coc_h.data();
  for (int c = 0; c < NC; ++c)
    for (int d = 0; d < 6; ++d) {
      const int n = coc[6 * (size_t)c + d];
      if (coc[6 * (size_t)n + (d + 3) % 6] != c) return;
      if (coc[6 * (size_t)n + (d + 2) % 6] != coc[6 * (size_t)c + (d + 1) % 6]) return;
    }
  // the lattice's places as tables
  int ce[6], pe[3][10];
  hl::Edge ed[3];
  hl::Vert ve[2];
  for (int d = 0; d < 6; ++d) ce[d] = hl::cell_edge(0, d);
  for (int K = 0; K < 3; ++K) {
    ed[K] = hl::edge(K);
    for (int j = 0; j < 10; ++j) pe[K][j] = hl::pv_edge(K, j);
  }
  for (int x = 0; x < 2; ++x) ve[x] = hl::vert(x);
  dm.hexc_h.resize((size_t)NC * hl::kRec);
  for (int c = 0; c < NC; ++c) {
    int *r = &dm.hexc_h[(size_t)c * hl::kRec];
    r[0] = c;
    for (int d = 0; d < 6; ++d) r[1 + d] = coc[6 * (size_t)c + d];
    for (int d = 0; d < 6; ++d) {
      r[7 + 2 * d] = coc[6 * (size_t)r[1 + d] + d];
      r[8 + 2 * d] = coc[6 * (size_t)r[1 + d] + (d + 1) % 6];
    }
    r[19] = 0;
    auto eid = [&](int e) { return 3 * r[e / 3] + e % 3; };
    auto vid = [&](int v) { return 2 * r[v / 2] + v % 2; };
    bool ok = true;
    for (int d = 0; d < 6; ++d) ok = ok && dm.eoc_h[(size_t)c * ME + d] == eid(ce[d]);
    for (int K = 0; K < 3; ++K) {
      const size_t e = 3 * (size_t)c + K;
      for (int s = 0; s < 2; ++s)
        ok = ok && dm.coe_h[2 * e + s] == r[ed[K].c[s]] && dm.voe_h[2 * e + s] == vid(ed[K].v[s]);
      for (int j = 0; j < 10; ++j) ok = ok && dm.eoe_h[e * 10 + j] == eid(pe[K][j]);
    }
    for (int x = 0; x < 2; ++x) {
      const size_t v = 2 * (size_t)c + x;
      for (int j = 0; j < 3; ++j)
        ok = ok && dm.eov_h[3 * v + j] == eid(ve[x].e[j]) && dm.cov_h[3 * v + j] == r[ve[x].c[j]];
    }
    if (!ok) {
      dm.hexc_h.clear();
      return;
    }
  }
  q.crv = R;
  q.cth = th;
  q.w = w1;
  q.w2 = w1 / 2;
  q.cke = ke;
  q.cdiv = C;
  q.hdiv = C / 2;
  q.qdiv = C / 4;
  q.idc = dm.inv_dc_h[0];
  q.idv = dm.inv_dv_h[0];
  q.idv4 = dm.inv_dv4_h[0];
  q.s2 = dm.s2_h[0];
  q.ml = dm.maxlev_h[0];
  // place every cell on the lattice: rows of nx cells running E, the next row
  // NE of an even one and NW of an odd one
  int nx = 0;
  for (int c = 0; nx == 0 || c != 0; c = coc[6 * (size_t)c + 3], ++nx)
    if (nx > NC) return;
  if (NC % nx || (NC / nx) % 2) return;
  const int ny = NC / nx;
  std::vector<int> at((size_t)NC), seen((size_t)NC, 0);
  for (int r = 0, first = 0; r < ny; ++r) {
    for (int i = 0, c = first; i < nx; ++i, c = coc[6 * (size_t)c + 3]) {
      at[(size_t)r * nx + i] = c;
      if (seen[c]++) return;
    }
    first = coc[6 * (size_t)first + (r % 2 ? 5 : 4)];
    if (r + 1 == ny && first != 0) return; // the rows close without a shift
  }
  // block shape: four lanes of two levels and 8 x 8 cells; with fewer lanes
  // of levels more cells
  TileView &t = dm.tile;
  const int lanes = m.nlayers % 2 == 0 ? m.nlayers / 2 : m.nlayers;
  t.lx = lanes >= 3 ? 4 : lanes;
  t.tw = t.lx == 4 ? 8 : 16;
  t.th = t.lx == 1 ? 16 : 8;
  t.nx = nx;
  t.ny = ny;
  const int tx = (nx + t.tw - 1) / t.tw, ty = (ny + t.th - 1) / t.th;
  dm.tile_h.resize((size_t)tx * ty * (t.tw + 4) * (t.th + 4));
  int *id = dm.tile_h.data();
  for (int j = 0; j < ty; ++j)
    for (int i = 0; i < tx; ++i)
      for (int y = -2; y < t.th + 2; ++y) {
        const int *row = &at[(size_t)(((j * t.th + y) % ny + ny) % ny) * nx];
        int q = ((i * t.tw - 2) % nx + nx) % nx;
        for (int x = 0; x < t.tw + 4; ++x) {
          *id++ = row[q];
          if (++q == nx) q = 0;
        }
      }
  dm.stage_ok = true;
}

} // namespace omega_hip
