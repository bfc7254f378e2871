// Static tables of the fused flux / draining / update kernel (swe_fused.hip).
//
// The cells are cut into tiles of kTileCells consecutive (Morton-ordered)
// cells.  A tile's kernel needs the fluxes of every edge of its own cells
// (the update) and of every edge of their outside neighbours, the tile's
// ring (their draining time steps, which the update of a cell next to them
// reads).  Its local cells are the tile's own cells (local ids 0 ..
// kTileCells - 1) followed by the ring (kTileCells + j, in order of first
// appearance).  Every edge of a local cell is evaluated once per tile, by
// its et0 cell when that cell is local, else by its local cell; the
// evaluations are numbered in order (local cell, then k) and their number
// is the LDS slot of that edge's flux.  Per (local cell, k) the tables hold
//   code = slot << 16 | nb
// with nb the local id of the neighbour across edge k, or kNbWall /
// kNbFree (boundary edge of that tag) or kNbOut (a ring cell's neighbour
// outside the tile: its global id is tt's).  Each evaluation also records
// its edge's index: a storing launch writes an edge's flux from the one
// evaluation whose et0 cell is a tile cell (the edge's et0 cell evaluates
// it in that cell's own tile, and no other tile holds that cell).
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <exception>
#include <thread>
#include <vector>

#include "swe_tiles.h"

namespace swe {

namespace {

// local ids of one tile: a small open-addressing table, emptied by a new stamp
class LocalIds {
 public:
  void next_tile() { ++stamp_; }
  // the slot of id g; its value is valid when found
  int* find(int g, bool& found) {
    uint32_t h = (uint32_t(g) * 2654435761u) >> (32 - kBits);
    while (mark_[h] == stamp_ && key_[h] != g) h = (h + 1) & (kSize - 1);
    found = mark_[h] == stamp_;
    mark_[h] = stamp_;
    key_[h] = g;
    return &val_[h];
  }
  int get(int g) const {  // -1: not there
    uint32_t h = (uint32_t(g) * 2654435761u) >> (32 - kBits);
    while (mark_[h] == stamp_ && key_[h] != g) h = (h + 1) & (kSize - 1);
    return mark_[h] == stamp_ ? val_[h] : -1;
  }

 private:
  static constexpr int kBits = 13;
  static constexpr uint32_t kSize = 1u << kBits;  // 6 kTileCells cells at most (own, ring, beyond): under half full
  static_assert(2 * 6 * kTileCells <= int(kSize), "table of local ids");
  std::vector<int> key_ = std::vector<int>(kSize), val_ = std::vector<int>(kSize);
  std::vector<uint32_t> mark_ = std::vector<uint32_t>(kSize, 0u);
  uint32_t stamp_ = 0u;
};

// build_tiles over tiles [t0, t1); tables relative to the first
bool build_range(int64_t T, int64_t t0, int64_t t1, const int* tt, const int* te, const uint32_t* cflag, const int* et0,
                 const int* et1, const int* ep0, const int* ep1, TileTables& out) {
  const int64_t nt = t1 - t0, b0 = t0 * kTileCells, nb = std::min<int64_t>(T, t1 * kTileCells) - b0;
  out = TileTables{};
  out.ntiles = nt;
  out.code.assign(size_t(3 * nb), 0u);
  out.ring_off.assign(size_t(nt) + 1, 0);
  out.ev_off.assign(size_t(nt) + 1, 0);
  const size_t guess = size_t(nb) * 2 + size_t(nb) / 16 + 64;
  out.ev.reserve(guess);
  out.evrec.reserve(guess);
  out.evedge.reserve(guess);
  LocalIds ids;  // ring cells; the tile's own are c0 .. c0 + nc - 1
  std::vector<int> ring;
  std::vector<uint32_t> codes;          // [local][k] of the current tile
  std::vector<int> slot;                // [local][k]: evaluation slot
  for (int64_t t = 0; t < nt; ++t) {
    const int64_t c0 = b0 + t * kTileCells, c1 = std::min<int64_t>(T, c0 + kTileCells);
    const int nc = int(c1 - c0);
    ring.clear();
    ids.next_tile();
    auto local = [&](int64_t y) -> int { return y >= c0 && y < c1 ? int(y - c0) : ids.get(int(y)); };
    for (int64_t i = c0; i < c1; ++i)
      for (int k = 0; k < 3; ++k) {
        const int y = tt[size_t(k * T + i)];
        if (y < 0 || (y >= c0 && y < c1)) continue;
        bool found;
        int* v = ids.find(y, found);
        if (!found) {
          *v = kTileCells + int(ring.size());
          ring.push_back(y);
        }
      }
    const int nl = kTileCells + int(ring.size());
    if (nl > kTileMaxLocal) return false;
    auto global = [&](int l) -> int64_t { return l < kTileCells ? c0 + l : ring[size_t(l - kTileCells)]; };
    auto local_ok = [&](int l) { return l < nc || l >= kTileCells; };
    // neighbour codes and evaluators
    codes.assign(size_t(3 * nl), 0u);
    slot.assign(size_t(3 * nl), -1);
    int nev = 0;
    for (int l = 0; l < nl; ++l) {
      if (!local_ok(l)) continue;
      const int64_t x = global(l);
      for (int k = 0; k < 3; ++k) {
        const int y = tt[size_t(k * T + x)];
        uint32_t nbc;
        bool evaluator;
        if (y < 0) {
          nbc = et1[te[size_t(k * T + x)]] == -1 ? kNbWall : kNbFree;
          evaluator = true;
        } else if (const int ly = local(y); ly >= 0) {
          nbc = uint32_t(ly);
          evaluator = (cflag[x] >> k) & 1u;  // the et0 side of a local pair
        } else {
          nbc = kNbOut;  // ring cell's outside neighbour
          evaluator = true;
        }
        codes[size_t(3 * l + k)] = nbc;
        if (evaluator) {
          slot[size_t(3 * l + k)] = nev++;
          out.ev.push_back(uint16_t((l << 2) | k));
          const int e = te[size_t(k * T + x)];
          out.evrec.push_back(EdgeRec{et0[e], et1[e], ep0[e], ep1[e]});
          out.evedge.push_back(e);
        }
      }
    }
    // the other side of every local pair reads its twin's slot
    for (int l = 0; l < nl; ++l) {
      if (!local_ok(l)) continue;
      const int64_t x = global(l);
      for (int k = 0; k < 3; ++k) {
        if (slot[size_t(3 * l + k)] >= 0) continue;
        const int ly = int(codes[size_t(3 * l + k)]);
        const int64_t y = global(ly);
        const int e = te[size_t(k * T + x)];
        for (int q = 0; q < 3; ++q)
          if (te[size_t(q * T + y)] == e) slot[size_t(3 * l + k)] = slot[size_t(3 * ly + q)];
        if (slot[size_t(3 * l + k)] < 0) return false;  // inconsistent tables
      }
    }
    if (nev > kTileMaxEval) return false;
    out.max_eval = std::max(out.max_eval, nev);
    out.max_ring = std::max(out.max_ring, int(ring.size()));
    for (int l = 0; l < nl; ++l) {
      if (!local_ok(l)) continue;
      for (int k = 0; k < 3; ++k) {
        const uint32_t c = (uint32_t(slot[size_t(3 * l + k)]) << 16) | codes[size_t(3 * l + k)];
        if (l < kTileCells) out.code[size_t(k * nb + (c0 - b0) + l)] = c;
        else out.ring_code.push_back(c);  // [ring entry][k], 3 per entry
      }
    }
    for (int y : ring) out.ring_cell.push_back(y);
    out.ring_off[size_t(t) + 1] = int(out.ring_cell.size());
    out.ev_off[size_t(t) + 1] = int(out.ev.size());
  }
  return true;
}

}  // namespace

bool build_tiles(int64_t T, const int* tt, const int* te, const uint32_t* cflag, const int* et0, const int* et1,
                 const int* ep0, const int* ep1, TileTables& out) {
  return build_range(T, 0, (T + kTileCells - 1) / kTileCells, tt, te, cflag, et0, et1, ep0, ep1, out);
}

namespace {

// the stage tables of one range of tiles, before their lists are cut to the
// strides of the whole mesh
struct StageRange {
  int64_t t0 = 0;
  std::vector<int> xcell, node, edges;  // tile by tile
  std::vector<EvalCode> evs;
  std::vector<RingCode> xcode;
  std::vector<int> x0, n0, r0, e0;  // [tiles + 1]
  int sx = 0, sr = 0, sn = 0, se = 0, lo = 0, la = 0;
};

// heads and cells of the range go to their place in `out`
bool build_stage_range(int64_t T, int64_t t0, int64_t t1, const int* tp, const int* tt, const int* te,
                       const uint32_t* cflag, const int* et0, const int* et1, const int* ep0, const int* ep1,
                       StageTables& out, StageRange& R) {
  TileTables P;
  if (!build_range(T, t0, t1, tt, te, cflag, et0, et1, ep0, ep1, P)) return false;
  const int64_t b0 = t0 * kTileCells, nb = int64_t(P.code.size() / 3);
  R.t0 = t0;
  R.evs.resize(P.ev.size());
  R.edges.resize(P.ev.size());
  R.xcode.resize(P.ring_cell.size());
  R.x0.assign(size_t(P.ntiles) + 1, 0);
  R.n0.assign(size_t(P.ntiles) + 1, 0);
  R.xcell.reserve(2 * P.ring_cell.size() + P.ring_cell.size() / 4);
  R.node.reserve(size_t(nb));
  LocalIds cells, nodes;
  std::vector<int> order;
  std::vector<uint32_t> slot;
  for (int64_t t = 0; t < P.ntiles; ++t) {
    const int64_t c0 = b0 + t * kTileCells;
    const int nc = int(std::min<int64_t>(kTileCells, T - c0));
    const int rg0 = P.ring_off[size_t(t)], nr = P.ring_off[size_t(t) + 1] - rg0;
    const int e0 = P.ev_off[size_t(t)], ne = P.ev_off[size_t(t) + 1] - e0;
    cells.next_tile();
    nodes.next_tile();
    int nl = kTileCells, nn = 0;
    auto add_cell = [&](int y) {
      if (y >= c0 && y < c0 + nc) return;
      bool found;
      int* v = cells.find(y, found);
      if (found) return;
      *v = nl++;
      R.xcell.push_back(y);
    };
    auto cell_of = [&](int y) { return uint32_t(y >= c0 && y < c0 + nc ? int(y - c0) : cells.get(y)); };
    auto node_of = [&](int g) {
      bool found;
      int* v = nodes.find(g, found);
      if (!found) {
        *v = nn++;
        R.node.push_back(g);
      }
      return uint32_t(*v);
    };
    for (int q = 0; q < nr; ++q) add_cell(P.ring_cell[size_t(rg0 + q)]);
    for (int q = 0; q < nr; ++q)  // the cells beyond the ring
      for (int k = 0; k < 3; ++k) {
        const int y = tt[size_t(k * T + P.ring_cell[size_t(rg0 + q)])];
        if (y >= 0) add_cell(y);
      }
    // the evaluations: the tile's own edges, its cells' other edges, the
    // ring's outer edges
    order.clear();
    slot.assign(size_t(ne), 0);
    int ne0 = 0, na = 0;
    for (int pass = 0; pass < 3; ++pass) {
      for (int j = 0; j < ne; ++j) {
        const EdgeRec& r = P.evrec[size_t(e0 + j)];
        const bool own0 = r.et0 >= c0 && r.et0 < c0 + nc, own1 = r.et1 >= c0 && r.et1 < c0 + nc;
        if (pass != (own0 ? 0 : (own1 ? 1 : 2))) continue;
        slot[size_t(j)] = uint32_t(order.size());
        order.push_back(j);
      }
      if (pass == 0) ne0 = int(order.size());
      if (pass == 1) na = int(order.size());
    }
    for (int l = 0; l < nc; ++l) {
      const int64_t x = c0 + l;
      TileCell c{0u, 0u, 0u, cflag[x] & 0xffffu};
      for (int k = 0; k < 3; ++k) {
        const int y = tt[size_t(k * T + x)];
        const uint32_t n = y >= 0 ? cell_of(y) : (et1[te[size_t(k * T + x)]] == -1 ? kLocalWall : kLocalFree);
        const uint32_t sh = kLocalBits * uint32_t(k);
        c.nodes |= node_of(tp[size_t(k * T + x)]) << sh;
        c.nbs |= n << sh;
        c.slots |= slot[P.code[size_t(k * nb + (c0 - b0) + l)] >> 16] << sh;
      }
      out.cell[size_t(x)] = c;
    }
    const int nn0 = nn;
    for (int q = 0; q < nr; ++q) {
      RingCode c{0u, cflag[P.ring_cell[size_t(rg0 + q)]] & 0xffffu};
      for (int k = 0; k < 3; ++k)
        c.slots |= slot[P.ring_code[size_t(3 * (rg0 + q) + k)] >> 16] << (kLocalBits * uint32_t(k));
      R.xcode[size_t(rg0 + q)] = c;
    }
    for (int j = 0; j < ne; ++j) {
      const EdgeRec& r = P.evrec[size_t(e0 + order[size_t(j)])];
      const uint32_t f = cell_of(r.et0);
      const uint32_t g = r.et1 >= 0 ? cell_of(r.et1) : (r.et1 == -1 ? kLocalWall : kLocalFree);
      R.evs[size_t(e0 + j)] = EvalCode{f | (g << kLocalBits), node_of(r.ep0) | (node_of(r.ep1) << kLocalBits)};
      R.edges[size_t(e0 + j)] = P.evedge[size_t(e0 + order[size_t(j)])];
    }
    if (uint32_t(nl) > kLocalMax || uint32_t(nn) > kLocalMax || uint32_t(ne) > kLocalMax) return false;
    out.head[size_t(t0 + t)] = TileHead{uint16_t(nr), uint16_t(nl - kTileCells), uint16_t(nn0), uint16_t(nn),
                                        uint16_t(ne0), uint16_t(na), uint16_t(ne), 0};
    R.x0[size_t(t) + 1] = int(R.xcell.size());
    R.n0[size_t(t) + 1] = int(R.node.size());
    R.sx = std::max(R.sx, nl - kTileCells);
    R.sr = std::max(R.sr, nr);
    R.sn = std::max(R.sn, nn);
    R.se = std::max(R.se, ne);
    R.lo = std::max(R.lo, nn0);
    R.la = std::max(R.la, na);
  }
  R.r0 = std::move(P.ring_off);
  R.e0 = std::move(P.ev_off);
  return true;
}

// f(0) .. f(n - 1), each on a thread of its own; the first exception is thrown on
template <class F>
void on_threads(int n, F f) {
  std::vector<std::exception_ptr> err(static_cast<size_t>(n));
  auto call = [&](int k) {
    try {
      f(k);
    } catch (...) {
      err[size_t(k)] = std::current_exception();
    }
  };
  std::vector<std::thread> th;
  th.reserve(size_t(n));
  int k = 1;
  try {
    for (; k < n; ++k) th.emplace_back(call, k);
  } catch (...) {  // no more threads: the rest here
  }
  call(0);
  for (; k < n; ++k) call(k);
  for (auto& t : th) t.join();
  for (auto& e : err)
    if (e) std::rethrow_exception(e);
}

}  // namespace

bool build_stage_tables(int64_t T, const int* tp, const int* tt, const int* te, const uint32_t* cflag, const int* et0,
                        const int* et1, const int* ep0, const int* ep1, StageTables& out) {
  out = StageTables{};
  const int64_t nt = (T + kTileCells - 1) / kTileCells;
  out.ntiles = nt;
  out.head.resize(size_t(nt));
  out.cell.resize(size_t(T));
  // a range of tiles per thread, at least 16 (half a ms) each
  const int hw = int(std::max(1u, std::min(8u, std::thread::hardware_concurrency())));
  const int n = int(std::max<int64_t>(1, std::min<int64_t>(hw, nt / 16)));
  std::vector<StageRange> R(static_cast<size_t>(n));
  std::vector<char> ok(size_t(n), 0);
  on_threads(n, [&](int k) {
    ok[size_t(k)] = build_stage_range(T, nt * k / n, nt * (k + 1) / n, tp, tt, te, cflag, et0, et1, ep0, ep1, out,
                                      R[size_t(k)]) ? 1 : 0;
  });
  for (char o : ok)
    if (!o) return false;
  for (const StageRange& r : R) {
    out.sx = std::max(out.sx, r.sx);
    out.sr = std::max(out.sr, r.sr);
    out.sn = std::max(out.sn, r.sn);
    out.se = std::max(out.se, r.se);
    out.max_own_nodes = std::max(out.max_own_nodes, r.lo);
    out.max_own_ev = std::max(out.max_own_ev, r.la);
  }
  out.xcell.resize(size_t(nt) * size_t(out.sx));
  out.xcode.resize(size_t(nt) * size_t(out.sr));
  out.node.resize(size_t(nt) * size_t(out.sn));
  out.ev.resize(size_t(nt) * size_t(out.se));
  out.evedge.resize(size_t(nt) * size_t(out.se));
  on_threads(n, [&](int k) {
    const StageRange& r = R[size_t(k)];
    for (size_t t = 0; t + 1 < r.x0.size(); ++t) {
      const int64_t g = r.t0 + int64_t(t);
      std::copy(r.xcell.begin() + r.x0[t], r.xcell.begin() + r.x0[t + 1], out.xcell.begin() + g * out.sx);
      std::copy(r.node.begin() + r.n0[t], r.node.begin() + r.n0[t + 1], out.node.begin() + g * out.sn);
      std::copy(r.xcode.begin() + r.r0[t], r.xcode.begin() + r.r0[t + 1], out.xcode.begin() + g * out.sr);
      std::copy(r.evs.begin() + r.e0[t], r.evs.begin() + r.e0[t + 1], out.ev.begin() + g * out.se);
      std::copy(r.edges.begin() + r.e0[t], r.edges.begin() + r.e0[t + 1], out.evedge.begin() + g * out.se);
    }
  });
  return true;
}

bool plain_geometry(const double* px, const double* py, int64_t E, const int* ep0, const int* ep1) {
  const double lo = std::ldexp(1., -400), hi = std::ldexp(1., 400);
  for (int64_t e = 0; e < E; ++e) {
    const double dx = std::fabs(px[ep1[e]] - px[ep0[e]]), dy = std::fabs(py[ep1[e]] - py[ep0[e]]);
    if (dx == 0. && dy == 0.) return false;
    for (double d : {dx, dy})  // one that is no number is refused here
      if (d != 0. && !(d >= lo && d <= hi)) return false;
  }
  return true;
}

}  // namespace swe
