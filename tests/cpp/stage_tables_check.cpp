// Host check of the stage kernels' tile tables (build_stage_tables) and of
// the rule that leaves the cells beyond the ring out of LDS: replays the
// kernels' index arithmetic over every tile against the mesh.  Built with g++
// into a shared library by tests/test_stage_tables_host.py.
#include <cstdint>
#include <cstdio>
#include <string>
#include <vector>

#include "../../swe_fvm_amd/csrc/swe_tiles.h"

using namespace swe;

extern "C" int stage_tables_check(int64_t T, const int* tp, const int* tt, const int* te, const uint32_t* cflag,
                                  const int* et0, const int* et1, const int* ep0, const int* ep1, int64_t* out,
                                  char* msg, int msglen) {
  auto bad = [&](const std::string& m) {
    std::snprintf(msg, size_t(msglen), "%s", m.c_str());
    return 1;
  };
  StageTables S;
  if (!build_stage_tables(T, tp, tt, te, cflag, et0, et1, ep0, ep1, S)) return bad("refused");
  DevTiles D{};
  D.ntiles = S.ntiles;
  D.sx = S.sx; D.sr = S.sr; D.sn = S.sn; D.se = S.se;
  D.lo = S.max_own_nodes; D.la = S.max_own_ev;
  for (int64_t t = 0; t < S.ntiles; ++t) {
    const TileHead h = S.head[size_t(t)];
    const int64_t c0 = t * kTileCells;
    const int nc = int(T - c0 < kTileCells ? T - c0 : kTileCells);
    if (h.nr > S.sr || h.nx > S.sx || h.nn > S.sn || h.ne > S.se || h.nn0 > D.lo || h.na > D.la || h.nr > h.nx ||
        h.nn0 > h.nn || h.ne0 > h.na || h.na > h.ne || h.nr > kTileCells)
      return bad("counts");
    const int* const xl = S.xcell.data() + t * S.sx;
    const int* const nl = S.node.data() + t * S.sn;
    auto cell = [&](int l) -> int64_t {
      return l < nc ? c0 + l : (l >= kTileCells && l < kTileCells + h.nx ? xl[l - kTileCells] : -1);
    };
    auto at = [](uint32_t w, int k) { return int((w >> (kLocalBits * uint32_t(k))) & kLocalMask); };
    const EvalCode* const ev = S.ev.data() + t * S.se;
    const int* const ee = S.evedge.data() + t * S.se;
    auto slot_is = [&](uint32_t slots, int64_t c, int lim) {
      for (int k = 0; k < 3; ++k)
        if (at(slots, k) >= lim || ee[at(slots, k)] != te[k * T + c]) return false;
      return true;
    };
    for (int l = 0; l < nc; ++l) {
      const int64_t i = c0 + l;
      const TileCell c = S.cell[size_t(i)];
      if (c.flags != (cflag[i] & 0xffffu) || !slot_is(c.slots, i, h.na)) return bad("own cell");
      for (int k = 0; k < 3; ++k) {
        if (at(c.nodes, k) >= h.nn0 || nl[at(c.nodes, k)] != tp[k * T + i]) return bad("own cell's node");
        const int n = at(c.nbs, k), y = tt[k * T + i];
        const bool ok = y >= 0 ? n < kTileCells + h.nr && cell(n) == y
                               : n == int(et1[te[k * T + i]] == -1 ? kLocalWall : kLocalFree);
        if (!ok) return bad("own cell's neighbour");
      }
    }
    for (int q = 0; q < h.nr; ++q) {
      const RingCode c = S.xcode[size_t(t * S.sr + q)];
      if (c.flags != (cflag[xl[q]] & 0xffffu) || !slot_is(c.slots, xl[q], h.ne)) return bad("ring cell");
    }
    for (int j = 0; j < h.ne; ++j) {
      const int e = ee[j], f = at(ev[j].cells, 0), g = at(ev[j].cells, 1);
      const int a = at(ev[j].nodes, 0), b = at(ev[j].nodes, 1);
      if (cell(f) != et0[e]) return bad("evaluation's first cell");
      if (et1[e] >= 0 ? cell(g) != et1[e] : g != int(et1[e] == -1 ? kLocalWall : kLocalFree))
        return bad("evaluation's second cell");
      if (a >= h.nn || b >= h.nn || nl[a] != ep0[e] || nl[b] != ep1[e]) return bad("evaluation's nodes");
      const bool own = (et0[e] >= c0 && et0[e] < c0 + nc) || (et1[e] >= c0 && et1[e] < c0 + nc);
      if (own != (j < h.na) || (j < h.ne0) != (et0[e] >= c0 && et0[e] < c0 + nc)) return bad("order of evaluations");
      // what a tile without the cells beyond the ring finds in LDS
      const int in = kTileCells + h.nr, lg = et1[e] < 0 ? f : g;
      if (own && (f >= in || lg >= in || a >= h.nn0 || b >= h.nn0)) return bad("own edge reaches beyond the ring");
      if (f >= in && lg >= in) return bad("an edge of two cells beyond the ring");
    }
  }
  int n = 0;
  out[n++] = S.ntiles;
  for (int len = 0; len < 2; ++len) {
    out[n++] = int64_t(stage_lds(D, false, false, len != 0));
    out[n++] = int64_t(stage_lds(D, false, true, len != 0));
    out[n++] = stage_far(D, len != 0, S.ntiles) ? 1 : 0;
  }
  return 0;
}
