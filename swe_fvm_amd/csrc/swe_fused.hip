// Fused second half of a stage: ComputeFluxes, the draining time steps and
// the update (src/SpaceDisc.cpp:54-74, src/TimeDisc.cpp:3-66,
// src/Solvers.cpp:5-59) in one kernel per tile of kTileCells cells.
//
// A workgroup evaluates the flux of every edge of its tile's cells and of
// the cells around the tile (the ring) once, into LDS; then the draining
// time step of every local cell from those fluxes; then the update of its
// own cells.  Fluxes and draining steps never go to HBM: the separate flux,
// draining and update kernels write 24 B per edge and 8 B per cell and read
// them back by gathers.  Edges between two tiles are evaluated by both
// (each tile needs them), and so are the ring cells' other edges; every
// evaluation and every update is the same sequence of operations as in the
// separate kernels (the same device functions), so the results are
// identical bit for bit.
//
// The stage step size must be known before the kernel: a fixed dt, or the
// CFL step of an earlier flux pass of the same step (stages 2 and 3).  The
// pass's own CFL length-to-wavespeed minimum is not taken: the solver
// recomputes it with the fluxes when a getter asks for them.
//
// The first stage of a CFL step learns its step size from its own flux pass,
// so the separate flux kernel runs first; the FF instance of this kernel
// then loads the listed edges' fluxes from memory instead of evaluating them
// (the same values: the separate flux kernel is the same device functions
// in the same orientation) and runs the draining and update phases as
// usual, in place of the separate draining and update kernels.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "swe_common.h"
#include "swe_tiles.h"

namespace swe {

// waves per SIMD the register allocation must allow; a build-time knob
#ifndef SWE_FUSED_MIN_WAVES
#define SWE_FUSED_MIN_WAVES 4
#endif
__device__ __forceinline__ int local3(uint32_t word, int k) { return (int)((word >> (kLocalBits * k)) & kLocalMask); }

// A launch of no more tiles than the card has CUs leaves a CU one tile, whose
// ~560 evaluations take a wave per SIMD three rounds one after the other,
// bound by the latency of its arithmetic: three waves per SIMD take a round
// each.  Us per fused stage, 256 / 768 threads: 9.6 / 9.0 (1,600 cells), 13.3 /
// 11.9 (40,000), 11.9 / 11.1 (62,000).  Beyond, a CU has several tiles, which
// hide each other's latency (and 24 waves would not fit it).  The instance
// that reads its fluxes has nothing to spread.
constexpr int kWideThreads = 768, kWideTiles = kCus;

// Gathered per edge from memory, the cells and nodes took 65 gathers of ~26
// lines per wave (the L1 busy 63 % of the time, its return path 91 %).
// Staged in LDS, a tile reads its own cells and a copy of its nodes once,
// coalesced, and gathers only the ~130 cells around it; every further use is
// an LDS read by local index, and the tables shrink to one 16-byte record
// per cell and 8 bytes per evaluation.  What bounds it now is the FP64 VALU
// (75 % busy) and, before the first barrier, two levels of loads (the lists
// are read at fixed strides so that they wait for nothing): 40.5 KB of LDS
// for a Delaunay mesh's 256-cell tile, so four workgroups share a CU
// (three, at 42.6 KB with F1 and F2 kept of every edge, took 255 us at 4M
// cells; 240 cells per tile 221).  The edges that only the ring's draining
// steps need come last and give their mass flux alone.  Us per launch,
// gathering / staged, dam break: fused stage 283 / 219 (4M cells), 73.3 /
// 62.1 (1M), 23.1 / 21.5 (250k); after the flux pass 164 / 139, 41.7 / 38.5,
// 13.7 / 12.6; of 24 ensemble members (0.7M cells) 57.3 / 50.6 and 33.1 / 31.5.
//
// Those are tiles of Morton-ordered cells.  One that is a strip of a row-ordered
// mesh has two to three times the cells around it (StructTriangMesh: 130 in
// the ring and 260 beyond, 56.9 KB, two workgroups to a CU), and one such tile
// sets the strides of all.  FAR (stage_far) leaves out of LDS what the outer
// edges of the ring alone need, each once: the cells beyond the ring, gathered
// from memory by a number that is loaded an evaluation ahead, and the outer
// nodes, read from the tile's copy (39.2 KB, four workgroups).  Us per fused
// stage of such a mesh, gathering / staged whole / FAR: 340 / 385 / 288 (4M
// cells), 83.7 / 100.9 / 79.1 (1M), 35.5 / 40.9 / 34.7 (360,000); with the
// draining step's edge lengths 357 / 423 / 335, 89.5 / 106.6 / 85.4, 38.2 /
// 44.0 / 38.0.
template <int FLUX, int WS, bool LEN, bool NT, bool FF, bool FAR, int TH>
__global__ void __launch_bounds__(TH, TH == kTileCells ? SWE_FUSED_MIN_WAVES : TH / 256) k_fused(DevMesh M, DevTiles P, DevState S, DevState U0,
                                                      DevOut O, DevWork W, StageArgs A, int64_t t0, int64_t t1,
                                                      int store) {
  extern __shared__ double lds[];
  // the evaluating instance walks the tiles backwards (it follows a
  // forward reconstruction); the FF instance forwards (it follows k_flux)
  const int64_t tile = t0 + (FF ? logical_block() : logical_block_reversed());
  if (A.pw_clear && blockIdx.x == 0 && threadIdx.x == 0) *A.pw_clear = 0u;
  if (tile >= t1) return;  // padding workgroups of the XCD-aware grid
  const TileHead h = P.head[tile];
  const int64_t c0 = tile * kTileCells;
  const int nc = (int)(M.T - c0 < kTileCells ? M.T - c0 : kTileCells);
  const int tid = threadIdx.x;
  const int ns = FAR ? P.sr : P.sx;  // of the cells around the tile, those in LDS
  const int lc = kTileCells + ns;
  double* const cw = lds;  // w0 of the local cells, then the draining steps
  double* const cgx = cw + lc;
  double* const cgy = cgx + lc;
  double* const cu = cgy + lc;
  double* const cv = cu + lc;
  double* const ccx = cv + lc;
  double* const ccy = ccx + lc;
  double* const sD = lds;
  const int ln = (FF && !LEN) || FAR ? P.lo : P.sn;
  double* const nx_ = lds + (FF ? kTileCells + P.sr : 7 * lc);
  double* const ny_ = nx_ + ln;
  double* const nz_ = ny_ + ln;
  double* const sF0 = nz_ + ln;
  double* const sF1 = sF0 + P.se;
  double* const sF2 = sF1 + P.la;
  auto lnode = [&](int l) { return V3{nx_[l], ny_[l], nz_[l]}; };
  const double* const tn = P.tnode + tile * 3 * P.sn;
  const int* const xl = P.xcell + tile * P.sx;

  // Every load that waits for no other comes first: the cells around the
  // tile by number, its nodes, its own cells.
  const bool mine = tid < nc;
  const int i = (int)(c0 + (mine ? tid : 0));
  const bool comb = A.a0 != 0.;
  const int xc = tid < (FF ? P.sr : ns) ? xl[tid] : i;
  const TileCell tc = P.cell[i];
  V3 nd{0., 0., 0.};
  if (tid < ln) nd = V3{tn[tid], tn[P.sn + tid], tn[2 * P.sn + tid]};
  const bool ringed = tid < h.nr;  // the ring cell whose draining step this thread takes (nr <= kTileCells)
  RingCode rc{0u, 0u};
  double rbc = 0., arear = 0., hr = 0.;
  if (ringed) {
    rc = P.xcode[tile * P.sr + tid];
    const double* const r = P.tring + 2 * (tile * P.sr + tid);
    rbc = r[0];
    arear = r[1];
  }
  RhsCell q;
  if (TH > kTileCells && !mine) q.mu = Muscl{0., 0., 0., 0., 0.};
  else q.mu = load_muscl(S, W, i);
  double w, u, v, w0 = 0., u0 = 0., v0 = 0.;
  w = S.w[S.at(i)];
  u = S.u[S.at(i)];
  v = S.v[S.at(i)];
  if (comb) {
    w0 = U0.w[U0.at(i)];
    u0 = U0.u[U0.at(i)];
    v0 = U0.v[U0.at(i)];
  }
  const int nn = (FF && !LEN) || FAR ? h.nn0 : h.nn;
  const double* const xo = P.txc + 2 * tile * P.sx;
  if constexpr (FF) {
    // fluxes of the stage's flux pass, written by the separate flux kernel;
    // ne <= kTileMaxEval: at most kFE evaluations per thread, every load of
    // them issued before the first LDS write
    constexpr int kFE = (kTileMaxEval + TH - 1) / TH;
    int ev[kFE];
#pragma unroll
    for (int it = 0; it < kFE; ++it) {
      const int j = tid + it * TH;
      ev[it] = j < P.se ? P.evedge[tile * P.se + j] : 0;
    }
    if (ringed) hr = S.w[S.at(xc)] - rbc;
    double f0[kFE], f1[kFE], f2[kFE];
#pragma unroll
    for (int it = 0; it < kFE; ++it) {
      f0[it] = W.f0[ev[it]];
      if (tid + it * TH < h.na) {
        f1[it] = W.f1[ev[it]];
        f2[it] = W.f2[ev[it]];
      }
    }
#pragma unroll
    for (int it = 0; it < kFE; ++it) {
      const int j = tid + it * TH;
      if (j < h.ne) sF0[j] = f0[it];
      if (j < h.na) {
        sF1[j] = f1[it];
        sF2[j] = f2[it];
      }
    }
  } else {
    auto stage_cell = [&](int l, const Muscl& m, double cx, double cy) {
      cw[l] = m.w0;
      cgx[l] = m.gx;
      cgy[l] = m.gy;
      cu[l] = m.u0;
      cv[l] = m.v0;
      ccx[l] = cx;
      ccy[l] = cy;
    };
    const int nx = FAR && h.nx > P.sr ? P.sr : h.nx;
    if (tid < nx) {
      const Muscl m = load_muscl(S, W, xc);
      if (ringed) hr = S.w[S.at(xc)] - rbc;
      stage_cell(kTileCells + tid, m, xo[2 * tid], xo[2 * tid + 1]);
    }
    for (int j = tid + TH; j < nx; j += TH)
      stage_cell(kTileCells + j, load_muscl(S, W, xl[j]), xo[2 * j], xo[2 * j + 1]);
  }
  if (tid < nn) {
    nx_[tid] = nd.x;
    ny_[tid] = nd.y;
    nz_[tid] = nd.z;
  }
  for (int j = tid + TH; j < nn; j += TH) {
    nx_[j] = tn[j];
    ny_[j] = tn[P.sn + j];
    nz_[j] = tn[2 * P.sn + j];
  }
  const EvalCode* const evl = P.ev + tile * P.se;
  EvalCode rn{0u, 0u};
  if (!FF && tid < P.se) rn = evl[tid];
  __syncthreads();
  if constexpr (!FF) {
    if (mine) {  // the centroid as the setup kernel computes M.cxy
      const V3 c = centroid(lnode(local3(tc.nodes, 0)), lnode(local3(tc.nodes, 1)), lnode(local3(tc.nodes, 2)));
      cw[tid] = q.mu.w0;
      cgx[tid] = q.mu.gx;
      cgy[tid] = q.mu.gy;
      cu[tid] = q.mu.u0;
      cv[tid] = q.mu.v0;
      ccx[tid] = c.x;
      ccy[tid] = c.y;
    }
    __syncthreads();
    // ---- edge fluxes (k_flux's operations), one evaluation per LDS slot;
    // the next evaluation's code is loaded before this one's arithmetic
    auto lmuscl = [&](int l) { return Muscl{cw[l], cgx[l], cgy[l], cu[l], cv[l]}; };
    // FAR: the cell beyond the ring of the next evaluation's edge, by number
    auto beyond = [&](const EvalCode& r) {
      const int f = local3(r.cells, 0), t = local3(r.cells, 1);
      return f >= lc ? f - kTileCells : (t >= lc && t < (int)kLocalMax ? t - kTileCells : -1);
    };
    int xn = -1, gn = 0;
    if (FAR && tid < h.ne && (xn = beyond(rn)) >= 0) gn = xl[xn];
    for (int j = tid; j < h.ne; j += TH) {
      const EvalCode r = rn;
      const int x = xn, gx = gn;
      if (j + TH < h.ne) {
        rn = evl[j + TH];
        if (FAR && (xn = beyond(rn)) >= 0) gn = xl[xn];
      }
      const int f = local3(r.cells, 0), t = local3(r.cells, 1);
      const bool wall = t == (int)kLocalWall;
      const bool all = j < h.na;
      const int tr = t >= (int)kLocalMax ? f : t;  // boundary edges read their own cell twice: R = L
      auto end = [&](int l) {  // FAR: the nodes that only the ring's outer edges have are not staged
        return FAR && !all ? V3{tn[l], tn[P.sn + l], tn[2 * P.sn + l]} : lnode(l);
      };
      const V3 Pa = end(local3(r.nodes, 0)), Pb = end(local3(r.nodes, 1));
      Muscl mo{0., 0., 0., 0., 0.};
      double cxo = 0., cyo = 0.;
      if (FAR && x >= 0) {
        mo = load_muscl(S, W, gx);
        cxo = xo[2 * x];
        cyo = xo[2 * x + 1];
      }
      auto cell = [&](int l, double& cx, double& cy) {
        if (FAR && l >= lc) {
          cx = cxo;
          cy = cyo;
          return mo;
        }
        cx = ccx[l];
        cy = ccy[l];
        return lmuscl(l);
      };
      double cxf, cyf;
      const Muscl mf = cell(f, cxf, cyf);
      const V3 E = midpoint(Pa, Pb);
      double le, tx, ty;
      PlainGeometry::edge(Pa, Pb, V3{cxf, cyf, 0.}, le, tx, ty);
      const double nx = ty, ny = -tx;
      double F[3];
      double lw = 1.0;  // the CFL candidate is not taken here (unused)
      if (wall) {
        // the cell average; SWE_OPT_EXACT_BALANCE: the inside edge depth
        double hw;
        if (M.eb) {
          hw = slot_value(mf, cxf, cyf, E).w - E.z;
        } else {
          const int g = f < kTileCells ? (int)c0 + f : xl[f - kTileCells];
          hw = S.w[S.at(g)] - M.bc[g];
        }
        elem_flux(nx, ny, hw, 0., 0., F[0], F[1], F[2]);
      } else {
        const Slot L = slot_value(mf, cxf, cyf, E);
        double cxt, cyt;
        const Muscl mt = cell(tr, cxt, cyt);
        const Slot R = slot_value(mt, cxt, cyt, E);
        if (FLUX == 0) flux_hll<WS>(nx, ny, E.z, L, R, 1.0, A.cor, lw, F, M.eb != 0, all);
        else flux_hllc<WS>(tx, ty, E.z, L, R, 1.0, A.cor, lw, F, M.eb != 0, all);
      }
      sF0[j] = FAR && LEN && !all ? F[0] * le : F[0];
      if (all) {
        sF1[j] = F[1];
        sF2[j] = F[2];
      }
      if (store && j < h.ne0) {  // the edge's one owning evaluation: its et0 cell is ours
        const int e = P.evedge[tile * P.se + j];
        out_store<NT>(&W.f0[e], F[0]);
        out_store<NT>(&W.f1[e], F[1]);
        out_store<NT>(&W.f2[e], F[2]);
      }
    }
    __syncthreads();
    q.mu = lmuscl(mine ? tid : 0);  // read before the draining steps take w0's place
  }

  // ---- draining time steps of every local cell (k_drain's operations)
  auto drain_dt = [&](double hh, uint32_t slots, uint32_t fl, double area) -> double {
    if (!is_wet(hh)) return 0.;
    double sum = 0.;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int s = local3(slots, k);
      const double fe = sF0[s];
      double out = sgn_pos(fl, k) ? fe : -fe;
      if (LEN && (!FAR || s < h.na)) {  // FAR: the outer edges' slots hold the product
        const uint32_t en = evl[s].nodes;
        out = out * edge_len(lnode(local3(en, 0)), lnode(local3(en, 1)));
      }
      sum += dmax(0., out);
    }
    return sum > kTol ? area * hh / sum : INFINITY;
  };
  q.fl = tc.flags;
  q.wi = w;
#pragma unroll
  for (int k = 0; k < 3; ++k) q.p[k] = mine ? lnode(local3(tc.nodes, k)) : V3{0., 0., 0.};
  const double bc = centroid(q.p[0], q.p[1], q.p[2]).z;
  if (mine) {
    // the centroid bathymetry and area from the vertices, as the setup
    // kernel computes M.bc and M.area (the same functions: the same bits)
    const double d = drain_dt(w - bc, tc.slots, tc.flags, tri_area(q.p[0], q.p[1], q.p[2]));
    sD[tid] = d;
    q.dti = d;
    if (store) out_store<NT>(&W.dtd[i], d);
  }
  if (ringed) sD[kTileCells + tid] = drain_dt(hr, rc.slots, rc.flags, arear);
  __syncthreads();

  // ---- update of the tile's cells (k_update's operations; the fluxes and
  // neighbour draining steps are read from LDS edge by edge)
  if (!mine) return;
  const double dt = M.cinst ? 0. : stage_dt(A);
  if (A.dts_log && tile == 0 && tid == 0) A.dts_log[0] = dt;
  double dts = A.coef * dt;
  if (M.cinst) {  // ensembles: the member's own step size (k_update's rule)
    const int inst = M.cinst[i];
    if (!M.bactive[inst]) {
      // finished member, or a cell of a tile that straddles the edge of the
      // active window: the stage leaves its state unchanged
      const int64_t o = O.at(i);
      O.w[o] = comb ? w0 : w;
      O.u[o] = comb ? u0 : u;
      O.v[o] = comb ? v0 : v;
      return;
    }
    dts = A.coef * member_dt(M, A, inst);
  }
  double R0, R1, R2;
  rhs_compute_by<PlainGeometry>(
      q,
      [&](int k, double& F0, double& F1, double& F2, double& dtik) {
        const int s = local3(tc.slots, k), nb = local3(tc.nbs, k);
        F0 = sF0[s];
        F1 = sF1[s];
        F2 = sF2[s];
        dtik = nb >= (int)kLocalMax ? INFINITY : sD[nb];
      },
      [&](int k, V3& Pa, V3& Pb) {
        Pa = lnode((int)((tc.nodes >> (kLocalBits * (uint32_t)ep0_local(tc.flags, k))) & kLocalMask));
        Pb = lnode((int)((tc.nodes >> (kLocalBits * (uint32_t)ep1_local(tc.flags, k))) & kLocalMask));
      },
      dts, A.cor, A.fric, M.eb != 0, R0, R1, R2);
  const double hh = w - bc;
  const double Uc0 = hh, Uc1 = hh * u, Uc2 = hh * v;
  double r0, r1, r2;
  if (comb) {
    const double h0 = w0 - bc;
    const double Ua0 = h0, Ua1 = h0 * u0, Ua2 = h0 * v0;
    const bool cvx = M.eb && A.a0 + A.a1 == 1.;
    r0 = stage_combine(cvx, A.a0, A.a1, Ua0, Uc0, R0);
    r1 = stage_combine(cvx, A.a0, A.a1, Ua1, Uc1, R1);
    r2 = stage_combine(cvx, A.a0, A.a1, Ua2, Uc2, R2);
  } else {
    r0 = Uc0 + R0;
    r1 = Uc1 + R1;
    r2 = Uc2 + R2;
  }
  double ow, ou, ov;
  cons_assign(bc, r0, r1, r2, ow, ou, ov);
  out_store<NT>(&O.w[O.at(i)], ow);
  out_store<NT>(&O.u[O.at(i)], ou);
  out_store<NT>(&O.v[O.at(i)], ov);
}

bool fused_fits(const DevTiles& P) {
  return stage_lds(P, false, true, true) <= kTileMaxLds && stage_lds(P, true, false, true) <= kTileMaxLds;
}

hipError_t launch_fused(const DevMesh& M, const DevTiles& P, const DevState& S, const DevState& U0,
                        const DevOut& O, const DevWork& W, const StageArgs& A, int flux, int ws, int opts,
                        hipStream_t st, bool store, bool from_fluxes) {
  // the tiles that hold cells of the visited window [c0, c1): the whole mesh,
  // or an ensemble's running members (cells of finished members in the
  // first and last tile are copied unchanged, as every finished member's)
  if (!M.cinst && (M.c0 != 0 || M.c1 != M.T)) return hipErrorInvalidValue;
  const int64_t t0 = M.c0 / kTileCells, t1 = (M.c1 + kTileCells - 1) / kTileCells;
  if (t1 <= t0) return hipGetLastError();
  const dim3 g = grid_for_bs(t1 - t0, 1), b(kTileCells);
  const bool wide = !M.nt && t1 - t0 <= kWideTiles;
  const bool len = (opts & kOptDrainLength) != 0;
  const int sto = store ? 1 : 0;
  const bool far = !from_fluxes && stage_far(P, len, t1 - t0);
  const unsigned lds = (unsigned)stage_lds(P, from_fluxes, far, len);
  if (from_fluxes) {  // the flux scheme does not enter: one instance per drain / store variant
    if (len && M.nt) hipLaunchKernelGGL((k_fused<0, 0, true, true, true, false, kTileCells>), g, b, lds, st, M, P, S, U0, O, W, A, t0, t1, sto);
    else if (len) hipLaunchKernelGGL((k_fused<0, 0, true, false, true, false, kTileCells>), g, b, lds, st, M, P, S, U0, O, W, A, t0, t1, sto);
    else if (M.nt) hipLaunchKernelGGL((k_fused<0, 0, false, true, true, false, kTileCells>), g, b, lds, st, M, P, S, U0, O, W, A, t0, t1, sto);
    else hipLaunchKernelGGL((k_fused<0, 0, false, false, true, false, kTileCells>), g, b, lds, st, M, P, S, U0, O, W, A, t0, t1, sto);
    return hipGetLastError();
  }
#define SWE_FUSED_TH(F, Wv, LEN, NT, FAR, TH)                                                                         \
  hipLaunchKernelGGL((k_fused<F, Wv, LEN, NT, false, FAR, TH>), g, dim3(TH), lds, st, M, P, S, U0, O, W, A, t0, t1, sto)
#define SWE_FUSED(F, Wv)                                                                                             \
  if (flux == F && ws == Wv) {                                                                                       \
    if (far && len && M.nt) SWE_FUSED_TH(F, Wv, true, true, true, kTileCells);                                       \
    else if (far && M.nt) SWE_FUSED_TH(F, Wv, false, true, true, kTileCells);                                        \
    else if (far && len) SWE_FUSED_TH(F, Wv, true, false, true, kTileCells);                                         \
    else if (far) SWE_FUSED_TH(F, Wv, false, false, true, kTileCells);                                               \
    else if (len && M.nt) SWE_FUSED_TH(F, Wv, true, true, false, kTileCells);                                        \
    else if (M.nt) SWE_FUSED_TH(F, Wv, false, true, false, kTileCells);                                              \
    else if (len && wide) SWE_FUSED_TH(F, Wv, true, false, false, kWideThreads);                                     \
    else if (wide) SWE_FUSED_TH(F, Wv, false, false, false, kWideThreads);                                           \
    else if (len) SWE_FUSED_TH(F, Wv, true, false, false, kTileCells);                                               \
    else SWE_FUSED_TH(F, Wv, false, false, false, kTileCells);                                                       \
    return hipGetLastError();                                                                                        \
  }
  SWE_FUSED(0, 0) SWE_FUSED(0, 1) SWE_FUSED(0, 2) SWE_FUSED(1, 0) SWE_FUSED(1, 1) SWE_FUSED(1, 2)
#undef SWE_FUSED_TH
#undef SWE_FUSED
  return hipErrorInvalidValue;
}

}  // namespace swe
