// Whole Runge-Kutta stage in one kernel (included by fvs_api.hip inside its
// anonymous namespace, after fused.hpp).
//
// A workgroup owns a block of consecutive cells.  It stages, in LDS, the state
// and centre of every cell its gradients read, forms the gradients (and limiter
// values) of its own cells and of the cells across its faces, the fluxes of its
// faces, and the gather and update of its own cells.  Gradients and limiter
// values never travel through HBM: per cell and stage that is 128 B of gradient
// traffic and two more reads of the state less than the two-kernel path, for 25%
// more gradients (those of the cells across the faces, at 128 cells a block).
//
// The arithmetic and the order of every sum are those of k_grad_lsqh and
// k_flux_update (the same inlined functions), so the states are theirs bit for
// bit.

// Block shape: at most BS cells and NT threads; C1 bounds the local cells with a
// gradient (own cells, then the cells across the block's faces: ring 1), and
// also the further cells of their stencils (ring 2); F bounds the block's faces.
//
// LDS, in planes of 16 B per local cell or face (lane-consecutive accesses are
// free of bank conflicts; as records of 32 and 64 B, conflicts were 62% of the
// LDS cycles): states W0 (rho, u), W1 (v, p) and centres X of the gradient
// cells, the same three planes of ring 2 a fixed distance behind, four gradient
// planes, and where they are needed limiter values P and wave speeds S.  A cell
// is addressed by its byte offset o alone: its planes lie at o, o + PS, o + 2 PS
// (immediate offsets of the LDS reads).  Ring 2 is dead once the gradients are
// formed, and the face fluxes F0, F1 take its place.  160 C1 + 8 C1 bytes: five
// blocks of 128 cells on a CU.
template <int BS_, int NT_, int C1_, int F_, int WAVES_>
struct StageShape {
  static constexpr int BS = BS_, NT = NT_, C1 = C1_, F = F_, WAVES = WAVES_;
  static constexpr int PS = 16 * C1, R2 = 3 * PS, FAR = 6 * PS;
  static constexpr int F0 = R2, F1 = R2 + 16 * F, G = 6 * PS, P = 10 * PS, S = P + 8 * C1, END = S + 8 * F;
  static constexpr int NSL = C1 / kSlice;  // stencil slices
  static_assert(32 * NT <= 4 * PS, "the node values fit where the gradients go");
  static_assert(C1 % kSlice == 0 && C1 <= NT && F <= NT && 32 * F <= 3 * PS && BS % kSlice == 0, "block shape");
};

// One block: cells [i0, i0 + n0), base = n0 rounded up to whole slices, ring-1
// cells at local indices base .. base + nr1 - 1, nh halo cells in all (ring 1,
// ring 2; those past the C1 that ring 2 holds are far: read from HBM)
// With node-based gradients nn nodes of up to 2 nkw cells each.  more: where the
// block's far cells start, or its nodes' words past the first kNodeRegs (a block
// with the one has none of the other).
struct StageBlock {
  int i0, n0, base, nr1, nh, nn, nkw, more;
};

constexpr int kCodeRegs = 8;  // code words a thread holds in registers
constexpr int kNodeRegs = 3;  // words of a node's cells

// Per-block lists at fixed strides, so that a block's first loads wait on no
// offset: halo cells id | periodic shift << 27 (-1 after the last); stencil
// codes, per slice of 64 gradient cells cw words of two byte offsets each;
// faces as byte offsets of their two gradient cells (R side: | periodic shift of
// its centre; 0xffff on a boundary; ~0 after the last) with 5 geometry values
// (planes nx,ny | xf,yf | area); boundary code (type | instance << 2) of a face.
// Green-Gauss gradients: four byte offsets per gradient cell in two words, of its
// face neighbours' states or of its nodes' values (16 n for the block's node n);
// nodes: the byte offsets of their cells two to a word, and the cells' weights.
// What a thread does not load at the start is packed instead, so that one node of
// many cells does not widen the lists of every block: a slice's code words past
// the first kCodeRegs, a block's far cells, its nodes' words (planes of nn) past
// the first kNodeRegs with their weights.
struct StageLists {
  const StageBlock *blk;
  const int *halo;
  const unsigned *code;
  const int *width;  // per slice: words used
  const int *mstart;  // where its packed ones start, in 64s
  const unsigned *face;
  const double *geo;
  const int *bcode;
  const short *lgat;
  int hs, cw, fs;  // strides: halo entries, code words per cell, faces
  const unsigned *gcode, *ncode;
  const double *nwt;
  int ns, nkw;  // strides: nodes, words of cells per node
  const unsigned *morecode, *morenode;
  const double *morewt;
  const int *far;
};

struct StageIn {
  int N, nb, gw;
  Phys P;
  double t;
  StageLists S;
  const double2 *cxy;
  const double *ginv;
  const double2 *gg0, *ggc;  // Green-Gauss: own coefficient (cell-based) and ngg per cell, planes
  int ngg;
  ShiftTable st;
  double p;
  int phisrc;  // without LIM: 0 limiter values 1, 1 read phi (frozen)
  double *phi;
  int lt;
  const double2 *loff;
  const double *vol;
  const int *ioff, *frz;
  int ninst;
  double *Ua, *Ub, *Facc, *dtl;
  NormOut norm;
  const int *blist;
  const unsigned *amask;
  const double *pinf_inst;
  // residual evaluation (mode M_RESID): where the residual and the summed wave
  // speeds go, in the caller's cell order (ref[device cell])
  double *rout, *wsout;
  const int *ref;
  // sweep direction: blocks in ascending or descending order.  Alternating
  // stages start where the last one ended, whose lists and states the 256 MB
  // memory-side cache still holds: 7% of a stage on 2,097,152 cells (now 125 us)
  int down;
  // phase timers: per block the clock cycles its launches spent until the gradients
  // were there, and in all
  unsigned long long *clk;
};

// The shapes in use.  128-cell blocks: five wavefronts per SIMD and five blocks on
// a CU (7% per step faster than four on 2,097,152 cells; now 375 us).  256-cell blocks:
// two blocks of 8 wavefronts on a CU, for meshes whose 128-cell blocks exceed the shape
// (the rule is with setup_stage).
using StageSmall = StageShape<128, 256, 192, 256, 5>;
using StageLarge = StageShape<256, 512, 384, 512, 4>;

// Block lb of a whole stage.  LIM: the limiter is evaluated (and written for the
// own cells).  PMODE: the LSQ weights as in lsq_term, or a Green-Gauss gradient,
// cell-based (kGGCB) or node-based (kGGNB).  With cons (SSP-RK3 and the two-register form), Win holds
// conservative states, converted once as they are staged, and the new stage
// state goes to Ub (a buffer other than Win; no primitive state is written).
// With mode M_RESID the block ends in the residual instead of an update.
// Green-Gauss stages in this kernel: 320,000 cells, cell-based, 45 -> 24 us per
// stage (gradient kernel and fused fluxes before); 181,202 cells, node-based and
// limited, 43 -> 29 (node values, gradient and fluxes before).  They take
// it on every size that was measured (3,200 to 819,200 cells).
constexpr int kGGCB = 4, kGGNB = 5;

// TIMED: the phase timers are on (a run-time switch cost 2,097,152 cells 1.3%).
template <class SH, int LIM, int PMODE, bool TIMED = false>
__device__ __forceinline__ void stage_block(const StageIn &a, int lb, const Upd &A, const double *__restrict__ Win,
                                            double *__restrict__ Wout, int cons) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int NT = SH::NT, PS = SH::PS;
  constexpr bool GG = PMODE >= kGGCB;
  auto at = [&](int o) __attribute__((always_inline)) -> double2 & { return *reinterpret_cast<double2 *>(smem + o); };
  auto at1 = [&](int o) __attribute__((always_inline)) -> double & { return *reinterpret_cast<double *>(smem + o); };
  const StageLists &S = a.S;
  const StageBlock d = S.blk[lb];
  const int tid = threadIdx.x, N = a.N;
  unsigned long long t0 = 0, t1 = 0;
  if (TIMED) t0 = __builtin_readcyclecounter();
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  // face record and geometry, stencil codes
  const int *hl = S.halo + long(lb) * S.hs;
  const unsigned rec = tid < S.fs ? S.face[long(lb) * S.fs + tid] : ~0u;
  const unsigned *lc = S.code + (long(lb) * SH::NSL + wv) * S.cw * kSlice + (tid & 63);
  unsigned cr[kCodeRegs];
  if (wv < SH::NSL) {
#pragma unroll
    for (int k = 0; k < kCodeRegs; ++k) cr[k] = (k < S.cw) ? lc[k * kSlice] : 0u;
  }
  const int nw = wv < SH::NSL ? S.width[lb * SH::NSL + wv] : 0;
  // the local cells: own and ring 1 at their index, ring 2 behind
  constexpr int R = (2 * SH::C1 + NT - 1) / NT;
  int jd[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int h = tid + r * NT - d.base;
    jd[r] = h < 0 ? (h + d.base < d.n0 ? d.i0 + h + d.base : -1) : (h < d.nh && h < d.nr1 + SH::C1 ? hl[h] : -1);
  }
  const bool mine = tid < d.n0, act = mine || (tid >= d.base && tid < d.base + d.nr1);
  const int id = jd[0] & 0x07ffffff;
  // Green-Gauss: the cell's four offsets, its coefficients and volume; the first
  // cells of the thread's node
  unsigned gc[2] = {0u, 0u}, nc[kNodeRegs];
  double2 gk[4], gown = make_double2(0.0, 0.0);
  double nw8[2 * kNodeRegs], GV = 1.0;
  const unsigned *ncl = S.ncode + long(lb) * S.nkw * S.ns + tid;
  const double *nwl = S.nwt + 2 * long(lb) * S.nkw * S.ns + tid;
  if (GG && act) {
    gc[0] = S.gcode[2 * long(lb) * SH::C1 + tid];
    gc[1] = S.gcode[(2 * long(lb) + 1) * SH::C1 + tid];
  }
  if (PMODE == kGGNB) {
#pragma unroll
    for (int k = 0; k < kNodeRegs; ++k) {
      const bool on = tid < d.nn && k < d.nkw;
      nc[k] = on ? ncl[k * S.ns] : 0u;
      nw8[2 * k] = on ? nwl[2 * k * S.ns] : 0.0;
      nw8[2 * k + 1] = on ? nwl[(2 * k + 1) * S.ns] : 0.0;
    }
  }
  double g[8];
  g[7] = 0.0;
  if (rec != ~0u) {
    const double *b = S.geo + 5 * (long(lb) * S.fs);
    const double2 n = reinterpret_cast<const double2 *>(b)[tid], x = reinterpret_cast<const double2 *>(b)[S.fs + tid];
    g[0] = n.x; g[1] = n.y;
    g[5] = x.x; g[6] = x.y;
    g[2] = b[4 * S.fs + tid];
  }
  // limiter: the cell's face offsets (zero past its last face, where they give
  // the candidate 1) and volume, or its frozen value
  const bool phi_one = !LIM && !a.phisrc;
  double2 fo[4];
  double V = 1.0, ph = 1.0;
  bool keep = !LIM;
  double Gi[3] = {0.0, 0.0, 0.0};
  double u[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (jd[r] == -1) continue;
    const int j = jd[r] & 0x07ffffff, sh = unsigned(jd[r]) >> 27, q = tid + r * NT;
    double2 xy = a.cxy[j];
    double w[4];
    ld4(Win, j, w);
    if (r == 0) {
      if (act && GG) {
        if (PMODE == kGGCB) gown = a.gg0[j];
#pragma unroll
        for (int k = 0; k < 4; ++k) gk[k] = (k < a.ngg) ? a.ggc[long(k) * N + j] : make_double2(0.0, 0.0);
        GV = a.vol[j];
      } else if (act) {
        Gi[0] = a.ginv[j];
        Gi[1] = a.ginv[N + j];
        Gi[2] = a.ginv[2 * long(N) + j];
      }
      for (int v = 0; v < 4; ++v) u[v] = w[v];
    }
    if (sh) {
      xy.x = xy.x + a.st.sx[sh - 1];
      xy.y = xy.y + a.st.sy[sh - 1];
    }
    const int r2 = q - d.base - d.nr1, o = r2 < 0 ? 16 * q : SH::R2 + 16 * r2;
    at(o + 2 * PS) = xy;
    make_prim(cons, A.gamma, w);
    at(o) = make_double2(w[0], w[1]);
    at(o + PS) = make_double2(w[2], w[3]);
  }
  if (!phi_one && act) {
    if (LIM) {
      V = a.vol[id];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        fo[k] = (k < a.gw) ? a.loff[long(k) * N + id] : make_double2(0.0, 0.0);
      if (a.ioff) keep = a.frz[instance_of(a.ioff, a.ninst, id)] != 0;
    }
    if (keep) ph = a.phi[id];
  }
  __syncthreads();
  if (PMODE == kGGNB) {
    // node values where the gradients go afterwards: one node per thread
    if (tid < d.nn) {
      double f[4] = {0.0, 0.0, 0.0, 0.0};
      auto add = [&](unsigned o, double c) __attribute__((always_inline)) {
        const double2 qa = at(o), qb = at(o + PS);
        const double q[4] = {qa.x, qa.y, qb.x, qb.y};
        node_term(c, q, f);
      };
#pragma unroll
      for (int k = 0; k < kNodeRegs; ++k)
        if (k < d.nkw) {
          add(nc[k] & 0xffffu, nw8[2 * k]);
          add(nc[k] >> 16, nw8[2 * k + 1]);
        }
      for (int k = kNodeRegs; k < d.nkw; ++k) {
        const long q = d.more + long(k - kNodeRegs) * d.nn;
        const unsigned w = S.morenode[q + tid];
        add(w & 0xffffu, S.morewt[2 * q + tid]);
        add(w >> 16, S.morewt[2 * q + d.nn + tid]);
      }
      at(SH::G + 16 * tid) = make_double2(f[0], f[1]);
      at(SH::G + 16 * NT + 16 * tid) = make_double2(f[2], f[3]);
    }
    __syncthreads();
  }
  double gx[4] = {0.0, 0.0, 0.0, 0.0}, gy[4] = {0.0, 0.0, 0.0, 0.0};
  if (act) {
    const int o0 = 16 * tid;
    const double2 ci = at(o0 + 2 * PS), wa = at(o0), wb = at(o0 + PS);
    const double w[4] = {wa.x, wa.y, wb.x, wb.y};
    double sx[4] = {0, 0, 0, 0}, sy[4] = {0, 0, 0, 0}, mn[4], mx[4];
    for (int v = 0; v < 4; ++v) mn[v] = mx[v] = w[v];
    auto term = [&](unsigned o) __attribute__((always_inline)) {
      const double2 cj = at(o + 2 * PS), qa = at(o), qb = at(o + PS);
      const double q[4] = {qa.x, qa.y, qb.x, qb.y};
      if (GG) stencil_bounds(q, mn, mx);
      else lsq_term<LIM, PMODE>(cj.x, cj.y, ci, q, w, a.p, sx, sy, mn, mx);
    };
    // the code words past those in registers (the offset is loaded only here: with
    // the widths at the start it cost every small stage 0.2 us)
    const auto packed = [&]() __attribute__((always_inline)) {
      return S.morecode + (long(S.mstart[lb * SH::NSL + wv]) - kCodeRegs) * kSlice + (tid & 63);
    };
    if (GG && !LIM) {
      // no stencil beyond the faces or nodes
    } else if (GG || d.nh <= d.nr1 + SH::C1) {
#pragma unroll
      for (int k = 0; k < kCodeRegs; ++k)
        if (k < nw) {
          term(cr[k] & 0xffffu);
          term(cr[k] >> 16);
        }
      if (nw > kCodeRegs) {
        const unsigned *lm = packed();
        for (int k = kCodeRegs; k < nw; ++k) {
          const unsigned c = lm[k * kSlice];
          term(c & 0xffffu);
          term(c >> 16);
        }
      }
    } else {
      // ring 2 does not fit: the codes past it are far cells, from HBM
      const unsigned *lm = packed();
      for (int k = 0; k < 2 * nw; ++k) {
        const int word = k >> 1;
        const unsigned o = ((word < kCodeRegs ? lc : lm)[word * kSlice] >> (16 * (k & 1))) & 0xffffu;
        if (o < unsigned(SH::FAR)) {
          term(o);
          continue;
        }
        const int e = S.far[d.more + int((o - SH::FAR) >> 4)], j = e & 0x07ffffff, sh = unsigned(e) >> 27;
        double2 xy = a.cxy[j];
        double q[4];
        ld4(Win, j, q);
        if (sh) {
          xy.x = xy.x + a.st.sx[sh - 1];
          xy.y = xy.y + a.st.sy[sh - 1];
        }
        make_prim(cons, A.gamma, q);
        lsq_term<LIM, PMODE>(xy.x, xy.y, ci, q, w, a.p, sx, sy, mn, mx);
      }
    }
    if (GG) {
      constexpr int B = PMODE == kGGNB ? SH::G : 0, BP = PMODE == kGGNB ? 16 * NT : PS;
      if (PMODE == kGGCB) gg_own(gown, w, gx, gy);
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (k < a.ngg) {
          const int o = B + int((gc[k >> 1] >> (16 * (k & 1))) & 0xffffu);
          const double2 qa = at(o), qb = at(o + BP);
          const double q[4] = {qa.x, qa.y, qb.x, qb.y};
          gg_term(gk[k], q, gx, gy);
        }
      gg_divide(GV, gx, gy);
    } else {
      lsq_apply_ginv(Gi[0], Gi[1], Gi[2], sx, sy, gx, gy);
    }
    if (LIM && !keep) {
      ph = cell_limiter_v(a.lt, a.gw, fo, V, w, mn, mx, gx, gy);
      if (mine) a.phi[id] = ph;
    }
    if (!phi_one) at1(SH::P + 8 * tid) = ph;
  }
  if (PMODE == kGGNB) __syncthreads();  // the node values have been read
  if (act) {
    const int o0 = SH::G + 16 * tid;
    at(o0) = make_double2(gx[0], gx[1]);
    at(o0 + PS) = make_double2(gx[2], gx[3]);
    at(o0 + 2 * PS) = make_double2(gy[0], gy[1]);
    at(o0 + 3 * PS) = make_double2(gy[2], gy[3]);
  }
  __syncthreads();
  if (TIMED) t1 = __builtin_readcyclecounter();
  const bool resid = A.mode == M_RESID, ws = resid || (A.steady && A.first);
  auto side = [&](unsigned o, double w[4], double gr[8], double &ph, double2 &c) __attribute__((always_inline)) {
    const double2 wa = at(o), wb = at(o + PS);
    c = at(o + 2 * PS);
    w[0] = wa.x; w[1] = wa.y; w[2] = wb.x; w[3] = wb.y;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const double2 q = at(SH::G + k * PS + o);
      gr[2 * k] = q.x;
      gr[2 * k + 1] = q.y;
    }
    ph = phi_one ? 1.0 : at1(SH::P + (o >> 1));
  };
  if (rec != ~0u) {
    double fa[4], wsa, wL[4], gL[8], phL;
    double2 c;
    side(rec & 0xffffu, wL, gL, phL, c);
    const double xf = g[5], yf = g[6];
    g[3] = xf - c.x;
    g[4] = yf - c.y;
    const unsigned rr = rec >> 16;
    if (rr != 0xffffu) {
      double wR[4], gR[8], phR;
      side(rr & 0xfff0u, wR, gR, phR, c);
      const int sh = int(rr & 15u);
      if (sh) {
        c.x = c.x + a.st.sx[sh - 1];
        c.y = c.y + a.st.sy[sh - 1];
      }
      g[5] = xf - c.x;
      g[6] = yf - c.y;
      interior_flux_v(a.P, g, wL, wR, gL, gR, phL, phR, fa, wsa);
    } else {
      const int code = S.bcode[long(lb) * S.fs + tid];
      boundary_flux_v(a.P, a.t, code & 3, g, wL, gL, phL, fa, wsa,
                      a.pinf_inst ? a.pinf_inst + 4 * (code >> 2) : a.P.pinf);
    }
    at(SH::F0 + 16 * tid) = make_double2(fa[0], fa[1]);
    at(SH::F1 + 16 * tid) = make_double2(fa[2], fa[3]);
    if (ws) at1(SH::S + 8 * tid) = wsa;
  }
  UpdIn in;
  if (mine && resid) {
#pragma unroll
    for (int k = 0; k < 4; ++k) in.sv[k] = (k < a.gw) ? S.lgat[long(k) * N + id] : 0;
    in.V = a.vol[id];
  } else if (mine) {
    block_update_load(N, id, a.gw, A, S.lgat, a.vol, a.Ua, a.Ub, a.Facc, a.dtl, in, cons != 0);
    if (cons) {  // the stage input (the step-start state too on the first stage)
      for (int v = 0; v < 4; ++v) in.x[v] = u[v];
      if (A.first)
        for (int v = 0; v < 4; ++v) in.u0[v] = u[v];
    }
  }
  __syncthreads();
  auto flux = [&](int f, double fa[4]) __attribute__((always_inline)) {
    const double2 q0 = at(SH::F0 + 16 * f), q1 = at(SH::F1 + 16 * f);
    fa[0] = q0.x; fa[1] = q0.y; fa[2] = q1.x; fa[3] = q1.y;
  };
  auto speed = [&](int f) __attribute__((always_inline)) { return at1(SH::S + 8 * f); };
  if (resid) {
    if (mine) {
      double acc[4], wacc;
      cell_gather(in.sv, flux, speed, true, acc, wacc);
      const double iV = recip(in.V);  // as in the stage update
      for (int v = 0; v < 4; ++v) acc[v] = -acc[v] * iV;
      const int c = a.ref[id];
      st4(a.rout, c, acc);
      a.wsout[c] = wacc;
    }
    return;
  }
  if (tid < d.base)
    cell_update(N, d.i0 + tid, mine, A, in, flux, speed, a.Ua, a.Ub, a.Facc, Wout, a.dtl, a.norm, a.amask);
  if (TIMED && tid == 0) {
    a.clk[2 * lb] += t1 - t0;
    a.clk[2 * lb + 1] += __builtin_readcyclecounter() - t0;
  }
}

// four wavefronts per SIMD with the limiter (its registers spill at five, 11%
// slower on 522,242 cells) and with the weights that need a division or pow,
// SH::WAVES without them
template <class SH, int LIM, int PMODE, bool TIMED>
__global__ __launch_bounds__(SH::NT, LIM || PMODE == 2 || PMODE == 3 ? 4 : SH::WAVES) void k_stage(StageIn a, Upd A,
                                                                       const double *__restrict__ Win,
                                                                       double *__restrict__ Wout, int cons) {
  const int nbl = a.nb < 0 ? -a.nb : a.nb;  // with a block list, its length
  int lb = a.blist ? int(blockIdx.x) : xcd_block(a.nb);
  if (lb >= nbl) return;  // the whole workgroup leaves before any barrier
  if (a.down) lb = nbl - 1 - lb;
  if (a.blist) lb = a.blist[lb];
  stage_block<SH, LIM, PMODE, TIMED>(a, lb, A, Win, Wout, cons);
}

// ---------------------------------------------------------------------------
// Persistent whole-step kernel: one cooperative launch runs nsteps time steps
// of the whole-stage block body over the launch-block list (the ragged batch's
// active blocks, or every block), with a grid-wide barrier after each stage
// and the step's residual norms reduced in the same launch.
// ---------------------------------------------------------------------------

// Grid-wide barrier of a co-resident launch: thread 0 of each workgroup
// counts itself in bar[0]; the last one resets the count and advances the
// generation bar[kBarGen] (a line of its own); the others poll the generation.
// What a workgroup wrote is released once before it arrives and the others'
// acquired once after the wait: a poll that acquires (or a full fence on either
// side) invalidates caches that workgroups still at work are reading.  With such
// polls the barrier cost 10 to 100 us and grew with the workgroups; us per step
// before / now: 8,192 cells 36 / 27, 34,848 cells 117 / 56, 320,000 cells 410 /
// 172, 65,536 limited steady cells 464 / 148.  Each wait is bounded
// (spin polls, or as soon as another workgroup has given up and set *err):
// a workgroup that gives up records it in *err and returns false, so every
// wave of the launch ends.
constexpr int kBarGen = 32, kBarWords = 2 * kBarGen;
__device__ __forceinline__ bool grid_barrier(unsigned *bar, unsigned nwg, unsigned &gen, unsigned spin, int *err) {
  __shared__ int ok;
  __syncthreads();
  if (threadIdx.x == 0) {
    ok = 1;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    const unsigned arrived = atomicAdd(&bar[0], 1u);
    if (arrived == nwg - 1) {
      atomicExch(&bar[0], 0u);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "agent");
      atomicAdd(&bar[kBarGen], 1u);
    } else {
      unsigned n = 0;
      while (__hip_atomic_load(&bar[kBarGen], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gen) {
        __builtin_amdgcn_s_sleep(2);
        if (++n >= spin || __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) {
          atomicExch(err, 1);
          ok = 0;
          break;
        }
      }
    }
    gen = gen + 1;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
  return ok != 0;
}

struct PersistCtl {
  Upd A[4];                 // the stages of one step
  int nst, nsteps, nlaunch;  // stages per step, steps, launch blocks
  double *W0, *W1;          // primitive states: stage k of the launch reads W0 when k is even
  double *dn;               // whole-mesh norms, one row per step (NULL: none)
  int ng;                   // 64-cell slices
  double *dinst;            // per-instance norms (NULL: the last step's are only kept)
  InstNorms inst;           // no instances on a single mesh
  int *ctr;                 // output row of the first step; advanced by nsteps at the end
  unsigned *bar;
  int *err;
  unsigned spin;
};

template <class SH, int LIM, int PMODE>
__global__ __launch_bounds__(SH::NT, SH::NT > 256 ? 4 : 3) void k_steps_persistent(StageIn a, PersistCtl c) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  double *lds = reinterpret_cast<double *>(smem);
  unsigned gen = 0;
  if (threadIdx.x == 0) gen = __hip_atomic_load(&c.bar[kBarGen], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int row0 = c.ctr[0];  // block 0 writes the counter only after the last barrier
  int par = 0;
  bool ok = true;
  for (int s = 0; s < c.nsteps && ok; ++s) {
    for (int k = 0; k < c.nst && ok; ++k) {
      const Upd A = c.A[k];
      const double *Win = par ? c.W1 : c.W0;
      double *Wout = par ? c.W0 : c.W1;
      for (int q = blockIdx.x; q < c.nlaunch; q += gridDim.x) {
        const int lb = a.blist ? a.blist[q] : q;
        stage_block<SH, LIM, PMODE>(a, lb, A, Win, Wout, 0);
        __syncthreads();  // the next block's staging overwrites this one's LDS
      }
      ok = grid_barrier(c.bar, gridDim.x, gen, c.spin, c.err);
      par ^= 1;
    }
    if (!ok) break;
    // this step's norms; the partials and increments they read are next
    // written by the last stage of the next step, two or more barriers later
    const long row = long(row0) + s;
    if (c.dn && blockIdx.x == 0) norm_row<SH::NT>(c.ng, a.N, a.norm.part, c.dn + 4 * row, lds);
    if (c.dinst || s == c.nsteps - 1)
      for (int k = blockIdx.x; k < c.inst.ninst; k += gridDim.x)
        inst_norm_row(c.inst, k, a.norm.part, a.norm.d2, s == c.nsteps - 1,
                      c.dinst ? c.dinst + 4 * (row * c.inst.ninst + k) : nullptr, lds);
  }
  if (ok) ok = grid_barrier(c.bar, gridDim.x, gen, c.spin, c.err);
  if (ok && blockIdx.x == 0 && threadIdx.x == 0) c.ctr[0] = row0 + c.nsteps;
}

// the blocks' clocks, added up and set to zero
__global__ __launch_bounds__(256) void k_phase_clocks(int nb, unsigned long long *__restrict__ clk,
                                                      double *__restrict__ out) {
  __shared__ double red[2][256];
  const int t = threadIdx.x;
  double s[2] = {0.0, 0.0};
  for (int b = t; b < nb; b += 256)
    for (int k = 0; k < 2; ++k) {
      s[k] += double(clk[2 * b + k]);
      clk[2 * b + k] = 0;
    }
  for (int k = 0; k < 2; ++k) red[k][t] = s[k];
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (t < h)
      for (int k = 0; k < 2; ++k) red[k][t] += red[k][t + h];
    __syncthreads();
  }
  if (t < 2) out[t] = red[t][0];
}

__global__ void k_barrier_reset(unsigned *bar, int *err) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    bar[0] = 0u;
    err[0] = 0;
  }
}
