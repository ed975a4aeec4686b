// Host side of the whole-stage kernel: its block lists (included by fvs_api.hip
// after the context).

// the mesh as the block lists read it (device cell order)
struct StageMesh {
  const std::vector<int> &gat;       // gw x N signed face slots
  const std::vector<int2> &fic;      // interior faces' cells
  const std::vector<double> &fig;    // and geometry, 8 per face
  const std::vector<int> &fbc, &fbt;  // boundary faces
  const std::vector<double> &fbg;
  const std::vector<int> &off, &wid;  // stencils in 64-cell slices
  const std::vector<unsigned> &code;  // id | periodic shift << 27
  // Green-Gauss gradients: ngg face neighbours (planes) or nodes per cell; the
  // nodes' cells and weights in 64-node slices
  const std::vector<int> *fnb = nullptr, *cnode = nullptr;
  int ngg = 0;
  const std::vector<int> *noff = nullptr, *nwid = nullptr, *ncell = nullptr;
  const std::vector<double> *ncoef = nullptr;
};

// the blocks cut from one contiguous part of the cells
template <class SH>
struct StageCut {
  const fvs_ctx &C;
  const StageMesh &M;
  const int cw;       // code words per cell at a fixed stride
  short *const lgat;  // gw x N signed 1-based local faces
  std::vector<StageBlock> blk;
  std::vector<unsigned> halo, face, code, morecode, gcode;
  std::vector<int> slot, nf;
  std::vector<int2> width;
  std::vector<unsigned short> ncode;  // per block nn x 2 nkw
  std::vector<double> nwt;
  bool shift_ok = true;  // every periodic shift of a face is in the table

  // byte offset of the local cell with index q, of which the first n1 have gradients
  static int offset(int q, int n1) {
    if (q < n1) return 16 * q;
    const int r = q - n1;
    return r < SH::C1 ? SH::R2 + 16 * r : SH::FAR + 16 * (r - SH::C1);
  }

  // cells [i0, i1) as one block; false (nothing added) when it does not fit.
  // Ring 2 may spill to far cells only where the block cannot be cut.
  bool block(int i0, int i1) {
    const int N = C.N, Fi = C.Fi, gw = C.GW;
    loc.clear();
    for (int i = i0; i < i1; ++i)
      for (int k = 0; k < gw; ++k)
        if (const int sg = M.gat[size_t(k) * N + i]) loc.push_back((sg > 0 ? sg : -sg) - 1);
    std::sort(loc.begin(), loc.end());
    loc.erase(std::unique(loc.begin(), loc.end()), loc.end());
    if (int(loc.size()) > SH::F) return false;
    r1.clear();
    for (int f : loc) {
      if (f >= Fi) continue;
      for (int c : {M.fic[f].x, M.fic[f].y})
        if (c < i0 || c >= i1) r1.push_back(c);
    }
    std::sort(r1.begin(), r1.end());
    r1.erase(std::unique(r1.begin(), r1.end()), r1.end());
    const int base = nblk(i1 - i0, kSlice) * kSlice, n1 = base + int(r1.size());
    if (n1 > SH::C1) return false;
    map.clear();
    bool fresh;
    for (int i = i0; i < i1; ++i) map.at(unsigned(i), fresh) = i - i0;
    hal.assign(r1.begin(), r1.end());
    for (size_t k = 0; k < r1.size(); ++k) map.at(unsigned(r1[k]), fresh) = base + int(k);
    const size_t c0 = code.size(), m0 = morecode.size();
    const auto drop_codes = [&] { code.resize(c0), morecode.resize(m0); };
    code.resize(c0 + size_t(SH::NSL) * cw * kSlice, 0u);
    int2 w2[SH::NSL];
    for (int s = 0; s < SH::NSL; ++s) {
      const auto cell = [&](int l) {
        const int q = s * kSlice + l;
        return q < base ? (i0 + q < i1 ? i0 + q : -1) : (q < n1 ? r1[q - base] : -1);
      };
      w2[s] = make_int2(0, int(morecode.size() / kSlice));
      for (int l = 0; l < kSlice && cw > 0; ++l)
        if (cell(l) >= 0) w2[s].x = std::max(w2[s].x, (M.wid[cell(l) / kSlice] + 1) / 2);
      morecode.resize(morecode.size() + size_t(std::max(0, w2[s].x - cw)) * kSlice, 0u);
      unsigned *const fixed = code.data() + c0 + size_t(s) * cw * kSlice;
      unsigned *const more = morecode.data() + size_t(w2[s].y) * kSlice;
      for (int l = 0; l < kSlice && cw > 0; ++l) {
        const int q = s * kSlice + l, i = cell(l);
        if (i < 0) continue;
        const int sg = i / kSlice, li = i % kSlice;
        for (int k = 0; k < 2 * w2[s].x; ++k) {
          int v = q;  // past the cell's own stencil: the cell itself (a zero term)
          if (k < M.wid[sg]) {
            const unsigned key = M.code[M.off[sg] + long(k) * kSlice + li];
            int &x = map.at(key, fresh);
            if (fresh) {
              x = base + int(hal.size());
              hal.push_back(key);
            }
            v = x;
          }
          unsigned *const word = k / 2 < cw ? fixed + k / 2 * kSlice : more + (k / 2 - cw) * kSlice;
          word[l] |= unsigned(offset(v, n1)) << (16 * (k & 1));
        }
      }
    }
    int nn = 0, nkw = 0;
    const size_t g0 = gcode.size();
    if (M.ngg > 0 && !green_gauss(i0, i1, base, n1, nn, nkw)) {
      drop_codes();
      gcode.resize(g0);
      return false;
    }
    const int nl = base + int(hal.size());
    if (nl - n1 > SH::C1 && (i1 - i0 > kSlice || offset(nl - 1, n1) > 0xfff0)) {
      drop_codes();
      return false;
    }
    blk.push_back({i0, i1 - i0, base, int(r1.size()), int(hal.size()), nn, nkw, 0});
    width.insert(width.end(), w2, w2 + SH::NSL);
    halo.insert(halo.end(), hal.begin(), hal.end());
    nf.push_back(int(loc.size()));
    slot.insert(slot.end(), loc.begin(), loc.end());
    for (int f : loc) {
      if (f >= Fi) {
        face.push_back(16 * unsigned(map.at(unsigned(M.fbc[f - Fi]), fresh)) | 0xffffu << 16);
        continue;
      }
      const unsigned l = unsigned(map.at(unsigned(M.fic[f].x), fresh)), r = unsigned(map.at(unsigned(M.fic[f].y), fresh));
      const double sx = C.mp.esx[C.mp.edge_intr[f]], sy = C.mp.esy[C.mp.edge_intr[f]];
      unsigned sh = 0;
      if (sx != 0.0 || sy != 0.0) {
        while (sh < 15 && !(C.shifts.sx[sh] == sx && C.shifts.sy[sh] == sy)) ++sh;
        shift_ok = shift_ok && sh < 15;
        ++sh;
      }
      face.push_back(16 * l | (16 * r | (sh & 15u)) << 16);
    }
    for (int i = i0; i < i1; ++i)
      for (int k = 0; k < gw; ++k)
        if (const int sg = M.gat[size_t(k) * N + i]) {
          const int li = int(std::lower_bound(loc.begin(), loc.end(), (sg > 0 ? sg : -sg) - 1) - loc.begin()) + 1;
          lgat[size_t(k) * N + i] = short(sg > 0 ? li : -li);
        }
    return true;
  }

  // offsets of the face neighbours or nodes of the block's gradient cells, and the
  // nodes' cells; false when there are too many nodes or local cells
  bool green_gauss(int i0, int i1, int base, int n1, int &nn, int &nkw) {
    const int N = C.N;
    const size_t g0 = gcode.size();
    gcode.resize(g0 + 2 * SH::C1, 0u);
    bool fresh;
    auto local = [&](int j) {
      int &x = map.at(unsigned(j), fresh);
      if (fresh) {
        x = base + int(hal.size());
        hal.push_back(unsigned(j));
      }
      return x;
    };
    nodes.clear();
    nmap.clear();
    for (int q = 0; q < n1; ++q) {
      const int i = q < base ? (i0 + q < i1 ? i0 + q : -1) : r1[q - base];
      if (i < 0) continue;
      for (int k = 0; k < M.ngg; ++k) {
        unsigned v;
        if (M.fnb) {
          v = unsigned(offset(local((*M.fnb)[size_t(k) * N + i]), n1));
        } else {
          const int n = (*M.cnode)[size_t(k) * N + i];
          int &x = nmap.at(unsigned(n), fresh);
          if (fresh) {
            x = int(nodes.size());
            nodes.push_back(n);
          }
          v = 16u * unsigned(x);
        }
        gcode[g0 + size_t(k / 2) * SH::C1 + q] |= v << (16 * (k & 1));
      }
    }
    if (int(nodes.size()) > SH::NT) return false;
    nn = int(nodes.size());
    cells.clear();
    for (int n : nodes) {
      const int sl = n / kSlice, at = (*M.noff)[sl] + n % kSlice;
      int w = (*M.nwid)[sl];
      while (w > 1 && (*M.ncoef)[size_t(at) + size_t(w - 1) * kSlice] == 0.0) --w;  // padding
      cells.push_back(make_int2(at, w));
      nkw = std::max(nkw, (w + 1) / 2);
    }
    const auto fits = [&] { return base + int(hal.size()) - n1 <= SH::C1; };  // every state in LDS
    for (int2 c : cells)
      for (int k = 0; k < c.y; ++k) {
        local((*M.ncell)[size_t(c.x) + size_t(k) * kSlice]);
        if (!fits()) return false;
      }
    if (!fits()) return false;
    for (int2 c : cells)
      for (int k = 0; k < 2 * nkw; ++k) {
        const size_t e = size_t(c.x) + size_t(k < c.y ? k : 0) * kSlice;
        ncode.push_back((unsigned short)(offset(local((*M.ncell)[e]), n1)));
        nwt.push_back(k < c.y ? (*M.ncoef)[e] : 0.0);
      }
    return true;
  }

  // cells [i0, i1) as one block or cut in two, down to one slice
  bool place(int i0, int i1) {
    if (block(i0, i1)) return true;
    if (i1 - i0 <= kSlice) return false;
    int h = kSlice;
    while (2 * h < i1 - i0) h *= 2;
    return place(i0, i0 + h) && place(i0 + h, i1);
  }
  bool place_range(long b) { return place(int(b) * SH::BS, std::min(C.N, int(b + 1) * SH::BS)); }

  StageCut(const fvs_ctx &c, const StageMesh &m, int w, short *g) : C(c), M(m), cw(w), lgat(g) {}

 private:
  LocalMap map, nmap;
  std::vector<int> loc, r1, nodes;
  std::vector<int2> cells;
  std::vector<unsigned> hal;
};

int code_words(const StageMesh &M) {
  if (M.wid.empty()) return 0;
  return std::min(kCodeRegs, std::max(1, (*std::max_element(M.wid.begin(), M.wid.end()) + 1) / 2));
}

// Blocks per range of SH::BS cells, from up to 256 ranges spread over the cells
// (a large number when one does not fit at all)
template <class SH>
double stage_blocks_per_range(const fvs_ctx &C, const StageMesh &M) {
  const long nr = nblk(C.N, SH::BS), step = std::max(1L, nr / 256);
  std::vector<short> lgat(size_t(C.GW) * C.N, 0);
  StageCut<SH> cut(C, M, code_words(M), lgat.data());
  long ranges = 0;
  for (long b = step / 2; b < nr; b += step, ++ranges)
    if (!cut.place_range(b)) return 1e9;
  return double(cut.blk.size()) / double(std::max(1L, ranges));
}

constexpr long kStageGrain = 8;  // ranges per worker thread at least (some 50 us each)

// Cuts all cells into blocks of shape SH and uploads the lists; C.stage_bs stays
// 0 when a slice does not fit, or when so many ranges had to be cut that the
// two-kernel path is faster.  With kernel_path 2 there are lists in that case too,
// for persistent launches, and C.use_stage is false.
template <class SH>
int setup_stage_blocks(fvs_ctx &C, const StageMesh &M) {
  const int N = C.N, Fi = C.Fi, cw = code_words(M);
  const long nr = nblk(N, SH::BS), np = parallel_parts(nr, kStageGrain);
  std::vector<short> lgat(size_t(C.GW) * N, 0);
  std::vector<StageCut<SH>> parts(np, StageCut<SH>(C, M, cw, lgat.data()));
  std::vector<char> ok(np, 1);
  parallel_for(nr, kStageGrain, [&](long t, long b0, long b1) {
    for (long b = b0; b < b1 && ok[t]; ++b) ok[t] = parts[t].place_range(b) && parts[t].shift_ok;
  });
  std::vector<size_t> start(np + 1, 0), mstart(np + 1, 0);
  int hs = 1, fs = 1, ns = 0, nkw = 0;
  size_t nmore = 0, nfar = 0;  // packed words of nodes and far cells so far
  for (long t = 0; t < np; ++t) {
    if (!ok[t]) return 0;
    start[t + 1] = start[t] + parts[t].blk.size();
    mstart[t + 1] = mstart[t] + parts[t].morecode.size() / kSlice;
    for (StageBlock &d : parts[t].blk) {
      hs = std::max(hs, std::min(d.nh, d.nr1 + SH::C1));
      ns = std::max(ns, d.nn);
      nkw = std::max(nkw, std::min(d.nkw, kNodeRegs));
      d.more = int(d.nn ? nmore : nfar);
      nmore += size_t(d.nn) * std::max(0, d.nkw - kNodeRegs);
      nfar += std::max(0, d.nh - d.nr1 - SH::C1);
    }
    for (int n : parts[t].nf) fs = std::max(fs, n);
  }
  const size_t nb = start[np];
  if (std::max({mstart[np], nmore, nfar}) > size_t(INT32_MAX)) return 0;
  const bool cut = N > kStageSmallMesh && double(nb) > kStageMostBlocks * double(nr);
  if (cut && C.opt.kernel_path != 2) return 0;
  hs = (hs + 31) / 32 * 32;  // strides of whole cache lines
  fs = (fs + 15) / 16 * 16;
  ns = (ns + 31) / 32 * 32;
  std::vector<StageBlock> blk(nb);
  std::vector<int> halo(nb * hs), far(nfar), bcode(nb * fs);
  std::vector<int> width(nb * SH::NSL), wstart(nb * SH::NSL);
  std::vector<unsigned> morecode(mstart[np] * kSlice), morenode(nmore);
  std::vector<double> morewt(2 * nmore);
  std::vector<unsigned> code(nb * SH::NSL * cw * kSlice), face(nb * fs);
  std::vector<double> geo(nb * fs * 5), nwt(nb * 2 * nkw * ns);
  std::vector<unsigned> gcode(M.ngg > 0 ? nb * 2 * SH::C1 : 0), ncode(nb * nkw * ns);
  run_threads(int(np), [&](int t) {
    const StageCut<SH> &p = parts[t];
    size_t ho = 0, fo = 0, no = 0;
    std::copy(p.gcode.begin(), p.gcode.end(), gcode.begin() + (M.ngg > 0 ? start[t] * 2 * SH::C1 : 0));
    std::copy(p.blk.begin(), p.blk.end(), blk.begin() + start[t]);
    for (size_t k = 0; k < p.width.size(); ++k) {
      width[start[t] * SH::NSL + k] = p.width[k].x;
      wstart[start[t] * SH::NSL + k] = p.width[k].y + int(mstart[t]);
    }
    std::copy(p.morecode.begin(), p.morecode.end(), morecode.begin() + mstart[t] * kSlice);
    std::copy(p.code.begin(), p.code.end(), code.begin() + start[t] * SH::NSL * cw * kSlice);
    for (size_t k = 0; k < p.blk.size(); ++k) {
      const size_t b = start[t] + k;
      const StageBlock &d = p.blk[k];
      const int nh = d.nh, nf = p.nf[k];
      const auto h0 = p.halo.begin() + ho, h1 = h0 + std::min(nh, d.nr1 + SH::C1);
      std::fill(std::copy(h0, h1, halo.begin() + b * hs), halo.begin() + (b + 1) * hs, -1);
      if (h1 != h0 + nh) std::copy(h1, h0 + nh, far.begin() + d.more);
      std::fill(std::copy(p.face.begin() + fo, p.face.begin() + fo + nf, face.begin() + b * fs),
                face.begin() + (b + 1) * fs, ~0u);
      double *q = &geo[b * fs * 5];
      for (int e = 0; e < nf; ++e) {
        const int f = p.slot[fo + e], bq = f - Fi;
        const double *g = f < Fi ? &M.fig[8 * size_t(f)] : &M.fbg[8 * size_t(bq)];
        q[2 * e] = g[0];
        q[2 * e + 1] = g[1];
        q[2 * (fs + e)] = f < Fi ? C.mp.ex[C.mp.edge_intr[f]] : g[5];
        q[2 * (fs + e) + 1] = f < Fi ? C.mp.ey[C.mp.edge_intr[f]] : g[6];
        q[4 * fs + e] = g[2];
        if (f >= Fi)
          bcode[b * fs + e] = M.fbt[bq] | ((C.ninst > 0 ? C.inst_of_real[C.perm[M.fbc[bq]]] : 0) << 2);
      }
      for (int n = 0; n < d.nn; ++n)
        for (int e = 0; e < 2 * d.nkw; ++e, ++no) {
          const unsigned v = unsigned(p.ncode[no]) << (16 * (e & 1));
          if (e / 2 < nkw) {
            ncode[(b * nkw + e / 2) * ns + n] |= v;
            nwt[(b * 2 * nkw + e) * ns + n] = p.nwt[no];
          } else {
            morenode[size_t(d.more) + size_t(e / 2 - nkw) * d.nn + n] |= v;
            morewt[2 * size_t(d.more) + size_t(e - 2 * nkw) * d.nn + n] = p.nwt[no];
          }
        }
      ho += size_t(nh);
      fo += size_t(nf);
    }
  });
  StageBlock *dblk;
  int *dhalo, *dbcode, *dfar;
  int *dwidth, *dwstart;
  unsigned *dcode, *dface, *dgcode, *dncode, *dmorecode, *dmorenode;
  double *dgeo, *dnwt, *dmorewt;
  short *dlgat;
  if (int rc = C.upload(dblk, blk)) return rc;
  if (int rc = C.upload(dhalo, halo)) return rc;
  if (int rc = C.upload(dbcode, bcode)) return rc;
  if (int rc = C.upload(dwidth, width)) return rc;
  if (int rc = C.upload(dwstart, wstart)) return rc;
  if (int rc = C.upload(dcode, code)) return rc;
  if (int rc = C.upload(dface, face)) return rc;
  if (int rc = C.upload(dgeo, geo)) return rc;
  if (int rc = C.upload(dlgat, lgat)) return rc;
  if (int rc = C.upload(dgcode, gcode)) return rc;
  if (int rc = C.upload(dncode, ncode)) return rc;
  if (int rc = C.upload(dnwt, nwt)) return rc;
  if (int rc = C.upload(dmorecode, morecode)) return rc;
  if (int rc = C.upload(dmorenode, morenode)) return rc;
  if (int rc = C.upload(dmorewt, morewt)) return rc;
  if (int rc = C.upload(dfar, far)) return rc;
  HIPC(hipStreamSynchronize(C.stream));  // the host arrays end here
  C.SL = {dblk, dhalo, dcode, dwidth, dwstart, dface, dgeo, dbcode, dlgat, hs, cw, fs, dgcode, dncode, dnwt, ns, nkw,
          dmorecode, dmorenode, dmorewt, dfar};
  C.stage_bs = SH::BS;
  C.use_stage = !cut;
  C.stage_words = C.stage_faces = C.stage_halo = C.stage_incidences = 0;
  for (const StageCut<SH> &p : parts) {
    C.stage_faces += long(p.face.size());
    C.stage_halo += long(p.halo.size());
    C.stage_incidences += long(p.nwt.size());
    for (int2 w : p.width) C.stage_words += long(w.x) * kSlice;
  }
  C.stage_cells.clear();
  for (const StageBlock &d : blk) C.stage_cells.push_back(make_int2(d.i0, d.n0));
  return 0;
}

// The block shape: 128-cell blocks, unless many of them do not fit (O-grids,
// whose stretched blocks have large halos) and the mesh is large enough for a
// 256-cell block on every CU.  Measured, us per step in 128- / 256-cell blocks:
// 2,097,152-cell vortex (nothing cut) 5% less / more; O-grids, limited, 128x64 (11%
// more blocks) 13% less / more, 256x128 63 / 64, 300x150 72 / 69, 384x192 100 / 91,
// 512x256 (19% more) 136 / 124; a batch of 12 O-grids (17% more) 416 / 371.  Room
// for 448 local cells in the large shape cuts 9 ranges of 512x256 instead of 86 and
// changes nothing.
int setup_stage(fvs_ctx &C, const StageMesh &M) {
  const bool large = C.opt.kernel_path != 2 && C.N >= 256 * StageLarge::BS;
  if (large && stage_blocks_per_range<StageSmall>(C, M) > 1.05) {
    if (int rc = setup_stage_blocks<StageLarge>(C, M)) return rc;
    if (C.stage_bs) return 0;
  }
  if (int rc = setup_stage_blocks<StageSmall>(C, M)) return rc;
  if (C.stage_bs || C.opt.kernel_path != 2) return 0;
  // persistent launches of cells whose 64-cell blocks exceed the small shape
  // (quadrilaterals in rows): 64 cells and their up to 256 neighbours fit the large
  if (int rc = setup_stage_blocks<StageLarge>(C, M)) return rc;
  C.use_stage = false;
  return 0;
}

// The same for a Green-Gauss gradient: the table of the faces' periodic shifts
// and the centres come first; without room for the shifts stage_bs stays 0.
int setup_gg_stage(fvs_ctx &C, const StageMesh &M) {
  const MeshPrep &m = C.mp;
  size_t n = 0;
  for (int e : m.edge_intr) {
    const double sx = m.esx[e], sy = m.esy[e];
    if (sx == 0.0 && sy == 0.0) continue;
    size_t q = 0;
    while (q < n && !(C.shifts.sx[q] == sx && C.shifts.sy[q] == sy)) ++q;
    if (q < n) continue;
    if (n == 15) return 0;
    C.shifts.sx[n] = sx;
    C.shifts.sy[n++] = sy;
  }
  std::vector<double2> cxy(C.N);
  for (int i = 0; i < C.N; ++i) cxy[i] = make_double2(m.cx[C.perm[i]], m.cy[C.perm[i]]);
  if (int rc = C.upload(C.cxy, cxy)) return rc;
  C.pmode = M.fnb ? kGGCB : kGGNB;
  return setup_stage(C, M);
}
