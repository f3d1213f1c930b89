// Construction of the device-resident cell-wise operator: validation of the
// cell -> dof map, greedy colouring of the cell-adjacency graph (cells that
// share a classical dof get different colours, so one colour's scatter-add is
// race-free), size classes, launch order, fragment offsets, the enriched-dof
// reduction lists and the dof -> slot lists of the stand-alone scatter.
#include <algorithm>
#include <numeric>
#include <unordered_map>

#include "api_util.hpp"
#include "kernels.hpp"

namespace dfx
{
  DevBuf &work(dfx_ctx *ctx, const char *name, size_t bytes)
  {
    DevBuf &b = ctx->work[name];
    b.ensure(bytes);
    return b;
  }

  template <class T>
  void colDotsView(dfx_ctx *ctx, View<const T> X, View<const T> Y, double *hostOut)
  {
    const u32 B = X.B;
    ctx->reducePartials.ensure((size_t)DOT_BLOCKS * B * sizeof(double) + B * sizeof(double));
    double *part = ctx->reducePartials.as<double>();
    double *out  = part + (size_t)DOT_BLOCKS * B;
    k::colDots<T>(ctx->stream, X, Y, part, out);
    DFX_HIP(hipMemcpyAsync(hostOut, out, B * sizeof(double), hipMemcpyDeviceToHost,
                           ctx->stream));
    DFX_HIP(hipStreamSynchronize(ctx->stream));
  }
  template void colDotsView<double>(dfx_ctx *, View<const double>, View<const double>,
                                    double *);
  template void colDotsView<float>(dfx_ctx *, View<const float>, View<const float>,
                                   double *);

  void colDotsHost(dfx_ctx *ctx, const dfx_mv *X, const dfx_mv *Y, double *out)
  {
    if (X->dtype == DFX_F64)
      colDotsView<double>(ctx, View<const double>{(const double *)X->d, X->N, X->B, X->B},
                          View<const double>{(const double *)Y->d, Y->N, Y->B, Y->B}, out);
    else
      colDotsView<float>(ctx, View<const float>{(const float *)X->d, X->N, X->B, X->B},
                         View<const float>{(const float *)Y->d, Y->N, Y->B, Y->B}, out);
  }

  namespace
  {
    u32 mtwOf(u32 n) { return (((n + 15) / 16) + 3) / 4; }

    // The slot apply's tables: launch records and cell metadata by (size
    // class, caller order), so that neighbours follow each other; the masked
    // map; per classical row its slots in launch order (the order in which
    // the colour-by-colour apply adds); the enriched dofs' slots in cell
    // order (eOff: their offsets).  Not built (slotsOk false) for rows of
    // more than 30 cells or more than 2^27 shared slots
    void buildSlots(dfx_op *op, const u32 *map, const std::vector<u32> &nc,
                    const std::vector<u32> &eOff, bool merge)
    {
      const u32   nCells = op->nCells, nClassical = op->nClassical;
      const auto &nd = op->hCellNdofs, &off = op->hMapOffset;
      hipStream_t st = op->ctx->stream;
      // slots per classical row; the first one is known from a row's head
      std::vector<unsigned char> cnt(nClassical, 0);
      u64                        others = 0;
      for (u32 e = 0; e < nCells; ++e)
        for (u32 s = off[e]; s < off[e] + nc[e]; ++s)
          {
            if (cnt[map[s]] == ROW_ZERO - 1)
              return;
            others += cnt[map[s]]++ != 0;
          }
      if (others >= (1ull << ROW_COUNT_SHIFT))
        return;
      const dfx_constraints *cons = op->cons;
      op->zeroRows = cons && cons->homDirichlet && !cons->hRows.empty() &&
                     *std::max_element(cons->hRows.begin(), cons->hRows.end()) < nClassical;
      std::vector<RowHead> heads(nClassical);
      std::vector<u32>     rest(others);
      u32                  pos = 0;
      for (u32 d = 0; d < nClassical; ++d)
        {
          heads[d] = {0u, ((u32)cnt[d] << ROW_COUNT_SHIFT) | pos};
          pos += cnt[d] ? cnt[d] - 1u : 0u;
        }
      std::vector<unsigned char> seen(nClassical, 0);
      for (u32 q = 0; q < nCells; ++q)
        {
          const u32 e = op->hOrder[q];
          for (u32 s = off[e]; s < off[e] + nc[e]; ++s)
            {
              RowHead       &h = heads[map[s]];
              unsigned char &k = seen[map[s]];
              if (k == 0)
                h.slot0 = s;
              else
                rest[(h.rest & ((1u << ROW_COUNT_SHIFT) - 1)) + k - 1] = s;
              ++k;
            }
        }
      if (op->zeroRows)
        {
          std::vector<u32> masked(map, map + op->sumNe);
          for (u32 r : cons->hRows)
            heads[r] = {0u, ROW_ZERO << ROW_COUNT_SHIFT};
          for (u32 e = 0; e < nCells; ++e)
            for (u32 s = off[e]; s < off[e] + nc[e]; ++s)
              if (heads[map[s]].rest >> ROW_COUNT_SHIFT == ROW_ZERO)
                masked[s] = ROW_NONE;
          upload(op->slotMap, masked, st);
        }
      // enriched dofs: the same lists as the colour apply's, as map slots
      std::vector<u32> eSlots(op->nEnrSlots), fp(eOff.begin(), eOff.end() - 1);
      for (u32 e = 0; e < nCells; ++e)
        for (u32 s = off[e] + nc[e]; s < off[e + 1]; ++s)
          eSlots[fp[map[s] - nClassical]++] = s;
      // launch order
      std::vector<u32> place(nCells), at(nCells);
      for (u32 q = 0; q < nCells; ++q)
        place[op->hOrder[q]] = q;
      std::iota(at.begin(), at.end(), 0u);
      std::stable_sort(at.begin(), at.end(),
                       [&](u32 a, u32 b) { return mtwOf(nd[a]) > mtwOf(nd[b]); });
      op->hSlotPos.resize(nCells);
      for (u32 q = 0; q < nCells; ++q)
        op->hSlotPos[q] = place[at[q]];
      for (int f64 = 0; f64 < 2; ++f64)
        {
          auto &out = f64 ? op->slotLaunches64 : op->slotLaunches32;
          out.clear();
          for (u32 q = 0; q < nCells;)
            {
              Launch l{};
              l.begin = q;
              l.mtw   = mtwOf(nd[at[q]]);
              for (; q < nCells && (merge || mtwOf(nd[at[q]]) == l.mtw); ++q)
                {
                  const u32 n = nd[at[q]];
                  l.kpadMax   = std::max(l.kpadMax, f64 ? 8 * ((n + 7) / 8) : 16 * ((n + 15) / 16));
                  l.sumN2 += (u64)n * n;
                  l.sumN += n;
                  l.sumNc += nc[at[q]];
                }
              l.end = q;
              out.push_back(l);
            }
        }
      upload(op->rowHeads, heads, st);
      if (!rest.empty())
        upload(op->slotRest, rest, st);
      if (!eSlots.empty())
        upload(op->enrMapSlots, eSlots, st);
      op->slotsOk = true;
    }
  } // namespace

  void buildCellwise(dfx_ctx *ctx, dfx_op *op, u32 nCells, const u32 *cellNdofs,
                     const u32 *map, u32 nDofs, u32 nClassical, dfx_constraints *cons,
                     u32 flags)
  {
    DFX_REQUIRE(nClassical <= nDofs, "nClassical > nDofs");
    DFX_REQUIRE(!cons || cons->nDofs == nDofs, "constraints built for another N");
    op->ctx        = ctx;
    op->kind       = OP_CELLWISE;
    op->nDofs      = nDofs;
    op->nClassical = nClassical;
    op->cons       = cons;
    consRetain(cons);
    op->nCells     = nCells;
    op->hasF32     = (flags & DFX_OP_KEEP_FP32) != 0;
    op->hCellNdofs.assign(cellNdofs, cellNdofs + nCells);
    op->hMapOffset.resize(nCells + 1);
    op->hMatOffset.resize(nCells + 1);
    op->hMapOffset[0] = 0;
    op->hMatOffset[0] = 0;
    u64 sumNe = 0, sumNe2 = 0;
    u32 maxN  = 0;
    for (u32 e = 0; e < nCells; ++e)
      {
        const u32 n = cellNdofs[e];
        DFX_REQUIRE(n > 0 && n <= 256, "cell dof count must be in 1..256");
        sumNe += n;
        sumNe2 += (u64)n * n;
        maxN = std::max(maxN, n);
        DFX_REQUIRE(sumNe < (1ull << 32), "cell->dof map longer than 2^32");
        op->hMapOffset[e + 1] = (u32)sumNe;
        op->hMatOffset[e + 1] = sumNe2;
      }
    op->sumNe  = sumNe;
    op->sumNe2 = sumNe2;
    op->maxN   = maxN;

    // classical entries first in every cell; nc = their count
    std::vector<u32> nc(nCells);
    for (u32 e = 0; e < nCells; ++e)
      {
        u32  cnt = 0;
        bool enr = false;
        for (u32 s = op->hMapOffset[e]; s < op->hMapOffset[e + 1]; ++s)
          {
            DFX_REQUIRE(map[s] < nDofs, "cell->dof map entry out of range");
            if (map[s] < nClassical)
              {
                DFX_REQUIRE(!enr, "classical dofs must precede enriched dofs in a cell");
                ++cnt;
              }
            else
              enr = true;
          }
        nc[e] = cnt;
      }
    {
      // a dof may appear once per cell (two lanes would update one row)
      std::vector<u32> last(nDofs, 0xffffffffu);
      for (u32 e = 0; e < nCells; ++e)
        for (u32 s = op->hMapOffset[e]; s < op->hMapOffset[e + 1]; ++s)
          {
            DFX_REQUIRE(last[map[s]] != e, "a dof appears twice in one cell's map");
            last[map[s]] = e;
          }
    }

    // ---- greedy colouring over shared classical dofs (cell order)
    std::vector<u32> dofCellOff(nClassical + 1, 0), dofCells;
    for (u32 e = 0; e < nCells; ++e)
      for (u32 s = op->hMapOffset[e]; s < op->hMapOffset[e] + nc[e]; ++s)
        ++dofCellOff[map[s] + 1];
    for (u32 d = 0; d < nClassical; ++d)
      dofCellOff[d + 1] += dofCellOff[d];
    dofCells.resize(dofCellOff[nClassical]);
    {
      std::vector<u32> fillp(dofCellOff.begin(), dofCellOff.end() - 1);
      for (u32 e = 0; e < nCells; ++e)
        for (u32 s = op->hMapOffset[e]; s < op->hMapOffset[e] + nc[e]; ++s)
          dofCells[fillp[map[s]]++] = e;
    }
    std::vector<int> color(nCells, -1);
    std::vector<u32> stamp(64, 0xffffffffu);
    int nColors = 0;
    for (u32 e = 0; e < nCells; ++e)
      {
        for (u32 s = op->hMapOffset[e]; s < op->hMapOffset[e] + nc[e]; ++s)
          for (u32 q = dofCellOff[map[s]]; q < dofCellOff[map[s] + 1]; ++q)
            {
              const int c = color[dofCells[q]];
              if (c >= 0)
                {
                  if ((size_t)c >= stamp.size())
                    stamp.resize(c + 1, 0xffffffffu);
                  stamp[c] = e;
                }
            }
        int c = 0;
        while ((size_t)c < stamp.size() && stamp[c] == e)
          ++c;
        color[e] = c;
        nColors  = std::max(nColors, c + 1);
      }
    op->nColors = (u32)nColors;

    // ---- launch order: (colour, M-tile class, cell)
    op->hOrder.resize(nCells);
    std::iota(op->hOrder.begin(), op->hOrder.end(), 0u);
    std::stable_sort(op->hOrder.begin(), op->hOrder.end(), [&](u32 a, u32 b) {
      if (color[a] != color[b])
        return color[a] < color[b];
      return mtwOf(cellNdofs[a]) > mtwOf(cellNdofs[b]);
    });

    // enriched partial rows, in caller cell order
    std::vector<u32> enrOff(nCells + 1, 0);
    for (u32 e = 0; e < nCells; ++e)
      enrOff[e + 1] = enrOff[e] + (cellNdofs[e] - nc[e]);
    op->nEnrSlots = enrOff[nCells];

    op->hMeta.resize(nCells);
    for (u32 q = 0; q < nCells; ++q)
      {
        const u32 e = op->hOrder[q];
        const u32 n = cellNdofs[e];
        CellMeta  m;
        m.n         = n;
        m.nc        = nc[e];
        m.mapOff    = op->hMapOffset[e];
        m.enrOff    = enrOff[e];
        m.fragOff64 = m.fragOff32 = 0; // placeCellMatrices
        u32 lo = 0xffffffffu, hi = 0;
        for (u32 i = 0; i < nc[e]; ++i)
          {
            lo = std::min(lo, map[op->hMapOffset[e] + i]);
            hi = std::max(hi, map[op->hMapOffset[e] + i]);
          }
        m.rowLo         = nc[e] ? lo : 0;
        m.pad_          = 0;
        op->maxRowSpan  = std::max(op->maxRowSpan, nc[e] ? hi - lo + 1 : 0u);
        op->hMeta[q] = m;
      }

    // one launch per (colour, size class); an operator of few cells (the
    // launches could not fill the GPU anyway, and every launch costs a
    // dispatch) runs each colour as one launch with the largest class's tile.
    // FP32 launches also merge the classes of a colour whenever the largest
    // class fits cells of up to 192 dofs (measured on C4: one launch per
    // colour instead of two side by side takes the FP32 apply from 1.39 to
    // 1.30 ms; the FP64 apply, whose classes use different column-chunk
    // widths, gets slower merged).  DFX_MERGE_CLASSES_BELOW sets the cell
    // count below which both merge (and nothing else does)
    const char *mergeEnv   = getenv("DFX_MERGE_CLASSES_BELOW");
    const u32   mergeBelow = mergeEnv ? (u32)atol(mergeEnv) : 4096u;
    u32         maxMtw     = 0;
    for (u32 e = 0; e < nCells; ++e)
      maxMtw = std::max(maxMtw, mtwOf(cellNdofs[e]));
    const bool merge64 = nCells < mergeBelow;
    const bool merge32 = mergeEnv ? merge64 : (merge64 || maxMtw <= 3);
    auto buildLaunches = [&](std::vector<Launch> &out, bool merge, bool f64) {
      out.clear();
      for (u32 q = 0; q < nCells;)
        {
          const u32 e0 = op->hOrder[q];
          u32       r  = q;
          u32 kp = 0, mtw = 0;
          u64 s2 = 0, s1 = 0, sc = 0;
          while (r < nCells && color[op->hOrder[r]] == color[e0] &&
                 (merge || mtwOf(cellNdofs[op->hOrder[r]]) == mtwOf(cellNdofs[e0])))
            {
              const u32 n = cellNdofs[op->hOrder[r]];
              kp          = std::max(kp, f64 ? 8 * ((n + 7) / 8) : 16 * ((n + 15) / 16));
              mtw         = std::max(mtw, mtwOf(n));
              s2 += (u64)n * n;
              s1 += n;
              sc += nc[op->hOrder[r]];
              ++r;
            }
          out.push_back({q, r, mtw, kp, s2, s1, sc, 0, (u32)color[e0]});
          q = r;
        }
    };
    buildLaunches(op->launches64, merge64, true);
    buildLaunches(op->launches32, merge32, false);
    op->merged192 = merge32 && maxMtw == 3;

    // first-touch bits in launch order: the first cell to reach a classical
    // dof stores its contribution, later cells add to it
    std::vector<u32> hFirst((size_t)nCells * 8, 0u);
    {
      std::vector<unsigned char> seen(nClassical, 0);
      for (u32 q = 0; q < nCells; ++q)
        {
          const u32 e = op->hOrder[q];
          for (u32 i = 0; i < nc[e]; ++i)
            {
              const u32 d = map[op->hMapOffset[e] + i];
              if (!seen[d])
                {
                  seen[d] = 1;
                  hFirst[(size_t)q * 8 + i / 32] |= 1u << (i % 32);
                }
            }
        }
      op->fillY = std::find(seen.begin(), seen.end(), 0) != seen.end();
      for (auto *L : {&op->launches64, &op->launches32})
        for (Launch &l : *L)
          {
            l.sumFirst = 0;
            for (u64 w = (u64)l.begin * 8; w < (u64)l.end * 8; ++w)
              l.sumFirst += (u64)__builtin_popcount(hFirst[w]);
          }
    }

    // last-touch bits in launch order (the residual step fused into the
    // cell apply): the last cell to reach an unconstrained classical dof
    // finishes it; every other row is listed for the stand-alone step
    std::vector<u32> hLast((size_t)nCells * 8, 0u), hResRows;
    {
      // 0: in no cell, 1: finished by a cell, 2: constrained
      std::vector<unsigned char> st(nClassical, 0);
      if (cons)
        for (u32 r : cons->hRows)
          if (r < nClassical)
            st[r] = 2;
      for (u32 q = nCells; q-- > 0;)
        {
          const u32 e = op->hOrder[q];
          for (u32 i = 0; i < nc[e]; ++i)
            {
              const u32 d = map[op->hMapOffset[e] + i];
              if (!st[d])
                {
                  st[d] = 1;
                  hLast[(size_t)q * 8 + i / 32] |= 1u << (i % 32);
                }
            }
        }
      // homogeneous Dirichlet rows are zero in every residual-filter buffer
      // from the seed on (A and M zero them) and the step keeps them zero,
      // so they are left out; other constrained rows and rows in no cell
      // are listed
      const bool zeroRows = cons && cons->homDirichlet;
      for (u32 d = 0; d < nClassical; ++d)
        if (st[d] == 0 || (st[d] == 2 && !zeroRows))
          hResRows.push_back(d);
      for (u32 d = nClassical; d < nDofs; ++d)
        hResRows.push_back(d);
      op->nResRows = (u32)hResRows.size();
    }

    // enriched dof -> slots (cell order)
    const u32 nE = nDofs - nClassical;
    std::vector<u32> eOff(nE + 1, 0), eSlots(op->nEnrSlots);
    for (u32 e = 0; e < nCells; ++e)
      for (u32 i = nc[e]; i < cellNdofs[e]; ++i)
        ++eOff[map[op->hMapOffset[e] + i] - nClassical + 1];
    for (u32 g = 0; g < nE; ++g)
      eOff[g + 1] += eOff[g];
    {
      std::vector<u32> fp(eOff.begin(), eOff.end() - 1);
      for (u32 e = 0; e < nCells; ++e)
        for (u32 i = nc[e]; i < cellNdofs[e]; ++i)
          eSlots[fp[map[op->hMapOffset[e] + i] - nClassical]++] = enrOff[e] + (i - nc[e]);
    }

    // dof -> map slots (slot order = cell order)
    std::vector<u32> sOff(nDofs + 1, 0), sList(sumNe);
    for (u64 s = 0; s < sumNe; ++s)
      ++sOff[map[s] + 1];
    for (u32 d = 0; d < nDofs; ++d)
      sOff[d + 1] += sOff[d];
    {
      std::vector<u32> fp(sOff.begin(), sOff.end() - 1);
      for (u64 s = 0; s < sumNe; ++s)
        sList[fp[map[s]]++] = (u32)s;
    }

    hipStream_t st = ctx->stream;
    upload(op->map, map, sumNe, st);
    buildSlots(op, map, nc, eOff, mergeEnv ? merge64 : nCells < 1024u);
    upload(op->first, hFirst, st);
    upload(op->last, hLast, st);
    if (!hResRows.empty())
      upload(op->resRows, hResRows, st);
    upload(op->enrSlotOffsets, eOff, st);
    upload(op->enrSlots, eSlots, st);
    upload(op->dofSlotOffsets, sOff, st);
    upload(op->dofSlots, sList, st);
  }

  namespace
  {
    // elements of a cell matrix in fragment order: whole 16-row tiles and
    // blocks of 4 G columns
    template <class T>
    u64 fragLength(u64 n)
    {
      constexpr u64 KB = 64 / sizeof(T);
      return 16 * ((n + 15) / 16) * (KB * ((n + KB - 1) / KB));
    }

    // Where the cell matrices of an upload go: per launch position the metadata
    // with the fragment offsets, the launch positions whose matrices are stored
    // (`stored`), and the lengths that they take
    struct Placement
    {
      std::vector<CellMeta> meta;
      std::vector<u32>      stored;
      u64                   len64 = 0, len32 = 0;
    };

    // Fragment offsets of the cell matrices, those of cells with the same
    // matrix (bit for bit) shared.  On a uniform mesh the mass and stiffness
    // matrices of all unenriched cells are one matrix: their applies then read
    // it from the L2 instead of streaming a copy per cell (K apply of 16^3 cells
    // at p = 3, 8 columns FP64: cell kernel 29 -> 19 us; 134 MB of copies).
    // Candidates come from a content hash and are compared in full
    Placement placeCellMatrices(const dfx_op *op, const double *raw, const u64 *rawOff)
    {
      const u32   nCells = op->nCells;
      hipStream_t st     = op->ctx->stream;
      std::vector<u32> rep(nCells), a, b;
      std::iota(rep.begin(), rep.end(), 0u);
      if (nCells)
        {
          DevBuf           dh((size_t)nCells * sizeof(u64));
          std::vector<u64> h(nCells);
          k::cellHashes(st, nCells, raw, rawOff, dh.as<u64>());
          DFX_HIP(hipMemcpyAsync(h.data(), dh.p, dh.bytes, hipMemcpyDeviceToHost, st));
          DFX_HIP(hipStreamSynchronize(st));
          std::unordered_map<u64, u32> seen;
          for (u32 e = 0; e < nCells; ++e)
            {
              const auto it = seen.emplace(h[e], e).first;
              if (it->second != e && op->hCellNdofs[it->second] == op->hCellNdofs[e])
                {
                  a.push_back(e);
                  b.push_back(it->second);
                }
            }
        }
      if (!a.empty())
        {
          DevBuf           da, db, dd(a.size() * sizeof(u32));
          std::vector<u32> d(a.size());
          upload(da, a, st);
          upload(db, b, st);
          k::cellsDiffer(st, (u32)a.size(), raw, rawOff, da.as<u32>(), db.as<u32>(), dd.as<u32>());
          DFX_HIP(hipMemcpyAsync(d.data(), dd.p, dd.bytes, hipMemcpyDeviceToHost, st));
          DFX_HIP(hipStreamSynchronize(st));
          for (size_t i = 0; i < a.size(); ++i)
            if (!d[i])
              rep[a[i]] = b[i];
        }
      Placement P;
      P.meta = op->hMeta;
      std::vector<u32> at(nCells, 0xffffffffu); // representative -> launch position
      for (u32 q = 0; q < nCells; ++q)
        {
          u32 &r = at[rep[op->hOrder[q]]];
          if (r == 0xffffffffu)
            {
              r = q;
              P.stored.push_back(q);
              P.meta[q].fragOff64 = P.len64;
              P.meta[q].fragOff32 = P.len32;
              P.len64 += fragLength<double>(P.meta[q].n);
              P.len32 += fragLength<float>(P.meta[q].n);
            }
          else
            {
              P.meta[q].fragOff64 = P.meta[r].fragOff64;
              P.meta[q].fragOff32 = P.meta[r].fragOff32;
            }
        }
      return P;
    }
  } // namespace

  namespace
  {
    // per launch over `meta`, the n_e^2 of the matrices it reads, each once
    std::vector<u64> distinctN2(const std::vector<Launch> &L, const std::vector<CellMeta> &meta)
    {
      std::vector<u64>                 out;
      std::vector<std::pair<u64, u64>> m; // (offset, n^2)
      for (const Launch &l : L)
        {
          m.clear();
          for (u32 q = l.begin; q < l.end; ++q)
            m.emplace_back(meta[q].fragOff64, (u64)meta[q].n * meta[q].n);
          std::sort(m.begin(), m.end());
          m.erase(std::unique(m.begin(), m.end()), m.end());
          u64 s = 0;
          for (const auto &x : m)
            s += x.second;
          out.push_back(s);
        }
      return out;
    }
  } // namespace

  // The stores have room for a matrix per cell and, like the metadata, stay
  // where they are from the operator's creation on: an update needs no memory
  // for them however many matrices differ, and a graph that a caller captured
  // an apply into stays valid.  What can fail for want of memory comes first: a
  // refused update leaves the operator as it was
  void uploadCellMatrices(dfx_op *op, const double *mats, bool device)
  {
    hipStream_t st = op->ctx->stream;
    DevBuf      raw, rawOff, order, stored;
    const double *dmats = mats;
    if (!device)
      {
        upload(raw, mats, op->sumNe2, st);
        dmats = raw.as<double>();
      }
    upload(rawOff, op->hMatOffset, st);
    Placement P = placeCellMatrices(op, dmats, rawOff.as<u64>());
    upload(order, op->hOrder, st);
    upload(stored, P.stored, st);
    std::vector<CellMeta> ms(op->slotsOk ? op->nCells : 0); // slot order
    for (u32 q = 0; q < ms.size(); ++q)
      ms[q] = P.meta[op->hSlotPos[q]];
    std::vector<Launch> *const lists[] = {&op->launches64, &op->launches32, &op->slotLaunches64,
                                          &op->slotLaunches32};
    std::vector<u64> distinct[4];
    for (int i = 0; i < 4; ++i)
      distinct[i] = distinctN2(*lists[i], i < 2 ? P.meta : ms);
    const size_t metaBytes = P.meta.size() * sizeof(CellMeta), msBytes = ms.size() * sizeof(CellMeta);
    if (!op->frag64.p) // the operator is being made
      {
        u64 cap64 = 0, cap32 = 0;
        for (const CellMeta &m : P.meta)
          {
            cap64 += fragLength<double>(m.n);
            cap32 += fragLength<float>(m.n);
          }
        op->meta.alloc(metaBytes);
        op->metaSlots.alloc(msBytes);
        op->frag64.alloc(cap64 * sizeof(double));
        if (op->hasF32)
          op->frag32.alloc(cap32 * sizeof(float));
      }

    ++op->gen;
    for (int i = 0; i < 4; ++i)
      for (size_t j = 0; j < lists[i]->size(); ++j)
        (*lists[i])[j].distinctN2 = distinct[i][j];
    op->hMeta.swap(P.meta);
    op->fragLen64 = P.len64;
    op->fragLen32 = P.len32;
    if (metaBytes)
      DFX_HIP(hipMemcpyAsync(op->meta.p, op->hMeta.data(), metaBytes, hipMemcpyHostToDevice, st));
    if (msBytes)
      DFX_HIP(hipMemcpyAsync(op->metaSlots.p, ms.data(), msBytes, hipMemcpyHostToDevice, st));
    const u32 nStored = (u32)P.stored.size();
    k::repackCells<double>(st, op, nStored, stored.as<u32>(), order.as<u32>(), dmats,
                           rawOff.as<u64>(), op->frag64.as<double>());
    if (op->hasF32)
      k::repackCells<float>(st, op, nStored, stored.as<u32>(), order.as<u32>(), dmats,
                            rawOff.as<u64>(), op->frag32.as<float>());
    DFX_HIP(hipStreamSynchronize(st));
  }
} // namespace dfx
