// mesh_host.cpp -- fvMesh geometry and addressing for the device path.
//
// The reference reads Sf, magSf, Cf, C, V, weights and deltaCoeffs from
// foam-extend's fvMesh (e.g. Roe.C:79, :195-197; timeDST.C:237); this file
// computes the same quantities from the polyMesh primitives on the host
// (face centres/areas by triangle decomposition about the point average,
// cell centres/volumes by face pyramids about the face-centre average,
// linear weights from the face-normal distances, stabilised deltaCoeffs
// 1/max(n.d, 0.05|d|) as the comment at timeDST.C:237 states) and derives
// the device addressing: the ELL cell->face map the cell-centric face loop
// walks, the owner/neighbour-sorted block-CSR with its face->slot maps, a
// greedy face colouring, and the level sets of the natural-order ILU sweeps.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>

#include "rdst_internal.hpp"

namespace rdst {

namespace {
struct P3 { double x, y, z; };
inline P3 add(P3 a, P3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
inline P3 sub(P3 a, P3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
inline P3 scl(double s, P3 a) { return {s * a.x, s * a.y, s * a.z}; }
inline double dotp(P3 a, P3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
inline P3 crossp(P3 a, P3 b) { return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x}; }
inline double norm(P3 a) { return std::sqrt(dotp(a, a)); }
}  // namespace

namespace {

// Recursive coordinate bisection: split the cell set at the median of its
// longest extent (ties broken by cell index) until a set holds at most
// maxCells cells.
void rcb(const std::vector<double>& C, std::vector<int>& idx, int lo, int hi, int maxCells, std::vector<int32_t>& part,
         int& nParts) {
    if (hi - lo <= maxCells) {
        for (int k = lo; k < hi; ++k) part[idx[k]] = nParts;
        ++nParts;
        return;
    }
    double mn[3] = {1e300, 1e300, 1e300}, mx[3] = {-1e300, -1e300, -1e300};
    for (int k = lo; k < hi; ++k)
        for (int d = 0; d < 3; ++d) {
            mn[d] = std::min(mn[d], C[3 * (size_t)idx[k] + d]);
            mx[d] = std::max(mx[d], C[3 * (size_t)idx[k] + d]);
        }
    int ax = 0;
    for (int d = 1; d < 3; ++d) if (mx[d] - mn[d] > mx[ax] - mn[ax]) ax = d;
    const int mid = lo + (hi - lo) / 2;
    std::nth_element(idx.begin() + lo, idx.begin() + mid, idx.begin() + hi, [&](int a, int b) {
        double ca = C[3 * (size_t)a + ax], cb = C[3 * (size_t)b + ax];
        return ca < cb || (ca == cb && a < b);
    });
    rcb(C, idx, lo, mid, maxCells, part, nParts);
    rcb(C, idx, mid, hi, maxCells, part, nParts);
}

}  // namespace

// The partitions of an ILU(0) apply as build_stream reads them (PartSet).
struct PartView {
    int nParts;
    const std::vector<int32_t>&rowStart, &rows, &levStart, &levPtr, &localCol;
};

// The record stream of an ILU(0) apply, in the layout StreamSet describes.
// tiles: the set is a TileSet; if it is more than one tile, the two sweeps are
// read by separate launches, so the backward records start a ring of their own.
// Left empty (kmax = 0) when a row has more than kStreamKD off-diagonal blocks in
// one sweep.
static void build_stream(const Mesh& m, const PartView& pv, bool tiles, bool fp32, StreamSet& ps) {
    ps.clear();
    const bool split = tiles && pv.nParts > 1;
    int kmax = 1;
    for (int i = 0; i < m.nC; ++i) {
        int lo = 0, up = 0;
        for (int s = m.rowPtr[i]; s < m.rowPtr[i + 1]; ++s)
            if (pv.localCol[s] >= 0 && s != m.slotDiag[i]) (s < m.slotDiag[i] ? lo : up)++;
        kmax = std::max(kmax, std::max(lo, up));
    }
    if (kmax > kStreamKD) return;
    ps.ent = stream_entry(kmax);
    const int ring = stream_ring(fp32), cap = stream_record(fp32), blk = 25 * (fp32 ? 4 : 8);
    struct Row {
        int t, i, cnt;
    };
    std::vector<Row> rows;
    ps.recBeg.assign(1, 0);
    ps.recRows.assign(1, 0);
    ps.recBlk.assign(1, 0);
    size_t pos = 0;
    std::vector<uint32_t> lDst(m.nnzb, 0), dDst(m.nC, 0);  // of forward blocks and Dinv, 4-byte units from the partition's start
    auto size_of = [&](int nr, int nb) { return nr * ps.ent + ((nb * blk + 15) & ~15); };
    for (int p = 0; p < pv.nParts; ++p) {
        const int rs = pv.rowStart[p], nOwn = pv.rowStart[p + 1] - rs;
        const int l0 = pv.levStart[p], nl = pv.levStart[p + 1] - l0 - 1;
        const size_t origin = pos;
        size_t base = pos;
        for (int sweep = 0; sweep < 2; ++sweep) {
            if (sweep == 1) {
                ps.recMid.push_back((int32_t)ps.hdr.size());
                if (split) base = pos = (pos + 1023) & ~(size_t)1023;
            }
            int need = 0;  // halo cells read so far
            for (int li = 0; li < nl; ++li) {
                const int L = sweep ? nl - 1 - li : li;
                rows.clear();
                for (int t = pv.levPtr[l0 + L]; t < pv.levPtr[l0 + L + 1]; ++t) {
                    const int i = pv.rows[t];
                    const int s0 = sweep ? m.slotDiag[i] + 1 : m.rowPtr[i], s1 = sweep ? m.rowPtr[i + 1] : m.slotDiag[i];
                    int cnt = 0;
                    for (int s = s0; s < s1; ++s) cnt += pv.localCol[s] >= 0;
                    if (sweep || cnt || split) rows.push_back({t - rs, i, cnt});  // forward: y = r on a row without L
                }
                // rows of one block count together: a wavefront's rows run the same products
                std::stable_sort(rows.begin(), rows.end(), [](const Row& a, const Row& b) { return a.cnt > b.cnt; });
                for (size_t r0 = 0; r0 < rows.size();) {
                    // as many rows as a record, and the ring up to its end, hold
                    int room = ring - (int)((pos - base) % ring);
                    if (size_of(1, rows[r0].cnt + sweep) > room) {
                        pos += room;
                        ps.hdr.back() += (uint32_t)(room / 16) << 16;
                        room = ring;
                    }
                    room = std::min(room, cap);
                    size_t r1 = r0;
                    int nb = 0;
                    while (r1 < rows.size() && r1 - r0 < (size_t)kStreamRows &&
                           size_of((int)(r1 - r0) + 1, nb + rows[r1].cnt + sweep) <= room)
                        nb += rows[r1++].cnt + sweep;
                    const int nr = (int)(r1 - r0), bytes = size_of(nr, nb);
                    int first = 0;
                    for (size_t q = r0; q < r1; ++q) {
                        const Row& w = rows[q];
                        const size_t e0 = ps.entries.size();
                        ps.entries.resize(e0 + ps.ent / 2, 0);
                        uint16_t* e = ps.entries.data() + e0;
                        e[0] = (uint16_t)(5 * w.t);
                        e[1] = (uint16_t)(first | w.cnt << 8);
                        const size_t at = (pos - origin + (size_t)nr * ps.ent + (size_t)blk * first) / 4;
                        if (sweep) {
                            dDst[w.i] = (uint32_t)at;
                            ps.src.push_back(-(w.i + 1));
                            ps.rowCell.push_back(w.i);
                        }
                        int k = 2;
                        const int s0 = sweep ? m.slotDiag[w.i] + 1 : m.rowPtr[w.i],
                                  s1 = sweep ? m.rowPtr[w.i + 1] : m.slotDiag[w.i];
                        for (int s = s0; s < s1; ++s)
                            if (pv.localCol[s] >= 0) {
                                if (!sweep) lDst[s] = (uint32_t)(at + (size_t)blk / 4 * (k - 2));
                                ps.src.push_back(s);
                                ps.rowCell.push_back(sweep ? w.i : -1);
                                e[k++] = (uint16_t)(5 * pv.localCol[s]);
                                need = std::max(need, pv.localCol[s] - nOwn + 1);
                            }
                        first += w.cnt + sweep;
                    }
                    ps.start.push_back((int64_t)(pos / 16));
                    ps.hdr.push_back((uint32_t)nr | (uint32_t)(bytes / 16) << 16);
                    ps.recRows.push_back(ps.recRows.back() + nr);
                    ps.recBlk.push_back((int32_t)ps.src.size());
                    if (split) ps.need.push_back(need);
                    pos += bytes;
                    r0 = r1;
                }
            }
        }
        ps.recBeg.push_back((int32_t)ps.hdr.size());
        pos = (pos + 1023) & ~(size_t)1023;  // the loader copies 1 KB pieces
    }
    ps.start.push_back((int64_t)(pos / 16));
    ps.nRec = (int)ps.hdr.size();
    ps.kmax = kmax;
    // the factor as a chain: a bipartite mesh has no triangle, any other is looked through
    int K = 1;
    bool tri = false;
    for (int i = 0; i < m.nC && !tri; ++i) {
        int lo = 0;
        for (int p = m.rowPtr[i]; p < m.slotDiag[i]; ++p) {
            if (pv.localCol[p] < 0) continue;
            ++lo;
            if (m.nCellColours <= 2) continue;
            const int k = m.cols[p];
            for (int q = m.slotDiag[k] + 1; q < m.rowPtr[k + 1] && !tri; ++q)
                if (pv.localCol[q] >= 0 && m.cols[q] != i)
                    for (int s = m.rowPtr[i]; s < m.rowPtr[i + 1]; ++s)
                        if (m.cols[s] == m.cols[q] && pv.localCol[s] >= 0) tri = true;
        }
        K = std::max(K, lo);
    }
    if (tri || K > 4) return;
    ps.chainK = K <= 3 ? 3 : 4;
    const int stride = 4 + 4 * ps.chainK;
    ps.chain.assign((size_t)stride * pv.rows.size(), 0);
    std::vector<int32_t> trans(m.nnzb, 0);
    for (int f = 0; f < m.nI; ++f) {
        trans[m.slotUpper[f]] = m.slotLower[f];
        trans[m.slotLower[f]] = m.slotUpper[f];
    }
    for (size_t t = 0; t < pv.rows.size(); ++t) {
        const int i = pv.rows[t];
        int32_t* e = ps.chain.data() + stride * t;
        e[0] = i;
        e[2] = m.slotDiag[i];
        e[3] = (int32_t)dDst[i];
        for (int k = 0; k < ps.chainK; ++k) {  // unused places read the diagonal
            e[4 + 4 * k] = e[5 + 4 * k] = m.slotDiag[i];
            e[6 + 4 * k] = tiles ? 0 : i;
        }
        for (int s = m.rowPtr[i]; s < m.slotDiag[i]; ++s) {
            if (pv.localCol[s] < 0) continue;
            int32_t* q = e + 4 + 4 * e[1]++;
            q[0] = s;
            q[1] = trans[s];
            q[2] = tiles ? pv.localCol[s] : m.cols[s];
            q[3] = (int32_t)lDst[s];
        }
    }
}

void StreamSet::clear() {
    kmax = nRec = chainK = 0;
    for (std::vector<int32_t>* v : {&recBeg, &recMid, &recRows, &recBlk, &need, &src, &rowCell, &chain}) v->clear();
    hdr.clear();
    start.clear();
    entries.clear();
}

void StreamSet::upload() {
    if (kmax == 0) return;
    d_recBeg.upload(recBeg);
    d_recMid.upload(recMid);
    d_recRows.upload(recRows);
    d_recBlk.upload(recBlk);
    d_entries.upload(entries);
    d_hdr.upload(hdr);
    d_start.upload(start);
    d_startLow.upload(std::vector<uint32_t>(start.begin(), start.end()));
    d_need.upload(need);
    d_src.upload(src);
    d_rowCell.upload(rowCell);
    d_chain.upload(chain);
}

StreamSet& mesh_stream(Mesh& m, bool fp32) {
    std::lock_guard<std::mutex> lock(m.planMutex);
    StreamSet& ps = m.ps[fp32];
    if (!ps.tried) {
        build_stream(m, {m.nParts, m.partRowStart, m.partRows, m.partLevStart, m.partLevPtr, m.localCol}, false, fp32, ps);
        ps.upload();
        ps.tried = true;
    }
    return ps;
}

// Partition-local level of every cell (longest chain of in-partition lower
// neighbours, cells in increasing index); returns the deepest level count.
static int partition_levels(const Mesh& m, std::vector<int32_t>& lev) {
    int deepest = 0;
    for (int c = 0; c < m.nC; ++c) {
        int l = 0;
        for (int s = m.rowPtr[c]; s < m.slotDiag[c]; ++s)
            if (m.part[m.cols[s]] == m.part[c]) l = std::max(l, lev[m.cols[s]] + 1);
        lev[c] = l;
        deepest = std::max(deepest, l + 1);
    }
    return deepest;
}

// The apply of a partition is a chain of its levels; a partition deeper than
// maxLevels is cut at its middle level (the cells of the upper half form a
// new partition), until none is.
static void split_deep_partitions(Mesh& m, int maxLevels) {
    std::vector<int32_t> lev(m.nC, 0);
    for (int pass = 0; pass < 16; ++pass) {
        partition_levels(m, lev);
        std::vector<int> depth(m.nParts, 0);
        for (int c = 0; c < m.nC; ++c) depth[m.part[c]] = std::max(depth[m.part[c]], lev[c] + 1);
        std::vector<int> newId(m.nParts, -1);
        int added = 0;
        for (int p = 0; p < m.nParts; ++p)
            if (depth[p] > maxLevels) newId[p] = m.nParts + added++;
        if (!added) return;
        for (int c = 0; c < m.nC; ++c) {
            const int p = m.part[c];
            if (newId[p] >= 0 && lev[c] >= depth[p] / 2) m.part[c] = newId[p];
        }
        m.nParts += added;
    }
}

// Rows of each partition in (partition-local level, cell) order, the level
// offsets, and per block-CSR slot the partition-local column (-1 outside).
static void order_partitions(const Mesh& m, const std::vector<int32_t>& part, int nParts, PartSet& ps) {
    const int n = m.nC;
    std::vector<std::vector<int>> cellsOf(nParts);
    for (int c = 0; c < n; ++c) cellsOf[part[c]].push_back(c);
    std::vector<int32_t> lev(n, 0), local(n, -1);
    ps.nParts = nParts;
    ps.rowStart.assign(nParts + 1, 0);
    ps.levStart.assign(nParts + 1, 0);
    ps.rows.clear();
    ps.levPtr.clear();
    ps.maxRows = 0;
    ps.maxLevels = 0;
    for (int p = 0; p < nParts; ++p) {
        const std::vector<int>& cs = cellsOf[p];
        int nl = 0;
        for (int c : cs) {
            int l = 0;
            for (int s = m.rowPtr[c]; s < m.slotDiag[c]; ++s)
                if (part[m.cols[s]] == p) l = std::max(l, lev[m.cols[s]] + 1);
            lev[c] = l;
            nl = std::max(nl, l + 1);
        }
        std::vector<int> order(cs.begin(), cs.end());
        std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return lev[a] < lev[b]; });
        ps.rowStart[p + 1] = ps.rowStart[p] + (int)order.size();
        for (size_t k = 0; k < order.size(); ++k) {
            local[order[k]] = (int)k;
            ps.rows.push_back(order[k]);
        }
        // level offsets (absolute positions in rows)
        int pos = ps.rowStart[p];
        for (int l = 0; l < nl; ++l) {
            ps.levPtr.push_back(pos);
            while (pos < ps.rowStart[p + 1] && lev[ps.rows[pos]] == l) ++pos;
        }
        ps.levPtr.push_back(ps.rowStart[p + 1]);
        ps.levStart[p + 1] = (int)ps.levPtr.size();
        ps.maxRows = std::max(ps.maxRows, (int)order.size());
        ps.maxLevels = std::max(ps.maxLevels, nl);
    }
    ps.localCol.assign(m.nnzb, -1);
    ps.maxOff = 0;
    for (int c = 0; c < n; ++c) {
        int off = -1;
        for (int s = m.rowPtr[c]; s < m.rowPtr[c + 1]; ++s)
            if (part[m.cols[s]] == part[c]) {
                ps.localCol[s] = local[m.cols[s]];
                ++off;
            }
        ps.maxOff = std::max(ps.maxOff, off);
    }
}

// Tiles of the natural-order ILU(0).  Every lower neighbour of a row gets a
// class by how far back in the numbering it lies (next to it, or one of two
// groups of larger distances; i, j and k neighbours of a structured numbering);
// coordinate c of a row is the largest number of class-c steps on a chain of
// dependencies ending there.  All three never decrease along a dependency, so
// boxes in them form an acyclic tile graph whatever the mesh, and on a
// structured numbering they are boxes of its indices, the shape with the
// shortest chain of tiles.  A box of more than kTileCells rows is cut by level.
static void build_tiles(const Mesh& m, TileSet& ts) {
    const int n = m.nC;
    double lmin = 1e300, lmax = 0.0;
    std::vector<double> hist(32 * 8, 0.0);
    auto bin_of = [&](int d) { return std::min((int)hist.size() - 1, (int)(8.0 * std::log2((double)d))); };
    for (int i = 0; i < n; ++i)
        for (int s = m.rowPtr[i]; s < m.slotDiag[i]; ++s) {
            const int d = i - m.cols[s];
            if (d <= 1) continue;
            hist[bin_of(d)] += 1.0;
            lmin = std::min(lmin, std::log2((double)d));
            lmax = std::max(lmax, std::log2((double)d));
        }
    // two groups of log(distance) by 2-means; one group when they are within a factor of four
    double c0 = lmin, c1 = lmax;
    for (int it = 0; it < 20; ++it) {
        double s0 = 0, w0 = 0, s1 = 0, w1 = 0;
        for (size_t q = 0; q < hist.size(); ++q) {
            const double x = (q + 0.5) / 8.0;
            if (std::fabs(x - c0) <= std::fabs(x - c1)) { s0 += hist[q] * x; w0 += hist[q]; }
            else { s1 += hist[q] * x; w1 += hist[q]; }
        }
        if (w0 > 0) c0 = s0 / w0;
        if (w1 > 0) c1 = s1 / w1;
    }
    const bool three = c1 - c0 > 2.0;
    const double cut = 0.5 * (c0 + c1);
    std::vector<int32_t> x(3 * (size_t)n, 0), lev(n, 0);
    for (int i = 0; i < n; ++i)
        for (int s = m.rowPtr[i]; s < m.slotDiag[i]; ++s) {
            const int j = m.cols[s], d = i - j;
            const int cl = d <= 1 ? 0 : (three && std::log2((double)d) > cut ? 2 : 1);
            for (int c = 0; c < 3; ++c) x[3 * (size_t)i + c] = std::max(x[3 * (size_t)i + c], x[3 * (size_t)j + c] + (c == cl ? 1 : 0));
            lev[i] = std::max(lev[i], lev[j] + 1);
        }
    // Box sides.  Small boxes hand on sooner, but more of them cross more halos (1-2 us
    // each) and the whole mesh's worth must be held by 256 workgroups.  Measured, step
    // of a 321 k wing: 8x8x8 45.9 ms, 6x6x6 38.1, 8x8x4 35.7, 8x4x2 32.6, 4x4x4 31.0,
    // 8x4x4 30.9; RAE2822 (two classes): 16x16 and 8x8 20.8, 16x8 18.9.
    const int T[3] = {three ? 8 : 16, three ? 4 : 8, 4};
    std::vector<int32_t> tile(n, 0);
    int nT = 0;
    if (n <= kPartCells) {
        nT = n ? 1 : 0;
    } else {
        // cells by (wavefront of boxes, box, level, index)
        struct Key {
            int32_t sum, k0, k1, k2, lev, c;
        };
        std::vector<Key> key(n);
        for (int i = 0; i < n; ++i) {
            const int32_t k0 = x[3 * (size_t)i] / T[0], k1 = x[3 * (size_t)i + 1] / T[1], k2 = x[3 * (size_t)i + 2] / T[2];
            key[i] = {k0 + k1 + k2, k0, k1, k2, lev[i], i};
        }
        std::sort(key.begin(), key.end(), [](const Key& a, const Key& b) {
            if (a.sum != b.sum) return a.sum < b.sum;
            if (a.k0 != b.k0) return a.k0 < b.k0;
            if (a.k1 != b.k1) return a.k1 < b.k1;
            if (a.k2 != b.k2) return a.k2 < b.k2;
            return a.lev != b.lev ? a.lev < b.lev : a.c < b.c;
        });
        int cnt = 0;
        for (int q = 0; q < n; ++q) {
            const Key &k = key[q], &p = key[q ? q - 1 : 0];
            const bool box = q == 0 || k.sum != p.sum || k.k0 != p.k0 || k.k1 != p.k1 || k.k2 != p.k2;
            if (box || cnt == kTileCells) {
                ++nT;
                cnt = 0;
            }
            tile[k.c] = nT - 1;
            ++cnt;
        }
    }
    order_partitions(m, tile, nT, ts);
    // columns outside the tile: halo cells, each once per tile and sweep
    ts.haloF.clear();
    ts.haloB.clear();
    ts.maxSlots = 0;
    ts.haloFStart.assign(1, 0);
    ts.needF.assign(ts.levPtr.size(), 0);
    ts.haloBStart.assign(1, 0);
    std::vector<int32_t> seen(n, -1), slot(n, 0);
    for (int sweep = 0; sweep < 2; ++sweep) {
        std::vector<int32_t>&hs = sweep ? ts.haloBStart : ts.haloFStart, &h = sweep ? ts.haloB : ts.haloF;
        std::fill(seen.begin(), seen.end(), -1);
        for (int t = 0; t < nT; ++t) {
            const int rs = ts.rowStart[t], nr = ts.rowStart[t + 1] - rs;
            for (int q0 = 0; q0 < nr; ++q0) {  // in the sweep's order of levels
                const int i = ts.rows[sweep ? rs + nr - 1 - q0 : rs + q0];
                const int s0 = sweep ? m.slotDiag[i] + 1 : m.rowPtr[i], s1 = sweep ? m.rowPtr[i + 1] : m.slotDiag[i];
                for (int s = s0; s < s1; ++s) {
                    const int j = m.cols[s];
                    if (tile[j] == t) continue;
                    if (seen[j] != t) {
                        seen[j] = t;
                        slot[j] = nr + (int)h.size() - hs.back();
                        h.push_back(j);
                    }
                    ts.localCol[s] = slot[j];
                }
            }
            hs.push_back((int32_t)h.size());
            ts.maxSlots = std::max(ts.maxSlots, nr + hs[t + 1] - hs[t]);
            if (sweep) continue;
            int need = 0;
            for (int L = ts.levStart[t]; L + 1 < ts.levStart[t + 1]; ++L) {
                for (int q = ts.levPtr[L]; q < ts.levPtr[L + 1]; ++q)
                    for (int s = m.rowPtr[ts.rows[q]]; s < m.slotDiag[ts.rows[q]]; ++s)
                        need = std::max(need, ts.localCol[s] - nr + 1);
                ts.needF[L] = need;
            }
        }
    }
}

// Whether the sweeps go by tiles or by one launch per level, from what each is
// expected to cost (us, both sweeps).  Tiles: the longest chain of tiles, each
// 0.7 per level and 1.6 per 256 halo values (the halo wavefront asks for those one
// window after the other).  Levels: 4 per launch and 0.5 per 100 rows of a level.
// A structured numbering has many levels and thin halos; cells numbered at random
// have a dozen levels, and tiles whose halo is several times the tile.  Step of
// 20 vectors FP64, levels / tiles, with the two predictions per sweep: wing
// 67.6 k 44.5 / 7.9 ms (906, 312 us), the same in the order of 4x4x4 tiles 45.2 / 32.4
// (906, 641), hybrid airfoil 9.1 k numbered at random within 100 cells 31.8 / 16.3
// (614, 425); 2.7 k quads at random 3.8 / 5.9 (62, 129), 10.8 k at random within 1000
// cells 6.1 / 10.1 (122, 262), 1.5 k tetrahedra 2.8 / 3.2 (44, 49).
bool tiles_pay(const Mesh& m, const TileSet& ts) {
    if (ts.nParts <= 1) return true;  // no halo: one workgroup and no launches between the levels
    std::vector<int32_t> tile(m.nC);
    for (int t = 0; t < ts.nParts; ++t)
        for (int q = ts.rowStart[t]; q < ts.rowStart[t + 1]; ++q) tile[ts.rows[q]] = t;
    double tiles = 0.0;
    for (int sweep = 0; sweep < 2; ++sweep) {
        const std::vector<int32_t>&hs = sweep ? ts.haloBStart : ts.haloFStart, &h = sweep ? ts.haloB : ts.haloF;
        std::vector<double> end(ts.nParts, 0.0);
        double longest = 0.0;
        for (int k = 0; k < ts.nParts; ++k) {
            const int t = sweep ? ts.nParts - 1 - k : k;
            double begin = 0.0;
            for (int q = hs[t]; q < hs[t + 1]; ++q) begin = std::max(begin, end[tile[h[q]]]);
            end[t] = begin + 0.7 * (ts.levStart[t + 1] - ts.levStart[t] - 1) + 1.6 * ((5 * (hs[t + 1] - hs[t]) + 255) / 256);
            longest = std::max(longest, end[t]);
        }
        tiles += longest;
    }
    return tiles <= 4.0 * (m.nLevL + m.nLevU) + 2 * 0.005 * m.nC;
}

TileSet& mesh_tiles(Mesh& m, bool fp32) {
    std::lock_guard<std::mutex> lock(m.planMutex);
    TileSet& ts = m.tiles;
    if (!ts.tried) {
        build_tiles(m, ts);
        ts.d_rowStart.upload(ts.rowStart);
        ts.d_rows.upload(ts.rows);
        ts.d_haloFStart.upload(ts.haloFStart);
        ts.d_haloF.upload(ts.haloF);
        ts.d_haloBStart.upload(ts.haloBStart);
        ts.d_haloB.upload(ts.haloB);
        ts.d_needF.upload(ts.needF);
        ts.d_levStart.upload(ts.levStart);
        ts.d_levPtr.upload(ts.levPtr);
        // the tile's vector and its halo, and where the vector's entries belong, next to the
        // ring in 160 KB of LDS (16-bit columns), and the sweeps the faster by it
        ts.ok = 40 * (size_t)ts.maxSlots + 20 * kTileCells + stream_ring(false) + 4096 <= 160 * 1024 && tiles_pay(m, ts);
        ts.tried = true;
    }
    StreamSet& ps = ts.ps[fp32];
    if (!ps.tried && ts.ok) {
        build_stream(m, {ts.nParts, ts.rowStart, ts.rows, ts.levStart, ts.levPtr, ts.localCol}, true, fp32, ps);
        ps.upload();
    }
    ps.tried = true;
    return ts;
}

// Partitions for the block-Jacobi ILU(0): couplings between partitions are
// dropped, inside a partition the factor is the natural-order ILU(0) of the
// partition's diagonal block, scheduled by local levels.  The RCB boxes as
// they come (at most maxCells cells, no level cut) also drive the
// Spalart-Allmaras Gauss-Seidel sweep: a mesh of at most maxCells cells is
// one box, i.e. the serial natural-order sweep.
void build_partitions(Mesh& m, int maxCells) {
    const int n = m.nC;
    m.part.assign(n, 0);
    std::vector<int> idx(n);
    std::iota(idx.begin(), idx.end(), 0);
    m.nParts = 0;
    rcb(m.C, idx, 0, n, maxCells, m.part, m.nParts);
    m.saPart = m.part;
    order_partitions(m, m.saPart, m.nParts, m.sa);
    split_deep_partitions(m, kMaxPartLevels);
    PartSet ps;
    order_partitions(m, m.part, m.nParts, ps);
    m.partRowStart.swap(ps.rowStart);
    m.partRows.swap(ps.rows);
    m.partLevStart.swap(ps.levStart);
    m.partLevPtr.swap(ps.levPtr);
    m.localCol.swap(ps.localCol);
    m.maxPartRows = ps.maxRows;
    m.maxPartLevels = ps.maxLevels;
}

void mesh_build(Mesh& m, const rdst_mesh_desc* d, const rdst_mesh_geometry* g) {
    if (!d || d->n_cells <= 0 || d->n_faces <= 0 || d->n_internal_faces < 0 || d->n_internal_faces > d->n_faces)
        throw ArgError("rdst_mesh_create: bad mesh sizes");
    if (!d->points || !d->face_offsets || !d->face_points || !d->owner || (d->n_internal_faces && !d->neighbour))
        throw ArgError("rdst_mesh_create: null array");
    const int nFaces = d->n_faces, nInt = d->n_internal_faces, nCells = d->n_cells;
    for (int f = 0; f < nFaces; ++f) {
        if (d->owner[f] < 0 || d->owner[f] >= nCells) throw ArgError("rdst_mesh_create: owner out of range");
        if (d->face_offsets[f + 1] - d->face_offsets[f] < 3) throw ArgError("rdst_mesh_create: face with < 3 points");
    }
    for (int f = 0; f < nInt; ++f) {
        if (d->neighbour[f] < 0 || d->neighbour[f] >= nCells) throw ArgError("rdst_mesh_create: neighbour out of range");
        if (d->neighbour[f] <= d->owner[f]) throw ArgError("rdst_mesh_create: internal faces must have owner < neighbour");
    }
    m.patches.assign(d->patches, d->patches + d->n_patches);
    m.nPatches = d->n_patches;
    m.nC = nCells;
    m.nI = nInt;

    // --- face centres and areas
    std::vector<P3> fSf(nFaces), fCf(nFaces);
    std::vector<double> fmag(nFaces);
    auto pt = [&](int i) { return P3{d->points[3 * i], d->points[3 * i + 1], d->points[3 * i + 2]}; };
    for (int f = 0; f < nFaces; ++f) {
        const int s = d->face_offsets[f], n = d->face_offsets[f + 1] - s;
        const int32_t* fp = d->face_points + s;
        for (int k = 0; k < n; ++k)
            if (fp[k] < 0 || fp[k] >= d->n_points) throw ArgError("rdst_mesh_create: face point out of range");
        if (n == 3) {
            P3 p0 = pt(fp[0]), p1 = pt(fp[1]), p2 = pt(fp[2]);
            fCf[f] = scl(1.0 / 3.0, add(add(p0, p1), p2));
            fSf[f] = scl(0.5, crossp(sub(p1, p0), sub(p2, p0)));
        } else {
            P3 c = pt(fp[0]);
            for (int k = 1; k < n; ++k) c = add(c, pt(fp[k]));
            c = {c.x / n, c.y / n, c.z / n};
            P3 sN = {0, 0, 0}, sAc = {0, 0, 0};
            double sA = 0;
            for (int k = 0; k < n; ++k) {
                P3 a = pt(fp[k]), b = pt(fp[(k + 1) % n]);
                P3 cc = add(add(a, b), c);
                P3 nv = crossp(sub(b, a), sub(c, a));
                double ar = norm(nv);
                sN = add(sN, nv);
                sA += ar;
                sAc = add(sAc, scl(ar, cc));
            }
            if (sA < 1e-150) {
                fCf[f] = c;
                fSf[f] = {0, 0, 0};
            } else {
                P3 t = scl(1.0 / 3.0, sAc);  // (1/3)*sumAc/sumA, left to right
                fCf[f] = {t.x / sA, t.y / sA, t.z / sA};
                fSf[f] = scl(0.5, sN);
            }
        }
        fmag[f] = norm(fSf[f]);
    }
    // --- wall triangles (the surface the wall distance is measured to): each
    // wall face fanned from the mean of its points, one triangle per edge, so
    // a warped quad is followed on both of its diagonals (a fan from one
    // corner can pass a first-cell centre at many times its height)
    for (int pi = 0; pi < d->n_patches; ++pi) {
        const rdst_patch& pa = d->patches[pi];
        if (pa.type != RDST_PATCH_WALL) continue;
        if (pa.start < nInt || pa.size < 0 || pa.start + pa.size > nFaces) throw ArgError("rdst_mesh_create: patch range");
        for (int f = pa.start; f < pa.start + pa.size; ++f) {
            const int s = d->face_offsets[f], n = d->face_offsets[f + 1] - s;
            const int32_t* fp = d->face_points + s;
            double c[3] = {d->points[3 * fp[0]], d->points[3 * fp[0] + 1], d->points[3 * fp[0] + 2]};
            for (int k = 1; k < n; ++k)
                for (int x = 0; x < 3; ++x) c[x] = c[x] + d->points[3 * fp[k] + x];
            for (int x = 0; x < 3; ++x) c[x] = c[x] / n;
            for (int k = 0; k < n; ++k) {
                for (int x = 0; x < 3; ++x) m.wallTri.push_back(c[x]);
                for (int q : {fp[k], fp[(k + 1) % n]})
                    for (int x = 0; x < 3; ++x) m.wallTri.push_back(d->points[3 * q + x]);
            }
        }
    }
    // --- cell centres and volumes
    std::vector<P3> cEst(nCells, P3{0, 0, 0}), cC(nCells, P3{0, 0, 0});
    std::vector<int> nCF(nCells, 0);
    std::vector<double> vol(nCells, 0.0);
    for (int f = 0; f < nFaces; ++f) { cEst[d->owner[f]] = add(cEst[d->owner[f]], fCf[f]); nCF[d->owner[f]]++; }
    for (int f = 0; f < nInt; ++f) { cEst[d->neighbour[f]] = add(cEst[d->neighbour[f]], fCf[f]); nCF[d->neighbour[f]]++; }
    for (int c = 0; c < nCells; ++c) cEst[c] = {cEst[c].x / nCF[c], cEst[c].y / nCF[c], cEst[c].z / nCF[c]};
    for (int f = 0; f < nFaces; ++f) {
        int o = d->owner[f];
        double v3 = std::max(dotp(fSf[f], sub(fCf[f], cEst[o])), 1e-300);
        P3 pc = add(scl(0.75, fCf[f]), scl(0.25, cEst[o]));
        cC[o] = add(cC[o], scl(v3, pc));
        vol[o] += v3;
    }
    for (int f = 0; f < nInt; ++f) {
        int nb = d->neighbour[f];
        double v3 = std::max(dotp(fSf[f], sub(cEst[nb], fCf[f])), 1e-300);
        P3 pc = add(scl(0.75, fCf[f]), scl(0.25, cEst[nb]));
        cC[nb] = add(cC[nb], scl(v3, pc));
        vol[nb] += v3;
    }
    for (int c = 0; c < nCells; ++c) {
        cC[c] = {cC[c].x / vol[c], cC[c].y / vol[c], cC[c].z / vol[c]};
        vol[c] *= (1.0 / 3.0);
        if (!(vol[c] > 0)) throw ArgError("rdst_mesh_create: non-positive cell volume");
    }
    // --- compacted boundary faces (empty patches have fvPatch size 0)
    m.bPatch.clear();
    m.bPolyFace.clear();
    for (int p = 0; p < m.nPatches; ++p) {
        const rdst_patch& pp = m.patches[p];
        if (pp.start < nInt || pp.start + pp.size > nFaces) throw ArgError("rdst_mesh_create: patch range");
        if (pp.type == RDST_PATCH_EMPTY) continue;
        for (int i = 0; i < pp.size; ++i) { m.bPatch.push_back(p); m.bPolyFace.push_back(pp.start + i); }
    }
    m.nB = (int)m.bPatch.size();
    m.nF = m.nI + m.nB;
    const int nF = m.nF;
    m.Sf.resize(3 * (size_t)nF); m.Cf.resize(3 * (size_t)nF); m.magSf.resize(nF); m.w.assign(nF, 1.0); m.dc.resize(nF);
    m.owner.resize(nF); m.neigh.assign(d->neighbour, d->neighbour + nInt);
    for (int k = 0; k < nF; ++k) {
        int f = k < nInt ? k : m.bPolyFace[k - nInt];
        m.Sf[3 * k] = fSf[f].x; m.Sf[3 * k + 1] = fSf[f].y; m.Sf[3 * k + 2] = fSf[f].z;
        m.Cf[3 * k] = fCf[f].x; m.Cf[3 * k + 1] = fCf[f].y; m.Cf[3 * k + 2] = fCf[f].z;
        m.magSf[k] = fmag[f];
        m.owner[k] = d->owner[f];
    }
    m.C.resize(3 * (size_t)nCells); m.V = vol;
    for (int c = 0; c < nCells; ++c) { m.C[3 * c] = cC[c].x; m.C[3 * c + 1] = cC[c].y; m.C[3 * c + 2] = cC[c].z; }
    for (int f = 0; f < nInt; ++f) {
        P3 sf = fSf[f], cf = fCf[f], co = cC[d->owner[f]], cn = cC[d->neighbour[f]];
        double dOwn = std::fabs(dotp(sf, sub(cf, co)));
        double dNei = std::fabs(dotp(sf, sub(cn, cf)));
        m.w[f] = dNei / (dOwn + dNei);
        P3 delta = sub(cn, co);
        P3 ua = {sf.x / fmag[f], sf.y / fmag[f], sf.z / fmag[f]};
        m.dc[f] = 1.0 / std::max(dotp(ua, delta), 0.05 * norm(delta));
    }
    for (int b = 0; b < m.nB; ++b) {
        int f = m.bPolyFace[b];
        P3 delta = sub(fCf[f], cC[d->owner[f]]);
        m.dc[nInt + b] = 1.0 / norm(delta);
    }
    // the host fvMesh's own geometry, kept bit for bit (faces of empty
    // patches, which have no fvPatch faces, are dropped)
    if (g) {
        if (!g->Sf || !g->Cf || !g->C || !g->V || !g->weights || !g->delta_coeffs)
            throw ArgError("rdst_mesh_create_geometry: null geometry array");
        for (int k = 0; k < nF; ++k) {
            const int f = k < nInt ? k : m.bPolyFace[k - nInt];
            for (int x = 0; x < 3; ++x) {
                m.Sf[3 * k + x] = g->Sf[3 * (size_t)f + x];
                m.Cf[3 * k + x] = g->Cf[3 * (size_t)f + x];
            }
            m.magSf[k] = g->mag_sf ? g->mag_sf[f] : std::sqrt(m.Sf[3 * k] * m.Sf[3 * k] + m.Sf[3 * k + 1] * m.Sf[3 * k + 1] +
                                                             m.Sf[3 * k + 2] * m.Sf[3 * k + 2]);
            m.w[k] = k < nInt ? g->weights[f] : 1.0;
            m.dc[k] = g->delta_coeffs[f];
            if (!(m.magSf[k] > 0)) throw ArgError("rdst_mesh_create_geometry: face of zero area");
        }
        for (int c = 0; c < nCells; ++c) {
            for (int x = 0; x < 3; ++x) m.C[3 * (size_t)c + x] = g->C[3 * (size_t)c + x];
            m.V[c] = g->V[c];
            if (!(m.V[c] > 0)) throw ArgError("rdst_mesh_create_geometry: non-positive cell volume");
        }
    }
    // correction vectors n - d deltaCoeffs of the corrected snGrad
    m.corr.resize(3 * (size_t)nInt);
    for (int f = 0; f < nInt; ++f) {
        const int o = d->owner[f], nb = d->neighbour[f];
        P3 delta = {m.C[3 * (size_t)nb] - m.C[3 * (size_t)o], m.C[3 * (size_t)nb + 1] - m.C[3 * (size_t)o + 1],
                    m.C[3 * (size_t)nb + 2] - m.C[3 * (size_t)o + 2]};
        P3 ua = {m.Sf[3 * f] / m.magSf[f], m.Sf[3 * f + 1] / m.magSf[f], m.Sf[3 * f + 2] / m.magSf[f]};
        P3 cv = sub(ua, scl(m.dc[f], delta));
        m.corr[3 * f] = cv.x; m.corr[3 * f + 1] = cv.y; m.corr[3 * f + 2] = cv.z;
    }

    // --- ELL cell->face map, faces of a cell in surface-field order
    std::vector<int> deg(nCells, 0);
    for (int f = 0; f < nInt; ++f) { deg[m.owner[f]]++; deg[m.neigh[f]]++; }
    for (int b = 0; b < m.nB; ++b) deg[m.owner[nInt + b]]++;
    m.ellW = nCells ? *std::max_element(deg.begin(), deg.end()) : 0;
    const size_t E = (size_t)m.ellW * nCells;
    m.ellCode.assign(E, (ELL_NONE << 30));
    m.ellFace.assign(E, -1);
    std::vector<int> fill(nCells, 0);
    // faces in increasing surface-field index: internal faces then boundary
    for (int f = 0; f < nInt; ++f) {
        int o = m.owner[f], nb = m.neigh[f];
        size_t eo = (size_t)fill[o]++ * nCells + o;
        m.ellCode[eo] = (ELL_OWNER << 30) | (uint32_t)nb;
        m.ellFace[eo] = f;
        size_t en = (size_t)fill[nb]++ * nCells + nb;
        m.ellCode[en] = (ELL_NEIGH << 30) | (uint32_t)o;
        m.ellFace[en] = f;
    }
    for (int b = 0; b < m.nB; ++b) {
        int c = m.owner[nInt + b];
        size_t e = (size_t)fill[c]++ * nCells + c;
        m.ellCode[e] = (ELL_BOUNDARY << 30) | (uint32_t)b;
        m.ellFace[e] = nInt + b;
    }

    // --- block-CSR (owner/neighbour-sorted): row i holds the diagonal, the
    // upper coefficients of faces it owns (column = neighbour) and the lower
    // coefficients of faces it neighbours (column = owner), columns ascending
    std::vector<std::vector<std::pair<int, int>>> rows(nCells);  // (col, tag) tag: -1 diag, 2f upper, 2f+1 lower
    for (int c = 0; c < nCells; ++c) rows[c].push_back({c, -1});
    for (int f = 0; f < nInt; ++f) {
        rows[m.owner[f]].push_back({m.neigh[f], 2 * f});
        rows[m.neigh[f]].push_back({m.owner[f], 2 * f + 1});
    }
    m.rowPtr.assign(nCells + 1, 0);
    for (int c = 0; c < nCells; ++c) {
        std::sort(rows[c].begin(), rows[c].end());
        m.rowPtr[c + 1] = m.rowPtr[c] + (int)rows[c].size();
    }
    m.nnzb = m.rowPtr[nCells];
    m.cols.resize(m.nnzb);
    m.slotUpper.resize(nInt); m.slotLower.resize(nInt); m.slotDiag.resize(nCells);
    for (int c = 0; c < nCells; ++c)
        for (size_t k = 0; k < rows[c].size(); ++k) {
            int s = m.rowPtr[c] + (int)k;
            m.cols[s] = rows[c][k].first;
            int tag = rows[c][k].second;
            if (tag == -1) m.slotDiag[c] = s;
            else if ((tag & 1) == 0) m.slotUpper[tag >> 1] = s;
            else m.slotLower[tag >> 1] = s;
        }
    for (int c = 0; c < nCells; ++c)
        for (int s = m.rowPtr[c] + 1; s < m.rowPtr[c + 1]; ++s)
            if (m.cols[s] == m.cols[s - 1]) throw ArgError("rdst_mesh_create: duplicate internal face between two cells");

    // --- ELL slot of the off-diagonal block each cell writes: the owner
    // writes the lower coefficient (row neighbour, column owner), the
    // neighbour writes the upper one (row owner, column neighbour)
    m.ellSlot.assign(E, -1);
    for (size_t e = 0; e < E; ++e) {
        uint32_t kind = m.ellCode[e] >> 30;
        int f = m.ellFace[e];
        if (kind == ELL_OWNER) m.ellSlot[e] = m.slotLower[f];
        else if (kind == ELL_NEIGH) m.ellSlot[e] = m.slotUpper[f];
    }

    // --- greedy face colouring in face order (deterministic)
    m.faceColour.assign(nInt, -1);
    {
        std::vector<uint64_t> used(nCells, 0);
        int maxc = 0;
        for (int f = 0; f < nInt; ++f) {
            uint64_t u = used[m.owner[f]] | used[m.neigh[f]];
            int col = 0;
            while (col < 64 && (u >> col & 1ull)) ++col;
            if (col >= 64) throw ArgError("rdst_mesh_create: face colouring needs more than 64 colours");
            m.faceColour[f] = col;
            used[m.owner[f]] |= 1ull << col;
            used[m.neigh[f]] |= 1ull << col;
            maxc = std::max(maxc, col + 1);
        }
        m.nColours = maxc;
    }
    // --- greedy cell colouring (distance-1) in cell order
    m.cellColour.assign(nCells, -1);
    {
        int maxc = 0;
        for (int c = 0; c < nCells; ++c) {
            uint64_t u = 0;
            for (int s = m.rowPtr[c]; s < m.rowPtr[c + 1]; ++s) {
                int j = m.cols[s];
                if (j != c && m.cellColour[j] >= 0) u |= 1ull << m.cellColour[j];
            }
            int col = 0;
            while (col < 64 && (u >> col & 1ull)) ++col;
            if (col >= 64) throw ArgError("rdst_mesh_create: cell colouring needs more than 64 colours");
            m.cellColour[c] = col;
            maxc = std::max(maxc, col + 1);
        }
        m.nCellColours = maxc;
    }
    // --- level sets of the natural-order triangular sweeps
    m.levL.assign(nCells, 0);
    for (int c = 0; c < nCells; ++c) {
        int lv = 0;
        for (int s = m.rowPtr[c]; s < m.rowPtr[c + 1]; ++s)
            if (m.cols[s] < c) lv = std::max(lv, m.levL[m.cols[s]] + 1);
        m.levL[c] = lv;
    }
    m.levU.assign(nCells, 0);
    for (int c = nCells - 1; c >= 0; --c) {
        int lv = 0;
        for (int s = m.rowPtr[c]; s < m.rowPtr[c + 1]; ++s)
            if (m.cols[s] > c) lv = std::max(lv, m.levU[m.cols[s]] + 1);
        m.levU[c] = lv;
    }
    auto bucket = [&](const std::vector<int32_t>& lev, int& nLev, std::vector<int32_t>& ptr, std::vector<int32_t>& rowsOut) {
        nLev = nCells ? *std::max_element(lev.begin(), lev.end()) + 1 : 0;
        ptr.assign(nLev + 1, 0);
        for (int c = 0; c < nCells; ++c) ptr[lev[c] + 1]++;
        for (int l = 0; l < nLev; ++l) ptr[l + 1] += ptr[l];
        rowsOut.resize(nCells);
        std::vector<int> pos(ptr.begin(), ptr.end() - 1);
        for (int c = 0; c < nCells; ++c) rowsOut[pos[lev[c]]++] = c;
    };
    bucket(m.levL, m.nLevL, m.levLPtr, m.levLRows);
    bucket(m.levU, m.nLevU, m.levUPtr, m.levURows);
    auto runs = [&](const std::vector<int32_t>& ptr, int nLev, std::vector<LevelRun>& out) {
        out.clear();
        for (int L = 0; L < nLev;) {
            const bool small = ptr[L + 1] - ptr[L] <= kIluSegRows;
            int E = L + 1;
            while (E < nLev && ((ptr[E + 1] - ptr[E] <= kIluSegRows) == small)) ++E;
            out.push_back({L, E, small});
            L = E;
        }
    };
    runs(m.levLPtr, m.nLevL, m.runL);
    runs(m.levUPtr, m.nLevU, m.runU);
    build_partitions(m, kPartCells);
    // sliced ELL (64 rows per slice)
    m.nSlices = (nCells + 63) / 64;
    m.sellPtr.assign(m.nSlices + 1, 0);
    m.sellWidth.assign(m.nSlices, 0);
    for (int sl = 0; sl < m.nSlices; ++sl) {
        int w = 0;
        for (int r = 64 * sl; r < std::min(nCells, 64 * sl + 64); ++r) w = std::max(w, m.rowPtr[r + 1] - m.rowPtr[r]);
        m.sellWidth[sl] = w;
        m.sellPtr[sl + 1] = m.sellPtr[sl] + 64 * (int64_t)w;
    }
    m.sellBlocks = m.sellPtr[m.nSlices];
    m.sellCol.assign(m.sellBlocks, -1);
    m.sellOfSlot.assign(m.nnzb, 0);
    for (int r = 0; r < nCells; ++r) {
        const int sl = r / 64, lane = r % 64;
        for (int s = m.rowPtr[r]; s < m.rowPtr[r + 1]; ++s) {
            const int p = s - m.rowPtr[r];
            const int64_t pos = m.sellPtr[sl] + 64 * (int64_t)p + lane;
            m.sellCol[pos] = m.cols[s];
            m.sellOfSlot[s] = 25 * (m.sellPtr[sl] + 64 * (int64_t)p) + lane;
        }
        // padding blocks point at the row itself with zero values
        for (int p = m.rowPtr[r + 1] - m.rowPtr[r]; p < m.sellWidth[sl]; ++p) m.sellCol[m.sellPtr[sl] + 64 * (int64_t)p + lane] = r;
    }
    for (int64_t q = 0; q < m.sellBlocks; ++q)
        if (m.sellCol[q] < 0) m.sellCol[q] = 0;  // lanes past the last row of the last slice
}

void mesh_upload(Mesh& m) {
    std::lock_guard<std::mutex> lock(m.planMutex);
    if (m.uploaded) return;
    const int nC = m.nC, nF = m.nF, W = m.ellW;
    m.d_owner.upload(m.owner.data(), m.nI);
    m.d_neigh.upload(m.neigh);
    std::vector<int32_t> bcell(m.nB), bwall(m.nB);
    for (int b = 0; b < m.nB; ++b) {
        bcell[b] = m.owner[m.nI + b];
        bwall[b] = m.patches[m.bPatch[b]].type == RDST_PATCH_WALL ? 1 : 0;
    }
    m.d_bcell.upload(bcell);
    m.d_bpatch.upload(m.bPatch);
    m.d_bWall.upload(bwall);
    std::vector<double> soa(3 * (size_t)nF);
    for (int k = 0; k < nF; ++k)
        for (int d = 0; d < 3; ++d) soa[(size_t)d * nF + k] = m.Sf[3 * (size_t)k + d];
    m.d_Sf.upload(soa);
    for (int k = 0; k < nF; ++k)
        for (int d = 0; d < 3; ++d) soa[(size_t)d * nF + k] = m.Cf[3 * (size_t)k + d];
    m.d_Cf.upload(soa);
    m.d_magSf.upload(m.magSf);
    m.d_w.upload(m.w);
    m.d_dc.upload(m.dc);
    m.d_V.upload(m.V);
    {
        std::vector<double> cs(3 * (size_t)m.nC);
        for (int c = 0; c < m.nC; ++c)
            for (int d = 0; d < 3; ++d) cs[(size_t)d * m.nC + c] = m.C[3 * (size_t)c + d];
        m.d_C.upload(cs);
    }
    m.d_ellCode.upload(m.ellCode);
    m.d_ellFace.upload(m.ellFace);
    m.d_ellSlot.upload(m.ellSlot);
    const size_t E = (size_t)W * nC;
    std::vector<double> esf(3 * E, 0.0), emag(E, 0.0), ew(E, 0.0), edc(E, 0.0), ecorr(3 * E, 0.0);
    for (size_t e = 0; e < E; ++e) {
        int k = m.ellFace[e];
        if (k < 0) continue;
        for (int d = 0; d < 3; ++d) esf[(size_t)d * E + e] = m.Sf[3 * (size_t)k + d];
        if (k < m.nI)
            for (int d = 0; d < 3; ++d) ecorr[(size_t)d * E + e] = m.corr[3 * (size_t)k + d];
        emag[e] = m.magSf[k];
        ew[e] = m.w[k];
        edc[e] = m.dc[k];
    }
    m.d_ellSf.upload(esf);
    m.d_ellMagSf.upload(emag);
    m.d_ellWt.upload(ew);
    m.d_ellDc.upload(edc);
    m.d_ellCorr.upload(ecorr);
    m.d_rowPtr.upload(m.rowPtr);
    m.d_cols.upload(m.cols);
    m.d_slotUpper.upload(m.slotUpper);
    m.d_slotLower.upload(m.slotLower);
    m.d_slotDiag.upload(m.slotDiag);
    m.d_levLRows.upload(m.levLRows);
    m.d_levLPtr.upload(m.levLPtr);
    m.d_levUPtr.upload(m.levUPtr);
    m.d_levURows.upload(m.levURows);
    m.d_partRowStart.upload(m.partRowStart);
    m.d_partRows.upload(m.partRows);
    m.d_partLevStart.upload(m.partLevStart);
    m.d_partLevPtr.upload(m.partLevPtr);
    m.d_localCol.upload(m.localCol);
    m.sa.d_rowStart.upload(m.sa.rowStart);
    m.sa.d_rows.upload(m.sa.rows);
    m.sa.d_levStart.upload(m.sa.levStart);
    m.sa.d_levPtr.upload(m.sa.levPtr);
    m.sa.d_localCol.upload(m.sa.localCol);
    m.d_sellPtr.upload(m.sellPtr);
    m.d_sellOfSlot.upload(m.sellOfSlot);
    m.d_sellWidth.upload(m.sellWidth);
    m.d_sellCol.upload(m.sellCol);
    m.uploaded = true;
}

}  // namespace rdst
