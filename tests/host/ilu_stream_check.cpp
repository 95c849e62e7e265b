// Host-side check of the ILU(0) record streams and of the tiles of the
// natural-order sweeps: replays the streams on the CPU with one number per
// block and compares with the plain sweeps over the block-CSR pattern.  Device
// memory is host memory here, and an allocation can be made to fail.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdlib>
#include <cstring>
#include <thread>

static std::atomic<int> g_mallocs{0};
static int g_mallocsLeft = -1;  // allocations until one fails (negative: none does)
static hipError_t g_last = hipSuccess;  // the runtime's last error
static hipError_t test_malloc(void** p, size_t n) {
    ++g_mallocs;
    if (g_mallocsLeft >= 0 && g_mallocsLeft-- == 0) return g_last = hipErrorOutOfMemory;
    *p = std::malloc(n);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
static hipError_t test_free(void* p) {
    std::free(p);
    return hipSuccess;
}
static hipError_t test_last() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
static hipError_t test_memcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
#define hipMalloc test_malloc
#define hipFree test_free
#define hipMemcpy test_memcpy
#define hipGetLastError test_last
#include "../../rhodst_amd/csrc/mesh_host.cpp"

#include <cstdio>

namespace rdst {
void set_error(const std::string&) {}
}  // namespace rdst
using namespace rdst;

static std::string g_what;
static int fail(const char* what, long a = 0, long b = 0) {
    char s[200];
    std::snprintf(s, sizeof s, "%s (%ld, %ld)", what, a, b);
    g_what = s;
    return 1;
}
static double coef(int s) { return 0.05 + 0.1 * ((s * 2654435761u) % 1000) / 1000.0; }
static double dinv(int c) { return 0.5 + 0.3 * ((c * 40503u) % 1000) / 1000.0; }

// one sweep's records over a partition's vector y (rows, then halo values)
static int replay(const Mesh& m, const StreamSet& ps, bool fp32, int q0, int q1, bool bwd, int own, int slots,
                  std::vector<double>& y) {
    const int blk = 25 * (fp32 ? 4 : 8);
    const bool tiles = !ps.need.empty();
    int need = 0;
    std::vector<char> done(own, 0);
    for (int q = q0; q < q1; ++q) {
        const int nr = ps.recRows[q + 1] - ps.recRows[q], b0 = ps.recBlk[q], nb = ps.recBlk[q + 1] - b0;
        if ((int)(ps.hdr[q] & 0xffff) != nr || nr < 1 || nr > kStreamRows) return fail("rows of a record", q, nr);
        if (nr * ps.ent + ((nb * blk + 15) & ~15) > stream_record(fp32)) return fail("record too large", q);
        std::vector<double> nw(nr);
        if (tiles && (ps.need[q] < need || ps.need[q] > slots - own)) return fail("halo count", q, ps.need[q]);
        if (tiles) need = ps.need[q];
        for (int j = 0; j < nr; ++j) {
            const uint16_t* e = ps.entries.data() + (size_t)(ps.recRows[q] + j) * (ps.ent / 2);
            const int t = e[0] / 5, cnt = e[1] >> 8;
            int b = b0 + (e[1] & 0xff);
            double a = y[t];
            double d = 1.0;
            if (bwd) {
                if (ps.src[b] >= 0) return fail("no Dinv first", q, j);
                d = dinv(-ps.src[b] - 1);
                if (ps.rowCell[b] != -ps.src[b] - 1) return fail("row cell", q, j);
                a *= d;
                ++b;
            }
            for (int k = 0; k < cnt; ++k, ++b) {
                if (b >= ps.recBlk[q + 1]) return fail("block outside its record", q, j);
                if (e[2 + k] % 5 || e[2 + k] / 5 >= slots) return fail("column out of range", q, e[2 + k]);
                if (e[2 + k] >= 5 * own && e[2 + k] / 5 - own >= need) return fail("a halo value before it is there", q, j);
                if (bwd != (ps.rowCell[b] >= 0)) return fail("sweep of a block", q, j);
                a -= d * coef(ps.src[b]) * y[e[2 + k] / 5];
            }
            nw[j] = a;
        }
        // rows of a record are independent: storing them together changes nothing
        for (int j = 0; j < nr; ++j) {
            const int t = ps.entries[(size_t)(ps.recRows[q] + j) * (ps.ent / 2)] / 5;
            y[t] = nw[j];
            ++done[t];
        }
    }
    for (int t = 0; t < own && tiles; ++t)
        if (done[t] != 1) return fail("a tile's row is not in one record", t);
    return 0;
}

static int check(const rdst_mesh_desc* desc, bool fp32, bool natural) {
    Mesh m;
    mesh_build(m, desc);
    const int n = m.nC;
    TileSet ts;
    StreamSet ps;
    std::vector<int32_t> part(m.part);
    if (natural) {
        build_tiles(m, ts);
        build_stream(m, {ts.nParts, ts.rowStart, ts.rows, ts.levStart, ts.levPtr, ts.localCol}, true, fp32, ps);
        std::fill(part.begin(), part.end(), 0);
    } else {
        build_stream(m, {m.nParts, m.partRowStart, m.partRows, m.partLevStart, m.partLevPtr, m.localCol}, false, fp32, ps);
    }
    if (ps.kmax == 0) return fail("not built");
    const int nP = natural ? ts.nParts : m.nParts;
    const std::vector<int32_t>&rowStart = natural ? ts.rowStart : m.partRowStart, &rows = natural ? ts.rows : m.partRows;
    // what the loader relies on: partitions at 1 KB, records inside the ring, three of them at once
    const int ring = stream_ring(fp32) / 16;
    const bool split = natural && nP > 1;  // each sweep a launch of its own
    for (int p = 0; p < nP; ++p)
        for (int part2 = 0; part2 < (split ? 2 : 1); ++part2) {
            const int q0 = part2 ? ps.recMid[p] : ps.recBeg[p], q1 = split && !part2 ? ps.recMid[p] : ps.recBeg[p + 1];
            if (q0 == q1) continue;
            const int64_t base = ps.start[q0];
            if (base % 64) return fail("start of a sweep", p);
            // the last 1 KB piece ends inside the stream
            if (16 * (size_t)(base + (ps.start[q1] - base + 63) / 64 * 64) > ps.bytes()) return fail("past the stream's end", p);
            int64_t off = 0;
            for (int q = q0; q < q1; ++q) {
                const int nr = ps.recRows[q + 1] - ps.recRows[q], nb = ps.recBlk[q + 1] - ps.recBlk[q];
                const int len = (nr * ps.ent + ((nb * 25 * (fp32 ? 4 : 8) + 15) & ~15)) / 16;
                if (off != ps.start[q] - base) return fail("distances do not add up", q);
                off += ps.hdr[q] >> 16;
                if ((int)((ps.start[q] - base) % ring) + len > ring) return fail("record crosses the ring's end", q);
                // while record q + 1 is read, record q + 3 arrives
                const int64_t a = ps.start[std::min(q + 1, q1)] - base, b = ps.start[std::min(q + 4, q1)] - base;
                if ((b + 63) / 64 > a / 64 + ring / 64) return fail("three records do not fit the ring", q);
            }
        }
    // the factor chain: each row's blocks, their transposed couplings and their places in the stream
    if (ps.chainK) {
        // (from the partition's first record: nothing in the plan bounds the stream's length to 32 bits)
        static_assert(sizeof(ps.start[0]) == 8, "the start of a record in a stream of more than 64 GiB");
        std::vector<uint32_t> place(m.nnzb, 0), placeD(n, 0);
        for (int q = 0, p = 0; q < ps.nRec; ++q) {
            while (q >= ps.recBeg[p + 1]) ++p;
            const size_t v = 16 * (size_t)(ps.start[q] - ps.start[ps.recBeg[p]]) +
                             (size_t)ps.ent * (ps.recRows[q + 1] - ps.recRows[q]);
            for (int b = ps.recBlk[q]; b < ps.recBlk[q + 1]; ++b) {
                const uint32_t at = (uint32_t)((v + (size_t)(25 * (fp32 ? 4 : 8)) * (b - ps.recBlk[q])) / 4);
                if (ps.src[b] < 0) placeD[-ps.src[b] - 1] = at;
                else if (ps.rowCell[b] < 0) place[ps.src[b]] = at;
            }
        }
        const int stride = 4 + 4 * ps.chainK;
        std::vector<int> rowOf(m.nnzb);
        for (int i = 0; i < n; ++i)
            for (int s = m.rowPtr[i]; s < m.rowPtr[i + 1]; ++s) rowOf[s] = i;
        for (size_t t = 0; t < rows.size(); ++t) {
            const int32_t* e = ps.chain.data() + stride * t;
            const int i = rows[t];
            int cnt = 0;
            if (e[0] != i || e[2] != m.slotDiag[i] || (uint32_t)e[3] != placeD[i]) return fail("chain row", i);
            for (int s = m.rowPtr[i]; s < m.slotDiag[i]; ++s) {
                if (part[m.cols[s]] != part[i]) continue;
                const int32_t* q = e + 4 + 4 * cnt++;
                if (q[0] != s || rowOf[q[1]] != m.cols[s] || m.cols[q[1]] != i ||
                    q[2] != (natural ? ts.localCol[s] : m.cols[s]) || (uint32_t)q[3] != place[s])
                    return fail("chain block", i, cnt);
            }
            if (cnt != e[1] || cnt > ps.chainK) return fail("chain count", i, cnt);
        }
    }
    // the halo cells that a tile's levels read are there: all of a level's below its count, in order
    for (int t = 0; t < nP && natural; ++t) {
        const int nr = rowStart[t + 1] - rowStart[t], nh = ts.haloFStart[t + 1] - ts.haloFStart[t];
        int last = 0;
        for (int L = ts.levStart[t]; L + 1 < ts.levStart[t + 1]; ++L) {
            if (ts.needF[L] < last || ts.needF[L] > nh) return fail("halo count of a level", t, L);
            last = ts.needF[L];
            for (int q = ts.levPtr[L]; q < ts.levPtr[L + 1]; ++q)
                for (int s = m.rowPtr[rows[q]]; s < m.slotDiag[rows[q]]; ++s)
                    if (ts.localCol[s] >= nr + last) return fail("a level's halo cell is not there", t, L);
        }
    }
    // a chain must be all of the factor: no lower neighbour shares another neighbour with the row
    for (int i = 0; i < n && ps.chainK; ++i)
        for (int p = m.rowPtr[i]; p < m.slotDiag[i]; ++p) {
            const int k = m.cols[p];
            if (part[k] != part[i]) continue;
            for (int q = m.slotDiag[k] + 1; q < m.rowPtr[k + 1]; ++q)
                for (int s = m.rowPtr[i]; s < m.rowPtr[i + 1]; ++s)
                    if (m.cols[q] != i && m.cols[s] == m.cols[q] && part[m.cols[s]] == part[i])
                        return fail("an update beyond the diagonal", i, k);
        }
    // the plain sweeps
    std::vector<double> r(n), y(n), x(n), yr(n), xr(n);
    for (int i = 0; i < n; ++i) r[i] = std::sin(1.0 + 0.37 * i);
    for (int i = 0; i < n; ++i) {
        yr[i] = r[i];
        for (int s = m.rowPtr[i]; s < m.slotDiag[i]; ++s)
            if (part[m.cols[s]] == part[i]) yr[i] -= coef(s) * yr[m.cols[s]];
    }
    for (int i = n - 1; i >= 0; --i) {
        double a = yr[i];
        for (int s = m.slotDiag[i] + 1; s < m.rowPtr[i + 1]; ++s)
            if (part[m.cols[s]] == part[i]) a -= coef(s) * xr[m.cols[s]];
        xr[i] = dinv(i) * a;
    }
    // the streams, tiles in ticket order: a halo value must have been stored before it is read
    std::vector<char> have(n, 0);
    for (int sweep = 0; sweep < 2; ++sweep) {
        std::fill(have.begin(), have.end(), 0);
        for (int t = 0; t < nP; ++t) {
            const int p = sweep ? nP - 1 - t : t;
            const int rs = rowStart[p], nr = rowStart[p + 1] - rs;
            std::vector<double> v(nr);
            for (int q = 0; q < nr; ++q) v[q] = sweep ? y[rows[rs + q]] : r[rows[rs + q]];
            if (natural) {
                const std::vector<int32_t>&hs = sweep ? ts.haloBStart : ts.haloFStart, &h = sweep ? ts.haloB : ts.haloF;
                for (int q = hs[p]; q < hs[p + 1]; ++q) {
                    if (!have[h[q]]) return fail("a tile reads a cell of a later tile", p, h[q]);
                    v.push_back((sweep ? x : y)[h[q]]);
                }
                if ((int)v.size() > ts.maxSlots) return fail("slots", p);
            }
            const int q0 = sweep ? ps.recMid[p] : ps.recBeg[p], q1 = sweep ? ps.recBeg[p + 1] : ps.recMid[p];
            if (int e = replay(m, ps, fp32, q0, q1, sweep != 0, nr, natural && nP > 1 ? (int)v.size() : nr, v)) return e;
            for (int q = 0; q < nr; ++q) {
                (sweep ? x : y)[rows[rs + q]] = v[q];
                have[rows[rs + q]] = 1;
            }
        }
        for (int i = 0; i < n; ++i)
            if (!have[i]) return fail("a cell is in no partition", i);
    }
    double scale = 1e-300;
    for (int i = 0; i < n; ++i) scale = std::max(scale, std::fabs(xr[i]));
    for (int i = 0; i < n; ++i)
        if (!(std::fabs(x[i] - xr[i]) <= 1e-12 * scale)) return fail("sweep result differs", i);
    return 0;
}

extern "C" long long ilu_entry_unit(int row, int ent) { return (long long)entry_unit(row, ent); }

extern "C" long long ilu_cell_value(int cell, int nv, int q) { return (long long)cell_value(cell, nv, q); }

// device allocations of n threads that all ask for the mesh's device copies and plans
extern "C" int mesh_upload_mallocs(const rdst_mesh_desc* desc, int n) {
    Mesh m;
    mesh_build(m, desc);
    g_mallocs = 0;
    std::vector<std::thread> th;
    for (int t = 0; t < n; ++t)
        th.emplace_back([&] {
            mesh_upload(m);
            mesh_stream(m, false);
            mesh_tiles(m, false);
        });
    for (std::thread& t : th) t.join();
    return g_mallocs;
}

// the plan made after an attempt that ran out of device memory at every one of
// its allocations in turn: the same as one made at once
static int check_retry(const rdst_mesh_desc* desc, bool fp32, bool natural) {
    DBuf<double> buf;
    g_mallocsLeft = 0;
    try {
        buf.alloc(8);
        return fail("the allocation did not fail");
    } catch (const HipError&) {
    }
    g_mallocsLeft = -1;
    if (buf.p || buf.n) return fail("a failed allocation leaves a size");
    if (g_last != hipSuccess) return fail("a failed allocation leaves its error to the next check");
    auto plan = [&](Mesh& m) -> StreamSet& { return natural ? mesh_tiles(m, fp32).ps[fp32] : mesh_stream(m, fp32); };
    Mesh ref;
    mesh_build(ref, desc);
    const StreamSet& a = plan(ref);
    for (int k = 0;; ++k) {
        Mesh m;
        mesh_build(m, desc);
        bool threw = false;
        g_mallocsLeft = k;
        try {
            plan(m);
        } catch (const HipError&) {
            threw = true;
        }
        g_mallocsLeft = -1;
        if (!threw) return k > 3 ? 0 : fail("too few allocations", k);
        const StreamSet& b = plan(m);
        if (a.kmax != b.kmax || a.ent != b.ent || a.nRec != b.nRec || a.chainK != b.chainK) return fail("plan numbers", k);
        if (a.recBeg != b.recBeg || a.recMid != b.recMid || a.recRows != b.recRows || a.recBlk != b.recBlk ||
            a.entries != b.entries || a.hdr != b.hdr || a.start != b.start || a.need != b.need || a.src != b.src ||
            a.rowCell != b.rowCell || a.chain != b.chain)
            return fail("plan records", k);
        if (b.d_hdr.n != b.hdr.size() || b.d_start.n != b.start.size() || b.d_chain.n != b.chain.size())
            return fail("device copies", k);
        const TileSet &s = ref.tiles, &t = m.tiles;
        if (s.ok != t.ok || s.maxSlots != t.maxSlots || s.nParts != t.nParts || s.rows != t.rows || s.haloF != t.haloF ||
            s.haloB != t.haloB || s.haloFStart != t.haloFStart || s.haloBStart != t.haloBStart || s.needF != t.needF ||
            s.localCol != t.localCol || s.d_levPtr.n != t.d_levPtr.n)
            return fail("tiles", k);
    }
}

extern "C" int sa_sgs_from_memory(int nParts, double levels, int columns, int lds) {
    return sgs_from_memory(nParts, levels, columns, (size_t)lds);
}

// kmax, chainK, partitions or tiles, and whether the natural order goes by tiles
extern "C" void ilu_plan_numbers(const rdst_mesh_desc* desc, int fp32, int natural, int* out) {
    Mesh m;
    mesh_build(m, desc);
    const StreamSet& ps = natural ? mesh_tiles(m, fp32 != 0).ps[fp32] : mesh_stream(m, fp32 != 0);
    out[0] = ps.kmax;
    out[1] = ps.chainK;
    out[2] = natural ? m.tiles.nParts : m.nParts;
    out[3] = m.tiles.ok;
}

extern "C" int ilu_plan_retry(const rdst_mesh_desc* desc, int fp32, int natural, char* what, int len) {
    g_what.clear();
    int rc = 2;
    try {
        rc = check_retry(desc, fp32 != 0, natural != 0);
    } catch (const std::exception& e) {
        g_what = e.what();
    }
    std::snprintf(what, len, "%s", g_what.c_str());
    return rc;
}

extern "C" int ilu_stream_check(const rdst_mesh_desc* desc, int fp32, int natural, char* what, int len) {
    g_what.clear();
    int rc = 2;
    try {
        rc = check(desc, fp32 != 0, natural != 0);
    } catch (const std::exception& e) {
        g_what = e.what();
    }
    std::snprintf(what, len, "%s", g_what.c_str());
    return rc;
}
