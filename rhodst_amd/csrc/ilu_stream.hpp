// ilu_stream.hpp -- the triangular sweeps of a block ILU(0) from a record
// stream (StreamSet, rdst_internal.hpp): a loader wavefront copies the stream
// linearly into an LDS ring (global -> LDS loads, no registers), four compute
// wavefronts work through it record by record with the partition's vector in
// LDS.
//
// What bounds it: a partition is a chain of at most 32 dependent levels per
// sweep (a mesh that is one tile: of all its levels), each with 2-50 rows, so on
// small and mid-size meshes a level costs the latency of whatever it waits for;
// from about 1e6 cells on, the stream itself (HBM).  Loading a level's blocks when the level is reached cost one memory
// round trip per level (0.75 us); here the blocks of the following records are
// already in the ring, the next record's are in registers, and a level costs an
// LDS gather, the products and a barrier (0.35 us).  Measured, before and after,
// per apply: forward step 4 032 cells FP32 54 -> 33 us; airfoil 205 k FP32 85
// -> 42; wing 321 k FP32 116 -> 61, 117 k FP64 151 -> 67, 403 k FP64 156 -> 147,
// 2.03 M FP32 317 -> 288 (4.5 TB/s; a large copy reaches 4.7); tetrahedra and prisms
// 1.15 M FP32 172 -> 151.
#pragma once
#include "rdst_internal.hpp"

namespace rdst {

#ifdef __HIPCC__

constexpr int STREAM_WAVES = 4;                          // compute wavefronts, 12 rows of 5 lanes each
constexpr int STREAM_THREADS = 64 * (STREAM_WAVES + 1);  // + the loader
// 16 bytes per lane straight into LDS (lane l lands at l16 past the wavefront's base);
// NT: non-temporal, for a stream that no cache holds until the next apply
template <bool NT>
__device__ __forceinline__ void lds_dma16(const uint8_t* g, uint8_t* l) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g,
                                     (__attribute__((address_space(3))) void*)l, 16, 0, NT ? 2 : 0);
}
template <int N>
__device__ __forceinline__ void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// wait until at most `out` (rounded down) of this wavefront's loads are in flight
__device__ __forceinline__ void wait_in_flight(int out) {
    if (out >= 48) wait_vm<48>();
    else if (out >= 32) wait_vm<32>();
    else if (out >= 24) wait_vm<24>();
    else if (out >= 16) wait_vm<16>();
    else if (out >= 12) wait_vm<12>();
    else if (out >= 8) wait_vm<8>();
    else if (out >= 6) wait_vm<6>();
    else if (out >= 4) wait_vm<4>();
    else if (out >= 2) wait_vm<2>();
    else wait_vm<0>();
}
// the loader's barrier: its loads are waited for by count, not by a fence
__device__ __forceinline__ void barrier_raw() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
// the compute wavefronts' barrier: LDS accesses of all of them ordered
__device__ __forceinline__ void barrier_lds() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// The loader: records [r0, r1) whose first bytes are start[r] (16-byte units;
// low: their low words, whose differences are all that the loop needs -- with
// the 64-bit starts in it an airfoil's step was 0.3 % longer).
// Barrier sequence (matched by stream_compute): one when records 0 and 1 are in
// the ring, one when record 2 is, then one per record s when record s + 3 is.
// Between the last two the compute wavefronts read the row entries of record
// s + 2 and the values of record s + 1 from the ring, so everything before
// record s + 1 may be overwritten.
template <int RING, bool NT>
__device__ __forceinline__ void stream_load(const uint8_t* stream, const int64_t* start, const uint32_t* low_, int r0, int r1,
                                            uint8_t* ring) {
    // scalar loads: the offsets must not wait behind the block loads
    const __attribute__((address_space(4))) uint32_t* low = (const __attribute__((address_space(4))) uint32_t*)low_;
    constexpr int RC = RING / 1024, MAXF = RC < 60 ? RC : 60;
    const int lane = threadIdx.x & 63;
    const uint32_t base = low[r0];
    const int n = r1 - r0, total = (int)((low[r1] - base + 63) / 64);
    const uint8_t* g = stream + 16 * start[r0] + 16 * lane;
    int issued = 0;
    auto issue = [&](int limit) {
        for (; issued < limit; ++issued) lds_dma16<NT>(g + (size_t)issued * 1024, ring + (issued & (RC - 1)) * 1024);
    };
    // 1 KB pieces that hold everything before the record starting at st
    auto pieces = [&](uint32_t st) { return (int)((st - base + 63) / 64); };
    issue(min(total, MAXF));
    uint32_t a1 = low[r0 + min(1, n)], a2 = low[r0 + min(2, n)], a3 = low[r0 + min(3, n)], a4 = low[r0 + min(4, n)];
    wait_in_flight(issued - pieces(a2));
    barrier_raw();
    issue(min(total, RC));
    wait_in_flight(issued - pieces(a3));
    barrier_raw();
    for (int s = 0; s < n; ++s) {
        // a1 .. a4: starts of records s + 1 .. s + 4
        const uint32_t a5 = low[r0 + min(s + 5, n)];
        issue(min(total, (int)((a1 - base) / 64) + RC));
        wait_in_flight(issued - pieces(a4));
        barrier_raw();
        a1 = a2; a2 = a3; a3 = a4; a4 = a5;
    }
}

// a row's product with a block's column vector, in one fixed order of rounding
__device__ __forceinline__ float dot5(const float* v, const float* y) {
    return __builtin_fmaf(v[4], y[4], __builtin_fmaf(v[3], y[3], __builtin_fmaf(v[2], y[2], __builtin_fmaf(v[0], y[0], v[1] * y[1]))));
}
__device__ __forceinline__ double dot5(const double* v, const double* y) {
    return __builtin_fma(v[4], y[4], __builtin_fma(v[3], y[3], __builtin_fma(v[2], y[2], __builtin_fma(v[0], y[0], v[1] * y[1]))));
}

// "not there yet" in a vector whose entries other workgroups wait for: a NaN of
// its own; a result with that bit pattern is stored as another NaN
template <class T>
struct Unset;
template <>
struct Unset<double> {
    using U = unsigned long long;
    static constexpr U bits = 0x7ffc5ad3e1b0972full;
};
template <>
struct Unset<float> {
    using U = unsigned int;
    static constexpr U bits = 0x7fe5ad3eu;
};
template <class T>
__device__ __forceinline__ typename Unset<T>::U load_dev(const T* p) {
    return __hip_atomic_load(reinterpret_cast<const typename Unset<T>::U*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void store_dev(T* p, T v) {
    using U = typename Unset<T>::U;
    U u = __builtin_bit_cast(U, v);
    if (u == Unset<T>::bits) u ^= 1;  // a NaN either way
    __hip_atomic_store(reinterpret_cast<U*>(p), u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Records [0, n) of the list starting at r0; the first nF are forward ones
// (y -= L y), the others backward ones (y = Dinv y - sum (Dinv U) y).  y holds
// the partition's rows (and, behind them, the values of rows outside it).
// Five lanes per row, lane r holds row r of the row's 5x5 blocks.  Called by
// the compute wavefronts, while the loader runs stream_load.  Per record: the
// row entries are read two records ahead and the values one ahead, so between
// two barriers only y's gather, the products and y's store depend on the
// barrier before.  PUB: each result also goes to out[to[its place in y]] at
// once, for the workgroups that wait for it.
template <class TM, class TV, int KDU, int RING, bool PUB>
__device__ __forceinline__ void stream_compute(const uint32_t* hdr, int r0, int nF, int n, const uint8_t* ring, TV* y,
                                               const int* to, TV* out) {
    constexpr int MASK = RING - 1, ENT = stream_entry(KDU), BLK = 25 * (int)sizeof(TM);
    // Rows of more than four blocks in a sweep.  A wavefront without one skips the
    // blocks past the fourth (K4), and FP64 with eight reads the next record's
    // values after this one's products (LATE): a wavefront has 256 registers, and
    // with all nine blocks of both records in them it spilled 356 of them.  Apply of
    // 403 k hexahedra numbered at random (six blocks): all of eight 292 us, six 142,
    // and so 125; FP32 with six gains nothing (77 / 104 us) and keeps all of them.  263 k
    // polyhedra, seven blocks: FP64 382 us with eight blocks, 270 so; FP32 263, 229.
    constexpr int K4 = KDU > 6 || (KDU > 4 && sizeof(TM) == 8) ? 4 : KDU;
    constexpr bool LATE = KDU > 6 && sizeof(TM) == 8;
    constexpr int KG = LATE ? KDU : K4;  // columns gathered before the products
    struct Ent {
        uint32_t w[ENT / 4];
        int eb, vb, nR;  // ring offset of the record's entries and values, rows (uniform)
        bool row;        // this lane has a row
        bool wide;       // a row of this wavefront has more than K4 off-diagonal blocks (uniform)
    };
    struct Val {
        TM d[5], v[KDU][5];
    };
    const int lane = threadIdx.x & 63, g = lane / 5, r = lane - 5 * g;
    const int w12 = 12 * (int)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = g < 12 ? w12 + g : kStreamRows;
    // header words, 64 records per vector load, the next 64 loaded ahead
    // (records past the last one have no rows)
    const uint32_t* hp = hdr + r0;
    uint32_t ha = lane < n ? hp[lane] : 0u, hb = 64 + lane < n ? hp[64 + lane] : 0u;
    int off = 0;  // of the next record, bytes
    // The steps of a record are free of branches (a taken branch costs as much
    // as several LDS accesses here): a lane without a row, and a block that a
    // row does not have, read something in bounds and drop it.
    auto head = [&](int s, Ent& E) {
        const uint32_t w = __builtin_amdgcn_readlane(ha, s & 63);
        E.nR = w & 0xffff;
        E.row = j < E.nR;
        E.eb = off & MASK;
        E.vb = E.eb + ENT * E.nR;
#pragma unroll
        for (int q = 0; q < ENT / 4; ++q) E.w[q] = 0u;  // in bounds also where entry() is skipped
        off += 16 * (int)(w >> 16);
        if ((s & 63) == 63) {
            ha = hb;
            hb = s + 65 + lane < n ? hp[s + 65 + lane] : 0u;
            // waited for here (vmcnt 0), not by the next records behind their stores
            if constexpr (PUB) __builtin_amdgcn_s_waitcnt(0x0f70);
        }
    };
    auto entry = [&](Ent& E) {
        const uint4* p = reinterpret_cast<const uint4*>(ring + E.eb + ENT * (E.row ? j : 0));
#pragma unroll
        for (int q = 0; q < ENT / 16; ++q) {
            const uint4 u = p[q];
            E.w[4 * q] = u.x; E.w[4 * q + 1] = u.y; E.w[4 * q + 2] = u.z; E.w[4 * q + 3] = u.w;
        }
    };
    // entry word 0: 5 x row | first block << 16 | off-diagonal blocks << 24; a
    // forward row has no Dinv, so what is read in its place precedes its blocks
    auto values = [&](int s, Ent& E, Val& V) {
#pragma unroll
        for (int q = 0; q < ENT / 4; ++q) E.w[q] = E.row ? E.w[q] : 0u;
        const int o = E.vb + BLK * ((int)((E.w[0] >> 16) & 0xff) + (s < nF ? 0 : 1));
        const TM* p = reinterpret_cast<const TM*>(ring + o) + 5 * r;
        const TM* pd = reinterpret_cast<const TM*>(ring + max(0, o - BLK)) + 5 * r;
#pragma unroll
        for (int c = 0; c < 5; ++c) V.d[c] = pd[c];
#pragma unroll
        for (int k = 0; k < K4; ++k)
#pragma unroll
            for (int c = 0; c < 5; ++c) V.v[k][c] = p[25 * k + c];
        if constexpr (KDU > K4) {
            // rows are in descending order of their blocks: lane 0 has the wavefront's longest
            E.wide = (int)(__builtin_amdgcn_readfirstlane(E.w[0]) >> 24) > K4;
            if (E.wide)
#pragma unroll
                for (int k = K4; k < KDU; ++k)
#pragma unroll
                    for (int c = 0; c < 5; ++c) V.v[k][c] = p[25 * k + c];
        }
    };
    struct Gat {
        TV a, d[5], v[KG][5];
        int to;
    };
    auto gather = [&](const Ent& E, Gat& G) {
        const TV* yr = y + (E.w[0] & 0xffff);
        G.a = yr[r];
        if constexpr (PUB) G.to = to[(E.w[0] & 0xffff) + r];
#pragma unroll
        for (int c = 0; c < 5; ++c) G.d[c] = yr[c];
#pragma unroll
        for (int k = 0; k < K4; ++k) {
            const uint32_t w = E.w[1 + k / 2];
            const TV* yv = y + ((k & 1) ? w >> 16 : w & 0xffff);
#pragma unroll
            for (int c = 0; c < 5; ++c) G.v[k][c] = yv[c];
        }
        if constexpr (KG > K4)
            if (E.wide)
#pragma unroll
                for (int k = K4; k < KG; ++k) {
                    const uint32_t w = E.w[1 + k / 2];
                    const TV* yv = y + ((k & 1) ? w >> 16 : w & 0xffff);
#pragma unroll
                    for (int c = 0; c < 5; ++c) G.v[k][c] = yv[c];
                }
    };
    auto apply = [&](int s, const Ent& E, const Val& V, const Gat& G) {
        const int cnt = (int)(E.w[0] >> 24);
        TV acc = dot5(V.d, G.d);
        acc = s < nF ? G.a : acc;
#pragma unroll
        for (int k = 0; k < K4; ++k) {
            const TV dot = dot5(V.v[k], G.v[k]);
            acc = k < cnt ? acc - dot : acc;
        }
        if constexpr (KDU > K4)
            if (E.wide)
#pragma unroll
                for (int k = K4; k < KDU; ++k) {
                    const uint32_t w = E.w[1 + k / 2];
                    const TV* yv = KG > K4 ? G.v[k < KG ? k : 0] : y + ((k & 1) ? w >> 16 : w & 0xffff);
                    const TV dot = dot5(V.v[k], yv);
                    acc = k < cnt ? acc - dot : acc;
                }
        if (E.row) {
            y[(E.w[0] & 0xffff) + r] = acc;
            if constexpr (PUB) store_dev(out + G.to, acc);
        }
    };
    Ent e0, e1, e2;
    Val A, B;
    Gat G;
    // one record: y first (it is what the next barrier waits for), then the
    // ring's parts of the next ones
    auto step = [&](int s, Ent& E0, Ent& E1, Ent& E2, Val& V0, Val& V1) {
        head(s + 2, E2);
        if (w12 < max(E0.nR, max(E1.nR, E2.nR))) {
            gather(E0, G);
            if constexpr (LATE) {
                apply(s, E0, V0, G);
                __builtin_amdgcn_sched_barrier(0);
            }
            entry(E2);
            values(s + 1, E1, V1);
            if constexpr (!LATE) apply(s, E0, V0, G);
        }
        barrier_lds();
    };
    barrier_lds();
    head(0, e0);
    entry(e0);
    values(0, e0, A);
    head(1, e1);
    entry(e1);
    barrier_lds();
    for (int s = 0;;) {
        step(s, e0, e1, e2, A, B);
        if (++s >= n) break;
        step(s, e1, e2, e0, B, A);
        if (++s >= n) break;
        step(s, e2, e0, e1, A, B);
        if (++s >= n) break;
        step(s, e0, e1, e2, B, A);
        if (++s >= n) break;
        step(s, e1, e2, e0, A, B);
        if (++s >= n) break;
        step(s, e2, e0, e1, B, A);
        if (++s >= n) break;
    }
}

// The partition's part of a vector into LDS and back: ten entries per thread
// and pass, so a partition costs a few memory round trips and not one (two
// with the row index) per entry.
template <class TV>
__device__ __forceinline__ void gather_rows(const int32_t* rows, int nl5, const TV* x, TV* y) {
    constexpr int U = 10, ST = 64 * STREAM_WAVES;
    for (int b = 0; b < nl5; b += U * ST) {
        int i[U];
        TV v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int t = min(b + u * ST + (int)threadIdx.x, nl5 - 1);
            i[u] = 5 * rows[t / 5] + t % 5;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = x[i[u]];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int t = b + u * ST + (int)threadIdx.x;
            if (t < nl5) y[t] = v[u];
        }
    }
}
template <class TV>
__device__ __forceinline__ void scatter_rows(const int32_t* rows, int nl5, const TV* y, TV* x) {
    constexpr int U = 10, ST = 64 * STREAM_WAVES;
    for (int b = 0; b < nl5; b += U * ST) {
        int i[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int t = min(b + u * ST + (int)threadIdx.x, nl5 - 1);
            i[u] = 5 * rows[t / 5] + t % 5;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int t = b + u * ST + (int)threadIdx.x;
            if (t < nl5) x[i[u]] = y[t];
        }
    }
}

// x = M^-1 r for the partitioned factor, one workgroup per partition
template <class TM, class TV, int KDU, bool NT>
__global__ __launch_bounds__(STREAM_THREADS) void k_stream_apply(const int32_t* __restrict__ rowStart,
                                                                 const int32_t* __restrict__ rows,
                                                                 const int32_t* __restrict__ recBeg,
                                                                 const int32_t* __restrict__ recMid,
                                                                 const uint32_t* __restrict__ hdr,
                                                                 const int64_t* __restrict__ start,
                                                                 const uint32_t* __restrict__ low,
                                                                 const uint8_t* __restrict__ stream,
                                                                 const TV* __restrict__ r, TV* __restrict__ x) {
    constexpr int RING = stream_ring(sizeof(TM) == 4);
    extern __shared__ __align__(1024) unsigned char smem_raw[];
    uint8_t* ring = smem_raw;
    TV* y = reinterpret_cast<TV*>(smem_raw + RING);
    const int pt = blockIdx.x;
    const int r0 = recBeg[pt], rm = recMid[pt], r1 = recBeg[pt + 1];
    if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) == STREAM_WAVES) {
        stream_load<RING, NT>(stream, start, low, r0, r1, ring);
        return;
    }
    const int rs = rowStart[pt], nl5 = (rowStart[pt + 1] - rs) * 5;
    gather_rows(rows + rs, nl5, r, y);
    stream_compute<TM, TV, KDU, RING, false>(hdr, r0, rm - r0, r1 - r0, ring, y, nullptr, (TV*)nullptr);
    scatter_rows(rows + rs, nl5, y, x);
}

// ---------------------------------------------------------------- natural order
// The sweeps of the natural-order ILU(0) by tiles (TileSet).  Workgroups take
// tiles in an order that respects their dependencies (a ticket counter), so a
// tile only waits for tiles that running workgroups already hold, and the
// launch ends whatever number of workgroups is resident.  A value another tile
// needs is its own flag: the vector is filled with Unset before the sweep, a
// row's result is stored the moment it is computed, and a wavefront of its own
// polls for the halo values (device-scope loads and stores) in the order in
// which the records read them.  A tile so runs a few levels behind the ones it
// depends on, and a sweep costs about the levels of the whole mesh, not tiles
// in a row times levels of a tile: with every halo value awaited at a tile's
// start the sweeps took 365 us (RAE2822, 23.5 k cells, 431 levels) and 765 (wing,
// 321 k, 260 levels), now 180 and 232.  By one launch per level (8-10 us
// each, or 3.3 us per level in a single-workgroup run of small levels) it was
// 1.5 ms and 2.3 ms.
template <class T>
__global__ __launch_bounds__(256) void k_fill_unset(long n, T* y, int* tickets) {
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        reinterpret_cast<typename Unset<T>::U*>(y)[i] = Unset<T>::bits;
    if (blockIdx.x == 0 && threadIdx.x < 2) tickets[threadIdx.x] = 0;
}

// The halo wavefront: the NV values of each cell outside the tile into LDS, each
// as soon as it has arrived, in step with the n records (barriers as in
// stream_load): before record s starts, those of the first need[s] cells are
// there.  A window of 64 U values is asked for at a time; what has not arrived is
// asked for again.
template <class TV, int NV, int U>
__device__ __forceinline__ void stream_halo(const int32_t* cells, int nh, const int32_t* need_, int n, const TV* x, TV* y) {
    constexpr int W = 64 * U;
    const __attribute__((address_space(4))) int32_t* need = (const __attribute__((address_space(4))) int32_t*)need_;
    const int lane = threadIdx.x & 63, nv = NV * nh;
    int b = 0, have = 0;
    uint32_t i[U];
    typename Unset<TV>::U v[U];
    auto ask = [&]() {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int t = min(b + 64 * u + lane, nv - 1);
            i[u] = (uint32_t)(t / NV);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) i[u] = (uint32_t)cells[i[u]];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            i[u] = cell_value((int)i[u], NV, min(b + 64 * u + lane, nv - 1) % NV);
            v[u] = load_dev(x + i[u]);
        }
    };
    auto until = [&](int k) {
        while (have < k) {
            int first = min(b + W, nv);
#pragma unroll
            for (int u = U - 1; u >= 0; --u) {
                const int t = b + 64 * u + lane;
                const bool ok = v[u] != Unset<TV>::bits;
                if (ok && t < nv) y[t] = __builtin_bit_cast(TV, v[u]);
                const unsigned long long miss = __ballot(!ok && t < nv);
                if (miss) first = b + 64 * u + (int)__builtin_ctzll(miss);
                if (!ok) v[u] = load_dev(x + i[u]);
            }
            have = first;
            if (first == b + W && first < nv) {
                b += W;
                ask();
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the values in LDS
    };
    if (nv > 0) ask();
    barrier_raw();
    until(NV * need[0]);
    barrier_raw();
    for (int s = 0; s < n; ++s) {
        until(NV * need[min(s + 1, n - 1)]);
        barrier_raw();
    }
}

// The tile's part of `in` into LDS, where each entry belongs in the vectors, and
// `reset` made unset (it may be `in`: each thread resets what it has read).
template <class TV>
__device__ __forceinline__ void gather_tile(const int32_t* rows, int nl5, const TV* in, TV* y, int* to, TV* reset) {
    constexpr int U = 10, ST = 64 * STREAM_WAVES;
    for (int b = 0; b < nl5; b += U * ST) {
        int i[U];
        TV v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int t = min(b + u * ST + (int)threadIdx.x, nl5 - 1);
            i[u] = 5 * rows[t / 5] + t % 5;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = in[i[u]];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int t = b + u * ST + (int)threadIdx.x;
            if (t < nl5) {
                y[t] = v[u];
                to[t] = i[u];
                reinterpret_cast<typename Unset<TV>::U*>(reset)[i[u]] = Unset<TV>::bits;
            }
        }
    }
}

// One sweep.  Forward: out = y from in = r, reset = x for the backward sweep.
// Backward: out = x from in = y, reset = y for the next forward sweep.  Each
// resets the other's ticket counter (the launches are ordered).
constexpr int TILE_THREADS = STREAM_THREADS + 64;  // + the halo wavefront
template <class TM, class TV, int KDU, bool BWD>
__global__ __launch_bounds__(TILE_THREADS) void k_tile_sweep(int nT, int* tickets, const int32_t* __restrict__ rowStart,
                                                             const int32_t* __restrict__ rows,
                                                             const int32_t* __restrict__ haloStart,
                                                             const int32_t* __restrict__ halo,
                                                             const int32_t* __restrict__ recBeg,
                                                             const int32_t* __restrict__ recMid,
                                                             const int32_t* __restrict__ need,
                                                             const uint32_t* __restrict__ hdr,
                                                             const int64_t* __restrict__ start,
                                                             const uint32_t* __restrict__ low,
                                                             const uint8_t* __restrict__ stream, const TV* in, TV* out,
                                                             TV* reset) {
    constexpr int RING = stream_ring(sizeof(TM) == 4);
    extern __shared__ __align__(1024) unsigned char smem_raw[];
    __shared__ int next[2];
    uint8_t* ring = smem_raw;
    int* to = reinterpret_cast<int*>(smem_raw + RING);
    TV* y = reinterpret_cast<TV*>(smem_raw + RING + 20 * kTileCells);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (threadIdx.x == 0) next[0] = atomicAdd(tickets + BWD, 1);
    __syncthreads();
    for (int round = 0;; ++round) {
        const int ticket = __builtin_amdgcn_readfirstlane(next[round & 1]);
        if (ticket >= nT) break;
        const int tl = BWD ? nT - 1 - ticket : ticket;
        const int r0 = BWD ? recMid[tl] : recBeg[tl], r1 = BWD ? recBeg[tl + 1] : recMid[tl];
        const int rs = rowStart[tl], nl5 = (rowStart[tl + 1] - rs) * 5;
        if (wave == STREAM_WAVES) {
            stream_load<RING, false>(stream, start, low, r0, r1, ring);
            if ((threadIdx.x & 63) == 0) next[(round + 1) & 1] = atomicAdd(tickets + BWD, 1);
        } else if (wave > STREAM_WAVES) {
            const int h0 = haloStart[tl];
            stream_halo<TV, 5, 4>(halo + h0, haloStart[tl + 1] - h0, need + r0, r1 - r0, (const TV*)out, y + nl5);
        } else {
            if (ticket == 0 && threadIdx.x == 0) tickets[!BWD] = 0;
            gather_tile(rows + rs, nl5, in, y, to, reset);
            stream_compute<TM, TV, KDU, RING, true>(hdr, r0, BWD ? 0 : r1 - r0, r1 - r0, ring, y, to, out);
        }
        __syncthreads();
    }
}
// the row entries of every record into the stream (once per buffer)
__global__ __launch_bounds__(64) void k_stream_entries(int ent, const int32_t* recRows, const uint4* entries,
                                                       const int64_t* start, uint8_t* stream) {
    const int q = blockIdx.x;
    const size_t b = entry_unit(recRows[q], ent), e = entry_unit(recRows[q + 1], ent);
    uint4* o = reinterpret_cast<uint4*>(stream + 16 * (size_t)start[q]);
    for (size_t t = b + threadIdx.x; t < e; t += 64) o[t - b] = entries[t];
}

// Scatter the factor into the stream, one wavefront per record and one thread
// per (block, block row).  src[b]: block-CSR slot, or -(cell + 1) for the
// row's Dinv; in a backward record (rowCell[b] >= 0) the slots' blocks are
// stored as Dinv U, formed in FP64.  uOnly: Dinv and the forward records are
// in place already (k_ilu_chain), and LU is the matrix itself.
template <class T>
__global__ __launch_bounds__(256) void k_stream_pack(int nRec, int ent, int uOnly, const int32_t* recRows, const int32_t* recBlk,
                                                    const int32_t* src, const int32_t* rowCell, const int64_t* start,
                                                    const T* LU, const T* Dinv, uint8_t* stream) {
    const int q = 4 * blockIdx.x + (threadIdx.x >> 6);
    if (q >= nRec) return;
    const int b0 = recBlk[q], n5 = 5 * (recBlk[q + 1] - b0);
    T* val = reinterpret_cast<T*>(stream + 16 * (size_t)start[q] + ent * (recRows[q + 1] - recRows[q]));
    if (n5 == 0 || (uOnly && rowCell[b0] < 0)) return;
    // Bound by the chain index -> blocks -> store of a step; the next step's
    // indices and blocks are asked for before this one's are used (2 M cells
    // FP32: one step after the other 905 us, so 534).
    struct Step {
        int sl, cell;
        T d[5], u[25];
    };
    auto index = [&](int e, Step& x) {
        const int b = min(e, n5 - 1) / 5;
        x.sl = src[b0 + b];
        x.cell = rowCell[b0 + b];
    };
    auto blocks = [&](int e, Step& x) {
        const int r = min(e, n5 - 1) % 5;
        const bool prod = x.sl >= 0 && x.cell >= 0;
        if (uOnly && !prod) return;
        const T* Dr = prod ? Dinv + 25 * (size_t)x.cell : x.sl < 0 ? Dinv + 25 * (size_t)(-x.sl - 1) : LU + 25 * (size_t)x.sl;
#pragma unroll
        for (int c = 0; c < 5; ++c) x.d[c] = Dr[5 * r + c];
        if (!prod) return;
        const T* U = LU + 25 * (size_t)x.sl;
#pragma unroll
        for (int c = 0; c < 25; ++c) x.u[c] = U[c];
    };
    auto store = [&](int e, const Step& x) {
        const bool prod = x.sl >= 0 && x.cell >= 0;
        if (e >= n5 || (uOnly && !prod)) return;
        T* dst = val + 5 * e;
#pragma unroll
        for (int c = 0; c < 5; ++c) {
            double a = 0.0;
#pragma unroll
            for (int p = 0; p < 5; ++p) a += (double)x.d[p] * (double)x.u[5 * p + c];
            dst[c] = prod ? (T)a : x.d[c];
        }
    };
    Step A = {}, B = {};
    int e = threadIdx.x & 63;
    index(e, A);
    index(e + 64, B);
    blocks(e, A);
    for (int n = 0; n < n5; n += 128) {
        blocks(e + 64, B);
        store(e, A);
        index(e + 128, A);
        blocks(e + 128, A);
        store(e + 64, B);
        index(e + 192, B);
        e += 128;
    }
}

#endif

}  // namespace rdst
