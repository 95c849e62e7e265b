// ilu_factor.hpp -- the block ILU(0) factor of a partition or tile whose
// couplings form no triangle (StreamSet::chain): every update then falls on a
// diagonal block, so the factor is a chain of D_i = A_ii - sum_k (A_ik Dinv_k)
// A_ki and its inverse, and L_ik = A_ik Dinv_k; U is A.
//
// What bounds it: the dependent levels of a partition, each two products of
// 5x5 blocks per lower neighbour and an inversion.  One thread per row spent
// 4-5 us per level on some 2000 dependent instructions at 30 busy lanes, with
// its blocks read after the level began and written back to the factor matrix.
// Here five lanes share a row (lane r holds row r of every block; the
// inversion is theirs together, rows exchanged by wavefront shuffles), the next
// level's blocks of A are loaded while this one is computed, and L and Dinv go
// straight into the sweeps' record stream: no copy of A, no factor matrix.
// Measured, this kernel with its pack against thread per row, copy and pack:
// FP32 partitions 2 M cells 1.80 / 5.8 ms, 24 k cells 0.25 / 0.52 ms; FP64 natural
// order 252 cells 0.19 / 0.52 ms, 23.5 k 2.2 / 9.5 ms, 321 k 2.1 / 9.9 ms.
#pragma once
#include "rdst_internal.hpp"

namespace rdst {

#ifdef __HIPCC__

template <class T>
__device__ __forceinline__ T row_shfl(T v, int src) {
    return __shfl(v, src, 64);
}

// Rows of the inverse of the 5x5 matrix whose row r is a in lane base + r
// (Gauss-Jordan, partial pivoting, the operations of inv5 in its order); returns
// which row of the inverse this lane holds in b, or -1 for a zero pivot.
template <class T>
__device__ __forceinline__ int inv5_lanes(T (&a)[5], T (&b)[5], int base, int r) {
#pragma unroll
    for (int c = 0; c < 5; ++c) b[c] = c == r ? T(1) : T(0);
    int perm = 0x43210;  // nibble q: the row that lane q holds by now
    bool ok = true;
#pragma unroll
    for (int col = 0; col < 5; ++col) {
        // the first largest entry of the column at or below the diagonal
        T v[5], pv = T(0), best = T(0);
        int bl = 0, bp = col;
#pragma unroll
        for (int q = 0; q < 5; ++q) {
            v[q] = row_shfl(a[col], base + q);
            const bool diag = ((perm >> (4 * q)) & 15) == col;
            pv = diag ? v[q] : pv;
            bl = diag ? q : bl;
        }
        best = pv < T(0) ? -pv : pv;  // a NaN there stays the pivot
#pragma unroll
        for (int q = 0; q < 5; ++q) {
            const T m = v[q] < T(0) ? -v[q] : v[q];
            const int p = (perm >> (4 * q)) & 15;
            // bitwise: as && and || these become branches, some 20 per column
            const bool take = (p > col) & ((m > best) | ((m == best) & (p < bp)));
            best = take ? m : best;
            pv = take ? v[q] : pv;
            bl = take ? q : bl;
            bp = take ? p : bp;
        }
        ok = ok & (pv != T(0));
        // lane bl's row becomes row col, the one that was row col takes bl's place
        int np = 0;
#pragma unroll
        for (int q = 0; q < 5; ++q) {
            const int p = (perm >> (4 * q)) & 15;
            np |= (q == bl ? col : (p == col ? bp : p)) << (4 * q);
        }
        perm = np;
        const T d = T(1) / pv;
        const T f = a[col];
        const bool piv = r == bl;
#pragma unroll
        for (int j = 0; j < 5; ++j) {
            if (j > col) {
                const T x = row_shfl(a[j], base + bl) * d;
                a[j] = piv ? x : (f == T(0) ? a[j] : a[j] - f * x);
            }
            const T y = row_shfl(b[j], base + bl) * d;
            b[j] = piv ? y : (f == T(0) ? b[j] : b[j] - f * y);
        }
    }
    return ok ? (perm >> (4 * r)) & 15 : -1;
}

constexpr int CHAIN_THREADS = 256;  // 4 wavefronts x 12 rows of 5 lanes

// A row of the chain (row entry t of StreamSet::chain) and its part of A, row r
// of each block in this lane.
template <int K>
struct ChainEntry {
    int4 h, n[K];
};
template <class T, int K>
struct ChainRegs {
    int cell, cnt, lk[K];  // lk: the neighbour's cell, or its column in the tile
    uint32_t dDst, lDst[K];
    T d[5], a[K][5], u[K][5];
};
template <int K>
__device__ __forceinline__ void chain_entry(const int32_t* __restrict__ rows, long t, ChainEntry<K>& E) {
    const int4* e = reinterpret_cast<const int4*>(rows + (4 + 4 * K) * (size_t)t);
    E.h = e[0];
#pragma unroll
    for (int k = 0; k < K; ++k) E.n[k] = e[1 + k];
}
template <class T, int K>
__device__ __forceinline__ void chain_load(const ChainEntry<K>& E, int r, const T* __restrict__ A, ChainRegs<T, K>& R) {
    R.cell = E.h.x;
    R.cnt = E.h.y;
    R.dDst = (uint32_t)E.h.w;
    const T* p = A + 25 * (size_t)E.h.z + 5 * r;
#pragma unroll
    for (int c = 0; c < 5; ++c) R.d[c] = p[c];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        R.lk[k] = E.n[k].z;
        R.lDst[k] = (uint32_t)E.n[k].w;
        const T* pa = A + 25 * (size_t)E.n[k].x + 5 * r;
        const T* pu = A + 25 * (size_t)E.n[k].y + 5 * r;
#pragma unroll
        for (int c = 0; c < 5; ++c) { R.a[k][c] = pa[c]; R.u[k][c] = pu[c]; }
    }
}
// own: the row's place in LDS (TILE), where the tile's Dinv and its halo's are
// kept; outside it they are read from Dinv itself.
template <class T, int K, bool TILE>
__device__ __forceinline__ void chain_row(const ChainRegs<T, K>& R, bool on, int base, int r, T* Dinv, T* lds, int own,
                                          uint8_t* stream, int* fail) {
    T d[5], l[K][5];
#pragma unroll
    for (int c = 0; c < 5; ++c) d[c] = R.d[c];
#pragma unroll
    for (int k = 0; k < K; ++k)
        if (k < R.cnt) {
            const T* Dk = (TILE ? lds : Dinv) + 25 * (size_t)R.lk[k];
#pragma unroll
            for (int j = 0; j < 5; ++j) {
                T s = 0;
#pragma unroll
                for (int q = 0; q < 5; ++q) s += R.a[k][q] * Dk[5 * q + j];
                l[k][j] = s;
            }
            T u[5][5];
#pragma unroll
            for (int q = 0; q < 5; ++q)
#pragma unroll
                for (int j = 0; j < 5; ++j) u[q][j] = row_shfl(R.u[k][j], base + q);
#pragma unroll
            for (int j = 0; j < 5; ++j) {
                T s = 0;
#pragma unroll
                for (int q = 0; q < 5; ++q) s += l[k][q] * u[q][j];
                d[j] -= s;
            }
        }
    T b[5];
    int row = inv5_lanes(d, b, base, r);
    // the next pass's blocks have arrived by now: waited for here (vmcnt 0), so
    // that using them does not wait behind the stores below
    __builtin_amdgcn_s_waitcnt(0x0f70);
    if (!on) return;
    if (row < 0) {  // the caller fails; whoever waits for this block goes on
        atomicExch(fail, 1);
        row = r;
#pragma unroll
        for (int c = 0; c < 5; ++c) b[c] = T(0);
    }
    T* g = Dinv + 25 * (size_t)R.cell + 5 * row;
    T* o = reinterpret_cast<T*>(stream + 4 * (size_t)R.dDst) + 5 * row;
#pragma unroll
    for (int c = 0; c < 5; ++c) {
        if constexpr (TILE) {
            lds[25 * own + 5 * row + c] = b[c];
            store_dev(g + c, b[c]);
        } else {
            g[c] = b[c];
        }
    }
#pragma unroll
    for (int c = 0; c < 5; ++c) o[c] = b[c];
#pragma unroll
    for (int k = 0; k < K; ++k)
        if (k < R.cnt) {
            T* p = reinterpret_cast<T*>(stream + 4 * (size_t)R.lDst[k]) + 5 * r;
#pragma unroll
            for (int j = 0; j < 5; ++j) p[j] = l[k][j];
        }
}

// One partition's (or tile's) rows level by level, NW wavefronts, for a tile two
// barriers before the first level, and one after each.  A pass is 12 NW rows of a
// level; the blocks of the pass after this one are loaded before this one is
// computed, and the entries of the one after that.
template <class T, int K, int NW, bool TILE>
__device__ __forceinline__ void chain_levels(int l0, int l1, const int32_t* __restrict__ levPtr,
                                             const int32_t* __restrict__ rows, const T* __restrict__ A, T* Dinv, T* lds,
                                             uint8_t* stream, int* fail) {
    const int lane = threadIdx.x & 63, g = lane / 5, r = lane - 5 * g, base = lane - r;
    const int w12 = 12 * (int)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6), slot = g < 12 ? w12 + g : 1 << 20;
    struct Pass {
        int L, s, e;  // level, its rows from this pass on
    };
    auto after = [&](Pass p) {
        if (p.s + 12 * NW < p.e) return Pass{p.L, p.s + 12 * NW, p.e};
        return Pass{p.L + 1, p.e, p.L + 2 < l1 ? levPtr[p.L + 2] : p.e};
    };
    // lanes without a row (past the last level: all) work on the last row there is and store nothing
    auto row_of = [&](Pass p) { return max(min(p.s + slot, p.e - 1), p.s - 1); };
    Pass p0 = {l0, levPtr[l0], levPtr[l0 + 1]};
    const int first = p0.s;
    Pass p1 = after(p0);
    ChainRegs<T, K> cur, nxt;
    ChainEntry<K> ent;
    chain_entry<K>(rows, row_of(p0), ent);
    chain_load<T, K>(ent, r, A, cur);
    chain_entry<K>(rows, row_of(p1), ent);
    if constexpr (TILE) {
        barrier_lds();
        barrier_lds();
    }
    while (p0.L + 1 < l1) {
        const Pass p2 = p1.L + 1 < l1 ? after(p1) : p1;
        chain_load<T, K>(ent, r, A, nxt);
        chain_entry<K>(rows, row_of(p2), ent);
        if (p0.s + w12 < p0.e)
            chain_row<T, K, TILE>(cur, p0.s + slot < p0.e, base, r, Dinv, lds, row_of(p0) - first, stream, fail);
        else
            __builtin_amdgcn_s_waitcnt(0x0f70);  // as in chain_row, or the next pass waits for its stores
        if (p1.L != p0.L) barrier_lds();  // rows of a later level read what this one stored
        p0 = p1;
        p1 = p2;
        cur = nxt;
    }
}

template <class T, int K>
__global__ __launch_bounds__(CHAIN_THREADS) void k_ilu_chain(const int32_t* __restrict__ levStart,
                                                             const int32_t* __restrict__ levPtr,
                                                             const int32_t* __restrict__ rows, const T* __restrict__ A,
                                                             T* Dinv, const int32_t* __restrict__ recBeg,
                                                             const int64_t* __restrict__ start, uint8_t* stream, int* fail) {
    const int p = blockIdx.x;
    chain_levels<T, K, CHAIN_THREADS / 64, false>(levStart[p], levStart[p + 1], levPtr, rows, A, Dinv, (T*)nullptr,
                                                  stream + 16 * start[recBeg[p]], fail);
}

// The natural-order factor by tiles, taken by ticket in an order that respects
// their dependencies and pipelined as k_tile_sweep's: Dinv is unset before, each
// row's is stored as it is computed, and a wavefront of its own polls for the
// halo's.  The tile's Dinv and its halo's are kept in LDS.  A level costs 4.6 us,
// nearly all of it the dependent instructions of a row.  With tiles that waited for
// their predecessors to end, and Dinv read back from memory, the factor took 3.9 ms
// (RAE2822, 23.5 k cells) and 4.35 (wing, 321 k), now 2.07 and 1.79.
// Three wavefronts compute (a level of a tile has 10-20 rows): with the halo's one
// per SIMD, so that all of a pass and the next one stay in registers.
constexpr int CHAIN_TILE_WAVES = 3, CHAIN_TILE_THREADS = 64 * (CHAIN_TILE_WAVES + 1);
template <class T, int K>
__global__ __launch_bounds__(CHAIN_TILE_THREADS) void k_ilu_chain_tiles(int nT, int* ticket,
                                                                        const int32_t* __restrict__ rowStart,
                                                                        const int32_t* __restrict__ haloStart,
                                                                        const int32_t* __restrict__ halo,
                                                                        const int32_t* __restrict__ need,
                                                                        const int32_t* __restrict__ levStart,
                                                                        const int32_t* __restrict__ levPtr,
                                                                        const int32_t* __restrict__ rows,
                                                                        const T* __restrict__ A, T* Dinv,
                                                                        const int32_t* __restrict__ recBeg,
                                                                        const int64_t* __restrict__ start,
                                                                        uint8_t* stream, int* fail) {
    extern __shared__ __align__(16) unsigned char chain_raw[];
    T* lds = reinterpret_cast<T*>(chain_raw);
    __shared__ int cur;
    if (threadIdx.x == 0) cur = atomicAdd(ticket, 1);
    __syncthreads();
    for (;;) {
        const int t = __builtin_amdgcn_readfirstlane(cur);
        if (t >= nT) break;
        const int l0 = levStart[t], l1 = levStart[t + 1];
        if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) == CHAIN_TILE_WAVES) {
            const int h0 = haloStart[t];
            stream_halo<T, 25, 12>(halo + h0, haloStart[t + 1] - h0, need + l0, l1 - l0 - 1, (const T*)Dinv,
                                   lds + 25 * (rowStart[t + 1] - rowStart[t]));
        } else {
            chain_levels<T, K, CHAIN_TILE_WAVES, true>(l0, l1, levPtr, rows, A, Dinv, lds, stream + 16 * start[recBeg[t]], fail);
        }
        __syncthreads();  // every wavefront has read cur
        if (threadIdx.x == 0) cur = atomicAdd(ticket, 1);
        __syncthreads();
    }
}

#endif

}  // namespace rdst
