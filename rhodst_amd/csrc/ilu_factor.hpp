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
// FP32 partitions 2 M cells 2.16 / 5.8 ms, 24 k cells 0.25 / 0.52 ms; FP64 natural
// order 252 cells 0.20 / 0.52 ms, 23.5 k 4.5 / 9.5 ms, 321 k 5.5 / 9.9 ms.
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

// A row of the chain and its part of A, row r of each block in this lane.
template <class T, int K>
struct ChainRegs {
    int cell, cnt, lk[K];
    uint32_t dDst, lDst[K];
    T d[5], a[K][5], u[K][5];
};
template <class T, int K>
__device__ __forceinline__ void chain_load(const int32_t* __restrict__ rows, long t, int r, const T* __restrict__ A,
                                           ChainRegs<T, K>& R) {
    const int4* e = reinterpret_cast<const int4*>(rows + (4 + 4 * K) * (size_t)t);
    const int4 h = e[0];
    int4 n[K];
#pragma unroll
    for (int k = 0; k < K; ++k) n[k] = e[1 + k];
    R.cell = h.x;
    R.cnt = h.y;
    R.dDst = (uint32_t)h.w;
    const T* p = A + 25 * (size_t)h.z + 5 * r;
#pragma unroll
    for (int c = 0; c < 5; ++c) R.d[c] = p[c];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        R.lk[k] = n[k].z;
        R.lDst[k] = (uint32_t)n[k].w;
        const T* pa = A + 25 * (size_t)n[k].x + 5 * r;
        const T* pu = A + 25 * (size_t)n[k].y + 5 * r;
#pragma unroll
        for (int c = 0; c < 5; ++c) { R.a[k][c] = pa[c]; R.u[k][c] = pu[c]; }
    }
}
template <class T, int K>
__device__ __forceinline__ void chain_row(const ChainRegs<T, K>& R, bool on, int base, int r, T* Dinv, uint8_t* stream,
                                          int* fail) {
    T d[5];
#pragma unroll
    for (int c = 0; c < 5; ++c) d[c] = R.d[c];
#pragma unroll
    for (int k = 0; k < K; ++k)
        if (k < R.cnt) {
            const T* Dk = Dinv + 25 * (size_t)R.lk[k];
            T l[5];
#pragma unroll
            for (int j = 0; j < 5; ++j) {
                T s = 0;
#pragma unroll
                for (int q = 0; q < 5; ++q) s += R.a[k][q] * Dk[5 * q + j];
                l[j] = s;
            }
            if (on) {
                T* o = reinterpret_cast<T*>(stream + 4 * (size_t)R.lDst[k]) + 5 * r;
#pragma unroll
                for (int j = 0; j < 5; ++j) o[j] = l[j];
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
                for (int q = 0; q < 5; ++q) s += l[q] * u[q][j];
                d[j] -= s;
            }
        }
    T b[5];
    const int row = inv5_lanes(d, b, base, r);
    if (!on) return;
    if (row < 0) {
        atomicExch(fail, 1);
        return;
    }
    T* g = Dinv + 25 * (size_t)R.cell + 5 * row;
    T* o = reinterpret_cast<T*>(stream + 4 * (size_t)R.dDst) + 5 * row;
#pragma unroll
    for (int c = 0; c < 5; ++c) { g[c] = b[c]; o[c] = b[c]; }
}

// One partition's (or tile's) rows level by level; the rows of the pass after
// this one are loaded before this one is computed.
template <class T, int K>
__device__ __forceinline__ void chain_levels(int l0, int l1, const int32_t* __restrict__ levPtr,
                                             const int32_t* __restrict__ rows, const T* __restrict__ A, T* Dinv,
                                             uint8_t* stream, int* fail) {
    const int lane = threadIdx.x & 63, g = lane / 5, r = lane - 5 * g, base = lane - r;
    const int w12 = 12 * (int)(threadIdx.x >> 6), slot = g < 12 ? w12 + g : 1 << 20;
    int L = l0, s = levPtr[l0], e = levPtr[l0 + 1];
    ChainRegs<T, K> cur, nxt;
    // lanes without a row work on the pass's last row and store nothing
    chain_load<T, K>(rows, min(s + slot, e - 1), r, A, cur);
    while (L + 1 < l1) {
        int nL = L, ns = s + CHAIN_THREADS / 64 * 12, ne = e;
        if (ns >= e) {
            nL = L + 1;
            ns = e;
            ne = nL + 1 < l1 ? levPtr[nL + 1] : e;
        }
        const bool more = nL + 1 < l1;
        if (more) chain_load<T, K>(rows, min(ns + slot, ne - 1), r, A, nxt);
        if (s + w12 < e) chain_row<T, K>(cur, s + slot < e, base, r, Dinv, stream, fail);
        if (nL != L) __syncthreads();  // rows of a later level read what this one stored
        L = nL; s = ns; e = ne;
        if (more) cur = nxt;
    }
}

template <class T, int K>
__global__ __launch_bounds__(CHAIN_THREADS) void k_ilu_chain(const int32_t* __restrict__ levStart,
                                                             const int32_t* __restrict__ levPtr,
                                                             const int32_t* __restrict__ rows, const T* __restrict__ A,
                                                             T* Dinv, uint8_t* stream, int* fail) {
    const int p = blockIdx.x;
    chain_levels<T, K>(levStart[p], levStart[p + 1], levPtr, rows, A, Dinv, stream, fail);
}

// The natural-order factor by tiles, taken by ticket in an order that respects
// their dependencies (see k_tile_sweep); done[t] = epoch releases tile t's Dinv.
template <class T, int K>
__global__ __launch_bounds__(CHAIN_THREADS) void k_ilu_chain_tiles(int nT, int* ticket, int* done, int epoch,
                                                                   const int32_t* __restrict__ predStart,
                                                                   const int32_t* __restrict__ pred,
                                                                   const int32_t* __restrict__ levStart,
                                                                   const int32_t* __restrict__ levPtr,
                                                                   const int32_t* __restrict__ rows,
                                                                   const T* __restrict__ A, T* Dinv, uint8_t* stream,
                                                                   int* fail) {
    __shared__ int cur;
    if (threadIdx.x == 0) cur = atomicAdd(ticket, 1);
    __syncthreads();
    for (;;) {
        const int t = __builtin_amdgcn_readfirstlane(cur);
        if (t >= nT) break;
        for (int q = predStart[t] + (int)threadIdx.x; q < predStart[t + 1]; q += CHAIN_THREADS)
            while (__hip_atomic_load(done + pred[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != epoch)
                __builtin_amdgcn_s_sleep(2);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        __syncthreads();
        chain_levels<T, K>(levStart[t], levStart[t + 1], levPtr, rows, A, Dinv, stream, fail);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        __syncthreads();
        // Flag and next ticket under one condition, the barrier behind it: split
        // over the loop's end, with no barrier between, the compiler joins the two
        // across the back edge and lane 0 leaves its wavefront to loop without it.
        if (threadIdx.x == 0) {
            __hip_atomic_store(done + t, epoch, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
            cur = atomicAdd(ticket, 1);
        }
        __syncthreads();
    }
}

#endif

}  // namespace rdst
