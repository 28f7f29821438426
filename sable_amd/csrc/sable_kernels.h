// Hand-written gfx950 kernels of the VBR SpMV / SpMM hot path.
//
// This header is compiled twice: ahead of time by hipcc into libsable_amd.so
// (generic instances, the fallback), and at run time by hipRTC with the
// SB_* macros set per plan (the per-matrix specialisations).  It therefore
// includes nothing under hipRTC and uses only compiler builtins.
//
// Work decomposition (see the plan builder): a tile is a row segment of one
// block row; it owns those output rows and writes each exactly once, so no
// atomics touch y/Y and results are deterministic.  A tile's pieces are the
// column groups of its block row (dense FP32, dense FP32 in MFMA order, or
// sparse) of at most xcap columns each.  SpMV and the MFMA kernel stage a
// piece's x slice or X rows in LDS; the FP32 SpMM kernel, whose tiles are cut
// into tasks, reads X from memory into registers.
#pragma once

#include "sable_device.h"

#ifndef SB_WG
#define SB_WG 256
#endif
#ifndef SB_XCAP
#define SB_XCAP 4096
#endif
#ifndef SB_UNROLL
#define SB_UNROLL 4
#endif
#ifndef SB_NRHS
#define SB_NRHS 0          // 0 = runtime RHS width (generic instance)
#endif

typedef float sb_f4 __attribute__((ext_vector_type(4)));
typedef unsigned int sb_u4 __attribute__((ext_vector_type(4)));
typedef unsigned int sb_u2 __attribute__((ext_vector_type(2)));

// Global-address-space views of the buffer pointers.  The pointers come
// from descriptor tables (SbMatBufs), so the compiler cannot tell they point
// to global memory and would emit FLAT loads and stores; those count against
// the LDS counter as well, so every wait for an LDS access would also wait
// for every global load in flight, defeating the software pipelining.
#define SB_G __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ SB_G T *sb_gp(T *p)
{
    return (SB_G T *)p;
}
template <typename T>
__device__ __forceinline__ const SB_G T *sb_gp(const T *p)
{
    return (const SB_G T *)p;
}

// Read-only descriptors through the constant address space: scalar loads.
#define SB_K __attribute__((address_space(4)))
template <typename T>
__device__ __forceinline__ const SB_K T *sb_kp(const T *p)
{
    return (const SB_K T *)p;
}
// element i of a descriptor table (uniform i): a copy in scalar registers
template <typename T>
__device__ __forceinline__ T sb_kload(const T *p, int i)
{
    static_assert(sizeof(T) % 8 == 0, "descriptors are whole 8-byte words");
    const SB_K uint64_t *s = (const SB_K uint64_t *)(p + i);
    uint64_t w[sizeof(T) / 8];
#pragma unroll
    for (unsigned k = 0; k < sizeof(T) / 8; ++k) w[k] = s[k];
    return __builtin_bit_cast(T, w);
}

// a compile-time index for generic lambdas
template <int V>
struct SbInt {
    static constexpr int value = V;
};

#define SB_MODE_GRID 0      // one workgroup per tile
#define SB_MODE_STATIC 1    // persistent, tile = wg + k * grid
#define SB_MODE_QUEUE 2     // persistent, atomic work queue (self-resetting)

// The device arrays of one matrix of a group: each member keeps its own
// arrays (the group copies none of them) and a tile finds them through its
// matrix slot.  Piece and tile offsets are relative to these arrays.
struct SbMatBufs {
    const float *dval;
    const float *sval;
    const uint16_t *sidx;
    const int32_t *srowptr;
    const int32_t *xmap;          // SpMV: the staging map; SpMM: scol
    const float *x;               // x (SpMV) or X [ncols x n_rhs] (SpMM)
    float *y;                     // y (SpMV) or Y [nrows x n_rhs] (SpMM)
    float *part;                  // SpMM: partial sums of the split MFMA tiles
};

struct SbSpmvArgs {
    const SbTile *tiles;
    const SbPiece *pieces;
    const SbXRange *xr;
    const float *dval;
    const float *sval;
    const uint16_t *sidx;
    const int32_t *srowptr;
    const int32_t *xmap;          // x column per staged slot (-1: zero pad)
    const SbMatBufs *mats;        // per matrix slot (groups), or null: the fields above
    const float *x0;              // single plan: x
    float *y0;                    // single plan: y
    float *part;                  // unused (SpMM only)
    int32_t *queue;               // [0] next tile, [1] retired workgroups
    int32_t ntiles;
    int32_t mode;
};

struct SbSpmmArgs {
    const SbTile *tiles;
    const SbPiece *pieces;
    const SbXRange *xr;
    const float *dval;            // FP32 dense pieces (column-major) and MFMA pieces (register order)
    const float *sval;
    const uint16_t *sidx;
    const int32_t *srowptr;
    const int32_t *scol;          // X row of every sparse entry
    const SbMatBufs *mats;        // per matrix slot (groups), or null: the fields above
    const float *x0;              // single plan: X
    float *y0;                    // single plan: Y
    float *part;                  // single plan: partial sums of the split MFMA tiles
    int32_t *queue;
    int32_t ntiles;
    int32_t mode;
    int32_t n_rhs;
    const SbTask *tasks;          // FP32 kernel: its work list (ntiles tasks)
};

// The arrays a tile reads: its matrix slot's in a group, else the plan's.
template <typename Args>
__device__ __forceinline__ SbMatBufs sb_mat_bufs(const Args &a, int mat, const int32_t *xmap)
{
    if (a.mats) return a.mats[mat];
    SbMatBufs b;
    b.dval = a.dval;
    b.sval = a.sval;
    b.sidx = a.sidx;
    b.srowptr = a.srowptr;
    b.xmap = xmap;
    b.x = a.x0;
    b.y = a.y0;
    b.part = a.part;
    return b;
}

// ---------------------------------------------------------------------------
// Work distribution helpers

// Runs body(t) over the tiles according to mode.  The queue counters are
// reset by the last workgroup to retire, so the kernel can be relaunched or
// replayed from a graph without a memset.
template <typename Body>
__device__ __forceinline__ void sb_for_tiles(int ntiles, int mode, int32_t *queue,
                                             int *next_tile, Body body)
{
    if (mode == SB_MODE_GRID) {
        if ((int)blockIdx.x < ntiles) body((int)blockIdx.x);
        return;
    }
    if (mode == SB_MODE_STATIC) {
        for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
            body(t);
            __syncthreads();
        }
        return;
    }
    for (;;) {
        if (threadIdx.x == 0) *next_tile = atomicAdd(&queue[0], 1);
        __syncthreads();
        const int t = *next_tile;
        __syncthreads();
        if (t >= ntiles) break;
        body(t);
    }
    if (threadIdx.x == 0) {
        __threadfence();
        const int done = atomicAdd(&queue[1], 1);
        if (done == (int)gridDim.x - 1) {
            atomicExch(&queue[0], 0);
            atomicExch(&queue[1], 0);
        }
    }
}

// ---------------------------------------------------------------------------
// SpMV
//
// A tile's pieces are processed in staging groups (formed by the host):
// consecutive pieces whose x slices (each followed by 4 zero pads) fit in the
// LDS buffer are staged in one pass through the group's slot map (x column
// per slot), then processed.  Sparse pieces come first in a group.
//
// Roles: lanes tid < T' stream the dense pieces.  In a tile with both kinds
// the last sp_waves wavefronts take the sparse pieces (their loads are
// latency-bound and run alongside the dense stream); otherwise every
// wavefront takes both in turn.
//
// Dense piece = column-major hs x ncols FP32 sub-panel, contiguous, 16-byte
// aligned, zero-padded to a multiple of 4 floats and followed by one zero
// float4, streamed as float4: lane t
// (t < T') reads float4 q = t + k*T'.  Because 4*T' = M*hs, lane t always
// sees the same four row indices (4t+s) % hs and walks columns (4t+s)/hs +
// k*M, so each lane accumulates four fixed rows in registers and every
// wavefront load is a fully coalesced 16-byte access.  Loads are software
// pipelined (two register batches of UNROLL float4).
//
// Sparse piece = wave slices (laid out by the host plan): the tile's rows,
// longest first, are cut into slices of C = 64/G rows, slice s going to
// sparse wavefront s % nsw, G lanes per row; at step j lane q*G+g holds
// entries 4(jG+g) .. 4(jG+g)+3 of its row (uint16 columns into the staged x
// slice).  A wavefront streams a slice's steps as one coalesced float4 + 4 x
// uint16 load per lane, accumulates in a register, folds the G lanes of a
// row with a fixed xor butterfly and adds the row sum to the row's LDS slot
// spy[r].  The same lane owns a row in every sparse piece of the tile, so
// spy needs no barrier between pieces.
//
// Row r's result is (dense partial sums of the M column groups, in group
// order) + (sparse sums, piece by piece): deterministic, no atomics.

struct SbStreamLane {
    int c0, c1, c2, c3;    // column offsets of this lane's four elements
};

// Loads are unconditional and nothing is applied to their values until the
// batch is consumed, so the compiler can wait for one batch while the next
// is still in flight: an index past the end reads the zero float4 the plan
// builder appends after every dense piece (P[nq]).
template <int UNROLL>
__device__ __forceinline__ void sb_dense_load(const SB_G sb_f4 *__restrict__ P, int nq, int q0, int tpar,
                                              sb_f4 *v)
{
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
        const int q = q0 + u * tpar;
        v[u] = __builtin_nontemporal_load(&P[q < nq ? q : nq]);
    }
}

// The x index is clamped to the slice's first zero pad (xs[ncols]): past the
// end of the stream the loaded value is zero and so is the x it meets.
template <int UNROLL>
__device__ __forceinline__ void sb_dense_fma(const sb_f4 *v, const float *xs, const SbStreamLane &L, int kc,
                                             int M, int ncols, float &a0, float &a1, float &a2, float &a3)
{
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
        const int k = kc + u * M;
        a0 += v[u].x * xs[min(L.c0 + k, ncols)];
        a1 += v[u].y * xs[min(L.c1 + k, ncols)];
        a2 += v[u].z * xs[min(L.c2 + k, ncols)];
        a3 += v[u].w * xs[min(L.c3 + k, ncols)];
    }
}

// Streams one dense piece whose x slice starts at xs; cur holds its first
// batch.
template <int UNROLL>
__device__ __forceinline__ void sb_dense_piece(const SB_G sb_f4 *__restrict__ P, int nq, int tpar, int M, int ncols,
                                               const float *xs, const SbStreamLane &L, sb_f4 *cur, float &a0,
                                               float &a1, float &a2, float &a3)
{
    const int tid = threadIdx.x;
    const int nmine = (nq - 1 - tid) / tpar + 1;             // float4 loads of this lane
    const int nbatch = (nmine + UNROLL - 1) / UNROLL;
    // The register copy cur = nxt waits for the batch it copies, so one
    // batch is in flight per round trip.  A copy-free form (two buffers that
    // trade roles) keeps two in flight but needs about 113 VGPRs (4 waves
    // per SIMD, two 512-thread workgroups per CU) and measured no faster on
    // the 100k matrix: the kernel runs at about 90 % of a cold streaming
    // read of the same bytes either way.
    sb_f4 nxt[UNROLL];
    for (int b = 0; b < nbatch; ++b) {
        // always prefetch (the batch after the last one reads the zero float4)
        sb_dense_load<UNROLL>(P, nq, tid + (b + 1) * UNROLL * tpar, tpar, nxt);
        sb_dense_fma<UNROLL>(cur, xs, L, b * UNROLL * M, M, ncols, a0, a1, a2, a3);
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) cur[u] = nxt[u];
    }
}

// Stages a group's x slices into xs through its slot map (x column per slot,
// -1 for the zero pads): two dependent loads per slot, 4 slots in flight per
// thread, no search over descriptors.  issue() runs while the first map
// loads are under way.
template <int WG, typename Issue>
__device__ __forceinline__ void sb_stage_map(const SB_G int32_t *__restrict__ map, int total,
                                             const SB_G float *__restrict__ x, float *xs, Issue issue)
{
    for (int i0 = 0; i0 < total; i0 += 4 * WG) {
        int m[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = i0 + u * WG + (int)threadIdx.x;
            m[u] = i < total ? __builtin_nontemporal_load(&map[i]) : -1;
        }
        if (i0 == 0) issue();
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = m[u] >= 0 ? x[m[u]] : 0.f;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = i0 + u * WG + (int)threadIdx.x;
            if (i < total) xs[i] = v[u];
        }
    }
}

// One slice of a sparse piece, streamed by one wavefront: its step range
// from the table (wave-uniform), loads unconditional (the step index is
// clamped to the last step) and software pipelined one batch ahead; steps
// past the slice's count are masked to value 0 at the zero pad slot xs[pad].
// The G lanes of a row are folded with a fixed xor butterfly and the
// row-owner lane adds the sum to spy[row].
template <int SU>
__device__ __forceinline__ void sb_sparse_slice(const SB_G float *__restrict__ sval,
                                                const SB_G uint16_t *__restrict__ sidx,
                                                const SB_G int32_t *__restrict__ tab, const SB_G int32_t *__restrict__ map,
                                                int hs, int glog, int slice, int pad, const float *xs, float *spy)
{
    const int lane = threadIdx.x & 63;
    const int off = tab[2 * slice];
    const int nst = tab[2 * slice + 1];
    if (nst <= 0) return;
    const int i = slice * (64 >> glog) + (lane >> glog);
    const bool owner = (lane & ((1 << glog) - 1)) == 0 && i < hs;
    const int row = owner ? map[i] : 0;
    const SB_G sb_f4 *__restrict__ V = reinterpret_cast<const SB_G sb_f4 *>(sval) + (int64_t)off * 64 + lane;
    const SB_G sb_u2 *__restrict__ I = reinterpret_cast<const SB_G sb_u2 *>(sidx) + (int64_t)off * 64 + lane;
    const unsigned padpair = (unsigned)pad | ((unsigned)pad << 16);
    sb_f4 cv[SU];
    sb_u2 ci[SU];
#pragma unroll
    for (int u = 0; u < SU; ++u) {
        const int j = min(u, nst - 1);
        cv[u] = __builtin_nontemporal_load(V + (int64_t)j * 64);
        ci[u] = __builtin_nontemporal_load(I + (int64_t)j * 64);
    }
    float acc = 0.f;
    for (int j0 = 0; j0 < nst; j0 += SU) {
        sb_f4 nv[SU];
        sb_u2 ni[SU];
#pragma unroll
        for (int u = 0; u < SU; ++u) {
            const int j = min(j0 + SU + u, nst - 1);
            nv[u] = __builtin_nontemporal_load(V + (int64_t)j * 64);
            ni[u] = __builtin_nontemporal_load(I + (int64_t)j * 64);
        }
#pragma unroll
        for (int u = 0; u < SU; ++u) {
            const bool ok = j0 + u < nst;
            const unsigned lo = ok ? ci[u].x : padpair;
            const unsigned hi = ok ? ci[u].y : padpair;
            acc += (ok ? cv[u].x : 0.f) * xs[lo & 0xffffu];
            acc += (ok ? cv[u].y : 0.f) * xs[lo >> 16];
            acc += (ok ? cv[u].z : 0.f) * xs[hi & 0xffffu];
            acc += (ok ? cv[u].w : 0.f) * xs[hi >> 16];
        }
#pragma unroll
        for (int u = 0; u < SU; ++u) {
            cv[u] = nv[u];
            ci[u] = ni[u];
        }
    }
    for (int m = 1; m < (1 << glog); m <<= 1) acc += __shfl_xor(acc, m, 64);
    if (owner) spy[row] += acc;
}

template <int WG, int UNROLL, int XCAP>
__device__ __forceinline__ void sb_spmv_tile(const SbSpmvArgs &a, int t, float *xs, float *red, float *spy)
{
    const int tid = threadIdx.x;
    const SbTile tile = sb_kload(a.tiles, __builtin_amdgcn_readfirstlane(t));
    const int hs = tile.nrows;
    const int tpar = tile.dense_tpar;
    const int M = tile.dense_mcols;
    const SbMatBufs mb = a.mats ? sb_kload(a.mats, tile.mat) : sb_mat_bufs(a, 0, a.xmap);
    const SB_G float *__restrict__ x = sb_gp(mb.x);
    SB_G float *__restrict__ y = sb_gp(mb.y);

    SbStreamLane L;
    float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
    if (tid < hs) spy[tid] = 0.f;   // before the first staging barrier; sparse row owners add after it
    // roles: lanes tid < tpar stream the dense pieces; the last nsw
    // wavefronts (all of them when sp_waves == 0) take the sparse slices
    constexpr int NW = WG / 64;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nsw = tile.sp_waves > 0 ? tile.sp_waves : NW;
    const int sw = wave - (NW - nsw);                     // sparse wavefront index, < 0: none
    const int nsl = (hs + (64 >> tile.sp_glog) - 1) / (64 >> tile.sp_glog);   // sparse slices
    int pb = tile.piece_begin;
    bool head = true;
    while (pb < tile.piece_end) {
        // staging group [pb, pe), formed by the host (stage_len <= XCAP + 4
        // slots); the first group's map offset and length come with the
        // tile, so its map loads need not wait for the piece descriptor
        const SbPiece first = sb_kload(a.pieces, pb);
        const SbPiece second = sb_kload(a.pieces, pb + 1);    // the array has slack behind it
        const int smap = head ? tile.stage_map : first.xmap_off;
        const int slen = head ? tile.stage_len : first.stage_len;
        if (slen > XCAP + 4) break;            // never built (the host and kernel choice check)
        __syncthreads();                       // previous group done with xs
        // A tile is a chain of round trips (tile, pieces, map, x, values), so
        // what needs no x goes ahead of it: the first batch of the group's
        // first dense piece (its first or second piece, else it is loaded
        // when its turn comes) is in flight while x is staged.  With the
        // descriptors in scalar registers (nothing spilled; 8 VGPRs were)
        // this took the kernel from 5.0 to 4.0 us at 1,000 rows, 9.8 to 7.6
        // at 30,011 and 49.8 to 47.8 at 100,000 (warm caches).
        const int ahead = first.kind == SB_PIECE_DENSE                                       ? pb
                          : second.kind == SB_PIECE_DENSE && first.grp_end > pb + 1 ? pb + 1
                                                                                             : -1;
        // (Without one, and on the lanes past tpar, the loads read some 16
        // bytes that exist: a branch here would make x wait for the batch.)
        const int64_t aoff = ahead == pb ? first.data_off : second.data_off;
        const int anq = ahead < 0 ? 0 : (hs * (ahead == pb ? first.ncols : second.ncols) + 3) >> 2;
        const SB_G sb_f4 *AP = ahead < 0 ? reinterpret_cast<const SB_G sb_f4 *>(sb_gp(a.tiles))
                                         : reinterpret_cast<const SB_G sb_f4 *>(sb_gp(mb.dval) + aoff);
        sb_f4 cur[UNROLL];
        sb_stage_map<WG>(sb_gp(mb.xmap) + smap, slen, x, xs, [&] {
            sb_dense_load<UNROLL>(AP, anq, tid < tpar ? tid : anq, tpar, cur);
            if (head) {
                const int p0 = 4 * tid;
                L.c0 = p0 / hs;
                L.c1 = (p0 + 1) / hs;
                L.c2 = (p0 + 2) / hs;
                L.c3 = (p0 + 3) / hs;
            }
        });
        head = false;
        __syncthreads();
        const int pe = first.grp_end;
        if (pe <= pb) break;                   // never built
        int base = 0;
        for (int p = pb; p < pe; ++p) {
            const SbPiece pc = sb_kload(a.pieces, p);
            if (pc.kind == SB_PIECE_DENSE) {
                const SB_G sb_f4 *P = reinterpret_cast<const SB_G sb_f4 *>(sb_gp(mb.dval) + pc.data_off);
                const int nq = (hs * pc.ncols + 3) >> 2;
                if (tid < tpar && tid < nq) {
                    if (p != ahead) sb_dense_load<UNROLL>(P, nq, tid, tpar, cur);
                    sb_dense_piece<UNROLL>(P, nq, tpar, M, pc.ncols, xs + base, L, cur, a0, a1, a2, a3);
                }
            } else if (sw >= 0) {
                // this wavefront's slices sw, sw + nsw, ...
                for (int sl = sw; sl < nsl; sl += nsw) {
                    sb_sparse_slice<SB_SPUNROLL>(sb_gp(mb.sval) + pc.data_off, sb_gp(mb.sidx) + pc.data_off,
                                                 sb_gp(mb.srowptr) + pc.rowptr_off, sb_gp(mb.srowptr) + tile.sp_map, hs,
                                                 tile.sp_glog, sl, pc.ncols, xs + base,
                                                 spy);
                }
            }
            base += pc.ncols + 4;
        }
        pb = pe;
    }

    __syncthreads();
    if (tid < tpar) {
        red[4 * tid] = a0;
        red[4 * tid + 1] = a1;
        red[4 * tid + 2] = a2;
        red[4 * tid + 3] = a3;
    }
    __syncthreads();
    // red holds M groups of hs partial sums: red[m*hs + r].  Fold halves while
    // there are many groups (short tiles), then each row owner sums in order.
    int m = M;
    while (m > 32) {
        const int half = (m + 1) >> 1;
        const int cnt = (m - half) * hs;
        for (int i = tid; i < cnt; i += WG) red[i] += red[i + half * hs];
        __syncthreads();
        m = half;
    }
    if (tid < hs) {
        float s = 0.f;
        for (int g = 0; g < m; ++g) s += red[g * hs + tid];
        y[tile.row0 + tid] = s + spy[tid];
    }
}

template <int WG, int UNROLL, int XCAP>
__device__ __forceinline__ void sb_spmv_body(const SbSpmvArgs &a)
{
    __shared__ float xs[XCAP + 4];
    __shared__ float red[4 * WG];
    __shared__ float spy[WG];
    __shared__ int next_tile;
    sb_for_tiles(a.ntiles, a.mode, a.queue, &next_tile,
                 [&](int t) { sb_spmv_tile<WG, UNROLL, XCAP>(a, t, xs, red, spy); });
}

// ---------------------------------------------------------------------------
// SpMM, FP32 (dense pieces on the FP32 matrix instructions, sparse pieces on
// the vector ALUs)
//
// A wavefront owns up to 32 rows x 64 columns of Y, keeps them in
// accumulators and streams its operands from memory into registers; no data
// goes through LDS.  The host's task list (SbTask) keeps the workgroups of a
// tile on one XCD, whose L2 then serves the panel and X rows they share.
//
// Dense pieces: v_mfma_f32_16x16x4_f32, whose lane l holds A[l%16][l/16] and
// B[l/16][l%16] (products and sums in FP32).  Which 16 rows and columns a
// fragment holds is free as long as loads and stores agree, so fragment u of
// U takes rows U*i + u and fragment t of T columns T*j + t (i, j = l%16): a
// lane's U rows of a panel column are one vector load and its T columns of
// an X row another, whole cache lines per wavefront, and its results are
// T-column vectors of Y.  Per 4 columns of A: two vector loads and U*T
// matrix instructions of 32 clocks each.
//
// Bound: the matrix instructions (256 FLOP per clock and CU, 157 TFLOP/s),
// twice the vector ALUs' rate without packed instructions.  The vector
// kernel this replaced (4 rows x 8 columns per thread, X staged in LDS) took
// 260 us on the 50,000-row SpMM at N = 128 (35 M dense values, 0.9 M
// entries) and 122 us on a 3,001-row one at N = 512; this one takes 173 and
// 35 us.  Uniform tiles (256 block rows of 16 blocks of 128 x 128) run at
// 113 TFLOP/s, the matrix units busy for 73 % of the launch, with 0.3 other
// vector instructions and 0.25 loads per matrix instruction and the
// wavefronts queued at the issue (72 % of their cycles).  On the 50,000-row
// SpMM they are busy for 37 %: 1.9 other vector instructions (the entries'
// products) and 0.45 loads per matrix instruction, 54 % of the wavefronts'
// cycles waiting for loads.  Measured slower there, dense blocks alone / with
// the entries, against 127 / 175 us: X staged through LDS (149 / 188 us),
// 32-column tasks (155 / 213 us), one wavefront per workgroup without the
// barrier (132 / 184 us).

// entries whose X rows are in flight in a task without dense pieces (4, 8 or 16)
#ifndef SB_F32_SPARSE_FLIGHT
#define SB_F32_SPARSE_FLIGHT 8
#endif
// waves per SIMD the launch bound asks of the compiler
#ifndef SB_F32_MINWAVES
#define SB_F32_MINWAVES 4
#endif

typedef float sb_f2 __attribute__((ext_vector_type(2)));
typedef float sb_c4 __attribute__((ext_vector_type(4)));      // accumulator fragment

// V consecutive floats at p (aligned to their size)
template <int V>
__device__ __forceinline__ void sb_load_v(const SB_G float *p, float (&o)[V])
{
    if constexpr (V == 4) {
        const sb_f4 v = *reinterpret_cast<const SB_G sb_f4 *>(p);
        o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
    } else if constexpr (V == 2) {
        const sb_f2 v = *reinterpret_cast<const SB_G sb_f2 *>(p);
        o[0] = v.x; o[1] = v.y;
    } else {
        o[0] = *p;
    }
}

// the same from a uniform base and a 32-bit byte offset (scalar-base loads)
template <int V>
__device__ __forceinline__ void sb_load_off(const SB_G float *base, uint32_t bytes, float (&o)[V])
{
    sb_load_v<V>(reinterpret_cast<const SB_G float *>(reinterpret_cast<const SB_G char *>(base) + bytes), o);
}

template <int V>
__device__ __forceinline__ void sb_store_v(SB_G float *p, const float (&o)[V])
{
    if constexpr (V == 4) *reinterpret_cast<SB_G sb_f4 *>(p) = sb_f4{o[0], o[1], o[2], o[3]};
    else if constexpr (V == 2) *reinterpret_cast<SB_G sb_f2 *>(p) = sb_f2{o[0], o[1]};
    else *p = o[0];
}

// Lane K of every 16-lane row (BATCH 16) or of every quad (BATCH 4), to all
// lanes of that row or quad.
template <int BATCH, int K>
__device__ __forceinline__ int sb_bcast(int v)
{
    if constexpr (BATCH == 16) return __builtin_amdgcn_update_dpp(0, v, 0x150 + K, 0xf, 0xf, true);   // row_newbcast:K
    else return __builtin_amdgcn_update_dpp(0, v, K * 0x55, 0xf, 0xf, true);                          // quad_perm:[K,K,K,K]
}

template <int I, int E, typename F>
__device__ __forceinline__ void sb_static_for(F f)
{
    if constexpr (I < E) {
        f(SbInt<I>{});
        sb_static_for<I + 1, E>(f);
    }
}

// Adds a batch of a row's entries (lane e of the batch holds entry e: value
// and X row) to the row's V columns at X + co: n entries of this lane's row
// are valid (n may differ between the rows of a wavefront), most is the
// largest n, least the smallest.  F entries' X rows are in flight at a time.
// Where some row has run out, its entries repeat its last X row and add
// nothing: the caller gives the value 0 there and X is taken as 0, so neither
// a value nor an X that is not finite gets into another entry's sum.  FAR: X
// is 4 GiB or more.
template <int BATCH, int F, int V, bool FAR>
__device__ __forceinline__ void sb_f32_entries(const SB_G float *__restrict__ X, int N, uint32_t co, float val, int col,
                                               int n, int least, int most, float (&acc)[V])
{
    const int off = FAR ? col : (int)((uint32_t)col * (uint32_t)N * 4u);
    sb_static_for<0, BATCH / F>([&](auto bc) {
        constexpr int b = decltype(bc)::value;
        if (F * b < most) {
            float x[F][V];
            sb_static_for<0, F>([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                const int o = sb_bcast<BATCH, F * b + k>(off);
                if (FAR) sb_load_v<V>(X + ((int64_t)o * N + co), x[k]);
                else sb_load_off<V>(X, (uint32_t)o + co * 4u, x[k]);
            });
            if (F * b + F > least) {
#pragma unroll
                for (int k = 0; k < F; ++k)
#pragma unroll
                    for (int j = 0; j < V; ++j) x[k][j] = F * b + k < n ? x[k][j] : 0.f;
            }
            sb_static_for<0, F>([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                const float v = __builtin_bit_cast(float, sb_bcast<BATCH, F * b + k>(__builtin_bit_cast(int, val)));
#pragma unroll
                for (int j = 0; j < V; ++j) acc[j] += v * x[k][j];
            });
        }
    });
}

// the largest and smallest of a value that is the same over every 2^LOGL lanes
template <int LOGL>
__device__ __forceinline__ void sb_range_of(int n, int &least, int &most)
{
    if constexpr (LOGL >= 4) {
        least = most = __builtin_amdgcn_readlane(n, 0);
#pragma unroll
        for (int l = 1 << LOGL; l < 64; l += 1 << LOGL) {
            const int v = __builtin_amdgcn_readlane(n, l);
            least = min(least, v);
            most = max(most, v);
        }
    } else {
        int a = n, b = n;
#pragma unroll
        for (int m = 1 << LOGL; m < 64; m <<= 1) {
            a = min(a, __shfl_xor(a, m, 64));
            b = max(b, __shfl_xor(b, m, 64));
        }
        least = __builtin_amdgcn_readfirstlane(a);
        most = __builtin_amdgcn_readfirstlane(b);
    }
}

// A task with dense pieces: rows [r0, r0 + 16U) of its tile, columns
// [n0, n0 + 16T) of Y.
template <int U, int T, bool FAR>
__device__ __forceinline__ void sb_f32_task(const SbSpmmArgs &a, const SbTask &tk, const SbMatBufs &mb, int r0, int N)
{
    const int lane = threadIdx.x & 63;
    const int i = lane & 15, g = lane >> 4;
    const int hs = tk.nrows, n0 = tk.n0;
    const int pitch = (hs + 3) & ~3;             // every dense piece of the tile
    const SB_G float *__restrict__ X = sb_gp(mb.x);
    const SB_K SbPiece *pieces = sb_kp(a.pieces);
    const SB_K SbXRange *xr = sb_kp(a.xr);
    // this lane's rows in a panel column and columns in an X row; past the
    // panel or the right-hand side they repeat the last ones (never stored)
    const uint32_t ro = min(r0 + U * i, pitch - U);
    const uint32_t co = min(n0 + T * i, N - T);
    const uint32_t va = 4u * (g * pitch + ro), vb = 4u * ((uint32_t)g * N + co);
    sb_c4 acc[U][T];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int t = 0; t < T; ++t) acc[u][t] = sb_c4{0.f, 0.f, 0.f, 0.f};

    // Each dense piece: the walk over its columns, 8 of one X range per step
    // (two products of 4), loads SB_F32_DEPTH steps ahead of the products.
    // Vector instructions take the matrix instructions' time (both run on the
    // FP32 lanes), so a full step has none: its loads are a scalar base plus
    // this lane's fixed offsets.  At the end of a range the lanes past it
    // repeat its last column and are zeroed before their products; past the
    // last range all are, so the loads are unconditional.
    constexpr int D = SB_F32_DEPTH;
    int pi = tk.piece_begin;
    for (; pi < tk.piece_end && pieces[pi].kind == SB_PIECE_DENSE; ++pi) {
        int r = pieces[pi].xr_begin;
        const int re = pieces[pi].xr_end;
        int left = xr[r].len;
        const SB_G float *pa = sb_gp(mb.dval) + pieces[pi].data_off;
        const SB_G float *px = X + (int64_t)xr[r].col0 * N;
        float av[D][2][U], bv[D][2][T];
        int rem[D];
        auto fetch = [&](int d) {
            rem[d] = left;
            uint32_t oa0 = va, ob0 = vb, oa1 = va + 16u * pitch, ob1 = vb + 16u * N;
            if (left < 8) {
                const int g0 = max(min(g, left - 1), 0), g1 = max(min(g + 4, left - 1), 0);
                oa0 = 4u * (g0 * pitch + ro);
                ob0 = 4u * ((uint32_t)g0 * N + co);
                oa1 = 4u * (g1 * pitch + ro);
                ob1 = 4u * ((uint32_t)g1 * N + co);
            }
            // 32-bit offsets of scalar-base loads, not hoisted to 64-bit adds
            asm volatile("" : "+v"(oa0), "+v"(ob0), "+v"(oa1), "+v"(ob1));
            sb_load_off<U>(pa, oa0, av[d][0]);
            sb_load_off<T>(px, ob0, bv[d][0]);
            sb_load_off<U>(pa, oa1, av[d][1]);
            sb_load_off<T>(px, ob1, bv[d][1]);
            if (left > 8) {
                left -= 8;
                pa += 8 * pitch;
                px += (int64_t)8 * N;
            } else if (r + 1 < re) {
                ++r;
                pa += left * pitch;
                left = xr[r].len;
                px = X + (int64_t)xr[r].col0 * N;
            } else {
                left = 0;
            }
        };
#pragma unroll
        for (int d = 0; d < D; ++d) fetch(d);
        // one exit per round of D steps (several would make the compiler wait
        // for every load in flight at the loop's head): the last round's
        // steps past the end multiply zeros
        do {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                if (rem[d] < 8) {
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const bool ok = g + 4 * h < rem[d];
#pragma unroll
                        for (int u = 0; u < U; ++u) av[d][h][u] = ok ? av[d][h][u] : 0.f;
#pragma unroll
                        for (int t = 0; t < T; ++t) bv[d][h][t] = ok ? bv[d][h][t] : 0.f;
                    }
                }
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int u = 0; u < U; ++u)
#pragma unroll
                        for (int t = 0; t < T; ++t)
                            acc[u][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[d][h][u], bv[d][h][t], acc[u][t], 0, 0, 0);
                fetch(d);
            }
            // the workgroup's wavefronts read the same X rows: a barrier per
            // round (no data passes) keeps them close, so all but the first
            // read find them in L1
            __builtin_amdgcn_s_barrier();
        } while (rem[0] > 0);
    }

    // Sparse pieces, into the same accumulators: lane (g, i) holds rows
    // U*(4g + q) + u (q < 4) and T columns of each, so the four 16-lane rows
    // of the wavefront walk the entries of four Y rows side by side.
    for (; pi < tk.piece_end; ++pi) {
        if (pieces[pi].kind != SB_PIECE_SPARSE) continue;
        const SB_G int32_t *__restrict__ rp = sb_gp(mb.srowptr) + pieces[pi].rowptr_off;
        const SB_G float *__restrict__ sv = sb_gp(mb.sval) + pieces[pi].data_off;
        const SB_G int32_t *__restrict__ sc = sb_gp(mb.xmap) + pieces[pi].data_off;
        int lo[U][4], n[U][4], c0[U][4];
        float v0[U][4];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int row = r0 + U * (4 * g + q) + u;
                lo[u][q] = rp[min(row, hs - 1)];
                n[u][q] = (row < hs ? rp[min(row, hs - 1) + 1] : lo[u][q]) - lo[u][q];
            }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                // past the row's end (an empty row's entry is not its own): 0
                const int e = lo[u][q] + max(min(i, n[u][q] - 1), 0);
                const float v = sv[e];
                v0[u][q] = i < n[u][q] ? v : 0.f;
                c0[u][q] = sc[e];
            }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float s[T];
#pragma unroll
                for (int t = 0; t < T; ++t) s[t] = acc[u][t][q];
                int least, most;
                sb_range_of<4>(n[u][q], least, most);
                float v = v0[u][q];
                int c = n[u][q] > 0 ? c0[u][q] : 0;
                for (int e0 = 0; e0 < most; e0 += 16) {
                    if (e0 > 0) {
                        const int e = lo[u][q] + max(min(e0 + i, n[u][q] - 1), 0);
                        v = sv[e];
                        v = e0 + i < n[u][q] ? v : 0.f;
                        c = n[u][q] > 0 ? sc[e] : 0;
                    }
                    sb_f32_entries<16, 4, T, FAR>(X, N, co, v, c, n[u][q] - e0, least - e0, most - e0, s);
                }
#pragma unroll
                for (int t = 0; t < T; ++t) acc[u][t][q] = s[t];
            }
    }

    if (n0 + T * i + T > N) return;
    SB_G float *__restrict__ Y = sb_gp(mb.y) + (int64_t)tk.row0 * N;
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int row = r0 + U * (4 * g + q) + u;
            if (row >= hs) continue;
            SB_G float *dst = Y + (int64_t)row * N + co;
            float o[T], w[T];
#pragma unroll
            for (int t = 0; t < T; ++t) o[t] = acc[u][t][q];
            if (tk.y_accum) {          // the rows' MFMA tile wrote Y in the previous launch
                sb_load_v<T>(dst, w);
#pragma unroll
                for (int t = 0; t < T; ++t) o[t] += w[t];
            }
            sb_store_v<T>(dst, o);
        }
}

// A task of a tile without dense pieces: 2^LOGL lanes per row, one float4 of
// X and Y each (the least that cover N, at least 4 and at most 64; column
// chunk ch beyond that), so the wavefront walks 64 >> LOGL rows side by side
// and every X row it meets is one contiguous read.  Its SB_F32_SPARSE_ITERS
// sets of rows are started together: row pointers of all, first entries of
// all, then the X rows, so three dependent loads are met once per task and
// not once per row.
template <int LOGL, bool FAR>
__device__ __forceinline__ void sb_f32_sparse_task(const SbSpmmArgs &a, const SbTask &tk, const SbMatBufs &mb, int N)
{
    constexpr int L = 1 << LOGL, G = 64 >> LOGL, BATCH = L >= 16 ? 16 : 4, IT = SB_F32_SPARSE_ITERS;
    constexpr int F = L >= 16 ? SB_F32_SPARSE_FLIGHT : 4;
    const int lane = threadIdx.x & 63;
    const int q = lane & (BATCH - 1);
    const int col = tk.n0 + 4 * (lane & (L - 1));
    const int r0 = tk.r0 + SB_F32_SPARSE_ROWS(N) * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (r0 >= tk.nrows) return;
    const uint32_t co = min(col, N - 4);
    const int hs = tk.nrows;
    const SB_G float *__restrict__ X = sb_gp(mb.x);
    SB_G float *__restrict__ Y = sb_gp(mb.y) + (int64_t)tk.row0 * N + co;
    const SB_K SbPiece *pieces = sb_kp(a.pieces);
    float s[IT][4];
#pragma unroll
    for (int k = 0; k < IT; ++k) s[k][0] = s[k][1] = s[k][2] = s[k][3] = 0.f;
    for (int pi = tk.piece_begin; pi < tk.piece_end; ++pi) {
        const SB_G int32_t *__restrict__ rp = sb_gp(mb.srowptr) + pieces[pi].rowptr_off;
        const SB_G float *__restrict__ sv = sb_gp(mb.sval) + pieces[pi].data_off;
        const SB_G int32_t *__restrict__ sc = sb_gp(mb.xmap) + pieces[pi].data_off;
        int lo[IT], n[IT], c0[IT];
        float v0[IT];
#pragma unroll
        for (int k = 0; k < IT; ++k) {
            const int row = r0 + k * G + (lane >> LOGL), rr = min(row, hs - 1);
            lo[k] = rp[rr];
            n[k] = (row < hs ? rp[rr + 1] : lo[k]) - lo[k];
        }
#pragma unroll
        for (int k = 0; k < IT; ++k) {
            // past the row's end (an empty row's entry is not its own): 0
            const int e = lo[k] + max(min(q, n[k] - 1), 0);
            const float v = sv[e];
            v0[k] = q < n[k] ? v : 0.f;
            c0[k] = sc[e];
        }
#pragma unroll
        for (int k = 0; k < IT; ++k) {
            int least, most;
            sb_range_of<LOGL>(n[k], least, most);
            float v = v0[k];
            int c = n[k] > 0 ? c0[k] : 0;
            for (int e0 = 0; e0 < most; e0 += BATCH) {
                // the next batch's entries, ahead of this one's X rows
                const int e = lo[k] + max(min(e0 + BATCH + q, n[k] - 1), 0);
                const float vn = sv[e];
                const int cn = sc[e];
                sb_f32_entries<BATCH, F, 4, FAR>(X, N, co, v, c, n[k] - e0, least - e0, most - e0, s[k]);
                v = e0 + BATCH + q < n[k] ? vn : 0.f;
                c = n[k] > 0 ? cn : 0;
            }
        }
    }
    if (col >= N) return;
#pragma unroll
    for (int k = 0; k < IT; ++k) {
        const int row = r0 + k * G + (lane >> LOGL);
        if (row >= hs) continue;
        SB_G float *dst = Y + (int64_t)row * N;
        if (tk.y_accum) {              // the row's MFMA tile wrote Y in the previous launch
            float w[4];
            sb_load_v<4>(dst, w);
#pragma unroll
            for (int j = 0; j < 4; ++j) s[k][j] += w[j];
        }
        sb_store_v<4>(dst, s[k]);
    }
}

// A task with dense pieces in fragments for its columns: 64, 32 or 16.
template <int U, int NRHS, bool FAR>
__device__ __forceinline__ void sb_f32_columns(const SbSpmmArgs &a, const SbTask &tk, const SbMatBufs &mb, int r0, int N)
{
    constexpr int rest = NRHS % 64;          // of N past its groups of 64 columns
    constexpr bool four = NRHS == 0 || NRHS >= 64 || rest > 32;
    constexpr bool less = NRHS == 0 || (rest > 0 && rest <= 32);
    if (four && (!less || tk.cols > 32)) sb_f32_task<U, 4, FAR>(a, tk, mb, r0, N);
    else if ((NRHS == 0 || rest > 16) && (NRHS != 0 || tk.cols > 16)) sb_f32_task<U, 2, FAR>(a, tk, mb, r0, N);
    else if (less) sb_f32_task<U, 1, FAR>(a, tk, mb, r0, N);
}

template <int NRHS, bool FAR>
__device__ __forceinline__ void sb_f32_work(const SbSpmmArgs &a, int v)
{
    const int N = NRHS ? NRHS : a.n_rhs;
    const SbTask tk = sb_kload(a.tasks, v);
    if (tk.nrows == 0) return;               // filler of the task list
    const SbMatBufs mb = a.mats ? sb_kload(a.mats, tk.mat) : sb_mat_bufs(a, 0, a.scol);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (tk.rounds > 0) {
        const int r0 = tk.r0 + tk.rows * wave;
        if (tk.rows > 16 && tk.nrows - r0 > 16) sb_f32_columns<2, NRHS, FAR>(a, tk, mb, r0, N);
        else if (tk.nrows > r0) sb_f32_columns<1, NRHS, FAR>(a, tk, mb, r0, N);
        else for (int k = 0; k < tk.rounds; ++k) __builtin_amdgcn_s_barrier();
        return;
    }
    if (NRHS) {
        sb_f32_sparse_task<SB_F32_SPARSE_LOGL(NRHS), FAR>(a, tk, mb, N);
    } else {
        switch (SB_F32_SPARSE_LOGL(N)) {
        case 2: sb_f32_sparse_task<2, FAR>(a, tk, mb, N); break;
        case 3: sb_f32_sparse_task<3, FAR>(a, tk, mb, N); break;
        case 4: sb_f32_sparse_task<4, FAR>(a, tk, mb, N); break;
        case 5: sb_f32_sparse_task<5, FAR>(a, tk, mb, N); break;
        default: sb_f32_sparse_task<6, FAR>(a, tk, mb, N);
        }
    }
}

// One call site for the three launch modes (the work is inlined once, on a
// scalar item number): sb_for_tiles' order and queue reset.
template <int NRHS, bool FAR>
__device__ __forceinline__ void sb_spmm_f32_body(const SbSpmmArgs &a)
{
    __shared__ int next_item;
    const int items = a.ntiles;
    const int mode = a.mode;
    int v = blockIdx.x;
    for (;;) {
        if (mode == SB_MODE_QUEUE) {
            if (threadIdx.x == 0) next_item = atomicAdd(&a.queue[0], 1);
            __syncthreads();
            v = __builtin_amdgcn_readfirstlane(next_item);
            __syncthreads();
        }
        if (v >= items) break;
        sb_f32_work<NRHS, FAR>(a, v);
        if (mode == SB_MODE_GRID) return;
        v += gridDim.x;
    }
    if (mode == SB_MODE_QUEUE && threadIdx.x == 0) {
        __threadfence();
        const int done = atomicAdd(&a.queue[1], 1);
        if (done == (int)gridDim.x - 1) {
            atomicExch(&a.queue[0], 0);
            atomicExch(&a.queue[1], 0);
        }
    }
}

// Expands a piece's x ranges into xrow[0..ncols): the X row of every column.
__device__ __forceinline__ void sb_expand_xrow(const SbXRange *__restrict__ xr, int r0, int r1, int *xrow)
{
    int base = 0;
    for (int r = r0; r < r1; r += 4) {
        // four ranges per round trip (the array has slack behind it)
        struct alignas(8) Four {
            SbXRange q[4];
        };
        const Four f = sb_kload(reinterpret_cast<const Four *>(xr + r), 0);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int len = r + k < r1 ? f.q[k].len : 0;
            for (int i = threadIdx.x; i < len; i += blockDim.x) xrow[base + i] = f.q[k].col0 + i;
            base += len;
        }
    }
}
