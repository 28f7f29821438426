// Device-visible plan descriptors shared by the host plan builder and the
// kernels.  Plain C layout (no HIP types) so the builder compiles with g++.
#pragma once
#ifdef __HIPCC_RTC__
// hipRTC: fixed-width types without system headers (LP64, as on the host)
typedef signed char int8_t;
typedef int int32_t;
typedef long int64_t;
typedef unsigned char uint8_t;
typedef unsigned short uint16_t;
typedef unsigned int uint32_t;
typedef unsigned long uint64_t;
#else
#include <stdint.h>
#endif

#define SB_PIECE_DENSE 0        // column-major hs x ncols FP32 sub-panel
#define SB_PIECE_SPARSE 1       // SpMV: wave slices, uint16 columns of the staged x;
                                // SpMM: CSR over hs rows, X rows in scol
#define SB_PIECE_MFMA 2         // FP32 sub-panel in MFMA A-operand order (SpMM)

// One unit of work: a row segment [row0, row0+nrows) of one block row of one
// matrix.  The tile owns those y rows (y is written once, by this tile).
struct SbTile {
    int32_t row0;
    int32_t nrows;
    int32_t piece_begin;     // pieces[piece_begin, piece_end)
    int32_t piece_end;
    int32_t mat;             // matrix slot (batched plans); 0 otherwise
    int32_t dense_tpar;      // T': active lanes of the flat dense stream
    int32_t dense_mcols;     // M : columns advanced per stream step (4T' = M*nrows)
    int32_t sp_glog;         // SpMV sparse: log2 of the lanes per row (G)
    int32_t sp_map;          // SpMV sparse: srowptr offset of the row order
                             // (nrows local rows, longest sparse row first); -1 if none
    int32_t sp_waves;        // SpMV: wavefronts reserved for the sparse pieces (the
                             // last ones; the rest stream the dense pieces), or 0
                             // when every wavefront does both in turn
    int32_t y_accum;         // SpMM: 1 = add to Y rows an MFMA tile wrote before
    int32_t stage_map;       // SpMV: xmap_off and stage_len of the first staging group
    int32_t stage_len;       // (copies, so its map loads follow the tile read directly)
    // SpMM MFMA row tiles split along k: this work item is chunk kpart of
    // ksplit (1 = not split).  Every chunk writes its partial sums to scratch
    // blocks part_blk + kpart * (16-row units * N/16) (1 KiB blocks, in
    // accumulator order); a fixup launch after the MFMA launch adds the
    // chunks of each split row tile in chunk order and writes its rows.
    int32_t ksplit;
    int32_t kpart;
    int32_t part_blk;
};

// SpMV sparse slices: steps per pipelined batch; and the batches the SpMV
// stream loops (dense and sparse) complete per round trip (their register
// copies of the next batch wait for it).  The plan builder balances the
// sparse and dense wavefronts' dependent chains with them.
#define SB_SPUNROLL 2
#define SB_SPMV_INFLIGHT 1

// The waves per SIMD the SpMV kernel is compiled for (its VGPR budget) given
// the dense unroll: 80 VGPRs (6 waves) at unroll 2, 96 (5 waves) at unroll 4.
// SB_SPMV_MINWAVES > 0 sets it for every unroll.
#ifndef SB_SPMV_MINWAVES
#define SB_SPMV_MINWAVES 0
#endif
#define SB_SPMV_WAVES(U) (SB_SPMV_MINWAVES > 0 ? SB_SPMV_MINWAVES : (U) <= 2 ? 6 : (U) <= 4 ? 5 : 1)

// SpMV row spans: runs of short block rows (at most SB_SPMV_SHORT_ROWS rows
// and SB_SPMV_SHORT_VALUES stored values each) are planned as one tile of at
// most SB_SPMV_SPAN_ROWS rows (and the workgroup size) and
// SB_SPMV_SPAN_VALUES stored values, every block on the sparse path.
#define SB_SPMV_SHORT_ROWS 32
#define SB_SPMV_SHORT_VALUES 8192
#define SB_SPMV_SPAN_ROWS 256
#define SB_SPMV_SPAN_VALUES 65536

// the device hands workgroups to its XCDs round robin
#define SB_XCDS 8
#define SB_SIMDS 1024
#define SB_CUS 256

// FP32 SpMM.  A tile with dense pieces is cut into workgroups of 64 columns
// of Y, each wavefront taking 32 (or 16) of its rows; a tile without, into workgroups
// whose wavefronts take SB_F32_SPARSE_ROWS rows x 4 << SB_F32_SPARSE_LOGL
// columns each.
#define SB_F32_WAVES(N) ((N) >= 64 ? 4 : 2)
#define SB_F32_WG(N) (64 * SB_F32_WAVES(N))
#define SB_F32_ROWS 32
#define SB_F32_COLS 64
#define SB_F32_SPARSE_LOGL(N) ((N) > 128 ? 6 : (N) > 64 ? 5 : (N) > 32 ? 4 : (N) > 16 ? 3 : 2)
#define SB_F32_SPARSE_ITERS 2
#define SB_F32_SPARSE_ROWS(N) (SB_F32_SPARSE_ITERS * (64 >> SB_F32_SPARSE_LOGL(N)))
// the tallest FP32 SpMM tile
#define SB_F32_MAX_ROWS(N) (SB_F32_ROWS * SB_F32_WAVES(N))
// steps (of 8 columns) of loads in flight per wavefront with dense pieces
#define SB_F32_DEPTH 3

// One task: rows [r0, ..) of a tile and columns [n0, ..) of Y, with what it
// needs of the tile (so a wavefront reads one descriptor before its pieces).
struct SbTask {
    int32_t row0;            // the tile's first row
    int32_t nrows;           // the tile's rows; 0: nothing to do (filler)
    int32_t piece_begin;     // the tile's pieces
    int32_t piece_end;
    int32_t mat;             // matrix slot
    int32_t r0;
    int32_t n0;
    int32_t rounds;          // rounds of SB_F32_DEPTH steps over the dense pieces; 0: none
    int32_t y_accum;         // add to the Y rows an MFMA tile wrote before
    uint16_t cols;           // with dense pieces: columns of the workgroup and
    uint16_t rows;           // rows of each wavefront (32 or 16)
};

// SpMM MFMA tiles: a workgroup takes SB_MFMA_COLS(N, WG) columns of Y (N over
// that many workgroups per tile): up to 64 in workgroups of at most 256
// threads, whose registers and LDS then leave room for two or three of them
// on a compute unit, all of N in larger ones.  On the 50,000-row SpMM at
// N = 128 (dense blocks alone) 64-column workgroups of 256 threads took
// 88 us and full-width ones 107 us; at 512 threads 100 us and 84 us.  Widths
// that are no multiple of 64 take groups of 48 or 32: the full-width kernels
// spill (500 to 1,300 bytes a lane above N = 144).  A 3,001-row matrix of
// dense blocks, full width and in groups, us: N = 96 43.7 and 24.1, N = 144
// 74.7 and 25.4, N = 160 74.8 and 26.9 (128 threads: 51 and 30, 102 and 31,
// 124 and 21); N = 224 31.0 and N = 240 34.2 in groups, N = 192 in 64s 24.0.
// A wavefront holds two 16-row units across the columns (their FP32
// accumulators plus the double-buffered A fragments), which bounds a tile at
// SB_MFMA_MAX_ROWS(N, WG) rows (and 256).
#define SB_MFMA_COLS(N, WG)                                                                                 \
    ((N) <= 64 || (WG) > 256 ? (N) : (N) % 64 == 0 ? 64 : (N) % 48 == 0 ? 48 : (N) % 32 == 0 ? 32 : (N))
#define SB_MFMA_UNITS(COLS) ((COLS) >= 256 ? 1 : 2)
#define SB_MFMA_MAX_ROWS(N, WG)                                     \
    (16 * ((WG) / 64) * SB_MFMA_UNITS(SB_MFMA_COLS(N, WG)) < 256    \
         ? 16 * ((WG) / 64) * SB_MFMA_UNITS(SB_MFMA_COLS(N, WG))    \
         : 256)

// A panel piece of a tile: the tile's rows restricted to a group of blocks of
// at most xcap columns together, which SpMV and the MFMA kernel stage in LDS.
struct SbPiece {
    int64_t data_off;        // dense: float offset (multiple of 4) into dval
                             // sparse: entry offset into sval and sidx (SpMV) or
                             // scol (SpMM)
                             // mfma: float offset (multiple of 8) into dval
    int32_t kind;            // SB_PIECE_*
    int32_t ncols;           // columns (x slice length)
    int32_t xr_begin;        // x ranges xr[xr_begin, xr_end)
    int32_t xr_end;
    int32_t rowptr_off;      // sparse, SpMM: CSR srowptr[rowptr_off .. +nrows] (relative
                             // to data_off); SpMV: per-wavefront {step offset,
                             // steps} pairs at srowptr[rowptr_off ..]
    int32_t ksteps;          // mfma: number of 32-wide k steps (ncols padded)
    // SpMV staging: pieces are staged in groups of consecutive pieces whose
    // slices (ncols + 4 zero pads each) fit the x buffer together.
    int32_t grp_end;         // first piece of a group: one past its last piece; else 0
    int32_t stage_len;       // first piece of a group: staged slots of the group
    int32_t xmap_off;        // xmap[xmap_off .. + ncols + 4): x column of each staged
                             // slot, -1 for the zero pads; consecutive pieces of a
                             // tile are consecutive in xmap
    int32_t pitch;           // dense: floats from one panel column to the next (SpMV:
                             // the tile's rows; SpMM: the rows rounded up to 4, the
                             // extra rows zero, so a column's row quads are float4s)
};

// A contiguous run of x (or X rows) that a piece's columns meet.
struct SbXRange {
    int32_t col0;
    int32_t len;
};
