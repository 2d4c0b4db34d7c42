// kernels.h -- launch wrappers of the libfastdose_hip kernels (host side).
#pragma once

#include <hip/hip_runtime.h>

#include "fd_internal.h"

namespace fdi {

// Destination of compacted CSR entries: columns, values and the entries they hold.
struct CsrDst {
    uint64_t* columns = nullptr;
    float* values = nullptr;
    uint64_t capacity = 0;
};

// Beamlet / PTV intersection flags of n bundles (d_beamletFlagInit, IMRTBeamBundle.cu:130-316);
// flags[beams[b].out_off + pixel], max_pixels = the largest fluence_dim^2; points: sample points of all
// beamlets; box: six u32 of scratch, all ones.
hipError_t launch_beamlet_flags(const FlagBeamDev* beams, int n, int max_pixels, uint64_t points, const uint8_t* mask,
                                const fd_volume& vol, uint32_t* box, uint8_t* flags, hipStream_t stream);

// Per-voxel trilinear corner records of the density (8 floats per base voxel of the zero-bordered
// volume, 4 x 4 x 4 bricks) for the Terma kernel; density_records_floats(vol) floats.
uint64_t density_records_floats(const fd_volume& vol);
hipError_t launch_expand_density(const float* density, const fd_volume& vol, float* records, hipStream_t stream);

// Terma + mean density along the 256 BEV rays of each beamlet (TermaComp.cu:179-253).
// density_pad: the corner records of launch_expand_density.
// scratch: 4 floats per BEV value (the layout of terma, 16-byte aligned), overwritten.
// segments: ray segments per ray (1, 2, 4, 8 or 16); a workgroup holds min(256, 1024 / segments)
// rays times `segments` threads, so with 8 or 16 a beamlet takes two or four workgroups.
// Beamlets with long_dim * long_spacing > rpl64_len [cm] accumulate the radiological path in FP64.
hipError_t launch_terma(const BeamletDev* beams, int n, const float* fluence, const float* density_pad,
                        const fd_volume& vol, const SpectrumDev& spec, float rpl64_len, float* terma,
                        float* dens_bev, float* scratch, int segments, hipStream_t stream);

// March tables of a batch (TabEntry): n_gt = (march geometries) x n_fwd entries, the record
// streams and chunk headers they index, and the flag a table that outgrows its capacity sets.
struct CccsTables {
    const TabEntry* ent;
    float4* rec;
    int* hdr;
    uint32_t* overflow;
    int n_gt;
};

// The march tables (one wavefront each); clears *overflow first.  n_phi <= cccs_table_max_phi().
hipError_t launch_cccs_tables(const CccsTables& tab, const ConeTable* cones_dev, int n_fwd, int n_phi,
                              hipStream_t stream);
int cccs_table_max_phi();
int cccs_chunk_steps();  // lattice steps of one azimuth per chunk at most

// Partial volumes per beamlet for a batch of n whose BEV buffers hold bev_floats floats: n_fwd, or more
// where the widest cone is split (never with march tables).
int cccs_volumes(int n, int n_fwd, int n_phi, uint64_t bev_floats, bool tables);

// CCCS over the forward cones (DoseComp.cu:217-392): per-cone partial BEV doses
// partial[v * bev_off_b + t * L_b * 256 + s * 256 + p] with v = n_vol volumes per beamlet, as cccs_volumes
// gives them (at least v times the batch's BEV floats), then their sum into dose (four floats per thread
// when vec4: every bev_off_b a multiple of four).
// ev (nullable): events recorded before the CCCS kernel, between it and the cone sum, and after.
// tab (nullable, n_phi <= cccs_table_max_phi()): the beamlets' march tables, built on this stream
// beforehand (launch_cccs_tables), beams[b].geom indexing them; the CCCS reads its chunks from
// them, with the results of the march wavefront.
hipError_t launch_cccs(const BeamletDev* beams, int n, int max_L, const ConeTable* cones_dev, int n_fwd,
                       int n_phi, int n_vol, bool exact_g, const float* terma, const float* dens_bev, float* partial,
                       float* dose, bool vec4, hipStream_t stream, hipEvent_t* ev = nullptr,
                       const CccsTables* tab = nullptr);

// Resampling into CSR rows.  Stage 1 counts candidate voxels per (beamlet, z-plane) segment and
// records the rows [y_lo, y_hi) of the segment that hold them in cand_rows ((0, 0) when none).  Clears
// overflow[0] for stage 2.
hipError_t launch_resample_count(const BeamletDev* beams, int n, const fd_volume& vol, uint32_t* cand_count,
                                 uint2* cand_rows, uint32_t* overflow, hipStream_t stream);
// Stage 2: values of every candidate, nonzeros compacted in voxel order into tmp_cols/tmp_vals
// at cand_off[b * Z + z]; nonzero counts into nnz_count.  A segment whose candidates would end
// beyond `cap` entries writes nothing, gets a zero count and sets overflow[0] = 1.
// rowmax_bits (nullable, zeroed by the caller): per-beamlet maximum value, as float bits.
// rcp_exact: launch_rcp_check found no mismatch on this device (see there).
hipError_t launch_resample_values(const BeamletDev* beams, int n, const fd_volume& vol, float extent,
                                  const float* dose_bev, const uint64_t* cand_off, const uint2* cand_rows,
                                  uint64_t cap, uint32_t* overflow, uint64_t* tmp_cols, float* tmp_vals,
                                  uint32_t* nnz_count, uint32_t* rowmax_bits, bool rcp_exact, hipStream_t stream);
// Adds to *mismatches (zeroed by the caller) the number of floats b with exponent in
// [exp0, exp0 + n_exp) for which the resampler's reciprocal (hardware reciprocal + one Newton
// step) differs from the IEEE quotient 1 / b.
hipError_t launch_rcp_check(int exp0, int n_exp, uint32_t* mismatches, hipStream_t stream);
// Relative threshold: per segment, the entries >= thr * rowmax of its beamlet.
hipError_t launch_resample_threshold_count(int n, int Z, const uint64_t* cand_off, const uint32_t* nnz_count,
                                           const float* tmp_vals, const uint32_t* rowmax_bits, float thr,
                                           uint32_t* keep_count, hipStream_t stream);
// Stage 3: copy the compacted nonzeros into the CSR arrays (with rowmax_bits and thr > 0 only
// those >= thr * rowmax); row offsets from nnz_off.  The entries go to dst0 when its capacity
// holds the total (nnz_off[n Z]), else to dst1 when that one does, else nowhere (the columns and
// values are left untouched; the offsets are still written).  A destination with a null array
// counts as capacity 0.  host_offsets (nullable) and host_totals: pinned host memory that receives the row
// offsets again, and the candidates (cand_off[n Z]), nonzeros, flags[0] and flags[2].
hipError_t launch_resample_compact(int n, int Z, const uint64_t* cand_off, const uint64_t* nnz_off,
                                   const uint32_t* nnz_count, const uint64_t* tmp_cols, const float* tmp_vals,
                                   const uint32_t* rowmax_bits, float thr, const uint32_t* flags, uint64_t* offsets,
                                   uint64_t* host_offsets, uint64_t* host_totals, CsrDst dst0, CsrDst dst1,
                                   hipStream_t stream);

// Exclusive scan of count[0..N) (u32) into off[0..N) (u64) plus total[0] = sum; large inputs by many
// workgroups (scratch: scan_scratch_size(N) u64, a sum per kScanTile counts).
constexpr uint64_t kScanTile = 4096;
constexpr uint64_t scan_scratch_size(uint64_t N) { return (N + kScanTile - 1) / kScanTile + 1; }
hipError_t launch_scan_u32(const uint32_t* count, uint64_t N, uint64_t* off, uint64_t* total, uint64_t* scratch,
                           hipStream_t stream);

// Dense (rows x cols, row-major) -> CSR, by segments of rows: nonzero counts per segment, then (after
// an exclusive scan of them) the fill.
struct DenseSplit {
    uint32_t per_row;  // segments per row
    uint32_t length;   // elements per segment (the row's last one may hold fewer)
};
// Segments for rows x cols with at most max(max_segments, rows) of them (cols < 2^32).
DenseSplit dense_split(uint64_t rows, uint64_t cols, uint64_t max_segments);
hipError_t launch_dense_count(const float* dense, uint64_t rows, uint64_t cols, const DenseSplit& s, uint32_t* count,
                              hipStream_t stream);
hipError_t launch_dense_fill(const float* dense, uint64_t rows, uint64_t cols, const DenseSplit& s,
                             const uint64_t* seg_off, uint64_t* columns, float* values, hipStream_t stream);
hipError_t launch_fill_u32(uint32_t* p, uint64_t n, uint32_t v, hipStream_t stream);
hipError_t launch_fill_u64(uint64_t* p, uint64_t n, uint64_t v, hipStream_t stream);
// offsets[r] = seg_off[r n_seg] (r < rows), offsets[rows] = total[0].
hipError_t launch_write_offsets(const uint64_t* seg_off, const uint64_t* total, uint64_t rows, uint32_t n_seg,
                                uint64_t* offsets, hipStream_t stream);

// Packing and D^T X products (kernels_spmm.hip).
hipError_t launch_global_rows(int n_mat, const uint64_t* row_first, const uint64_t* off_off, const uint64_t* nnz_off,
                              const uint64_t* offsets, uint64_t R, uint64_t total_nnz, uint64_t* rowptr,
                              hipStream_t stream);
// scale[r] = row maximum; q (nullable) = value / scale in BF16 or FP16
hipError_t launch_pack_rows(uint64_t R, const uint64_t* rowptr, const float* values, int vtype, float* scale,
                            uint16_t* q, hipStream_t stream);
// Voxel-major copy of rows whose columns ascend: n = csc_tiles(C, tile_cols) tiles of tile_cols consecutive
// columns (csc_tile_cols).  launch_row_tiles: tiles[r (n + 1) + t] = row r's entries before tile t; scale (nullable)
// = row maxima; *unsorted (zeroed by the caller) = 1 when a row's columns do not ascend below C (the
// table then must not be used).  launch_tile_totals: total[t] (zeroed by the caller) = entries of tile
// t.  launch_place_tiles: colptr (C + 1), crow and cval from the table and tile_base, the exclusive
// scan of total; order: csc_tile_groups(C, tile_cols) words of scratch.  C > 0, R <= 2^20 and every row's length
// below 2^32.
uint32_t csc_tile_cols(uint64_t R, uint64_t C, bool narrow);  // narrow: where narrow tiles are worth it
uint64_t csc_tiles(uint64_t C, uint32_t tile_cols);
uint64_t csc_tile_groups(uint64_t C, uint32_t tile_cols);
hipError_t launch_row_tiles(uint64_t R, const uint64_t* rowptr, const uint64_t* columns, const float* values,
                            uint64_t C, uint32_t tile_cols, uint32_t* tiles, float* scale, uint32_t* unsorted,
                            hipStream_t stream);
hipError_t launch_tile_totals(uint64_t R, uint64_t C, uint32_t tile_cols, const uint32_t* tiles, uint32_t* total, hipStream_t stream);
hipError_t launch_place_tiles(int vtype, uint64_t R, uint64_t C, uint32_t tile_cols, const uint32_t* tiles, const uint64_t* rowptr,
                              const uint64_t* columns, const float* values, const float* scale,
                              const uint64_t* tile_base, uint32_t* order, uint64_t* colptr, uint32_t* crow,
                              void* cval, hipStream_t stream);
hipError_t launch_col_count(uint64_t nnz, const uint64_t* columns, uint32_t* count, hipStream_t stream);
hipError_t launch_col_scatter(uint64_t R, const uint64_t* rowptr, const uint64_t* columns, const void* vals,
                              int vbytes, const uint64_t* colptr, uint32_t* cursor, uint32_t* crow, void* cval,
                              hipStream_t stream);
hipError_t launch_col_sort(uint64_t C, const uint64_t* colptr, uint32_t* crow, void* cval, int vbytes,
                           hipStream_t stream);
hipError_t launch_spmm(int vtype, uint64_t C, const uint64_t* colptr, const uint32_t* crow, const void* cval,
                       const float* scale, const float* X, int k, uint64_t R, uint64_t nnz, float* Y, hipStream_t stream);

}  // namespace fdi
