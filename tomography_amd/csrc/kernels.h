// kernels.h — host-callable launchers of the gfx950 kernels (kernels.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "setup.h"
#include "tomo_internal.h"

namespace tomo {

// Steps fused per launch that have a compiled kernel.
bool tblock_supported(int T);

// Time the next update, fold, projection or fitness launch made by the calling
// thread: its dispatch packet carries `start` and `stop` (hipExtLaunchKernelGGL),
// so timing puts no marker packets between kernels.  (nullptr, nullptr) disarms.
void arm_launch_events(hipEvent_t start, hipEvent_t stop);

// Time-blocked E/H update of every tile in `tiles` (T steps, one launch):
// the general kernel (CPML, contour samples, edges, ref-compat physics) and
// the interior kernel (physical mode, tiles away from every boundary).
hipError_t launch_tblock(int T, int mode, const TileItem* tiles, int ntiles, const LaunchItem* items,
                         const DevSim* sims, int ordinal, int waves, int grid, hipStream_t st);
hipError_t launch_tedge(int T, const TileItem* tiles, int ntiles, const LaunchItem* items, const DevSim* sims,
                        int ordinal, int waves, int grid, hipStream_t st);
hipError_t launch_trow(int T, const TileItem* tiles, int ntiles, const LaunchItem* items, const DevSim* sims,
                       int ordinal, int waves, int grid, hipStream_t st);
hipError_t launch_tcol(int T, const TileItem* tiles, int ntiles, const LaunchItem* items, const DevSim* sims,
                       int ordinal, int waves, int grid, hipStream_t st);
hipError_t launch_tinner(int T, const TileItem* tiles, int ntiles, const LaunchItem* items, const DevSim* sims,
                         int ordinal, int waves, int grid, hipStream_t st);
// Rows a row-sweep tile streams (its output rows y1 - y0 plus T ghost rows on
// each side) are at most kMaxTileRows: the sweeps of the interior, row-edge,
// column-edge and corner tiles hold the rows' dispersive spans one per lane.
constexpr int kMaxTileRows = 64;
// All tile classes of physical-mode simulations in one launch (TileItem::cls).
hipError_t launch_tfused(int T, const TileItem* tiles, int ntiles, const LaunchItem* items, const DevSim* sims,
                         int ordinal, int waves, int grid, hipStream_t st);

// Tile update form: one workgroup of kTileWaveCount waves per TileItem holds a
// 64-lane band x (kTileWaveCount * rows_per_wave) rows in registers and
// advances it one time block (T steps); every tile row span y1 - y0 must be
// at most kTileWaveCount * rows_per_wave - 2T.
constexpr int kTileWaveCount = 8;
bool twave_supported(int T, int rows_per_wave);
hipError_t launch_twave(int T, int rows_per_wave, const TileItem* tiles, int ntiles, const LaunchItem* items,
                        const DevSim* sims, int ordinal, int grid, hipStream_t st);

// Register-tile update: one workgroup of `waves` waves (8, or 16 in physical mode) per RegTile
// advances it one time block of `tsteps` steps.  Every held node is a node of
// the grid, and the owned nodes lie at least `tsteps` inside the held ones
// wherever those do not end at the grid's edge.  rows: kTileRowsTall for a tile
// of vacuum clear of the CPML strips and the grid's edge (held rows and columns
// and the row below); kTileRowsClean for vacuum at the strips of one axis, and
// for physical-mode material clear of them and of the source; else
// kTileRowsEdge.  The six field planes take less than 2 GiB together.
// A tile of item -1 is an unused place.
constexpr int kMaxTileSteps = 15;  // longest block that the planner asks for (runtime.cpp)
constexpr int kTileRowsEdge = 4, kTileRowsClean = 8, kTileRowsTall = 16;
// `fold`: the previous epoch's items (n of them, FP32 running DFT), whose
// samples further workgroups of the launch fold; this launch must write other
// sample rows (LaunchItem::samp0).  `lone`: the description of the launch's only
// simulation, null when there are several (a hint: it changes no result).
struct FoldRun {
    const LaunchItem* items;
    int n, max_p, max_f;
};
hipError_t launch_rtile(int mode, int waves, const RegTile* tiles, int ntiles, const LaunchItem* items, const DevSim* sims,
                        int ordinal, int tsteps, const DevSim* lone, const FoldRun& fold, hipStream_t st);

// Resident update form: one cooperative launch advances every simulation of
// `items` by its epoch (all time blocks), one workgroup per ResTile, all
// co-resident.  `done` (ntiles counters) must start at zero; `err` is set to 1
// if a workgroup gave up waiting (after spin_limit polls) and stays set.
constexpr int kResidentWaves = 8;  // waves per workgroup of the resident kernel
bool tres_supported(int T, int rows_per_wave);
// Tiles one cooperative launch can hold on `cus` compute units (0: none).
int tres_max_tiles(int T, int rows_per_wave, int mode, int cus);
hipError_t launch_tres(int T, int rows_per_wave, int mode, const ResTile* tiles, int ntiles,
                       const LaunchItem* items, const DevSim* sims, int* done, int* err, int spin_limit,
                       hipStream_t st);

// Fold one chunk of surface samples into the running DFT (Kahan FP32 or FP64).
hipError_t launch_fold(bool fp64, const LaunchItem* items, int nitems, const DevSim* sims, int max_p, int max_f,
                       hipStream_t st);

// Far-field projection of a group of simulations that share grid, contour and
// frequencies: D/P at [(sim * n_freq + f) * n_angles + a];
// kinv[f] = {wavenumber, far-field normaliser}.
hipError_t launch_project(const int* sim_idx, int n_sims, int n_freq, const DevSim* sims, const float2* kinv,
                               int n_angles, float eta0, float* D, float* Pph, hipStream_t st);

// FP64 fitness reduction, one block per evaluation:
// fit[e] = -sum_i (D[e*L+i] - tgt[i])^2 / norm  (+ optional wrapped phase term).
// terms bit 0: phase term; bit 1: relative misfit (divide each term by tgt^2).
hipError_t launch_fitness(const float* D, const float* Pph, const float* tgt, const float* tgt_phase, int L,
                          int n_eval, double norm, int terms, double* fit, hipStream_t st);

// Start state of one simulation, in one launch: copies its tables and its
// DevSim out of pinned host memory (src: table_bytes, then entry_bytes; both
// multiples of 8, any of them 0), zeroes [zero, zero + zero_bytes) (a multiple
// of 16) and, when mat is given, rasterises the phantom `g` of physical mode
// (bit-exact with the oracle).
struct SlotInit {
    const void* src;
    void* tables;
    size_t table_bytes;
    void* entry;
    size_t entry_bytes;
    void* zero;
    size_t zero_bytes;
    uint8_t* mat;
    int pitch, nx, ny;
    float dxf, dyf;
    PhantomGeom g;
};
hipError_t launch_slot_init(const SlotInit& a, hipStream_t st);

// Material map of the reference-compatible mode, from its uploaded tables
// (bit-exact with the oracle).
hipError_t launch_raster_ref(uint8_t* mat, int pitch, int nx, int ny, const int* lo, const int* hi,
                             const int* xc, const int* yc, int npatch, hipStream_t st);

// Dense copies of the rows [y0, y1) of a simulation's fields, written to
// pinned host memory: Ez and Jp nx + 1 wide over rows 0..ny, Hx and Hy nx wide
// over rows 0..ny - 1.  A null `out` skips that field.
struct FieldPack {
    const float *ez, *hx, *hy, *jp;  // device planes; jp is the compact row-span storage
    const int* span;
    int nx, ny, pitch, y0, y1;
    float* out[4];  // Ez, Hx, Hy, Jp: destination of row y0
};
hipError_t launch_field_pack(const FieldPack& a, hipStream_t st);

// Zero-fill (a kernel, so that it is safe inside captured graphs).
hipError_t launch_zero(void* p, size_t bytes, hipStream_t st);

}  // namespace tomo
