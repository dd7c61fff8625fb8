// hjm_kernels.h -- launchers of the HJM kernels (internal to libhjm_cva.so).
#pragma once
#include "hjm_common.h"

namespace hjm {

struct SelRowState;  // hjm_select.h

struct ExposureParams {
    int64_t paths;
    int ndates;
    int pad;
    double notional, K;
    double m;                // 1 / dtau (compounding frequency of the simple rate)
    double accrual[kTenors];
    double w[kTenors];       // CVA weights (1-R) x default probability shares
};

hipError_t launch_ref_paths_f64(const RefStepConsts<double>& k, const RefGrid& g,
                                const double* normals, double* nx, double* ny, hipStream_t st);
hipError_t launch_ref_paths_f32k(const RefStepConsts<float>& k, const RefGrid& g,
                                 const double* normals, double* nx, double* ny, hipStream_t st);
hipError_t launch_ref_exposure(const ExposureParams& e, const double* nx, const double* ny,
                               double* exposures, double* partials, hipStream_t st);
hipError_t launch_column_sum(const double* partials, int64_t rows, int cols, double* out,
                             hipStream_t st);
// k-th smallest of each row; ws: workspace of bracket_workspace_bytes (hjm_select.h) or null
hipError_t launch_radix_select(const double* x, int rows, int64_t n, int64_t k, void* ws,
                               double* out, hipStream_t st);
hipError_t launch_normals(uint64_t seed, int64_t path0, int64_t paths, int nsteps, int stride,
                          double* out, hipStream_t st);
hipError_t launch_box_muller_parts(const uint32_t* words, int64_t n, float* r, float* c, float* s,
                                   hipStream_t st);

// Matrix-core FP32 path kernels (50 steps per date); prepare once per plan (sets the
// kernels' dynamic LDS limits) before launching or capturing them.
hipError_t mfma_kernels_prepare();
// zs (optional): the forward's FP32 normals [step][factor][path] for a later reverse sweep
hipError_t launch_ref_paths_mfma(const MfmaGrid& g, const uint16_t* wfrag, double* nx, double* ny,
                                 float* zs, hipStream_t st);
// The FP64 matrix-core path kernel (reference semantics); wfrag: build_mfma64_block_map's
// fragments of ref_mfma_tiles(g.ndates) M-tiles; prepare once per plan.
hipError_t mfma64_kernels_prepare();
hipError_t launch_ref_paths_mfma64(const MfmaGrid& g, const double* wfrag, double* nx, double* ny,
                                   float* zs, hipStream_t st);
// The FP64 portfolio path kernel: curves [ndates][51][paths] and logb [ndates][paths];
// wfrag: build_mfma64_block_map's portfolio fragments.
hipError_t launch_pf_paths_mfma64(const MfmaGrid& g, const double* wfrag, double* curves, double* logb,
                                  float* zs, hipStream_t st);
// Launch shape of a matrix-core portfolio kernel (0 in a field: the kernel's default).
//   tiles: N-tiles of 16 paths per wave; waves: per workgroup;
//   stage (valuation): M-tiles of -gamma staged in LDS at a time;
//   max_blocks (paths): a persistent grid of at most this many workgroups.
struct MfmaShape {
    int tiles = 0, waves = 0, stage = 0;
    int64_t max_blocks = 0;
};
// path kernel: {tiles, waves} in {2, 8} (default: by path count), {2, 12}, {1, 12}, {1, 16};
// valuation: tiles 2 (default) or 4, waves 4 or 8 (default), stage 1..8 (default 2)
bool pf_path_shape_ok(int tiles, int waves);
bool pf_value_shape_ok(int tiles, int waves);
hipError_t launch_pf_paths_mfma(const MfmaGrid& g, const uint16_t* wfrag, float* curves,
                                double* logb, float* zs, const MfmaShape& shape, hipStream_t st);

// Pathwise adjoint of the reference-semantics CVA.
// sa_partials: [blocks of 256 paths][51] per-slot sums of gA over the block's paths
hipError_t launch_ref_adjoint_seed(const ExposureParams& e, double dt, const double* nx,
                                   const double* ny, float* gx, float* gA, double* sa_partials,
                                   hipStream_t st);
// One-pass VALU sweep, two lanes per path. normals: host FP64 [path][step][3]; zs: the
// forward's stored FP32 normals [step][3][path]; both null: regenerate. partials:
// [ref_adjoint_blocks(paths)][5 * 51]
// (loading gradients of factors 0, 1, 2, sum of the block-end adjoints, d J / d spot).
int64_t ref_adjoint_blocks(int64_t paths);
hipError_t launch_ref_adjoint(const RefGrid& rg, double c, double sqrt_dt, const double* normals,
                              const float* zs, const float* gx, const float* gA, double* partials,
                              hipStream_t st);

// The block map's fragments of an FP32 matrix plan, block_map_elems(prm.mtiles) elements; the
// reverse sweep's map and tables (hjm_map_kernels.hip).
struct BlockMapParams;
hipError_t launch_block_map(const BlockMapParams& prm, bool pf, uint16_t* frag, hipStream_t st);
hipError_t launch_sweep_map(double c, bool pf, uint16_t* frag, float* ptab, hipStream_t st);

// The reverse sweep on the matrix cores (50 steps per date, in-kernel normals; hjm_adjoint_mfma.hip).
struct SweepGrid {
    int hi, lo;               // blocks hi .. lo, swept downwards
    int units;                // units of 32 paths per pair of waves (sweep_units of the whole run)
    float dt;                 // portfolio: the bank account's step
    int64_t paths;            // row stride of the seeds
    int64_t begin, end;       // paths of this launch; begin a multiple of sweep_group
    int64_t zld;              // row stride of zs, whose column 0 is path begin
};
constexpr int64_t kSweepMaxPaths = (int64_t)1 << 26;   // 32-bit lane offsets: 48 B x paths
constexpr int kSweepSlack = 32;              // floats of zeros the sweep needs past zs
int sweep_row_tiles(bool pf, int ndates);    // rows of a partial: 16 x this, 160 columns
// units of a pair of waves, 1 or 2: its FP32 sums then cover at most 2 units' blocks, for any
// number of paths, before they join the FP64 ones
int sweep_units(int64_t paths);
int64_t sweep_group(int64_t paths);          // paths of a workgroup: one partial each
hipError_t launch_adjoint_mfma(const SweepGrid& g, bool pf, const uint16_t* map, const float* ptab,
                               const float* zs, const float* seed_a, const float* seed_b, float* partials,
                               hipStream_t st);
// out[c] = (add ? out[c] : 0) + the FP64 sum of partials[r][c] over the rows, in a fixed order
hipError_t launch_sweep_sum(const float* partials, int64_t rows, int cols, bool add, double* out,
                            hipStream_t st);
hipError_t launch_sweep_shocks(uint64_t seed, int64_t path0, const SweepGrid& g, float* zs, hipStream_t st);

// A book's swaps on the device, grouped by netting set (the caller's order within a set):
// maturity in periods, signed notional, notional x rate x dtau; set g owns [first[g], first[g + 1]).
struct BookSwaps {
    const int* first;
    const int* periods;
    const double* notional;
    const double* coupon;
};
// Coefficient tables [ndates][nsets][60], [ndates][nsets] of the set values a - gamma P and the
// sets' largest live period; from them the matrix-core tables of FP32 plans, and the adjoint's.
hipError_t launch_book_tables(const BookSwaps& b, int nsets, int ndates, double* coef, double* a, int* kmax,
                              hipStream_t st);
hipError_t launch_value_fragments(const double* coef, const double* a, const int* kmax, int nsets, int ndates,
                                  uint16_t* frag, float* apad, int* tilek, hipStream_t st);
hipError_t launch_adjoint_fragments(const double* coef, int nsets, int ndates, uint16_t* frag, hipStream_t st);
hipError_t launch_clear_matured(const int* kmax, int rows, int64_t paths, void* ex, int elem_bytes,
                                hipStream_t st);

// Portfolio semantics. FP64 with in-kernel normals: several lanes per path, the same for every
// block and grid.
hipError_t launch_pf_paths_lanes(const RefStepConsts<double>& k, const PfGrid& g, double* curves,
                                 double* logb, hipStream_t st);
hipError_t launch_pf_paths_f64(const RefStepConsts<double>& k, const PfGrid& g, const double* normals,
                               double* curves, double* logb, int block, int grid, hipStream_t st);
hipError_t launch_pf_paths_f32(const RefStepConsts<float>& k, const PfGrid& g, const double* normals,
                               float* curves, double* logb, int block, int grid, hipStream_t st);
hipError_t launch_pf_value_f64(const PfValueParams& v, const double* curves, const double* logb,
                               const double* coef, const double* a, const int* kmax, double* ex,
                               hipStream_t st);
// FP32 plans: the matrix-core valuation over launch_value_fragments' tables, of paths
// [0, count) (count < 0: all); filter (or null): only the rows (date, set) whose PFE
// bracket selection is unresolved for rank fk with fcap candidate slots
hipError_t launch_pf_value_mfma(const PfValueParams& v, const float* curves, const double* logb,
                                const uint16_t* gfrag, const float* apad, const int* tilek,
                                float* ex, const MfmaShape& shape, hipStream_t st, int64_t count = -1,
                                const SelRowState* filter = nullptr, int64_t fk = 0,
                                int64_t fcap = 0);
// FP32 plans: valuation, EE and per-path CVA moments (partials
// [set][pf_fused_blocks(paths)][ndates + 2], for the grouped column sums) and, with sel,
// the PFE bracket counting and candidates of every row, in one pass without exposures
// (groups of 128 sets)
int64_t pf_fused_blocks(int64_t paths);
hipError_t launch_pf_value_stats_mfma(const PfValueParams& v, const float* curves, const double* logb,
                                      const uint16_t* gfrag, const float* apad, const int* tilek,
                                      const double* w, double* partials, SelRowState* sel,
                                      float* cand, int64_t cap, int stage_slots, hipStream_t st);
// sums[set][c] = sum over blocks of partials[set][block][c] (fixed order)
hipError_t launch_grouped_column_sum(const double* partials, int nsets, int64_t blocks, int cols,
                                     double* sums, hipStream_t st);
// selws (or null): bracket-selection workspace whose counting this pass does, for rank
// pfe_rank of each (date, set) row, after launch_bracket_sample*; needs
// pf_stats_stage(...) > 0 (LDS staging slice per wave, in entries; *flush_dates, if given,
// receives the number of dates between the slice's flushes)
int pf_stats_stage(int64_t paths, int64_t pfe_rank, int ndates, int elem_bytes,
                   int* flush_dates = nullptr);
// lo_parts (or null; FP32 with selws): [ndates * nsets][pf_stats_blocks(paths)] counts
// below the bracket per row and statistics workgroup, stored plainly and added to the rows'
// states by one small launch after the pass (null, and FP64 rows: one atomic per row and
// workgroup instead)
int64_t pf_stats_blocks(int64_t paths);
hipError_t launch_pf_stats_f64(const PfValueParams& v, const double* ex, const double* w,
                               double* partials, double* sums, void* selws, int64_t pfe_rank,
                               uint32_t* lo_parts, hipStream_t st);
hipError_t launch_pf_stats_f32(const PfValueParams& v, const float* ex, const double* w,
                               double* partials, double* sums, void* selws, int64_t pfe_rank,
                               uint32_t* lo_parts, hipStream_t st);
hipError_t launch_radix_select_f32(const float* x, int rows, int64_t n, int64_t k, void* ws,
                                   double* out, hipStream_t st);
// the sampled-bracket selection split around a statistics pass that does its counting
hipError_t launch_bracket_sample(const double* x, int rows, int64_t n, int64_t k, void* ws,
                                 hipStream_t st);
hipError_t launch_bracket_sample_f32(const float* x, int rows, int64_t n, int64_t k, void* ws,
                                     hipStream_t st);
hipError_t launch_bracket_finish(const double* x, int rows, int64_t n, int64_t k, void* ws,
                                 double* out, hipStream_t st);
hipError_t launch_bracket_finish_f32(const float* x, int rows, int64_t n, int64_t k, void* ws,
                                     double* out, hipStream_t st);

// FP64 plans; partials: [blocks of 256 paths][2 ndates], the sums over the block's paths of
// beta at every date, then of sum_g w_ge E_ge (the CVA's numerator)
hipError_t launch_pf_adjoint_seed_f64(const PfValueParams& v, const double* curves,
                                      const double* logb, const double* coef, const double* a,
                                      const int* kmax, const double* w, float* gbar, float* beta,
                                      double* partials, hipStream_t st);
// FP32 plans: both products on the matrix cores over launch_value_fragments' and
// launch_adjoint_fragments' tables; partials: [pf_adjoint_seed_mfma_blocks(paths)][2 ndates]
int64_t pf_adjoint_seed_mfma_blocks(int64_t paths);
hipError_t launch_pf_adjoint_seed_mfma(const PfValueParams& v, const float* curves, const double* logb,
                                       const uint16_t* gfrag, const uint16_t* tfrag, const float* apad,
                                       const int* tilek, const double* w, float* gbar, float* beta,
                                       double* partials, hipStream_t st);
// One-pass sweep, two lanes per path; partials [pf_adjoint_blocks(paths)][5 * 51] as the
// reference sweep's.
int64_t pf_adjoint_blocks(int64_t paths);
hipError_t launch_pf_adjoint(const PfGrid& g, double c, const double* normals, const float* zs,
                             const float* gbar, const float* beta, double* partials, hipStream_t st);

// The reference's own GPU design (baseline form).
hipError_t launch_blockwise_paths(const RefStepConsts<double>& k, const RefGrid& g, int block_index,
                                  const double* normals, const double* state_in, double* state_out,
                                  double* integral, double* nx, double* ny, hipStream_t st);
hipError_t launch_blockwise_exposure(const ExposureParams& e, const double* nx, const double* ny,
                                     double* exposures, hipStream_t st);
hipError_t launch_column_mean_gemv(const double* exposures, int64_t paths, double* sums,
                                   hipStream_t st);

}  // namespace hjm
