// hjm_capi_portfolio.hip -- C ABI of the portfolio semantics: coefficient tables,
// persistent-grid tuning, hipGraph capture and replay, autotuner.
#include <math.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "hjm_host.h"
#include "hjm_kernels.h"
#include "hjm_mfma_plan.h"
#include "hjm_select.h"
#include "hjm_sweep.h"

using namespace hjm;
using namespace hjm_host;

struct hjm_pplan_s {
    int device = 0;
    ContextHolder ctx;
    hipStream_t stream = nullptr;   // the context's, as are the events
    hipEvent_t* ev = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    hjm_tuning tuning{256, 0, 0, 0, 0, 0, 0, 0, 0, 0};  // block size 256, the rest defaults
    MfmaShape path_shape{}, value_shape{};             // matrix-core kernels, from tuning
    int cus = 0;
    int precision = HJM_FP64;
    bool do_pfe = false;
    int64_t paths = 0;
    int nsets = 0, ndates = 0;
    int64_t pfe_rank = 1;
    int grid_blocks = 0;
    bool use_mfma = false;    // FP32 on the matrix cores (path kernel and valuation)
    bool use_mfma64 = false;  // FP64 path kernel on the matrix cores (HJM_KERNEL_MATRIX)
    MfmaGrid mg{};
    uint16_t* d_wfrag = nullptr;  // bf16 parts of the block map
    double* d_wfrag64 = nullptr;  // the block map's FP64 fragments
    RefStepConsts<double> kd{};
    RefStepConsts<float> kf{};
    PfGrid grid{};
    PfValueParams vp{};
    std::vector<double> w;  // [nsets][ndates] CVA weights
    double* d_normals = nullptr;
    void* d_curves = nullptr;
    double* d_logb = nullptr;
    void* d_ex = nullptr;
    double* d_partials = nullptr;
    double* d_sums = nullptr;
    double* d_pfe = nullptr;  // [date][set], after the sums
    char* d_selws = nullptr;  // bracket-selection workspace (PFE)
    uint32_t* d_loparts = nullptr;  // counts below the bracket per row and statistics workgroup
    double* d_coef = nullptr;
    double* d_a = nullptr;
    // the swap list: set offsets, periods; signed notionals, coupons. The host copies are the
    // plan's, since an asynchronous upload may still read them when its creation fails
    std::vector<int> book_ints;
    std::vector<double> book_reals;
    int* d_book_ints = nullptr;
    double* d_book_reals = nullptr;
    int* d_kmax = nullptr;
    double* d_w = nullptr;
    uint16_t* d_vfrag = nullptr;  // FP32: bf16 parts of -gamma (matrix-core valuation)
    float* d_apad = nullptr;
    int* d_tilek = nullptr;
};

namespace {

void pplan_release(hjm_portfolio_plan p)
{
    if (!p) return;
    int prev = -1;
    (void)hipGetDevice(&prev);
    (void)hipSetDevice(p->device);
    const bool clean = p->ctx.quiesce();
    if (p->exec) (void)hipGraphExecDestroy(p->exec);
    if (p->graph) (void)hipGraphDestroy(p->graph);
    dev_free(clean, p->d_normals, p->d_curves, p->d_logb, p->d_ex, p->d_partials, p->d_sums, p->d_selws,
             p->d_loparts, p->d_coef, p->d_book_ints, p->d_book_reals, p->d_vfrag, p->d_apad, p->d_tilek,
             p->d_a, p->d_kmax, p->d_w, p->d_wfrag, p->d_wfrag64);
    p->ctx.give();
    if (prev >= 0) (void)hipSetDevice(prev);
    delete p;
}

int check_portfolio(const hjm_portfolio* pf, int* ndates)
{
    if (!pf || !pf->periods || !pf->sign_notional || !pf->fixed_rate || !pf->netting_set ||
        !pf->hazard_rate)
        return HJM_ERR_NULL;
    if (pf->nswaps <= 0 || pf->nswaps > HJM_MAX_SWAPS || pf->nsets <= 0 || pf->nsets > HJM_MAX_SETS)
        return HJM_ERR_ARG;
    if (!(pf->dtau > 0.0) || !(pf->horizon > 0.0) || !(pf->recovery >= 0.0 && pf->recovery <= 1.0))
        return HJM_ERR_ARG;
    const double r = pf->horizon / pf->dtau;
    const int E = (int)llround(r);
    if (E < 1 || fabs(r - E) > 1e-9 * E || E > kMaxPeriods) return HJM_ERR_GRID;
    for (int s = 0; s < pf->nswaps; ++s) {
        if (pf->periods[s] < 1 || pf->periods[s] > E) return HJM_ERR_ARG;
        if (pf->netting_set[s] < 0 || pf->netting_set[s] >= pf->nsets) return HJM_ERR_ARG;
        if (!isfinite(pf->sign_notional[s]) || !isfinite(pf->fixed_rate[s])) return HJM_ERR_ARG;
    }
    for (int g = 0; g < pf->nsets; ++g)
        if (!(pf->hazard_rate[g] >= 0.0)) return HJM_ERR_ARG;
    *ndates = E + 1;
    return HJM_OK;
}

int check_tuning(const hjm_tuning& t)
{
    if (t.block_size != 64 && t.block_size != 128 && t.block_size != 256) return HJM_ERR_ARG;
    if (t.blocks_per_cu < 0 || t.blocks_per_cu > 64) return HJM_ERR_ARG;
    if (t.use_graph != 0 && t.use_graph != 1) return HJM_ERR_ARG;
    if (t.fuse_statistics != 0 && t.fuse_statistics != 1) return HJM_ERR_ARG;
    if (t.pfe_stage_slots < 0 || t.pfe_stage_slots > 32) return HJM_ERR_ARG;
    if (!pf_path_shape_ok(t.path_tiles ? t.path_tiles : 2, t.path_waves ? t.path_waves : 8))
        return HJM_ERR_ARG;
    if (!pf_value_shape_ok(t.value_tiles ? t.value_tiles : 2, t.value_waves ? t.value_waves : 8))
        return HJM_ERR_ARG;
    if (t.value_stage < 0 || t.value_stage > 8) return HJM_ERR_ARG;
    return HJM_OK;
}

// the kernels' launch shapes for a (checked) tuning
void pplan_apply_tuning(hjm_portfolio_plan p, const hjm_tuning& t)
{
    p->tuning = t;
    const int64_t tiles = (p->paths + t.block_size - 1) / t.block_size;
    p->grid_blocks = (int)std::min<int64_t>(
        tiles, t.blocks_per_cu > 0 ? (int64_t)t.blocks_per_cu * p->cus : tiles);
    p->path_shape = MfmaShape{t.path_tiles, t.path_waves, 0,
                              t.blocks_per_cu > 0 ? (int64_t)t.blocks_per_cu * p->cus : 0};
    p->value_shape = MfmaShape{t.value_tiles, t.value_waves, t.value_stage, 0};
}

// greeks: a plan of the Greeks call, whose seeds value the sets (no exposures, no statistics)
int pplan_init(hjm_portfolio_plan p, const hjm_market* market, const hjm_portfolio* pf,
               const hjm_config* cfg, const hjm_tuning* tuning, bool greeks = false)
{
    HJM_TRY(check_market(market));
    if (!cfg) return HJM_ERR_NULL;
    int nd = 0;
    HJM_TRY(check_portfolio(pf, &nd));
    if (cfg->paths <= 0 || cfg->path_offset < 0 || cfg->path_offset + cfg->paths > (1ll << 32))
        return HJM_ERR_ARG;
    if (cfg->precision != HJM_FP64 && cfg->precision != HJM_FP32_KAHAN) return HJM_ERR_ARG;
    if (cfg->rng != HJM_RNG_PHILOX && cfg->rng != HJM_RNG_HOST) return HJM_ERR_ARG;
    if (cfg->rng == HJM_RNG_HOST && !cfg->host_normals) return HJM_ERR_NULL;
    if (cfg->pfe_quantile > 1.0) return HJM_ERR_ARG;
    if (tuning) {
        HJM_TRY(check_tuning(*tuning));
        p->tuning = *tuning;
    }
    if (!(cfg->dt > 0.0)) return HJM_ERR_ARG;
    const double rs = pf->dtau / cfg->dt;
    const int stride = (int)llround(rs);
    if (stride <= 0 || fabs(rs - stride) > 1e-6 * stride) return HJM_ERR_GRID;
    const int S = stride * (nd - 1);
    if (cfg->path_kernel < HJM_KERNEL_AUTO || cfg->path_kernel > HJM_KERNEL_MATRIX) return HJM_ERR_ARG;
    if (cfg->adjoint_normals != HJM_ADJ_NORMALS_AUTO && cfg->adjoint_normals != HJM_ADJ_NORMALS_REGENERATE)
        return HJM_ERR_ARG;
    const bool mfma_ok = cfg->rng == HJM_RNG_PHILOX && stride == kMfmaStride;
    if (cfg->path_kernel == HJM_KERNEL_MATRIX && !mfma_ok) return HJM_ERR_UNSUPPORTED;
    // AUTO: the matrix cores for FP32; FP64 keeps the vector path kernel unless MATRIX is
    // asked for (its valuation and statistics stay on the vector ALUs either way)
    p->use_mfma = mfma_ok && cfg->precision == HJM_FP32_KAHAN && cfg->path_kernel != HJM_KERNEL_VECTOR;
    p->use_mfma64 = mfma_ok && cfg->precision == HJM_FP64 && cfg->path_kernel == HJM_KERNEL_MATRIX;

    p->device = cfg->device;
    p->precision = cfg->precision;
    p->paths = cfg->paths;
    p->nsets = pf->nsets;
    p->ndates = nd;
    p->do_pfe = cfg->pfe_quantile > 0.0;
    p->pfe_rank = quantile_rank(cfg->paths, cfg->pfe_quantile);
    fill_consts(p->kd, market, cfg->dt, pf->dtau);
    fill_consts(p->kf, market, cfg->dt, pf->dtau);
    PfGrid& g = p->grid;
    g.stride = stride;
    g.nsteps = S;
    g.ndates_m1 = nd - 1;
    g.paths = cfg->paths;
    g.path0 = cfg->path_offset;
    g.seed_lo = (uint32_t)cfg->seed;
    g.seed_hi = (uint32_t)(cfg->seed >> 32);
    g.dt = cfg->dt;
    p->vp.paths = cfg->paths;
    p->vp.nsets = pf->nsets;
    p->vp.ndates = nd;
    p->vp.dtau = pf->dtau;
    p->w.assign((size_t)pf->nsets * nd, 0.0);
    for (int s = 0; s < pf->nsets; ++s)
        cva_weights(nd, pf->dtau, pf->hazard_rate[s], pf->recovery, &p->w[(size_t)s * nd]);
    // the swaps grouped by set, in the caller's order within a set
    const int G = pf->nsets, N = pf->nswaps;
    std::vector<int> order((size_t)N);
    std::vector<int>& ints = p->book_ints;
    std::vector<double>& reals = p->book_reals;
    ints.assign((size_t)G + 1 + N, 0);
    reals.resize(2 * (size_t)N);
    int* first = ints.data();
    for (int s = 0; s < N; ++s) ++first[pf->netting_set[s] + 1];
    for (int g = 0; g < G; ++g) first[g + 1] += first[g];
    {
        std::vector<int> at(first, first + G);
        for (int s = 0; s < N; ++s) order[(size_t)at[pf->netting_set[s]]++] = s;
    }
    for (int i = 0; i < N; ++i) {
        const int s = order[(size_t)i];
        first[G + 1 + i] = pf->periods[s];
        reals[(size_t)i] = pf->sign_notional[s];
        reals[(size_t)N + i] = pf->sign_notional[s] * pf->fixed_rate[s] * pf->dtau;
    }

    DeviceGuard guard;
    HJM_TRY(guard.set(cfg->device));
    HJM_HIP(hipDeviceGetAttribute(&p->cus, hipDeviceAttributeMultiprocessorCount, cfg->device),
            HJM_ERR_DEVICE);
    pplan_apply_tuning(p, p->tuning);
    // pinned: the column sums and the PFE rows of one run, or a Greeks call's sums
    const size_t pinned = std::max<size_t>((size_t)pf->nsets * (2 * nd + 2), 64 * 160 + 5 * kTenors + 2 * (size_t)nd);
    HJM_TRY(p->ctx.take(cfg->device, sizeof(double) * pinned));
    p->stream = p->ctx.c->stream;
    p->ev = p->ctx.c->ev;
    const size_t rsz = (p->precision == HJM_FP64) ? sizeof(double) : sizeof(float);
    const size_t P = (size_t)cfg->paths;
    // workgroups of the statistics: 256 paths (exposure pass) or the fused pass's blocks
    const size_t nb = std::max<size_t>((P + kBlock - 1) / kBlock, (size_t)pf_fused_blocks(cfg->paths));
    char* raw = nullptr;
    HJM_TRY(dev_alloc(&raw, (size_t)nd * kTenors * P * rsz));
    p->d_curves = raw;
    HJM_TRY(dev_alloc(&p->d_logb, (size_t)nd * P));
    hipStream_t st = p->stream;
    const size_t rows = (size_t)G * nd;
    if (!greeks) {
        raw = nullptr;
        HJM_TRY(dev_alloc(&raw, rows * P * rsz));
        p->d_ex = raw;
        HJM_TRY(dev_alloc(&p->d_partials, (size_t)G * nb * (nd + 2)));
        HJM_TRY(dev_alloc(&p->d_sums, (size_t)G * (2 * nd + 2)));
        p->d_pfe = p->d_sums + (size_t)G * (nd + 2);
    }
    if (p->do_pfe) {
        const size_t wsb = bracket_workspace_bytes((int)rows, bracket_plan(cfg->paths, p->pfe_rank, (int)rsz),
                                                   (int)rsz);
        if (wsb) {
            HJM_TRY(dev_alloc(&p->d_selws, wsb));
            if (rsz == sizeof(float))
                HJM_TRY(dev_alloc(&p->d_loparts, rows * pf_stats_blocks(cfg->paths)));
        }
    }
    HJM_TRY(dev_alloc(&p->d_w, p->w.size()));
    HJM_HIP(hipMemcpyAsync(p->d_w, p->w.data(), p->w.size() * sizeof(double), hipMemcpyHostToDevice, st),
            HJM_ERR_DEVICE);
    // coefficient tables from the swap list
    HJM_TRY(dev_alloc(&p->d_book_ints, ints.size()));
    HJM_TRY(dev_alloc(&p->d_book_reals, reals.size()));
    HJM_HIP(hipMemcpyAsync(p->d_book_ints, ints.data(), ints.size() * sizeof(int), hipMemcpyHostToDevice, st),
            HJM_ERR_DEVICE);
    HJM_HIP(hipMemcpyAsync(p->d_book_reals, reals.data(), reals.size() * sizeof(double),
                           hipMemcpyHostToDevice, st),
            HJM_ERR_DEVICE);
    HJM_TRY(dev_alloc(&p->d_coef, rows * kMaxPeriods));
    HJM_TRY(dev_alloc(&p->d_a, rows));
    HJM_TRY(dev_alloc(&p->d_kmax, rows));
    p->vp.kmax = p->d_kmax;
    const BookSwaps book{p->d_book_ints, p->d_book_ints + G + 1, p->d_book_reals, p->d_book_reals + N};
    HJM_HIP(launch_book_tables(book, G, nd, p->d_coef, p->d_a, p->d_kmax, st), HJM_ERR_LAUNCH);
    // rows of matured sets are never written (their exposures are 0) and never read by the
    // statistics pass; they hold zeros for the PFE selection and the per-path copy
    if (!greeks)
        HJM_HIP(launch_clear_matured(p->d_kmax, (int)rows, (int64_t)P, p->d_ex, (int)rsz, st), HJM_ERR_LAUNCH);
    if (p->precision != HJM_FP64) {
        const size_t mt = (size_t)value_mtiles(G);
        HJM_TRY(dev_alloc(&p->d_vfrag, nd * mt * kValueFragsPerTile * kWave * 8));
        HJM_TRY(dev_alloc(&p->d_apad, nd * mt * 16));
        HJM_TRY(dev_alloc(&p->d_tilek, nd * mt));
        HJM_HIP(launch_value_fragments(p->d_coef, p->d_a, p->d_kmax, G, nd, p->d_vfrag, p->d_apad, p->d_tilek,
                                       st),
                HJM_ERR_LAUNCH);
    }
    if (cfg->rng == HJM_RNG_HOST) {
        const size_t n = P * (size_t)S * 3;
        HJM_TRY(dev_alloc(&p->d_normals, n));
        HJM_HIP(hipMemcpy(p->d_normals, cfg->host_normals, n * sizeof(double), hipMemcpyHostToDevice),
                HJM_ERR_DEVICE);
    }
    int scale = 0;
    if (p->use_mfma) {
        HJM_HIP(mfma_kernels_prepare(), HJM_ERR_DEVICE);
        const BlockMapParams bm = block_map_params(market->spot_rates, market->drifts, market->volatilities,
                                                   cfg->dt, pf->dtau, kMfmaPfMTiles, MfmaMap::kPortfolio);
        scale = bm.scale;
        HJM_TRY(dev_alloc(&p->d_wfrag, block_map_elems(bm.mtiles)));
        HJM_HIP(launch_block_map(bm, true, p->d_wfrag, p->stream), HJM_ERR_LAUNCH);
    }
    if (p->use_mfma64) {
        HJM_HIP(mfma64_kernels_prepare(), HJM_ERR_DEVICE);
        std::vector<double> wf;
        build_mfma64_block_map(market->drifts, market->volatilities, cfg->dt, pf->dtau,
                               kMfmaPfMTiles, wf, MfmaMap::kPortfolio);
        HJM_TRY(dev_alloc(&p->d_wfrag64, wf.size()));
        HJM_HIP(hipMemcpy(p->d_wfrag64, wf.data(), wf.size() * sizeof(double), hipMemcpyHostToDevice),
                HJM_ERR_DEVICE);
    }
    if (p->use_mfma || p->use_mfma64) {
        MfmaGrid& mg = p->mg;
        mg.ndates = nd;
        mg.paths = cfg->paths;
        mg.path0 = cfg->path_offset;
        mg.seed_lo = g.seed_lo;
        mg.seed_hi = g.seed_hi;
        mg.dt = ldexp(cfg->dt, -scale);
        mg.down = ldexpf(1.f, -scale);
        for (int j = 0; j < kTenors; ++j) {
            mg.spot[j] = ldexpf((float)market->spot_rates[j], scale);
            mg.spot64[j] = market->spot_rates[j];
        }
    }
    HJM_HIP(hipStreamSynchronize(st), HJM_ERR_DEVICE);
    return HJM_OK;
}

// FP32 plans value on the matrix cores. With tuning.fuse_statistics, unless the caller
// wants the per-path exposures (or the PFE needs whole rows: fewer than 4 x 16384 paths),
// valuation and statistics run fused, without writing the exposures: the PFE's bracket
// comes from the first 16384 paths valued on their own, the fused pass counts and
// collects every row's candidates, and only rows the counting leaves unresolved are
// valued again, whole, for the selection.
bool pplan_fused(hjm_portfolio_plan p, bool keep_exposures)
{
    if (p->precision == HJM_FP64 || keep_exposures || !p->tuning.fuse_statistics) return false;
    return !p->do_pfe || (p->d_selws && bracket_plan(p->paths, p->pfe_rank, (int)sizeof(float)).use);
}

// Enqueue the passes on the plan's stream, with timing events between them unless the
// sequence is being captured into a graph (a captured replay is timed as a whole).
// Timings: [0] paths, [1] valuation (+ statistics when fused), [2] statistics (the column
// sums when fused), [3] PFE selection.
int pplan_enqueue(hjm_portfolio_plan p, bool events = true, float* zs = nullptr,
                  bool keep_exposures = false)
{
    hipStream_t st = p->stream;
    const bool f64 = p->precision == HJM_FP64;
    const int rows = p->nsets * p->ndates;
    auto mark = [&](int i) { return events ? hipEventRecord(p->ev[i], st) : hipSuccess; };
    HJM_HIP(mark(0), HJM_ERR_DEVICE);
    hipError_t err;
    if (p->use_mfma)
        err = launch_pf_paths_mfma(p->mg, p->d_wfrag, (float*)p->d_curves, p->d_logb, zs,
                                   p->path_shape, st);
    else if (p->use_mfma64)
        err = launch_pf_paths_mfma64(p->mg, p->d_wfrag64, (double*)p->d_curves, p->d_logb, zs, st);
    else if (f64)
        err = launch_pf_paths_f64(p->kd, p->grid, p->d_normals, (double*)p->d_curves, p->d_logb,
                                  p->tuning.block_size, p->grid_blocks, st);
    else
        err = launch_pf_paths_f32(p->kf, p->grid, p->d_normals, (float*)p->d_curves, p->d_logb,
                                  p->tuning.block_size, p->grid_blocks, st);
    HJM_HIP(err, HJM_ERR_LAUNCH);
    HJM_HIP(mark(1), HJM_ERR_DEVICE);
    if (!p->d_ex) return HJM_OK;   // a plan of the Greeks call
    if (pplan_fused(p, keep_exposures)) {
        const float* curves = (const float*)p->d_curves;
        float* ex = (float*)p->d_ex;
        SelRowState* state = nullptr;
        float* cand = nullptr;
        BracketPlan bp{};
        if (p->do_pfe) {
            bp = bracket_plan(p->paths, p->pfe_rank, (int)sizeof(float));
            bracket_ws_split<float>(p->d_selws, rows, &state, &cand);
            // the sample: exposures of the first bp.m paths, then the rows' brackets
            HJM_HIP(launch_pf_value_mfma(p->vp, curves, p->d_logb, p->d_vfrag, p->d_apad, p->d_tilek,
                                         ex, p->value_shape, st, bp.m),
                    HJM_ERR_LAUNCH);
            HJM_HIP(launch_bracket_sample_f32(ex, rows, p->paths, p->pfe_rank, p->d_selws, st),
                    HJM_ERR_LAUNCH);
        }
        HJM_HIP(launch_pf_value_stats_mfma(p->vp, curves, p->d_logb, p->d_vfrag, p->d_apad,
                                           p->d_tilek, p->d_w, p->d_partials, state, cand, bp.cap,
                                           p->tuning.pfe_stage_slots, st),
                HJM_ERR_LAUNCH);
        HJM_HIP(mark(2), HJM_ERR_DEVICE);
        HJM_HIP(launch_grouped_column_sum(p->d_partials, p->nsets, pf_fused_blocks(p->paths),
                                          p->ndates + 2, p->d_sums, st),
                HJM_ERR_LAUNCH);
        HJM_HIP(mark(3), HJM_ERR_DEVICE);
        if (p->do_pfe) {
            // whole rows only where the counting did not resolve the rank
            HJM_HIP(launch_pf_value_mfma(p->vp, curves, p->d_logb, p->d_vfrag, p->d_apad, p->d_tilek,
                                         ex, p->value_shape, st, -1, state, p->pfe_rank, bp.cap),
                    HJM_ERR_LAUNCH);
            HJM_HIP(launch_bracket_finish_f32(ex, rows, p->paths, p->pfe_rank, p->d_selws, p->d_pfe, st),
                    HJM_ERR_LAUNCH);
        }
        HJM_HIP(mark(4), HJM_ERR_DEVICE);
        return HJM_OK;
    }
    err = f64 ? launch_pf_value_f64(p->vp, (const double*)p->d_curves, p->d_logb,
                                    p->d_coef, p->d_a, p->d_kmax,
                                    (double*)p->d_ex, st)
              : launch_pf_value_mfma(p->vp, (const float*)p->d_curves, p->d_logb, p->d_vfrag,
                                     p->d_apad, p->d_tilek, (float*)p->d_ex, p->value_shape, st);
    HJM_HIP(err, HJM_ERR_LAUNCH);
    HJM_HIP(mark(2), HJM_ERR_DEVICE);
    // With a bracket-selection workspace the statistics pass also does the PFE's counting
    // pass: the bracket sample runs before it and the selection's last launch after it.
    void* selws = (p->do_pfe && p->d_selws &&
                   pf_stats_stage(p->paths, p->pfe_rank, p->ndates, f64 ? 8 : 4) > 0)
                      ? p->d_selws
                      : nullptr;
    if (selws) {
        err = f64 ? launch_bracket_sample((const double*)p->d_ex, rows, p->paths, p->pfe_rank, selws, st)
                  : launch_bracket_sample_f32((const float*)p->d_ex, rows, p->paths, p->pfe_rank, selws,
                                              st);
        HJM_HIP(err, HJM_ERR_LAUNCH);
    }
    err = f64 ? launch_pf_stats_f64(p->vp, (const double*)p->d_ex, p->d_w, p->d_partials,
                                    p->d_sums, selws, p->pfe_rank, nullptr, st)
              : launch_pf_stats_f32(p->vp, (const float*)p->d_ex, p->d_w, p->d_partials,
                                    p->d_sums, selws, p->pfe_rank, p->d_loparts, st);
    HJM_HIP(err, HJM_ERR_LAUNCH);
    HJM_HIP(mark(3), HJM_ERR_DEVICE);
    if (p->do_pfe) {
        if (selws)
            err = f64 ? launch_bracket_finish((const double*)p->d_ex, rows, p->paths, p->pfe_rank,
                                              selws, p->d_pfe, st)
                      : launch_bracket_finish_f32((const float*)p->d_ex, rows, p->paths, p->pfe_rank,
                                                  selws, p->d_pfe, st);
        else
            err = f64 ? launch_radix_select((const double*)p->d_ex, rows, p->paths, p->pfe_rank,
                                            p->d_selws, p->d_pfe, st)
                      : launch_radix_select_f32((const float*)p->d_ex, rows, p->paths, p->pfe_rank,
                                                p->d_selws, p->d_pfe, st);
        HJM_HIP(err, HJM_ERR_LAUNCH);
    }
    HJM_HIP(mark(4), HJM_ERR_DEVICE);
    return HJM_OK;
}

int pplan_run(hjm_portfolio_plan p)
{
    if (!p->tuning.use_graph) return pplan_enqueue(p);
    if (!p->exec) {
        HJM_HIP(hipStreamBeginCapture(p->stream, hipStreamCaptureModeThreadLocal), HJM_ERR_DEVICE);
        const int rc = pplan_enqueue(p, false);
        hipGraph_t graph = nullptr;
        const hipError_t end = hipStreamEndCapture(p->stream, &graph);
        if (rc != HJM_OK) {
            if (graph) (void)hipGraphDestroy(graph);
            return rc;
        }
        HJM_HIP(end, HJM_ERR_DEVICE);
        p->graph = graph;
        HJM_HIP(hipGraphInstantiate(&p->exec, p->graph, nullptr, nullptr, 0), HJM_ERR_DEVICE);
    }
    HJM_HIP(hipEventRecord(p->ev[0], p->stream), HJM_ERR_DEVICE);
    HJM_HIP(hipGraphLaunch(p->exec, p->stream), HJM_ERR_LAUNCH);
    HJM_HIP(hipEventRecord(p->ev[4], p->stream), HJM_ERR_DEVICE);
    return HJM_OK;
}

int pplan_collect(hjm_portfolio_plan p, hjm_portfolio_results* r)
{
    const int G = p->nsets, nd = p->ndates, nc = nd + 2;
    double* sums = static_cast<double*>(p->ctx.c->host);
    const double* pf = sums + (size_t)G * nc;
    HJM_HIP(hipMemcpyAsync(sums, p->d_sums,
                           sizeof(double) * G * (nc + (r->pfe && p->do_pfe ? nd : 0)),
                           hipMemcpyDeviceToHost, p->stream),
            HJM_ERR_DEVICE);
    HJM_HIP(hipStreamSynchronize(p->stream), HJM_ERR_LAUNCH);
    const double P = (double)p->paths, inv = 1.0 / P;
    for (int g = 0; g < G; ++g) {
        const double* sg = &sums[(size_t)g * nc];
        double cva = 0.0;
        for (int e = 0; e < nd; ++e) {
            const double ee = inv * sg[e];
            if (r->expected_exposure) r->expected_exposure[(size_t)g * nd + e] = ee;
            cva += p->w[(size_t)g * nd + e] * ee;
        }
        if (r->cva) r->cva[g] = cva;
        if (r->cva_stderr) {
            const double s1 = sg[nd], s2 = sg[nd + 1];
            const double var = (p->paths > 1) ? (s2 - s1 * s1 / P) / (P - 1.0) : 0.0;
            r->cva_stderr[g] = sqrt((var > 0.0 ? var : 0.0) / P);
        }
    }
    // device rows are [date][set]; the results are [set][date]
    if (r->pfe) {
        if (p->do_pfe) {
            for (int e = 0; e < nd; ++e)
                for (int g = 0; g < G; ++g) r->pfe[(size_t)g * nd + e] = pf[(size_t)e * G + g];
        } else {
            for (int i = 0; i < G * nd; ++i) r->pfe[i] = 0.0;
        }
    }
    if (r->exposures) {
        const size_t cells = (size_t)G * nd * p->paths;
        std::vector<double> tmp(cells);
        if (p->precision == HJM_FP64) {
            HJM_HIP(hipMemcpy(tmp.data(), p->d_ex, cells * sizeof(double), hipMemcpyDeviceToHost),
                    HJM_ERR_DEVICE);
        } else {
            std::vector<float> tf(cells);
            HJM_HIP(hipMemcpy(tf.data(), p->d_ex, cells * sizeof(float), hipMemcpyDeviceToHost),
                    HJM_ERR_DEVICE);
            for (size_t i = 0; i < cells; ++i) tmp[i] = tf[i];
        }
        for (int e = 0; e < nd; ++e)
            for (int g = 0; g < G; ++g) {
                const double* src = &tmp[((size_t)e * G + g) * p->paths];
                for (int64_t i = 0; i < p->paths; ++i)
                    r->exposures[((size_t)i * G + g) * nd + e] = src[i];
            }
    }
    if (r->timings_ms) {
        float ms = 0.f;
        for (int i = 0; i < 4; ++i) {
            if (p->tuning.use_graph) {
                r->timings_ms[i] = NAN;  // one graph replay: only its total is timed
                continue;
            }
            HJM_HIP(hipEventElapsedTime(&ms, p->ev[i], p->ev[i + 1]), HJM_ERR_DEVICE);
            r->timings_ms[i] = ms;
        }
        HJM_HIP(hipEventElapsedTime(&ms, p->ev[0], p->ev[4]), HJM_ERR_DEVICE);
        r->timings_ms[4] = ms;
    }
    return HJM_OK;
}

int pplan_create(hjm_portfolio_plan* out, const hjm_market* market, const hjm_portfolio* portfolio,
                 const hjm_config* config, const hjm_tuning* tuning, bool greeks)
{
    if (!out) return HJM_ERR_NULL;
    *out = nullptr;
    hjm_portfolio_plan p = new (std::nothrow) hjm_pplan_s();
    if (!p) return HJM_ERR_ALLOC;
    const int rc = pplan_init(p, market, portfolio, config, tuning, greeks);
    if (rc != HJM_OK) {
        pplan_release(p);
        return rc;
    }
    *out = p;
    return HJM_OK;
}

}  // namespace

extern "C" {

int hjm_portfolio_plan_create(hjm_portfolio_plan* out, const hjm_market* market,
                              const hjm_portfolio* portfolio, const hjm_config* config,
                              const hjm_tuning* tuning)
{
    return pplan_create(out, market, portfolio, config, tuning, false);
}

int hjm_portfolio_plan_execute(hjm_portfolio_plan plan, hjm_portfolio_results* results)
{
    if (!plan || !results) return HJM_ERR_NULL;
    DeviceGuard guard;
    HJM_TRY(guard.set(plan->device));
    // per-path exposures asked for: an eager run that writes them (the graph, if any, is
    // the fused form)
    if (results->exposures) HJM_TRY(pplan_enqueue(plan, true, nullptr, true));
    else HJM_TRY(pplan_run(plan));
    return pplan_collect(plan, results);
}

void hjm_portfolio_plan_destroy(hjm_portfolio_plan plan) { pplan_release(plan); }

int hjm_simulate_portfolio(const hjm_market* market, const hjm_portfolio* portfolio,
                           const hjm_config* config, const hjm_tuning* tuning,
                           hjm_portfolio_results* results)
{
    if (!results) return HJM_ERR_NULL;
    hjm_portfolio_plan p = nullptr;
    HJM_TRY(hjm_portfolio_plan_create(&p, market, portfolio, config, tuning));
    const int rc = hjm_portfolio_plan_execute(p, results);
    hjm_portfolio_plan_destroy(p);
    return rc;
}

int hjm_portfolio_cva_greeks(const hjm_market* market, const hjm_portfolio* portfolio,
                             const hjm_config* config, const hjm_tuning* tuning, hjm_greeks* gr)
{
    if (!gr || !config) return HJM_ERR_NULL;
    hjm_config cfg = *config;
    cfg.pfe_quantile = 0.0;
    hjm_portfolio_plan p = nullptr;
    HJM_TRY(pplan_create(&p, market, portfolio, &cfg, tuning, true));
    constexpr int kOut = 5 * kTenors;  // VALU sweep: g0, g1, g2, sum of lambda_e, d spot
    struct Cleanup {
        hjm_portfolio_plan p;
        float *gbar = nullptr, *beta = nullptr, *zs = nullptr;
        double *part = nullptr, *sums = nullptr, *bp = nullptr;
        uint16_t* tfrag = nullptr;
        SweepBuffers sweep;
        ~Cleanup()
        {
            const bool clean = p->ctx.quiesce();
            dev_free(clean, zs, gbar, beta, part, sums, bp, tfrag);
            sweep.free(clean);
            hjm_portfolio_plan_destroy(p);
        }
    } c{p};
    DeviceGuard guard;
    HJM_TRY(guard.set(p->device));
    const int64_t P = p->paths;
    const int nd = p->ndates, E = nd - 1;
    const int64_t nb = pf_adjoint_blocks(P);
    HJM_TRY(dev_alloc(&c.gbar, (size_t)nd * kTenors * P));
    HJM_TRY(dev_alloc(&c.beta, (size_t)nd * P));
    // the VALU sweep's sums, then per date the sums of beta and of the CVA's terms
    const size_t nsum = (size_t)kOut + 2 * nd;
    HJM_TRY(dev_alloc(&c.sums, nsum));
    const bool f64 = p->precision == HJM_FP64;
    // rows of the seeds' partials: blocks of 256 paths (FP64) or the matrix-core kernel's
    // workgroups (FP32)
    const int64_t tiles = f64 ? (P + kBlock - 1) / kBlock : pf_adjoint_seed_mfma_blocks(P);
    HJM_TRY(dev_alloc(&c.bp, (size_t)tiles * 2 * nd));
    hipStream_t st = p->stream;
    if (!f64) {
        // -Gamma^T in the order the seed's second product reads it
        const size_t nch = (size_t)(value_mtiles(p->nsets) + 1) / 2;
        HJM_TRY(dev_alloc(&c.tfrag, (size_t)nd * 4 * nch * kMfmaParts * kWave * 8));
        HJM_HIP(launch_adjoint_fragments(p->d_coef, p->nsets, nd, c.tfrag, st), HJM_ERR_LAUNCH);
    }
    hipEvent_t e0 = p->ev[5], e1 = p->ev[6];
    // the matrix-core forward keeps its normals for the reverse sweep; without the memory
    // the sweep regenerates them
    if ((p->use_mfma || p->use_mfma64) && config->adjoint_normals == HJM_ADJ_NORMALS_AUTO &&
        dev_alloc(&c.zs, (size_t)p->grid.nsteps * 3 * (size_t)P + kSweepSlack) != HJM_OK)
        c.zs = nullptr;
    const double dt = p->grid.dt, cc = dt / portfolio->dtau;
    SweepGrid sg{};
    sg.hi = E - 1;
    sg.lo = 0;
    sg.dt = (float)dt;
    sg.paths = P;
    // the matrix-core sweep for FP32 runs of the path kernels' 50-step blocks with in-kernel
    // normals; the VALU sweep for the others, and where the matrix sweep's buffers cannot be had.
    // (Both sweep in FP32: FP64 runs keep the VALU sweep's sums, from which the matrix sweep's
    // differ by that sweep's own rounding, up to 1e-5, more than FP64 results may move.)
    const bool matrix = !f64 && p->grid.stride == kMfmaStride && !p->d_normals &&
                        c.sweep.take(sg, true, cc, p->grid.nsteps, c.zs != nullptr, st) == HJM_OK;
    HJM_TRY(pplan_enqueue(p, true, c.zs));
    HJM_HIP(hipEventRecord(e0, st), HJM_ERR_DEVICE);
    hipError_t err = f64 ? launch_pf_adjoint_seed_f64(p->vp, (const double*)p->d_curves, p->d_logb,
                                                      p->d_coef, p->d_a, p->d_kmax, p->d_w, c.gbar,
                                                      c.beta, c.bp, st)
                         : launch_pf_adjoint_seed_mfma(p->vp, (const float*)p->d_curves, p->d_logb,
                                                       p->d_vfrag, c.tfrag, p->d_apad, p->d_tilek,
                                                       p->d_w, c.gbar, c.beta, c.bp, st);
    HJM_HIP(err, HJM_ERR_LAUNCH);
    // over the paths at every date: beta (the drift gradient's bank-account terms), w E
    HJM_HIP(launch_column_sum(c.bp, tiles, 2 * nd, c.sums + kOut, st), HJM_ERR_LAUNCH);
    double* sums = static_cast<double*>(p->ctx.c->host);
    double* swept = sums + nsum;
    if (matrix) {
        HJM_TRY(c.sweep.run(sg, true, c.zs, p->grid.nsteps, cfg.seed, cfg.path_offset, c.gbar, c.beta, swept, st));
    } else {
        HJM_TRY(dev_alloc(&c.part, (size_t)nb * kOut));
        HJM_HIP(launch_pf_adjoint(p->grid, cc, p->d_normals, c.zs, c.gbar, c.beta, c.part, st), HJM_ERR_LAUNCH);
        HJM_HIP(launch_column_sum(c.part, nb, kOut, c.sums, st), HJM_ERR_LAUNCH);
    }
    HJM_HIP(hipEventRecord(e1, st), HJM_ERR_DEVICE);
    HJM_HIP(hipMemcpyAsync(sums, c.sums, sizeof(double) * nsum, hipMemcpyDeviceToHost, st), HJM_ERR_DEVICE);
    HJM_HIP(hipStreamSynchronize(st), HJM_ERR_LAUNCH);
    double total = 0.0;
    for (int e = 0; e < nd; ++e) total += sums[kOut + nd + e];
    if (gr->cva) *gr->cva = total / (double)P;
    if (gr->cva_stderr) *gr->cva_stderr = NAN;
    const double inv = 1.0 / (double)P;
    double ds[kTenors], dv[kFactors * kTenors], dm[kTenors];
    if (matrix) {
        sweep_gradients(swept, true, nd, cc, dt, p->grid.stride, inv, ds, dv, dm);
    } else {
        for (int k = 0; k < kFactors * kTenors; ++k) dv[k] = sums[k] * inv;
        for (int j = 0; j < kTenors; ++j) ds[j] = sums[4 * kTenors + j] * inv;
        // drift: dt (A Lambda + B mu_sum e_0) / P with Lambda the sum over dates and paths of
        // the date-end adjoints and mu_sum = dt sum_e e (sum over paths of beta_e): beta_e
        // feeds mu in the e intervals before date e
        std::vector<double> A((size_t)kTenors * kTenors), B((size_t)kTenors * kTenors);
        adjoint_block_sums((double)step_ratio_f32(cc), p->grid.stride, A.data(), B.data());
        double musum = 0.0;
        for (int e = 1; e <= E; ++e) musum += (double)e * sums[kOut + e];
        musum *= dt;
        const double* L = sums + 3 * kTenors;
        for (int j = 0; j < kTenors; ++j) {
            double a = B[(size_t)j * kTenors] * musum;
            for (int m = 0; m < kTenors; ++m) a += A[(size_t)j * kTenors + m] * L[m];
            dm[j] = dt * a * inv;
        }
    }
    if (gr->d_spot) memcpy(gr->d_spot, ds, sizeof(ds));
    if (gr->d_vol) memcpy(gr->d_vol, dv, sizeof(dv));
    if (gr->d_drift) memcpy(gr->d_drift, dm, sizeof(dm));
    if (gr->d_vol_total) {
        memcpy(gr->d_vol_total, dv, sizeof(dv));
        drift_vjp(market->volatilities, portfolio->dtau, dm, gr->d_vol_total);
    }
    if (gr->stored_normals_bytes)
        *gr->stored_normals_bytes = c.zs ? (int64_t)p->grid.nsteps * 3 * P * (int64_t)sizeof(float) : 0;
    if (gr->timings_ms) {
        float fwd = 0.f, adj = 0.f;
        HJM_HIP(hipEventElapsedTime(&fwd, p->ev[0], p->ev[1]), HJM_ERR_DEVICE);
        HJM_HIP(hipEventElapsedTime(&adj, e0, e1), HJM_ERR_DEVICE);
        gr->timings_ms[0] = fwd;
        gr->timings_ms[1] = adj;
        gr->timings_ms[2] = fwd + adj;
    }
    return HJM_OK;
}

int hjm_portfolio_autotune(const hjm_market* market, const hjm_portfolio* portfolio,
                           const hjm_config* config, hjm_tuning* best, double* best_ms)
{
    if (!best || !config || !portfolio) return HJM_ERR_NULL;
    hjm_config cfg = *config;
    // FP64 runs on host normals have a path kernel of their own, the one that FP64's launch fields
    // are for; it is tuned on the first of the caller's normals. The others are tuned on the
    // generator's.
    const bool host64 = cfg.precision == HJM_FP64 && cfg.path_kernel != HJM_KERNEL_MATRIX && cfg.host_normals;
    if (cfg.rng == HJM_RNG_HOST && !host64) cfg.rng = HJM_RNG_PHILOX;
    // the VALU path kernel's cost is linear in the horizon: it is tuned on two dates
    hjm_portfolio short_pf = *portfolio;
    std::vector<int32_t> per;
    // the plan's own choice of path kernel (pplan_init)
    const bool mfma = cfg.precision == HJM_FP32_KAHAN && cfg.path_kernel != HJM_KERNEL_VECTOR &&
                      cfg.dt > 0.0 && llround(portfolio->dtau / cfg.dt) == kMfmaStride;
    int nd = 0;
    HJM_TRY(check_portfolio(portfolio, &nd));
    if (!mfma) {
        short_pf.horizon = std::min(portfolio->horizon, 2.0 * portfolio->dtau);
        per.assign(portfolio->periods, portfolio->periods + portfolio->nswaps);
        for (auto& x : per) x = std::min(x, 2);
        short_pf.periods = per.data();
        cfg.pfe_quantile = 0.0;
    }
    hjm_portfolio_plan p = nullptr;
    HJM_TRY(hjm_portfolio_plan_create(&p, market, &short_pf, &cfg, nullptr));
    DeviceGuard guard;
    int rc = guard.set(p->device);
    // mean of 3 eager executes after one untimed, per timing slot
    auto measure = [&](const hjm_tuning& t, double (&ms)[5]) {
        pplan_apply_tuning(p, t);
        for (double& m : ms) m = 0.0;
        double tm[5];
        hjm_portfolio_results r{};
        r.timings_ms = tm;
        for (int rep = 0; rep < 4 && rc == HJM_OK; ++rep) {
            rc = pplan_enqueue(p);
            if (rc == HJM_OK) rc = pplan_collect(p, &r);
            if (rep > 0)
                for (int i = 0; i < 5; ++i) ms[i] += tm[i] / 3.0;
        }
    };
    hjm_tuning bt{256, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    double ms[5];
    if (p->use_mfma) {
        // path kernel: shape x {one workgroup per group, persistent (one per CU)}
        const int shapes[4][2] = {{2, 8}, {2, 12}, {1, 12}, {1, 16}};
        double bv = 1e300;
        hjm_tuning t = bt;
        for (const auto& sh : shapes)
            for (int bpc : {0, 1}) {
                t.path_tiles = sh[0];
                t.path_waves = sh[1];
                t.blocks_per_cu = bpc;
                measure(t, ms);
                if (rc == HJM_OK && ms[0] < bv) {
                    bv = ms[0];
                    bt.path_tiles = sh[0];
                    bt.path_waves = sh[1];
                    bt.blocks_per_cu = bpc;
                }
            }
        // valuation: tiles x waves x LDS stage (stages below the M-tile count only)
        const int mtiles = value_mtiles(p->nsets);
        bv = 1e300;
        t = bt;
        for (int tiles : {4, 2})
            for (int waves : {4, 8})
                for (int stage : {8, 4, 2}) {
                    if (stage != 8 && stage >= mtiles) continue;
                    t.value_tiles = tiles;
                    t.value_waves = waves;
                    t.value_stage = stage;
                    measure(t, ms);
                    if (rc == HJM_OK && ms[1] < bv) {
                        bv = ms[1];
                        bt.value_tiles = tiles;
                        bt.value_waves = waves;
                        bt.value_stage = stage;
                    }
                }
        // the exposure pass against the fused valuation-statistics pass (which keeps its
        // own shape): everything after the path kernel
        double passes[2] = {1e300, 1e300};
        for (int fuse : {0, 1}) {
            t = bt;
            t.fuse_statistics = fuse;
            measure(t, ms);
            if (rc == HJM_OK) passes[fuse] = ms[4] - ms[0];
        }
        bt.fuse_statistics = passes[1] < passes[0] ? 1 : 0;
    } else if (p->precision != HJM_FP64 || p->d_normals) {
        // (FP64 path kernels on the generator's normals have a shape by path count, or one shape)
        double bv = 1e300;
        for (int bs : {64, 128, 256})
            for (int bpc : {0, 1, 2, 4, 8}) {
                hjm_tuning t = bt;
                t.block_size = bs;
                t.blocks_per_cu = bpc;
                measure(t, ms);
                if (rc == HJM_OK && ms[0] < bv) {
                    bv = ms[0];
                    bt.block_size = bs;
                    bt.blocks_per_cu = bpc;
                }
            }
    }
    double total = 0.0;
    if (rc == HJM_OK) {
        measure(bt, ms);
        total = ms[4];
    }
    hjm_portfolio_plan_destroy(p);
    if (rc != HJM_OK) return rc;
    bt.use_graph = 1;
    *best = bt;
    if (best_ms) *best_ms = total;
    return HJM_OK;
}

}  // extern "C"
