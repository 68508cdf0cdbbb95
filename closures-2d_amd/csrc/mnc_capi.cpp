// mnc_capi.cpp -- the C-ABI (include/mnclosure.h): context, device memory,
// kernel sequencing and timing.  Host code compiled with hipcc.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "mnc_internal.h"

struct mnc_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    mnc::Tables tab;
    int num_cu = 256;
    // tables on device
    double *d_w = nullptr, *d_p = nullptr, *d_xi = nullptr, *d_eta = nullptr, *d_gv = nullptr;
    int *d_gptr = nullptr, *d_gk = nullptr;
    // solver state / stats
    int *d_ctl = nullptr;            // [0],[1] list counts, [2] tail queue, [3] error bits, [4] deferred
    long long *d_stats = nullptr;    // [kStatWords]
    // change-of-basis grid state: per-cell basis (column-major) and multipliers
    // in that basis, and the blocks' tables seen through their cells' bases
    double *d_cbB = nullptr, *d_cbaP = nullptr, *d_cbws = nullptr;
    size_t cb_cells = 0;
    int cb_blocks = 0;
    double *d_std = nullptr;         // per-cell solver state (doubles)
    int *d_sti = nullptr;            // per-cell solver state (ints)
    int *d_lists = nullptr;          // mnc::kNumLists lists of cell indices (see mnc_internal.h)
    // mixed precision operand tables (absent when the order/quadrature has none)
    mnc::MixTables mix;
    bool has_mix = false;
    bool ppn = false;                // moment type PPn (setup->moment_type == 1)
    double *d_mz = nullptr, *d_mg = nullptr, *d_mgv = nullptr;
    float *d_mpv = nullptr;          // Gaunt map in compile-time pattern order (mixed logic)
    unsigned short *d_mh = nullptr;
    int *d_mgptr = nullptr, *d_mgk = nullptr;
    // FP64 solve with a row of lanes per cell (moment orders up to 4)
    mnc::OrbitTables orb;
    double *d_ot = nullptr, *d_ogv = nullptr;
    unsigned char *d_opos = nullptr;
    int *d_ogoff = nullptr, *d_ogk = nullptr;
    // FP64 matrix-core operand tables of the high orders (M8)
    mnc::G64Tables g64;
    bool has_g64 = false;
    double *d_gz = nullptr, *d_gh = nullptr, *d_gmap = nullptr;
    int *d_gidx = nullptr, *d_gpos = nullptr;
    size_t state_cap = 0;
    int state_nm = 0;
    void *d_noalloc = nullptr;       // the library's fixed scratch array on this device (not owned)
    // tuning
    int rounds = -1;                 // -1 (not set): run_newton's choice, 6 or 0
    int tail_blocks = 0;             // 0: 2 per CU
    int tail_mode = 0;               // 0, 3: row of lanes per cell, 1: lane per cell, 2: wave sweep + serial logic
    int mix_cond_log10 = 9;          // mixed steps need cond(H) <= 10^this, else FP64
    int mix_defer = 0;               // 0: redone steps wait for the FP64 tail; 1: FP64 lockstep rounds
    int mix_split = 3;               // bf16 parts of e and of the table in the mixed Hessian products
    int mix_blocks = 0;              // 0: one per CU
    int flux_tile = 3;               // 0: ansatz to HBM + flux; 1: fused, 8x8 tiles; 2: fused, 16x16;
                                     // 3: fused, 16x16, directions split into flux_groups
    int flux_groups = 0;             // direction groups of flux_tile 3; 0: by the grid (auto_flux_groups)
    int flux_overlap = 1;            // flux_tile 3: the flux of tiles clear of the Newton tail runs beside it
    int learned_fused = 1;           // 1: network and judge in one kernel; 0: the network's kernel, then the FP64 judge
    int learned_fallback_iters = 10;   // a network-started cell failing at level 0 within this many
                                     // iterations restarts from isotropicAlpha at level 0
    int learned_gate_log10 = -2;     // the network is consulted when ||g(best start)|| > 10^this ||u||;
                                     // kGateOff: never (no network launches)
    // grid
    bool has_grid = false;
    mnc_grid_desc grid{};
    double *d_mom = nullptr, *d_alpha = nullptr, *d_old = nullptr, *d_st = nullptr, *d_ss = nullptr,
           *d_flux = nullptr, *d_ansatz = nullptr, *d_fpart = nullptr;
    int ansatz_chunk = 0;
    mnc::FluxTables ftab;            // orders 5 to 8
    double *d_foz = nullptr, *d_fop = nullptr, *d_fodir = nullptr;
    int *d_foidx = nullptr;
    int *d_tflag = nullptr;          // flux_tile 3 tile flags (flux_overlap)
    hipStream_t stream2 = nullptr;   // the second stream of flux_overlap (default priority)
    hipEvent_t ev_fork = nullptr, ev_join = nullptr;
    // flux_overlap: run_newton leaves the tail for the step to launch
    bool defer_tail = false, tail_saved = false, tail_mixed = false;
    mnc::NewtonArgs tail_a{};
    mnc::LaunchPlan tail_lp{};
    int tail_lin = 0, tail_flin = 2;
    // batch staging for host entry points
    double *d_bu = nullptr, *d_ba = nullptr;
    mnc_outs *d_bo = nullptr;
    size_t batch_cap = 0;
    int batch_n = 0;                 // cells staged by mnc_batch_set
    // learned warm start
    bool mlp_ready = false, mlp_stats_set = false;
    int mlp_step = 0;
    float *d_mlp = nullptr;          // parameters + standardisation, grad, m, v (4 blocks)
    float *d_mlp_scratch = nullptr, *d_mlp_loss = nullptr;
    size_t mlp_scratch_cap = 0, mlp_loss_cap = 0;
    double *d_cb_batch = nullptr;    // the host-array optcb entry's arrays and workspace, its outputs
    mnc_outs *d_cb_outs = nullptr;
    size_t cb_batch_cap = 0, cb_outs_cap = 0;
    double *d_mlp_io = nullptr;      // host-call staging (inputs, targets/outputs)
    size_t mlp_io_cap = 0;
    double *d_guess = nullptr;       // the unfused learned start's guesses
    size_t guess_cap = 0;
    // timing
    bool timing = false;
    struct Ev { int kc; hipEvent_t a, b; };
    std::vector<Ev> events;
    // hipGraphs of whole mnc_update steps, one per distinct (dt, options)
    int use_graph = 0;
    unsigned long long epoch = 1;    // bumped by every device (re)allocation and tuning change
    struct StepGraph {
        unsigned long long epoch = 0;
        double dt = 0.0;
        mnc_options o{};
        int eager_runs = 0;
        hipGraphExec_t exec = nullptr;
    };
    StepGraph graphs[4];
    int graph_next = 0;
    long long t_launch[MNC_NUM_KCLASS] = {};
    double t_ms[MNC_NUM_KCLASS] = {};
    std::string last_error;
};

namespace {

int ctx_fail(mnc_ctx *ctx, int code, const char *what, hipError_t e = hipSuccess) {
    if (ctx) {
        char buf[512];
        if (e != hipSuccess)
            snprintf(buf, sizeof buf, "%s failed: %s", what, hipGetErrorString(e));
        else
            snprintf(buf, sizeof buf, "%s", what);
        ctx->last_error = buf;
    }
    return code;
}

template <class T>
int dalloc(mnc_ctx *ctx, T **p, size_t n) {
    ++ctx->epoch;    // captured steps hold device addresses
    if (*p) { (void)hipFree(*p); *p = nullptr; }
    if (n == 0) return MNC_OK;
    MNC_HIP_CHECK(hipMalloc((void **)p, n * sizeof(T)));
    return MNC_OK;
}

void drop_graph(mnc_ctx::StepGraph &g) {
    if (g.exec) (void)hipGraphExecDestroy(g.exec);
    g = mnc_ctx::StepGraph{};
}

// Records an event pair around one launch when timing is on.
struct Timed {
    mnc_ctx *ctx;
    int kc;
    hipEvent_t a = nullptr, b = nullptr;
    bool on;
    Timed(mnc_ctx *c, int k, bool enable = true) : ctx(c), kc(k), on(enable && c->timing) {
        if (on) {
            (void)hipEventCreate(&a);
            (void)hipEventCreate(&b);
            (void)hipEventRecord(a, ctx->stream);
        }
    }
    ~Timed() {
        if (on) {
            (void)hipEventRecord(b, ctx->stream);
            ctx->events.push_back({kc, a, b});
        }
    }
};

int ensure_state(mnc_ctx *ctx, size_t ncells) {
    if (ncells <= ctx->state_cap) return MNC_OK;
    int df = 0, ifl = 0;
    mnc::newton_store_fields(ctx->tab.nm, ctx->tab.np2, &df, &ifl);
    const size_t cap = std::max<size_t>(ncells, 64);
    int st;
    if ((st = dalloc(ctx, &ctx->d_std, size_t(df) * cap)) || (st = dalloc(ctx, &ctx->d_sti, size_t(ifl) * cap)) ||
        (st = dalloc(ctx, &ctx->d_lists, size_t(mnc::kNumLists) * cap)))
        return st;
    ctx->state_cap = cap;
    return MNC_OK;
}

// Reads the kernels' error bits (synchronising the stream).
int check_errors(mnc_ctx *ctx, const int *d_ctl = nullptr) {
    int ctl[4] = {0, 0, 0, 0};
    MNC_HIP_CHECK(hipMemcpyAsync(ctl, d_ctl ? d_ctl : ctx->d_ctl, sizeof ctl, hipMemcpyDeviceToHost, ctx->stream));
    MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    if (ctl[3] & (1 << MNC_ERR_U0)) return ctx_fail(ctx, MNC_ERR_U0, "u[0] <= 0 in at least one cell");
    if (ctl[3] & (1 << MNC_ERR_MAXREG)) return ctx_fail(ctx, MNC_ERR_MAXREG, "Max regularization achieved");
    return MNC_OK;
}

// m_inf of the supplementary stop test (opt.cpp:61-62): the bound of the
// real spherical harmonics up to order floor(sqrt(n)) + 1.
double gamma_minf(int nm) {
    const int pn_order = int(std::floor(std::sqrt(double(nm)))) + 1;
    return std::sqrt((2 * pn_order + 1) / (2 * M_PI));
}

int check_opts(mnc_ctx *ctx, const mnc_options *o) {
    if (ctx->device < 0) return ctx_fail(ctx, MNC_ERR_STATE, "host-only context (device < 0)");
    if (!o) return ctx_fail(ctx, MNC_ERR_ARG, "options pointer is NULL");
    if (o->max_iter < 1) return ctx_fail(ctx, MNC_ERR_ARG, "max_iter must be >= 1");
    if (!(o->tol_rel >= 0.0)) return ctx_fail(ctx, MNC_ERR_ARG, "tol_rel must be >= 0");
    if (std::isnan(o->tol_gamma)) return ctx_fail(ctx, MNC_ERR_ARG, "tol_gamma is NaN");
    if (o->tol_gamma > 0.0 && o->opt_type != MNC_OPT_NEWTON)
        return ctx_fail(ctx, MNC_ERR_ARG, "tol_gamma is a stop test of the Newton optimiser (opt_type 0)");
    if (o->precision != MNC_PREC_FP64 && o->precision != MNC_PREC_MIXED)
        return ctx_fail(ctx, MNC_ERR_ARG, "unknown precision");
    if (o->warm_start < MNC_WARM_PREVIOUS || o->warm_start > MNC_WARM_LEARNED)
        return ctx_fail(ctx, MNC_ERR_ARG, "unknown warm_start");
    if (o->line_search != MNC_LS_REFERENCE && o->line_search != MNC_LS_ROBUST)
        return ctx_fail(ctx, MNC_ERR_ARG, "unknown line_search");
    if (ctx->ppn) {
        if (!(o->delta_ppn > 0.0)) return ctx_fail(ctx, MNC_ERR_ARG, "PPn needs delta_ppn > 0");
        if (o->precision != MNC_PREC_FP64 || o->warm_start == MNC_WARM_LEARNED)
            return ctx_fail(ctx, MNC_ERR_ARG, "PPn runs the FP64 form from the previous or isotropic alpha");
        if (ctx->tab.nm > 15) return ctx_fail(ctx, MNC_ERR_ARG, "PPn has kernels for moment orders up to 4");
    }
    if (o->opt_type != MNC_OPT_NEWTON && o->opt_type != MNC_OPT_CHANGE_BASIS && o->opt_type != MNC_OPT_BFGS)
        return ctx_fail(ctx, MNC_ERR_ARG, "unknown opt_type");
    if (o->opt_type == MNC_OPT_BFGS && (o->max_bfgs_iter < 1 || !(o->cond_h_max_bfgs > 1.0)))
        return ctx_fail(ctx, MNC_ERR_ARG, "the BFGS variant needs max_bfgs_iter >= 1 and cond_h_max_bfgs > 1 "
                                          "(else it takes no step)");
    if (o->opt_type != MNC_OPT_NEWTON &&
        (ctx->ppn || ctx->tab.use_gaunt || ctx->tab.np2 != ctx->tab.nm || ctx->tab.nm > 15 ||
         o->precision != MNC_PREC_FP64 || o->warm_start != MNC_WARM_PREVIOUS))
        return ctx_fail(ctx, MNC_ERR_ARG, "the change-of-basis optimiser runs Mn, direct Hessian, FP64, "
                                          "from the cell's own state");
    return MNC_OK;
}

// ---- learned warm start -------------------------------------------------------
mnc::MlpBuffers mlp_buffers(mnc_ctx *ctx) {
    const size_t np = size_t(mnc::mlp_param_count()) + mnc::kMlpStats;
    return {ctx->d_mlp, ctx->d_mlp + np, ctx->d_mlp + 2 * np, ctx->d_mlp + 3 * np,
            (unsigned short *)(ctx->d_mlp + 4 * np), ctx->d_mlp_scratch, ctx->d_mlp_loss};
}

int mlp_alloc(mnc_ctx *ctx) {
    if (ctx->d_mlp) return MNC_OK;
    return dalloc(ctx, &ctx->d_mlp, 4 * (size_t(mnc::mlp_param_count()) + mnc::kMlpStats) + mnc::mlp_operand_floats());
}

int mlp_train_alloc(mnc_ctx *ctx, int rows, size_t losses) {
    int st = mlp_alloc(ctx);
    if (st) return st;
    const size_t need = mnc::mlp_scratch_floats(rows);
    if (need > ctx->mlp_scratch_cap) {
        if ((st = dalloc(ctx, &ctx->d_mlp_scratch, need))) return st;
        ctx->mlp_scratch_cap = need;
    }
    if (losses > ctx->mlp_loss_cap) {
        if ((st = dalloc(ctx, &ctx->d_mlp_loss, losses))) return st;
        ctx->mlp_loss_cap = losses;
    }
    return MNC_OK;
}

int mlp_io(mnc_ctx *ctx, size_t doubles) {
    if (doubles <= ctx->mlp_io_cap) return MNC_OK;
    int st = dalloc(ctx, &ctx->d_mlp_io, doubles);
    if (st) return st;
    ctx->mlp_io_cap = doubles;
    return MNC_OK;
}

int mlp_check(mnc_ctx *ctx, bool need_ready) {
    if (ctx->device < 0) return ctx_fail(ctx, MNC_ERR_STATE, "host-only context (device < 0)");
    if (ctx->tab.nm != 15) return ctx_fail(ctx, MNC_ERR_ARG, "the learned warm start exists for moment order 4 only");
    if (need_ready && !ctx->mlp_ready)
        return ctx_fail(ctx, MNC_ERR_STATE, "no MLP parameters (mnc_mlp_init/mnc_mlp_set_params first)");
    return MNC_OK;
}

// Enqueues the batched Newton on device arrays (stats accumulate in d_stats).
// With check, synchronises and turns the kernels' error bits into a status.
// learned_gate_log10 at this value switches the network off
constexpr int kGateOff = 5;

// A solve whose path depends on the rounding of f: the reference's Armijo test below
// TOL 1e-6 compares values of f that differ by that rounding.
bool by_rounding(const mnc_options *o) { return o->line_search == MNC_LS_REFERENCE && o->tol_rel < 1e-6; }

// Lockstep rounds of a solve for which none are set.  FP64 cells go straight to the
// tail's kernel.  Not if the path depends on the rounding of f, and with it on the
// order of the sums: the lockstep kernels sum in the reference's.  Seven rounds are
// the fewest after which no more than one per cent of the cells that take the
// reference's iterations end elsewhere than it does (3,000 M3 closures, Q = 30, four
// draws: 1.27% without rounds, 1.05 after six, 0.84 after seven and after twelve; 0.88
// with six and the former tail of a wave per cell).  Against that form (ms, M4, Q = 16,
// means over draws): 2,049 closures from near starts 2.4 -> 1.6 (its best draws 1.5),
// cold 3.4 -> 1.8, 200,003 cold 16.3 -> 9.7, 150,001 with beams 19.5 -> 9.3, a step of a
// 133 x 101 lattice 7.9 -> 3.5; with twelve rounds 2.5, 2.8, 8.4, 9.6 and 5.4.
int auto_rounds(const mnc_ctx *ctx, const mnc_options *o) {
    const bool network = o->warm_start == MNC_WARM_LEARNED && ctx->learned_gate_log10 < kGateOff;
    return o->precision == MNC_PREC_MIXED || network ? 6 : (by_rounding(o) ? 7 : 0);
}

// na: the no-allocation entry point's state regions (the library's fixed
// scratch array) in place of the context's buffers; then nothing is allocated
// and no timing events are recorded.
int run_newton(mnc_ctx *ctx, int ncells, double *u, double *alpha, const mnc_options *o, mnc_outs *outs,
               const double *alpha_guess, bool check, const mnc::NoAllocState *na = nullptr) {
    if (ncells <= 0) return MNC_OK;
    if (o->opt_type != MNC_OPT_NEWTON)
        return ctx_fail(ctx, MNC_ERR_ARG, "batch solves run the Newton optimiser; the change-of-basis batch is "
                                          "mnc_optcb_batch_host");
    const auto &t = ctx->tab;
    const bool mixed = o->precision == MNC_PREC_MIXED;
    if (mixed && !ctx->has_mix)
        return ctx_fail(ctx, MNC_ERR_ARG, "mixed precision needs moment order <= 4 and quad order <= 16");
    if (ctx->has_g64 && (mixed || o->warm_start == MNC_WARM_LEARNED))
        return ctx_fail(ctx, MNC_ERR_ARG, "moment order 8 runs the FP64 form only");
    const bool learned = o->warm_start == MNC_WARM_LEARNED;
    if (na && learned) return ctx_fail(ctx, MNC_ERR_ARG, "the learned warm start allocates the network's buffers");
    int st = na ? MNC_OK : ensure_state(ctx, size_t(ncells));
    if (st) return st;
    const bool timed = na == nullptr;
    double *st_d = na ? na->st_d : ctx->d_std;
    int *st_i = na ? na->st_i : ctx->d_sti, *lists = na ? na->lists : ctx->d_lists, *ctl = na ? na->ctl : ctx->d_ctl;
    const size_t cap = na ? na->cap : ctx->state_cap;
    if (learned && ctx->learned_gate_log10 < kGateOff && (st = mlp_check(ctx, true))) return st;
    // the one-kernel network and judge holds the quadrature in LDS
    const bool net_fused = ctx->learned_fused && ctx->tab.nq <= mnc::kNetMaxQ;
    if (learned && ctx->learned_gate_log10 < kGateOff && !net_fused) {   // the unfused path's buffers
        if (size_t(ncells) > ctx->guess_cap) {
            if ((st = dalloc(ctx, &ctx->d_guess, size_t(ncells) * 15))) return st;
            ctx->guess_cap = size_t(ncells);
        }
        alpha_guess = ctx->d_guess;
    }
    mnc::NewtonArgs a{};
    a.ncells = ncells;
    a.u = u;
    a.alpha = alpha;
    a.outs = outs;
    a.w = ctx->d_w;
    a.p = ctx->d_p;
    a.nq = t.nq;
    a.gptr = ctx->d_gptr;
    a.gk = ctx->d_gk;
    a.gv = ctx->d_gv;
    a.ppn = ctx->ppn ? 1 : 0;
    a.delta = o->delta_ppn;
    a.max_iter = o->max_iter;
    a.tol = o->tol_rel;
    a.cond_h_max = o->cond_h_max;
    a.tol_gamma = o->tol_gamma;
    a.gamma_minf = gamma_minf(t.nm);
    a.warm = o->warm_start;
    a.ls_mode = o->line_search;
    a.stats = ctx->d_stats;
    a.alpha_guess = alpha_guess;
    a.st_d = st_d;
    a.st_i = st_i;
    a.lists = lists;
    a.ctl = ctl;
    a.cap = cap;
    a.mz = ctx->d_mz;
    a.mg = ctx->d_mg;
    a.mh = ctx->d_mh;
    a.mnt = ctx->mix.nt;
    a.mgptr = ctx->d_mgptr;
    a.mgk = ctx->d_mgk;
    a.mgv = ctx->d_mgv;
    a.mpv = ctx->d_mpv;
    a.cmix = std::pow(10.0, ctx->mix_cond_log10);
    a.gate = std::pow(10.0, ctx->learned_gate_log10);
    a.fallback_iters = ctx->learned_fallback_iters;
    a.mlp_w = ctx->d_mlp;
    a.ot = ctx->d_ot;
    a.opos = ctx->d_opos;
    a.ogoff = ctx->d_ogoff;
    a.ogk = ctx->d_ogk;
    a.ogv = ctx->d_ogv;
    a.no = ctx->orb.no;
    a.nop = ctx->orb.nop;
    a.gz = ctx->d_gz;
    a.gh = ctx->d_gh;
    a.gmap = ctx->d_gmap;
    a.gidx = ctx->d_gidx;
    a.gpos = ctx->d_gpos;
    a.gnt = ctx->g64.nt;
    mnc::LaunchPlan lp;
    lp.r0 = 0;
    const bool network = learned && ctx->learned_gate_log10 < kGateOff;
    const int rounds = ctx->rounds >= 0 ? ctx->rounds : auto_rounds(ctx, o);
    lp.r1 = rounds;
    lp.num_cu = ctx->num_cu;
    lp.fresh = rounds == 0 && !mixed && !network && (ctx->tail_mode == 0 || ctx->tail_mode == 3 || ctx->ppn);
    if (lp.fresh) lp.init = false;
    lp.tail_blocks = ctx->tail_blocks > 0 ? ctx->tail_blocks : 2 * ctx->num_cu;
    lp.tail_mode = ctx->tail_mode;
    lp.mix_blocks = ctx->mix_blocks > 0 ? ctx->mix_blocks : ctx->num_cu;
    lp.defer_rounds = ctx->mix_defer;
    lp.mix_split = ctx->mix_split;
    const bool gaunt = t.use_gaunt != 0;
    auto launch = [&](const mnc::NewtonArgs &aa, const mnc::LaunchPlan &p) -> int {
        if (mixed) {
            if (!mnc::launch_newton_mixed(aa, t.nm, t.np2, gaunt, p, ctx->stream))
                return ctx_fail(ctx, MNC_ERR_ARG, "no mixed-precision Newton kernel instance for this order");
        } else if (!mnc::launch_newton_fp64(aa, t.nm, t.np2, gaunt, p, ctx->stream)) {
            return ctx_fail(ctx, MNC_ERR_ARG, "no FP64 Newton kernel instance for this moment order");
        }
        return MNC_OK;
    };
    // The prologue and lockstep rounds, then the persistent tail, each in its
    // own timing class (the same launches as one plan).
    auto launch_timed = [&](const mnc::NewtonArgs &aa, const mnc::LaunchPlan &p, bool reset) -> int {
        mnc::LaunchPlan body = p, tail = p;
        body.tail = false;
        tail.init = false;
        tail.r0 = tail.r1 = p.r1;
        int s2;
        {
            Timed tm(ctx, MNC_KCLASS_NEWTON, timed);
            if (reset) mnc::launch_ctl_reset(ctl, ctx->stream);
            if ((s2 = launch(aa, body))) return s2;
        }
        if (p.tail && ctx->defer_tail && !p.fresh) {   // the step launches it (flux_overlap)
            ctx->tail_saved = true;
            ctx->tail_mixed = mixed;
            ctx->tail_a = aa;
            ctx->tail_lp = tail;
            ctx->tail_lin = p.r1 & 1;   // the lists the tail reads (launch_all, launch_mixed_all)
            ctx->tail_flin = mixed ? 2 + (p.defer_rounds ? (p.r1 & 1) : 0) : 2;
        } else if (p.tail) {
            Timed tm(ctx, MNC_KCLASS_TAIL, timed);
            if ((s2 = launch(aa, tail))) return s2;
        }
        return MNC_OK;
    };
    if (learned && ctx->learned_gate_log10 >= kGateOff) {
        // network off: every cell starts from the alpha passed in (isotropicAlpha
        // if it is not finite), as the gate would decide at any threshold above
        // the gradient norms, without the network's or judge_kernel's launches
        if (t.nm != 15) return ctx_fail(ctx, MNC_ERR_ARG, "the learned warm start is for moment order 4");
        if ((st = launch_timed(a, lp, true))) return st;
    } else if (learned) {
        // Round 1 evaluates every cell at its start and parks those failing the
        // gate on the network's list; the network runs on those rows only (the
        // count is read on the device), judge_kernel moves them to round 2's list.
        if (t.nm != 15) return ctx_fail(ctx, MNC_ERR_ARG, "the learned warm start is for moment order 4");
        mnc::LaunchPlan first = lp, rest = lp;
        first.r1 = 1;
        first.tail = false;
        rest.r0 = 1;
        rest.r1 = std::max(rounds, 1);
        rest.init = false;
        mnc::NewtonArgs ad = a;
        ad.divert = 1;
        {
            Timed tm(ctx, MNC_KCLASS_NEWTON);
            mnc::launch_ctl_reset(ctx->d_ctl, ctx->stream);
            if ((st = launch(ad, first))) return st;
        }
        if (net_fused) {
            // the network and the judge in one kernel on the parked cells
            Timed tm(ctx, MNC_KCLASS_MLP);
            if (!mnc::launch_newton_net_judge(a, t.nm, t.np2, gaunt, ncells, ctx->num_cu, ctx->stream))
                return ctx_fail(ctx, MNC_ERR_ARG, "no learned warm start for this order");
        } else {
            {
                Timed tm(ctx, MNC_KCLASS_MLP);
                mnc::mlp_predict_listed(mlp_buffers(ctx), u, ctx->d_lists + size_t(mnc::kMlpListIndex) * ctx->state_cap,
                                        ctx->d_ctl + mnc::kMlpListWord, ncells, ctx->d_guess, ctx->stream);
            }
            {
                Timed tm(ctx, MNC_KCLASS_NEWTON);
                if (!mnc::launch_newton_judge(a, t.nm, t.np2, gaunt, ctx->stream))
                    return ctx_fail(ctx, MNC_ERR_ARG, "no learned warm start for this order");
            }
        }
        if ((st = launch_timed(a, rest, false))) return st;
    } else if (ctx->has_g64) {
        Timed tm(ctx, MNC_KCLASS_NEWTON, timed);
        mnc::launch_ctl_reset(ctl, ctx->stream);
        {
            // lockstep rounds in batches until the active list is empty (the
            // count is read back between batches, so this path is not captured)
            if (!mnc::launch_newton_g64_init(a, t.nm, t.np2, ctx->stream))
                return ctx_fail(ctx, MNC_ERR_ARG, "no FP64 matrix-core Newton instance for this order");
            int lin = 0;
            for (int batch = 0;; ++batch) {
                if (batch > 4000) return ctx_fail(ctx, MNC_ERR_STATE, "closure solve did not finish");
                mnc::launch_newton_g64_rounds(a, t.nm, t.np2, lin, 4, ctx->num_cu, ctx->stream);
                int left = 0;
                MNC_HIP_CHECK(hipMemcpyAsync(&left, ctl + lin, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
                MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
                if (left == 0) break;
            }
        }
    } else if ((st = launch_timed(a, lp, true))) {
        return st;
    }
    MNC_HIP_CHECK(hipGetLastError());
    if (!check) return MNC_OK;
    return check_errors(ctx, ctl);
}

// The change-of-basis state as MomOptSolver::init leaves it
// (momopt_init.cpp:144-158): ones in the first nm entries of each cell's
// P2M (its first column) and isotropicAlpha as alphaP.
int cb_state_init(mnc_ctx *ctx) {
    const int nm = ctx->tab.nm;
    const size_t nc = ctx->cb_cells;
    std::vector<double> B(nc * nm * nm, 0.0), aP(nc * nm, 0.0);
    const double a0 = 2.0 * std::sqrt(M_PI) * std::log(0.5 / std::sqrt(M_PI));
    for (size_t c = 0; c < nc; ++c) {
        for (int k = 0; k < nm; ++k) B[c * nm * nm + k] = 1.0;
        aP[c * nm] = a0;
    }
    MNC_HIP_CHECK(hipMemcpy(ctx->d_cbB, B.data(), B.size() * sizeof(double), hipMemcpyHostToDevice));
    MNC_HIP_CHECK(hipMemcpy(ctx->d_cbaP, aP.data(), aP.size() * sizeof(double), hipMemcpyHostToDevice));
    return MNC_OK;
}

// optcb over every cell of the grid (solveOptimization with
// OPT_TYPE_CHANGE_BASIS, momopt_update.cpp:240-243): u = the moments, alphaM =
// the grid's alpha, the basis state kept on the device between solves.
// Allocates the change-of-basis state for nc cells and initialises it as
// momopt_init.cpp:144-158 (first use, or a larger grid; never inside a capture).
int cb_state_alloc(mnc_ctx *ctx, int nc) {
    if (size_t(nc) <= ctx->cb_cells) return MNC_OK;
    const int nm = ctx->tab.nm, nq = ctx->tab.nq;
    int st;
    ctx->cb_cells = size_t(nc);
    ctx->cb_blocks = std::min(nc, 16 * ctx->num_cu);
    if ((st = dalloc(ctx, &ctx->d_cbB, size_t(nc) * nm * nm)) || (st = dalloc(ctx, &ctx->d_cbaP, size_t(nc) * nm)) ||
        (st = dalloc(ctx, &ctx->d_cbws, size_t(ctx->cb_blocks) * nq * nm)) || (st = cb_state_init(ctx)))
        return st;
    return MNC_OK;
}

// The host-array change-of-basis entry's buffers.  The context keeps them from call to
// call (126 MB of workspace at M4, Q = 16, whose allocation and release took longer than
// the solve of 5,000 cells) up to a bound; beyond it (66,000 M4 cells) the solve outlasts
// the allocation, and they are given back with the call.  No captured step holds
// their addresses, so they do not end the captures.
constexpr size_t kCbKeepBytes = size_t(256) << 20;

void cb_batch_release(mnc_ctx *ctx) {
    if (ctx->d_cb_batch) (void)hipFree(ctx->d_cb_batch);
    if (ctx->d_cb_outs) (void)hipFree(ctx->d_cb_outs);
    ctx->d_cb_batch = nullptr;
    ctx->d_cb_outs = nullptr;
    ctx->cb_batch_cap = ctx->cb_outs_cap = 0;
}

int cb_batch_buffers(mnc_ctx *ctx, size_t doubles, size_t cells) {
    if (doubles <= ctx->cb_batch_cap && cells <= ctx->cb_outs_cap) return MNC_OK;
    cb_batch_release(ctx);
    if (hipMalloc((void **)&ctx->d_cb_batch, doubles * sizeof(double)) != hipSuccess ||
        hipMalloc((void **)&ctx->d_cb_outs, cells * sizeof(mnc_outs)) != hipSuccess) {
        (void)hipGetLastError();
        cb_batch_release(ctx);
        return ctx_fail(ctx, MNC_ERR_HIP, "hipMalloc failed");
    }
    ctx->cb_batch_cap = doubles;
    ctx->cb_outs_cap = cells;
    return MNC_OK;
}

int run_optcb_grid(mnc_ctx *ctx, int nc, const mnc_options *o, bool check) {
    const int nm = ctx->tab.nm, nq = ctx->tab.nq;
    int st;
    if ((st = cb_state_alloc(ctx, nc))) return st;
    (void)nq;
    mnc::CbArgs a{};
    a.ncells = nc;
    a.nm = nm;
    a.nq = nq;
    a.w = ctx->d_w;
    a.p = ctx->d_p;
    a.u = ctx->d_mom;
    a.P2M = ctx->d_cbB;
    a.alphaP = ctx->d_cbaP;
    a.alphaM = ctx->d_alpha;
    a.outs = nullptr;
    a.ws = ctx->d_cbws;
    a.max_iter = o->max_iter;
    a.ls_mode = o->line_search;
    a.tol = o->tol_rel;
    a.cond_h_max = o->cond_h_max;
    a.err = ctx->d_ctl + mnc::kErrWord;
    a.queue = ctx->d_ctl + mnc::kQueueWord;
    a.stats = ctx->d_stats;
    a.bfgs = o->opt_type == MNC_OPT_BFGS;
    a.max_bfgs_iter = o->max_bfgs_iter;
    a.cond_h_max_bfgs = o->cond_h_max_bfgs;
    {
        Timed tm(ctx, MNC_KCLASS_NEWTON);
        mnc::launch_ctl_reset(ctx->d_ctl, ctx->stream);
        if (mnc::launch_optcb(a, ctx->cb_blocks, ctx->num_cu, ctx->stream) < 0)
            return ctx_fail(ctx, MNC_ERR_ARG, "no change-of-basis kernel instance for this moment order");
    }
    MNC_HIP_CHECK(hipGetLastError());
    if (!check) return MNC_OK;
    return check_errors(ctx);
}

// Direction groups of the split flux: six, or on grids whose tiles are few as many
// as give three blocks per CU, up to 16 (each group's sums are one more pass
// through flux_sum_kernel).  Of 63 tiles (133 x 101 M4 cells) 45 + 7.5 and 40 + 9.8 us, of 16 (50 x 50
// M2) 22.3 + 5.3 and 12.6 + 6.6 us a stage, with six and by this rule.
int auto_flux_groups(const mnc_ctx *ctx) {
    const int T = mnc::kSplitTile;
    const int tiles = std::max(1, ((ctx->grid.num_cells_x + T - 1) / T) * ((ctx->grid.num_cells_y + T - 1) / T));
    const int half = ctx->tab.Q / 2, orbits = half * half;
    const int want = std::max(6, std::min(mnc::kMaxFluxGroups, 3 * ctx->num_cu / tiles));
    const int per = (orbits + want - 1) / want;          // no group without orbits
    return std::max(1, (orbits + per - 1) / per);
}
int flux_groups_of(const mnc_ctx *ctx) { return ctx->flux_groups > 0 ? ctx->flux_groups : auto_flux_groups(ctx); }

mnc::GridArgs grid_args(mnc_ctx *ctx) {
    mnc::GridArgs g{};
    const auto &t = ctx->tab;
    g.nx = ctx->grid.num_cells_x;
    g.ny = ctx->grid.num_cells_y;
    g.NX = g.nx + 4;
    g.NY = g.ny + 4;
    g.nm = t.nm;
    g.np2 = t.np2;
    g.nq = t.nq;
    g.half = t.Q / 2;
    g.dx = ctx->grid.dx;
    g.dy = ctx->grid.dy;
    g.theta = ctx->grid.theta;
    g.init_x = ctx->grid.init_x;
    g.init_y = ctx->grid.init_y;
    g.init_cond = ctx->grid.init_cond;
    g.w = ctx->d_w;
    g.p = ctx->d_p;
    g.xi = ctx->d_xi;
    g.eta = ctx->d_eta;
    g.moments = ctx->d_mom;
    g.alpha = ctx->d_alpha;
    g.moments_old = ctx->d_old;
    g.sigma_t = ctx->d_st;
    g.sigma_s = ctx->d_ss;
    g.flux = ctx->d_flux;
    g.ansatz = ctx->d_ansatz;
    g.fpart = ctx->d_fpart;
    g.groups = flux_groups_of(ctx);
    g.ppn = ctx->ppn ? 1 : 0;
    g.delta = ctx->grid.delta_ppn;
    g.tile_flag = ctx->d_tflag;
    g.tile_mode = 0;
    g.oz = ctx->d_foz;
    g.op = ctx->d_fop;
    g.odir = ctx->d_fodir;
    g.oidx = ctx->d_foidx;
    return g;
}

// Nodes the unfused flux's ansatz holds: whole tiles of 16 orbits above order 4.
int ansatz_nodes(const mnc_ctx *ctx) { return ctx->ftab.nt > 0 ? 64 * ctx->ftab.nt : ctx->tab.nq; }

// solveFlux (+ Euler stage when stage > 0) over all quadrature chunks.
int flux_stage(mnc_ctx *ctx, int stage, double dt) {
    mnc::GridArgs g = grid_args(ctx);
    if (ctx->flux_tile > 0) {
        Timed tm(ctx, MNC_KCLASS_FLUX);
        if (!mnc::launch_flux_fused(g, ctx->flux_tile, stage, dt, ctx->stream))
            return ctx_fail(ctx, MNC_ERR_ARG, "no flux kernel instance for this moment order");
        MNC_HIP_CHECK(hipGetLastError());
        return MNC_OK;
    }
    const int nq = ansatz_nodes(ctx), ch = ctx->ansatz_chunk;
    for (int q0 = 0; q0 < nq; q0 += ch) {
        const int nqc = std::min(ch, nq - q0);
        {
            Timed tm(ctx, MNC_KCLASS_FLUX);
            mnc::launch_ansatz(g, q0, nqc, ctx->stream);
        }
        {
            Timed tm(ctx, MNC_KCLASS_FLUX);
            if (!mnc::launch_flux_euler(g, q0, nqc, stage, dt, q0 == 0, q0 + nqc >= nq, ctx->stream))
                return ctx_fail(ctx, MNC_ERR_ARG, "no flux kernel instance for this moment order");
        }
    }
    MNC_HIP_CHECK(hipGetLastError());
    return MNC_OK;
}

}  // namespace

extern "C" {

int mnc_create(const mnc_setup *setup, mnc_ctx **out) {
    if (!out) return MNC_ERR_ARG;
    *out = nullptr;
    if (!setup) return MNC_ERR_ARG;
    if (setup->moment_type != 0 && setup->moment_type != 1) return MNC_ERR_ARG;   // Mn or PPn
    mnc_ctx *ctx = new mnc_ctx();
    ctx->device = setup->device;
    ctx->ppn = setup->moment_type == 1;
    int st = mnc::build_tables(setup->moment_order, setup->quad_order, setup->use_gaunt, ctx->tab);
    if (st != MNC_OK) { delete ctx; return st; }
    if (ctx->device < 0) {   // host-only context: tables, no device state
        *out = ctx;
        return MNC_OK;
    }
    hipError_t e = hipSetDevice(ctx->device);
    if (e != hipSuccess) { delete ctx; return MNC_ERR_HIP; }
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, ctx->device) == hipSuccess) ctx->num_cu = prop.multiProcessorCount;
    if (hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking) != hipSuccess) { delete ctx; return MNC_ERR_HIP; }
    if (hipStreamCreateWithFlags(&ctx->stream2, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&ctx->ev_fork, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&ctx->ev_join, hipEventDisableTiming) != hipSuccess) {
        mnc_destroy(ctx);
        return MNC_ERR_HIP;
    }
    // the no-allocation entry point's scratch array: its address on this
    // device, resolved once per device (the device is current)
    if (mnc::noalloc_scratch_address(ctx->device, &ctx->d_noalloc) != hipSuccess) {
        mnc_destroy(ctx);
        return MNC_ERR_HIP;
    }
    const auto &t = ctx->tab;
    auto up = [&](auto **dst, const auto &vec) -> int {
        using T = typename std::remove_reference<decltype(vec)>::type::value_type;
        size_t n = vec.size() ? vec.size() : 1;
        if (hipMalloc((void **)dst, n * sizeof(T)) != hipSuccess) return MNC_ERR_HIP;
        if (!vec.empty() && hipMemcpy(*dst, vec.data(), vec.size() * sizeof(T), hipMemcpyHostToDevice) != hipSuccess)
            return MNC_ERR_HIP;
        return MNC_OK;
    };
    if (up(&ctx->d_w, t.w) || up(&ctx->d_p, t.p) || up(&ctx->d_xi, t.xi) || up(&ctx->d_eta, t.eta) ||
        up(&ctx->d_gptr, t.gptr) || up(&ctx->d_gk, t.gk) || up(&ctx->d_gv, t.gv) ||
        hipMalloc((void **)&ctx->d_ctl, mnc::kCtlWords * sizeof(int)) != hipSuccess ||
        hipMemset(ctx->d_ctl, 0, mnc::kCtlWords * sizeof(int)) != hipSuccess ||
        hipMalloc((void **)&ctx->d_stats, mnc::kStatWords * sizeof(long long)) != hipSuccess ||
        hipMemset(ctx->d_stats, 0, mnc::kStatWords * sizeof(long long)) != hipSuccess) {
        mnc_destroy(ctx);
        return MNC_ERR_HIP;
    }
    if (t.nm <= 15) {
        if (mnc::build_orbit_tables(t, ctx->ppn, ctx->orb) != MNC_OK || up(&ctx->d_ot, ctx->orb.t) ||
            up(&ctx->d_opos, ctx->orb.pos) || up(&ctx->d_ogoff, ctx->orb.goff) || up(&ctx->d_ogk, ctx->orb.gk) ||
            up(&ctx->d_ogv, ctx->orb.gv)) {
            mnc_destroy(ctx);
            return MNC_ERR_HIP;
        }
    }
    // above n = 15 the fused flux's halo of alpha (20 x 20 cells does not fit,
    // 12 x 12 leaves two waves per CU) loses to the ansatz through HBM, whose two
    // passes go by orbits on the matrix cores (M8 96^2: 0.11 ms a stage)
    if (t.nm > 15) ctx->flux_tile = 0;
    if (t.N >= 5 && t.N <= 8 &&
        (mnc::build_flux_tables(t, ctx->ftab) != MNC_OK || up(&ctx->d_foz, ctx->ftab.z) || up(&ctx->d_fop, ctx->ftab.p) ||
         up(&ctx->d_fodir, ctx->ftab.dir) || up(&ctx->d_foidx, ctx->ftab.idx))) {
        mnc_destroy(ctx);
        return MNC_ERR_HIP;
    }
    if (!ctx->ppn && t.nm == 45 && mnc::build_g64_tables(setup->moment_order, setup->quad_order, ctx->g64) == MNC_OK) {
        if (up(&ctx->d_gz, ctx->g64.z) || up(&ctx->d_gh, ctx->g64.h) || up(&ctx->d_gmap, ctx->g64.map) ||
            up(&ctx->d_gidx, ctx->g64.idx) || up(&ctx->d_gpos, ctx->g64.pos)) {
            mnc_destroy(ctx);
            return MNC_ERR_HIP;
        }
        ctx->has_g64 = true;
    }
    if (!ctx->ppn && mnc::build_mix_tables(setup->moment_order, setup->quad_order, ctx->mix) == MNC_OK &&
        ctx->mix.nnt == mnc::mix_tiles(t.nm)) {
        if (up(&ctx->d_mz, ctx->mix.z) || up(&ctx->d_mg, ctx->mix.g) || up(&ctx->d_mh, ctx->mix.h) ||
            up(&ctx->d_mgptr, ctx->mix.gptr) || up(&ctx->d_mgk, ctx->mix.gk) || up(&ctx->d_mgv, ctx->mix.gv) ||
            (!ctx->mix.pv.empty() && up(&ctx->d_mpv, ctx->mix.pv))) {
            mnc_destroy(ctx);
            return MNC_ERR_HIP;
        }
        ctx->has_mix = true;
    }
    *out = ctx;
    return MNC_OK;
}

void mnc_destroy(mnc_ctx *ctx) {
    if (!ctx) return;
    if (ctx->device < 0) { delete ctx; return; }
    (void)hipSetDevice(ctx->device);
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    for (auto &g : ctx->graphs) drop_graph(g);
    for (auto &ev : ctx->events) { (void)hipEventDestroy(ev.a); (void)hipEventDestroy(ev.b); }
    void *ptrs[] = {ctx->d_w, ctx->d_p, ctx->d_xi, ctx->d_eta, ctx->d_gv, ctx->d_gptr, ctx->d_gk,
                    ctx->d_mz, ctx->d_mg, ctx->d_mh, ctx->d_mgptr, ctx->d_mgk, ctx->d_mgv, ctx->d_mpv, ctx->d_gz, ctx->d_gh, ctx->d_gmap, ctx->d_gidx, ctx->d_gpos,
                    ctx->d_ot, ctx->d_opos, ctx->d_ogoff, ctx->d_ogk, ctx->d_ogv,
                    ctx->d_foz, ctx->d_fop, ctx->d_fodir, ctx->d_foidx, ctx->d_cb_batch, ctx->d_cb_outs, ctx->d_mlp, ctx->d_mlp_scratch, ctx->d_mlp_loss, ctx->d_mlp_io, ctx->d_guess,
                    ctx->d_ctl, ctx->d_stats, ctx->d_std, ctx->d_sti, ctx->d_lists, ctx->d_mom, ctx->d_alpha, ctx->d_old,
                    ctx->d_st, ctx->d_ss, ctx->d_flux, ctx->d_ansatz, ctx->d_fpart, ctx->d_bu, ctx->d_ba, ctx->d_bo,
                    ctx->d_cbB, ctx->d_cbaP, ctx->d_cbws, ctx->d_tflag};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    if (ctx->ev_fork) (void)hipEventDestroy(ctx->ev_fork);
    if (ctx->ev_join) (void)hipEventDestroy(ctx->ev_join);
    if (ctx->stream2) (void)hipStreamDestroy(ctx->stream2);
    if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
    delete ctx;
}

int mnc_num_moments(const mnc_ctx *ctx) { return ctx ? ctx->tab.nm : 0; }
int mnc_num_quad(const mnc_ctx *ctx) { return ctx ? ctx->tab.nq : 0; }
int mnc_table_stride(const mnc_ctx *ctx) { return ctx ? ctx->tab.np2 : 0; }
int mnc_gaunt_nnz(const mnc_ctx *ctx) { return ctx ? int(ctx->tab.gv.size()) : 0; }

int mnc_get_tables(const mnc_ctx *ctx, double *w, double *p, double *xi, double *eta) {
    if (!ctx) return MNC_ERR_ARG;
    const auto &t = ctx->tab;
    if (w) std::memcpy(w, t.w.data(), t.w.size() * sizeof(double));
    if (p) std::memcpy(p, t.p.data(), t.p.size() * sizeof(double));
    if (xi) std::memcpy(xi, t.xi.data(), t.xi.size() * sizeof(double));
    if (eta) std::memcpy(eta, t.eta.data(), t.eta.size() * sizeof(double));
    return MNC_OK;
}

int mnc_get_gaunt(const mnc_ctx *ctx, int *ptr, int *k, double *v) {
    if (!ctx) return MNC_ERR_ARG;
    const auto &t = ctx->tab;
    if (!t.use_gaunt) return MNC_ERR_STATE;
    if (ptr) std::memcpy(ptr, t.gptr.data(), t.gptr.size() * sizeof(int));
    if (k) std::memcpy(k, t.gk.data(), t.gk.size() * sizeof(int));
    if (v) std::memcpy(v, t.gv.data(), t.gv.size() * sizeof(double));
    return MNC_OK;
}

int mnc_opt_batch(mnc_ctx *ctx, int ncells, double *u, double *alpha, const mnc_options *opt, mnc_outs *outs) {
    if (!ctx) return MNC_ERR_ARG;
    if (ncells < 0 || (ncells > 0 && (!u || !alpha))) return ctx_fail(ctx, MNC_ERR_ARG, "bad batch arguments");
    int st = check_opts(ctx, opt);
    if (st) return st;
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    return run_newton(ctx, ncells, u, alpha, opt, outs, nullptr, true);
}

int mnc_opt_batch_noalloc(mnc_ctx *ctx, int ncells, double *u, double *alpha, const mnc_options *opt,
                          mnc_outs *outs) {
    if (!ctx) return MNC_ERR_ARG;
    if (ncells < 0 || (ncells > 0 && (!u || !alpha))) return ctx_fail(ctx, MNC_ERR_ARG, "bad batch arguments");
    int st = check_opts(ctx, opt);
    if (st) return st;
    if (ncells > MNC_NOALLOC_MAX_CELLS)
        return ctx_fail(ctx, MNC_ERR_ARG, "mnc_opt_batch_noalloc takes at most MNC_NOALLOC_MAX_CELLS (16384) cells");
    if (ctx->has_g64 || ctx->tab.nm > 15)
        return ctx_fail(ctx, MNC_ERR_ARG, "mnc_opt_batch_noalloc serves moment orders up to 4");
    mnc::NoAllocState na;
    if (!ctx->d_noalloc || !mnc::noalloc_layout(ctx->tab.nm, ctx->tab.np2, ctx->d_noalloc, na))
        return ctx_fail(ctx, MNC_ERR_ARG, "this order's Newton state does not fit the no-allocation scratch");
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    return run_newton(ctx, ncells, u, alpha, opt, outs, nullptr, true, &na);
}

int mnc_opt_batch_host(mnc_ctx *ctx, int ncells, double *u, double *alpha, const mnc_options *opt, mnc_outs *outs) {
    if (!ctx) return MNC_ERR_ARG;
    if (ncells < 0 || (ncells > 0 && (!u || !alpha))) return ctx_fail(ctx, MNC_ERR_ARG, "bad batch arguments");
    int st = check_opts(ctx, opt);
    if (st) return st;
    if (ncells == 0) return MNC_OK;
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    const size_t n = size_t(ncells) * ctx->tab.nm;
    if (size_t(ncells) > ctx->batch_cap) {
        if ((st = dalloc(ctx, &ctx->d_bu, n)) || (st = dalloc(ctx, &ctx->d_ba, n)) ||
            (st = dalloc(ctx, &ctx->d_bo, size_t(ncells))))
            return st;
        ctx->batch_cap = ncells;
    }
    MNC_HIP_CHECK(hipMemcpyAsync(ctx->d_bu, u, n * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    MNC_HIP_CHECK(hipMemcpyAsync(ctx->d_ba, alpha, n * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    st = run_newton(ctx, ncells, ctx->d_bu, ctx->d_ba, opt, outs ? ctx->d_bo : nullptr, nullptr, true);
    // copy back whatever the kernel produced, also on MNC_ERR_U0 / MNC_ERR_MAXREG
    if (st != MNC_OK && st != MNC_ERR_U0 && st != MNC_ERR_MAXREG) return st;
    MNC_HIP_CHECK(hipMemcpyAsync(u, ctx->d_bu, n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    MNC_HIP_CHECK(hipMemcpyAsync(alpha, ctx->d_ba, n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    if (outs)
        MNC_HIP_CHECK(hipMemcpyAsync(outs, ctx->d_bo, size_t(ncells) * sizeof(mnc_outs), hipMemcpyDeviceToHost,
                                     ctx->stream));
    MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    return st;
}

int mnc_optcb_batch_host(mnc_ctx *ctx, int ncells, double *u, double *P2M, double *alphaP, double *alphaM,
                         const mnc_options *opt, mnc_outs *outs) {
    if (!ctx) return MNC_ERR_ARG;
    if (ncells < 0 || (ncells > 0 && (!u || !P2M || !alphaP || !alphaM)))
        return ctx_fail(ctx, MNC_ERR_ARG, "bad optcb batch arguments");
    int st = check_opts(ctx, opt);
    if (st) return st;
    if (ctx->ppn) return ctx_fail(ctx, MNC_ERR_ARG, "the change-of-basis optimiser runs Mn contexts only");
    if (ctx->tab.use_gaunt || ctx->tab.np2 != ctx->tab.nm)
        return ctx_fail(ctx, MNC_ERR_ARG, "the change-of-basis optimiser needs the direct Hessian (use_gaunt 0)");
    if (opt->precision != MNC_PREC_FP64 || opt->warm_start != MNC_WARM_PREVIOUS)
        return ctx_fail(ctx, MNC_ERR_ARG, "the change-of-basis optimiser is FP64 from the cell's own alphaP");
    if (ncells == 0) return MNC_OK;
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    const int nm = ctx->tab.nm, nq = ctx->tab.nq;
    const int blocks = std::min(ncells, 16 * ctx->num_cu);
    const size_t nv = size_t(ncells) * nm, nb = size_t(ncells) * nm * nm, nws = size_t(blocks) * nq * nm;
    const size_t nd = 3 * nv + nb + nws;
    if ((st = cb_batch_buffers(ctx, nd, size_t(ncells)))) return st;
    double *d = ctx->d_cb_batch;
    mnc_outs *d_outs = ctx->d_cb_outs;
    double *d_u = d, *d_aP = d + nv, *d_aM = d + 2 * nv, *d_B = d + 3 * nv, *d_ws = d_B + nb;
    mnc::CbArgs a{};
    a.ncells = ncells;
    a.nm = nm;
    a.nq = nq;
    a.w = ctx->d_w;
    a.p = ctx->d_p;
    a.u = d_u;
    a.P2M = d_B;
    a.alphaP = d_aP;
    a.alphaM = d_aM;
    a.outs = d_outs;
    a.ws = d_ws;
    a.stats = ctx->d_stats;
    a.max_iter = opt->max_iter;
    a.ls_mode = opt->line_search;
    a.tol = opt->tol_rel;
    a.cond_h_max = opt->cond_h_max;
    a.err = ctx->d_ctl + mnc::kErrWord;
    a.queue = ctx->d_ctl + mnc::kQueueWord;
    a.bfgs = opt->opt_type == MNC_OPT_BFGS;
    a.max_bfgs_iter = opt->max_bfgs_iter;
    a.cond_h_max_bfgs = opt->cond_h_max_bfgs;
    auto run = [&]() -> int {
        MNC_HIP_CHECK(hipMemcpyAsync(d_u, u, nv * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
        MNC_HIP_CHECK(hipMemcpyAsync(d_aP, alphaP, nv * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
        MNC_HIP_CHECK(hipMemcpyAsync(d_aM, alphaM, nv * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
        MNC_HIP_CHECK(hipMemcpyAsync(d_B, P2M, nb * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
        mnc::launch_ctl_reset(ctx->d_ctl, ctx->stream);
        {
            Timed tm(ctx, MNC_KCLASS_NEWTON);
            if (mnc::launch_optcb(a, blocks, ctx->num_cu, ctx->stream) < 0)
                return ctx_fail(ctx, MNC_ERR_ARG, "no change-of-basis kernel instance for this moment order");
        }
        MNC_HIP_CHECK(hipGetLastError());
        int s2 = check_errors(ctx);
        if (s2 != MNC_OK && s2 != MNC_ERR_U0 && s2 != MNC_ERR_MAXREG) return s2;
        MNC_HIP_CHECK(hipMemcpyAsync(u, d_u, nv * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
        MNC_HIP_CHECK(hipMemcpyAsync(alphaP, d_aP, nv * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
        MNC_HIP_CHECK(hipMemcpyAsync(alphaM, d_aM, nv * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
        MNC_HIP_CHECK(hipMemcpyAsync(P2M, d_B, nb * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
        if (outs)
            MNC_HIP_CHECK(hipMemcpyAsync(outs, d_outs, size_t(ncells) * sizeof(mnc_outs), hipMemcpyDeviceToHost,
                                         ctx->stream));
        MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
        return s2;
    };
    st = run();
    if (nd * sizeof(double) > kCbKeepBytes) cb_batch_release(ctx);
    return st;
}

int mnc_batch_set(mnc_ctx *ctx, int ncells, const double *u, const double *alpha) {
    if (!ctx) return MNC_ERR_ARG;
    if (ctx->device < 0) return ctx_fail(ctx, MNC_ERR_STATE, "host-only context (device < 0)");
    if (ncells < 1 || !u || !alpha) return ctx_fail(ctx, MNC_ERR_ARG, "bad batch arguments");
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    const size_t n = size_t(ncells) * ctx->tab.nm;
    int st;
    if (size_t(ncells) > ctx->batch_cap) {
        if ((st = dalloc(ctx, &ctx->d_bu, n)) || (st = dalloc(ctx, &ctx->d_ba, n)) ||
            (st = dalloc(ctx, &ctx->d_bo, size_t(ncells))))
            return st;
        ctx->batch_cap = ncells;
    }
    MNC_HIP_CHECK(hipMemcpyAsync(ctx->d_bu, u, n * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    MNC_HIP_CHECK(hipMemcpyAsync(ctx->d_ba, alpha, n * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    ctx->batch_n = ncells;
    return MNC_OK;
}

int mnc_batch_solve(mnc_ctx *ctx, const mnc_options *opt) {
    if (!ctx) return MNC_ERR_ARG;
    int st = check_opts(ctx, opt);
    if (st) return st;
    if (ctx->batch_n < 1) return ctx_fail(ctx, MNC_ERR_STATE, "no staged batch (mnc_batch_set first)");
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    return run_newton(ctx, ctx->batch_n, ctx->d_bu, ctx->d_ba, opt, ctx->d_bo, nullptr, true);
}

int mnc_batch_get(mnc_ctx *ctx, double *u, double *alpha, mnc_outs *outs) {
    if (!ctx) return MNC_ERR_ARG;
    if (ctx->batch_n < 1) return ctx_fail(ctx, MNC_ERR_STATE, "no staged batch (mnc_batch_set first)");
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    const size_t n = size_t(ctx->batch_n) * ctx->tab.nm;
    if (u) MNC_HIP_CHECK(hipMemcpyAsync(u, ctx->d_bu, n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    if (alpha) MNC_HIP_CHECK(hipMemcpyAsync(alpha, ctx->d_ba, n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    if (outs)
        MNC_HIP_CHECK(hipMemcpyAsync(outs, ctx->d_bo, size_t(ctx->batch_n) * sizeof(mnc_outs), hipMemcpyDeviceToHost,
                                     ctx->stream));
    MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    return MNC_OK;
}

int mnc_grid_create(mnc_ctx *ctx, const mnc_grid_desc *grid, const double *moments, const double *alpha,
                    const double *sigma_t, const double *sigma_s) {
    if (!ctx || !grid || !moments || !alpha || !sigma_t || !sigma_s) return MNC_ERR_ARG;
    if (ctx->device < 0) return ctx_fail(ctx, MNC_ERR_STATE, "host-only context (device < 0)");
    if (grid->num_cells_x < 2 || grid->num_cells_y < 2)
        return ctx_fail(ctx, MNC_ERR_ARG, "grid needs at least 2x2 interior cells");
    if (!(grid->dx > 0.0) || !(grid->dy > 0.0)) return ctx_fail(ctx, MNC_ERR_ARG, "dx, dy must be > 0");
    if (ctx->ppn && !(grid->delta_ppn > 0.0)) return ctx_fail(ctx, MNC_ERR_ARG, "PPn grid needs delta_ppn > 0");
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    ctx->grid = *grid;
    const size_t nc = size_t(grid->num_cells_x + 4) * (grid->num_cells_y + 4);
    const size_t n = nc * ctx->tab.nm;
    int st;
    if ((st = dalloc(ctx, &ctx->d_mom, n)) || (st = dalloc(ctx, &ctx->d_alpha, n)) ||
        (st = dalloc(ctx, &ctx->d_old, n)) || (st = dalloc(ctx, &ctx->d_flux, n)) ||
        (st = dalloc(ctx, &ctx->d_st, nc)) || (st = dalloc(ctx, &ctx->d_ss, nc)) ||
        (st = dalloc(ctx, &ctx->d_fpart, size_t(std::max(mnc::kTuneFluxGroups, auto_flux_groups(ctx))) * grid->num_cells_x *
                                             grid->num_cells_y * ctx->tab.nm)) ||
        (st = dalloc(ctx, &ctx->d_tflag, size_t((grid->num_cells_x + mnc::kSplitTile - 1) / mnc::kSplitTile) *
                                             ((grid->num_cells_y + mnc::kSplitTile - 1) / mnc::kSplitTile))))
        return st;
    // ansatz buffer: all q at once unless that exceeds 8 GiB
    const size_t max_elems = (size_t(8) << 30) / sizeof(double);
    int ch = ansatz_nodes(ctx);
    while (ch > 1 && size_t(ch) * nc > max_elems) ch = (ch + 1) / 2;
    if (ctx->ftab.nt > 0) ch = (ch + 63) / 64 * 64;
    ctx->ansatz_chunk = ch;
    if ((st = dalloc(ctx, &ctx->d_ansatz, size_t(ch) * nc))) return st;
    MNC_HIP_CHECK(hipMemcpy(ctx->d_mom, moments, n * sizeof(double), hipMemcpyHostToDevice));
    MNC_HIP_CHECK(hipMemcpy(ctx->d_alpha, alpha, n * sizeof(double), hipMemcpyHostToDevice));
    MNC_HIP_CHECK(hipMemcpy(ctx->d_st, sigma_t, nc * sizeof(double), hipMemcpyHostToDevice));
    MNC_HIP_CHECK(hipMemcpy(ctx->d_ss, sigma_s, nc * sizeof(double), hipMemcpyHostToDevice));
    MNC_HIP_CHECK(hipMemset(ctx->d_flux, 0, n * sizeof(double)));
    MNC_HIP_CHECK(hipMemset(ctx->d_old, 0, n * sizeof(double)));
    ctx->has_grid = true;
    if (ctx->d_cbB) return cb_state_init(ctx);   // a new grid starts the change-of-basis state afresh
    return MNC_OK;
}

int mnc_grid_get_basis(mnc_ctx *ctx, double *P2M, double *alphaP) {
    if (!ctx) return MNC_ERR_ARG;
    if (!ctx->has_grid) return ctx_fail(ctx, MNC_ERR_STATE, "no grid");
    const int nm = ctx->tab.nm;
    const size_t nc = size_t(ctx->grid.num_cells_x + 4) * (ctx->grid.num_cells_y + 4);
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    int st;
    if ((st = cb_state_alloc(ctx, int(nc)))) return st;   // before any change-of-basis solve: the initial state
    if (P2M)
        MNC_HIP_CHECK(hipMemcpyAsync(P2M, ctx->d_cbB, nc * nm * nm * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    if (alphaP)
        MNC_HIP_CHECK(hipMemcpyAsync(alphaP, ctx->d_cbaP, nc * nm * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    return MNC_OK;
}

int mnc_grid_set_basis(mnc_ctx *ctx, const double *P2M, const double *alphaP) {
    if (!ctx) return MNC_ERR_ARG;
    if (!ctx->has_grid) return ctx_fail(ctx, MNC_ERR_STATE, "no grid");
    if (!P2M || !alphaP) return ctx_fail(ctx, MNC_ERR_ARG, "mnc_grid_set_basis needs both P2M and alphaP");
    const int nm = ctx->tab.nm;
    const size_t nc = size_t(ctx->grid.num_cells_x + 4) * (ctx->grid.num_cells_y + 4);
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    int st;
    if ((st = cb_state_alloc(ctx, int(nc)))) return st;
    MNC_HIP_CHECK(hipMemcpyAsync(ctx->d_cbB, P2M, nc * nm * nm * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    MNC_HIP_CHECK(hipMemcpyAsync(ctx->d_cbaP, alphaP, nc * nm * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    return MNC_OK;
}

int mnc_grid_get(mnc_ctx *ctx, double *moments, double *alpha) {
    if (!ctx) return MNC_ERR_ARG;
    if (!ctx->has_grid) return ctx_fail(ctx, MNC_ERR_STATE, "no grid");
    const size_t n = size_t(ctx->grid.num_cells_x + 4) * (ctx->grid.num_cells_y + 4) * ctx->tab.nm;
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    if (moments) MNC_HIP_CHECK(hipMemcpyAsync(moments, ctx->d_mom, n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    if (alpha) MNC_HIP_CHECK(hipMemcpyAsync(alpha, ctx->d_alpha, n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    return MNC_OK;
}

int mnc_grid_set(mnc_ctx *ctx, const double *moments, const double *alpha) {
    if (!ctx) return MNC_ERR_ARG;
    if (!ctx->has_grid) return ctx_fail(ctx, MNC_ERR_STATE, "no grid");
    const size_t n = size_t(ctx->grid.num_cells_x + 4) * (ctx->grid.num_cells_y + 4) * ctx->tab.nm;
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    if (moments) MNC_HIP_CHECK(hipMemcpyAsync(ctx->d_mom, moments, n * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    if (alpha) MNC_HIP_CHECK(hipMemcpyAsync(ctx->d_alpha, alpha, n * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    if (ctx->d_cbB) return cb_state_init(ctx);        // a new state starts the change-of-basis state afresh
    return MNC_OK;
}

int mnc_ghost_fill(mnc_ctx *ctx) {
    if (!ctx) return MNC_ERR_ARG;
    if (!ctx->has_grid) return ctx_fail(ctx, MNC_ERR_STATE, "no grid");
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    {
        Timed tm(ctx, MNC_KCLASS_OTHER);
        mnc::launch_ghost_fill(grid_args(ctx), ctx->stream);
    }
    MNC_HIP_CHECK(hipGetLastError());
    return MNC_OK;
}

int mnc_solve_grid(mnc_ctx *ctx, const mnc_options *opt) {
    if (!ctx) return MNC_ERR_ARG;
    if (!ctx->has_grid) return ctx_fail(ctx, MNC_ERR_STATE, "no grid");
    int st = check_opts(ctx, opt);
    if (st) return st;
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    const int nc = (ctx->grid.num_cells_x + 4) * (ctx->grid.num_cells_y + 4);
    if (opt->opt_type != MNC_OPT_NEWTON) return run_optcb_grid(ctx, nc, opt, true);
    return run_newton(ctx, nc, ctx->d_mom, ctx->d_alpha, opt, nullptr, nullptr, true);
}

int mnc_flux(mnc_ctx *ctx, double *flux_host) {
    if (!ctx) return MNC_ERR_ARG;
    if (!ctx->has_grid) return ctx_fail(ctx, MNC_ERR_STATE, "no grid");
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    const size_t n = size_t(ctx->grid.num_cells_x + 4) * (ctx->grid.num_cells_y + 4) * ctx->tab.nm;
    MNC_HIP_CHECK(hipMemsetAsync(ctx->d_flux, 0, n * sizeof(double), ctx->stream));
    int st = flux_stage(ctx, 0, 0.0);
    if (st) return st;
    if (flux_host)
        MNC_HIP_CHECK(hipMemcpyAsync(flux_host, ctx->d_flux, n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    return MNC_OK;
}

}  // extern "C"

namespace {

// The tail of a grid solve and the stage's flux (flux_tile 3) overlapped:
// tiles whose stencil region holds no cell left for the tail take their flux
// on the second stream while the tail runs; the flagged tiles follow the tail.
// The two share no cell: the tail writes the alpha and moments of its own
// cells, a clear tile's flux reads alpha of cells the rounds finished and
// writes the moments of its own interior cells.
int overlap_tail_flux(mnc_ctx *ctx, int nc, int stage, double dt) {
    const size_t cap = ctx->state_cap;
    const int *lists = ctx->d_lists, *ctl = ctx->d_ctl;
    const int w0 = mnc::newton_list_word(ctx->tail_lin), w1 = mnc::newton_list_word(ctx->tail_flin);
    mnc::launch_tile_flags(lists + size_t(ctx->tail_lin) * cap, ctl + w0, lists + size_t(ctx->tail_flin) * cap,
                           ctl + w1, nc, ctx->grid.num_cells_x, ctx->grid.num_cells_y, ctx->d_tflag, ctx->stream);
    MNC_HIP_CHECK(hipEventRecord(ctx->ev_fork, ctx->stream));
    MNC_HIP_CHECK(hipStreamWaitEvent(ctx->stream2, ctx->ev_fork, 0));
    const auto &t = ctx->tab;
    const bool gaunt = t.use_gaunt != 0;
    const bool ok = ctx->tail_mixed ? mnc::launch_newton_mixed(ctx->tail_a, t.nm, t.np2, gaunt, ctx->tail_lp, ctx->stream)
                                    : mnc::launch_newton_fp64(ctx->tail_a, t.nm, t.np2, gaunt, ctx->tail_lp, ctx->stream);
    if (!ok) return ctx_fail(ctx, MNC_ERR_ARG, "no Newton tail instance for this moment order");
    mnc::GridArgs g = grid_args(ctx);
    g.tile_mode = 1;
    if (!mnc::launch_flux_fused(g, 3, stage, dt, ctx->stream2))
        return ctx_fail(ctx, MNC_ERR_ARG, "no flux kernel instance for this moment order");
    MNC_HIP_CHECK(hipEventRecord(ctx->ev_join, ctx->stream2));
    MNC_HIP_CHECK(hipStreamWaitEvent(ctx->stream, ctx->ev_join, 0));
    g.tile_mode = 2;
    if (!mnc::launch_flux_fused(g, 3, stage, dt, ctx->stream))
        return ctx_fail(ctx, MNC_ERR_ARG, "no flux kernel instance for this moment order");
    MNC_HIP_CHECK(hipGetLastError());
    return MNC_OK;
}

// One Heun step (MomOptSolver::update, momopt_update.cpp:283-382) enqueued on
// the context's stream with no host synchronisation and no allocation once the
// buffers exist, so that it can be captured.
int enqueue_step(mnc_ctx *ctx, double dt, const mnc_options *opt) {
    const int nc = (ctx->grid.num_cells_x + 4) * (ctx->grid.num_cells_y + 4);
    const size_t n = size_t(nc) * ctx->tab.nm;
    int st;
    // momentsOld <- moments before the first solve (momopt_update.cpp:299-308)
    MNC_HIP_CHECK(hipMemcpyAsync(ctx->d_old, ctx->d_mom, n * sizeof(double), hipMemcpyDeviceToDevice, ctx->stream));
    for (int stage = 1; stage <= 2; ++stage) {
        if ((st = mnc_ghost_fill(ctx))) return st;
        if (opt->opt_type != MNC_OPT_NEWTON) {
            if ((st = run_optcb_grid(ctx, nc, opt, false))) return st;
        } else {
            // flux_overlap: the tail is launched here, beside the flux of the
            // tiles whose stencil region it does not touch (eager timing
            // measures one stream, so it runs the plain sequence)
            ctx->defer_tail = ctx->flux_overlap && ctx->flux_tile == 3 && !ctx->timing && !ctx->has_g64 &&
                              ctx->tab.nm <= 15;
            ctx->tail_saved = false;
            st = run_newton(ctx, nc, ctx->d_mom, ctx->d_alpha, opt, nullptr, nullptr, false);
            ctx->defer_tail = false;
            if (st) return st;
            if (ctx->tail_saved) {
                ctx->tail_saved = false;
                if ((st = overlap_tail_flux(ctx, nc, stage, dt))) return st;
                continue;
            }
        }
        // errors of the first stage are seen at the end of the step (the
        // kernels flag them in device memory; the state is left as computed)
        if ((st = flux_stage(ctx, stage, dt))) return st;
    }
    return MNC_OK;
}

bool same_opts(const mnc_options &a, const mnc_options &b) {
    return a.max_iter == b.max_iter && a.tol_rel == b.tol_rel && a.cond_h_max == b.cond_h_max &&
           a.precision == b.precision && a.warm_start == b.warm_start && a.line_search == b.line_search &&
           a.delta_ppn == b.delta_ppn && a.opt_type == b.opt_type && a.max_bfgs_iter == b.max_bfgs_iter &&
           a.cond_h_max_bfgs == b.cond_h_max_bfgs && a.tol_gamma == b.tol_gamma;
}

// Captures enqueue_step into g.exec.  On any capture error the context falls
// back to eager launches of the same kernels for the rest of its life.
int capture_step(mnc_ctx *ctx, mnc_ctx::StepGraph &g, double dt, const mnc_options *opt) {
    hipGraph_t graph = nullptr;
    hipError_t e = hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal);
    int st = (e == hipSuccess) ? enqueue_step(ctx, dt, opt) : MNC_ERR_HIP;
    hipError_t e2 = (e == hipSuccess) ? hipStreamEndCapture(ctx->stream, &graph) : e;
    if (st == MNC_OK && e2 == hipSuccess && graph)
        e2 = hipGraphInstantiate(&g.exec, graph, nullptr, nullptr, 0);
    if (graph) (void)hipGraphDestroy(graph);
    (void)hipGetLastError();
    if (st != MNC_OK || e2 != hipSuccess || !g.exec) {
        drop_graph(g);
        ctx->use_graph = 0;
        return MNC_ERR_HIP;
    }
    return MNC_OK;
}

}  // namespace

extern "C" {

int mnc_update(mnc_ctx *ctx, double dt, const mnc_options *opt) {
    if (!ctx) return MNC_ERR_ARG;
    if (!ctx->has_grid) return ctx_fail(ctx, MNC_ERR_STATE, "no grid");
    int st = check_opts(ctx, opt);
    if (st) return st;
    if (ctx->ppn && opt->delta_ppn != ctx->grid.delta_ppn)   // one deck value in the reference
        return ctx_fail(ctx, MNC_ERR_ARG, "options.delta_ppn differs from the grid's delta_ppn");
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    if (ctx->use_graph && !ctx->timing && !ctx->has_g64) {   // timing needs eager launches; M8 syncs per batch
        mnc_ctx::StepGraph *g = nullptr;
        for (auto &c : ctx->graphs)
            if (c.epoch == ctx->epoch && c.dt == dt && same_opts(c.o, *opt)) g = &c;
        if (g && !g->exec && g->eager_runs >= 1 && capture_step(ctx, *g, dt, opt) != MNC_OK) g = nullptr;
        if (g && g->exec) {
            MNC_HIP_CHECK(hipGraphLaunch(g->exec, ctx->stream));
            return check_errors(ctx);
        }
        if (ctx->use_graph && !g) {   // first step with this key: eager, then captured from the next one
            g = &ctx->graphs[ctx->graph_next];
            ctx->graph_next = (ctx->graph_next + 1) % 4;
            drop_graph(*g);
            if ((st = enqueue_step(ctx, dt, opt))) return st;
            st = check_errors(ctx);
            g->epoch = ctx->epoch;     // after the step's own allocations
            g->dt = dt;
            g->o = *opt;
            g->eager_runs = 1;
            return st;
        }
    }
    if ((st = enqueue_step(ctx, dt, opt))) return st;
    return check_errors(ctx);
}

int mnc_get_stats(mnc_ctx *ctx, mnc_stats *st) {
    if (!ctx || !st) return MNC_ERR_ARG;
    if (ctx->device < 0) return ctx_fail(ctx, MNC_ERR_STATE, "host-only context (device < 0)");
    long long h[mnc::kStatWords];
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    MNC_HIP_CHECK(hipMemcpyAsync(h, ctx->d_stats, sizeof h, hipMemcpyDeviceToHost, ctx->stream));
    MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    st->max_iter = int(h[0]);
    st->iter_sum = h[1];
    st->num_dual_solves = h[2];
    for (int r = 0; r < 5; ++r) st->hist_reg[r] = h[3 + r];
    st->trial_sum = h[8];
    for (int r = 0; r < 3; ++r) st->warm_pick[r] = h[9 + r];
    st->mixed_deferred = h[12];
    st->tail_cells = h[13];
    st->tail_iter_sum = h[14];
    st->tail_trial_sum = h[15];
    st->warm_fallback = h[16];
    return MNC_OK;
}

int mnc_reset_stats(mnc_ctx *ctx) {
    if (!ctx) return MNC_ERR_ARG;
    if (ctx->device < 0) return ctx_fail(ctx, MNC_ERR_STATE, "host-only context (device < 0)");
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    MNC_HIP_CHECK(hipMemsetAsync(ctx->d_stats, 0, mnc::kStatWords * sizeof(long long), ctx->stream));
    MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    return MNC_OK;
}

int mnc_sync(mnc_ctx *ctx) {
    if (!ctx) return MNC_ERR_ARG;
    if (ctx->device < 0) return ctx_fail(ctx, MNC_ERR_STATE, "host-only context (device < 0)");
    MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    return MNC_OK;
}

int mnc_timing_enable(mnc_ctx *ctx, int on) {
    if (!ctx) return MNC_ERR_ARG;
    if (ctx->device < 0) return ctx_fail(ctx, MNC_ERR_STATE, "host-only context (device < 0)");
    MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    for (auto &ev : ctx->events) { (void)hipEventDestroy(ev.a); (void)hipEventDestroy(ev.b); }
    ctx->events.clear();
    for (int k = 0; k < MNC_NUM_KCLASS; ++k) { ctx->t_launch[k] = 0; ctx->t_ms[k] = 0.0; }
    ctx->timing = on != 0;
    return MNC_OK;
}

int mnc_timing_get(mnc_ctx *ctx, int kclass, long long *launches, double *ms) {
    if (!ctx || kclass < 0 || kclass >= MNC_NUM_KCLASS) return MNC_ERR_ARG;
    if (ctx->device < 0) return ctx_fail(ctx, MNC_ERR_STATE, "host-only context (device < 0)");
    MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    for (auto &ev : ctx->events) {
        float el = 0.f;
        MNC_HIP_CHECK(hipEventElapsedTime(&el, ev.a, ev.b));
        ctx->t_launch[ev.kc] += 1;
        ctx->t_ms[ev.kc] += el;
        (void)hipEventDestroy(ev.a);
        (void)hipEventDestroy(ev.b);
    }
    ctx->events.clear();
    if (launches) *launches = ctx->t_launch[kclass];
    if (ms) *ms = ctx->t_ms[kclass];
    return MNC_OK;
}

int mnc_tune(mnc_ctx *ctx, const char *key, int value) {
    if (!ctx || !key) return MNC_ERR_ARG;
    ++ctx->epoch;
    if (std::strcmp(key, "graph") == 0) {
        if (value < 0 || value > 1) return ctx_fail(ctx, MNC_ERR_ARG, "graph must be 0 or 1");
        ctx->use_graph = value;
        return MNC_OK;
    }
    if (std::strcmp(key, "rounds") == 0) {
        if (value < -1 || value > 512) return ctx_fail(ctx, MNC_ERR_ARG, "rounds out of range");
        ctx->rounds = value;
        return MNC_OK;
    }
    if (std::strcmp(key, "tail_blocks") == 0) {
        if (value < 1 || value > 65536) return ctx_fail(ctx, MNC_ERR_ARG, "tail_blocks out of range");
        ctx->tail_blocks = value;
        return MNC_OK;
    }
    if (std::strcmp(key, "tail_mode") == 0) {
        if (value < 0 || value > 3) return ctx_fail(ctx, MNC_ERR_ARG, "tail_mode out of range");
        ctx->tail_mode = value;
        return MNC_OK;
    }
    if (std::strcmp(key, "mix_cond_log10") == 0) {
        if (value < 0 || value > 10) return ctx_fail(ctx, MNC_ERR_ARG, "mix_cond_log10 out of range");
        ctx->mix_cond_log10 = value;
        return MNC_OK;
    }
    if (std::strcmp(key, "mix_defer") == 0) {
        if (value < 0 || value > 1) return ctx_fail(ctx, MNC_ERR_ARG, "mix_defer is 0 or 1");
        ctx->mix_defer = value;
        return MNC_OK;
    }
    if (std::strcmp(key, "mix_split") == 0) {
        if (value < 2 || value > 3) return ctx_fail(ctx, MNC_ERR_ARG, "mix_split is 2 or 3");
        ctx->mix_split = value;
        return MNC_OK;
    }
    if (std::strcmp(key, "mix_blocks") == 0) {
        if (value < 1 || value > 65536) return ctx_fail(ctx, MNC_ERR_ARG, "mix_blocks out of range");
        ctx->mix_blocks = value;
        return MNC_OK;
    }
    if (std::strcmp(key, "flux_tile") == 0) {
        if (value < 0 || value > 3) return ctx_fail(ctx, MNC_ERR_ARG, "flux_tile must be 0, 1, 2 or 3");
        ctx->flux_tile = value;
        return MNC_OK;
    }
    if (std::strcmp(key, "flux_groups") == 0) {
        if (value < 0 || value > mnc::kTuneFluxGroups) return ctx_fail(ctx, MNC_ERR_ARG, "flux_groups must be 0 to 8");
        ctx->flux_groups = value;
        return MNC_OK;
    }
    if (std::strcmp(key, "flux_overlap") == 0) {
        if (value != 0 && value != 1) return ctx_fail(ctx, MNC_ERR_ARG, "flux_overlap is 0 or 1");
        ctx->flux_overlap = value;
        ++ctx->epoch;
        return MNC_OK;
    }
    if (std::strcmp(key, "learned_fused") == 0) {
        if (value != 0 && value != 1) return ctx_fail(ctx, MNC_ERR_ARG, "learned_fused is 0 or 1");
        ctx->learned_fused = value;
        ++ctx->epoch;
        return MNC_OK;
    }
    if (std::strcmp(key, "learned_fallback_iters") == 0) {
        if (value < 0 || value > 100000) return ctx_fail(ctx, MNC_ERR_ARG, "learned_fallback_iters out of range");
        ctx->learned_fallback_iters = value;
        ++ctx->epoch;
        return MNC_OK;
    }
    if (std::strcmp(key, "learned_gate_log10") == 0) {
        if (value < -16 || value > kGateOff) return ctx_fail(ctx, MNC_ERR_ARG, "learned_gate_log10 out of range");
        ctx->learned_gate_log10 = value;
        return MNC_OK;
    }
    return ctx_fail(ctx, MNC_ERR_ARG, "unknown tuning key");
}

int mnc_get_tune(const mnc_ctx *ctx, const char *key, int *value) {
    if (!ctx || !key || !value) return MNC_ERR_ARG;
    if (std::strcmp(key, "rounds") == 0) { *value = ctx->rounds; return MNC_OK; }
    if (std::strcmp(key, "tail_mode") == 0) { *value = ctx->tail_mode; return MNC_OK; }
    if (std::strcmp(key, "mix_cond_log10") == 0) { *value = ctx->mix_cond_log10; return MNC_OK; }
    if (std::strcmp(key, "mix_defer") == 0) { *value = ctx->mix_defer; return MNC_OK; }
    if (std::strcmp(key, "mix_split") == 0) { *value = ctx->mix_split; return MNC_OK; }
    if (std::strcmp(key, "mix_blocks") == 0) {
        *value = ctx->mix_blocks > 0 ? ctx->mix_blocks : ctx->num_cu;
        return MNC_OK;
    }
    if (std::strcmp(key, "has_mixed") == 0) { *value = ctx->has_mix ? 1 : 0; return MNC_OK; }
    if (std::strcmp(key, "graph") == 0) { *value = ctx->use_graph; return MNC_OK; }
    if (std::strcmp(key, "flux_tile") == 0) { *value = ctx->flux_tile; return MNC_OK; }
    if (std::strcmp(key, "flux_groups") == 0) { *value = ctx->flux_groups; return MNC_OK; }
    if (std::strcmp(key, "learned_gate_log10") == 0) { *value = ctx->learned_gate_log10; return MNC_OK; }
    if (std::strcmp(key, "learned_fallback_iters") == 0) { *value = ctx->learned_fallback_iters; return MNC_OK; }
    if (std::strcmp(key, "learned_fused") == 0) { *value = ctx->learned_fused; return MNC_OK; }
    if (std::strcmp(key, "flux_overlap") == 0) { *value = ctx->flux_overlap; return MNC_OK; }
    if (std::strcmp(key, "tail_blocks") == 0) {
        *value = ctx->tail_blocks > 0 ? ctx->tail_blocks : 2 * ctx->num_cu;
        return MNC_OK;
    }
    return MNC_ERR_ARG;
}

const char *mnc_last_error(const mnc_ctx *ctx) { return ctx ? ctx->last_error.c_str() : "no context"; }

int mnc_autotune(mnc_ctx *ctx, double dt, const mnc_options *opt, int steps, char *report, int report_len) {
    if (!ctx) return MNC_ERR_ARG;
    if (!ctx->has_grid) return ctx_fail(ctx, MNC_ERR_STATE, "no grid");
    int st = check_opts(ctx, opt);
    if (st) return st;
    if (steps < 1 || steps > 1000 || !(dt > 0.0)) return ctx_fail(ctx, MNC_ERR_ARG, "bad autotune arguments");
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    const size_t n = size_t(ctx->grid.num_cells_x + 4) * (ctx->grid.num_cells_y + 4) * ctx->tab.nm;
    double *bk = nullptr;
    MNC_HIP_CHECK(hipMalloc((void **)&bk, 2 * n * sizeof(double)));
    long long stats[mnc::kStatWords];
    std::string rep;
    auto save = [&]() -> int {
        MNC_HIP_CHECK(hipMemcpyAsync(bk, ctx->d_mom, n * sizeof(double), hipMemcpyDeviceToDevice, ctx->stream));
        MNC_HIP_CHECK(hipMemcpyAsync(bk + n, ctx->d_alpha, n * sizeof(double), hipMemcpyDeviceToDevice, ctx->stream));
        MNC_HIP_CHECK(hipMemcpyAsync(stats, ctx->d_stats, sizeof stats, hipMemcpyDeviceToHost, ctx->stream));
        MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
        return MNC_OK;
    };
    auto restore = [&]() -> int {
        MNC_HIP_CHECK(hipMemcpyAsync(ctx->d_mom, bk, n * sizeof(double), hipMemcpyDeviceToDevice, ctx->stream));
        MNC_HIP_CHECK(hipMemcpyAsync(ctx->d_alpha, bk + n, n * sizeof(double), hipMemcpyDeviceToDevice, ctx->stream));
        MNC_HIP_CHECK(hipMemcpyAsync(ctx->d_stats, stats, sizeof stats, hipMemcpyHostToDevice, ctx->stream));
        MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
        return MNC_OK;
    };
    // One trial: a warm-up step (allocations, graph capture), then `steps` timed steps.
    auto trial = [&](double *ms) -> int {
        int s2;
        if ((s2 = restore()) || (s2 = mnc_update(ctx, dt, opt)) || (s2 = restore())) return s2;
        const auto t0 = std::chrono::steady_clock::now();
        for (int k = 0; k < steps; ++k)
            if ((s2 = mnc_update(ctx, dt, opt))) return s2;
        MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
        *ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count() / steps;
        return MNC_OK;
    };
    const bool timing = ctx->timing;
    ctx->timing = false;
    if ((st = save())) { (void)hipFree(bk); ctx->timing = timing; return st; }
    struct Knob { const char *key; std::vector<int> vals; int *slot; };
    const int cu = ctx->num_cu;
    // Knobs that change which work is done (the network gate, which steps run
    // in mixed precision) come first, so the launch shapes are tuned for the
    // work that is left.
    std::vector<Knob> knobs;
    if (opt->warm_start == MNC_WARM_LEARNED)
        knobs.push_back({"learned_gate_log10", {-3, -2, -1, 0, 1, kGateOff}, &ctx->learned_gate_log10});
    if (opt->precision == MNC_PREC_MIXED) {
        knobs.push_back({"mix_cond_log10", {5, 6, 7, 8, 9, 10}, &ctx->mix_cond_log10});
        knobs.push_back({"mix_split", {2, 3}, &ctx->mix_split});
        knobs.push_back({"mix_defer", {0, 1}, &ctx->mix_defer});
    }
    knobs.push_back({"graph", {0, 1}, &ctx->use_graph});
    knobs.push_back({"flux_tile", {0, 1, 2, 3}, &ctx->flux_tile});
    knobs.push_back({"flux_groups", {0, 2, 3, 4, 6, 8}, &ctx->flux_groups});
    knobs.push_back({"flux_overlap", {0, 1}, &ctx->flux_overlap});
    // -1 stands for each solve's own rule, which sends plain FP64 solves straight to the
    // tail's kernel.  A path that depends on rounding gets no fewer than that rule
    // gives; mixed and learned solves may also do without rounds (all FP64 then).
    const bool floor = by_rounding(opt);
    std::vector<int> rounds = floor && opt->precision != MNC_PREC_MIXED ? std::vector<int>{-1, 8, 12}
                                                                        : std::vector<int>{-1, 2, 4, 6, 8, 12};
    if (!floor && auto_rounds(ctx, opt) != 0) rounds.push_back(0);
    knobs.push_back({"rounds", rounds, &ctx->rounds});
    knobs.push_back({"tail_mode", {0, 1, 2}, &ctx->tail_mode});
    knobs.push_back({"tail_blocks", {cu, 2 * cu, 4 * cu}, &ctx->tail_blocks});
    if (opt->precision == MNC_PREC_MIXED) knobs.push_back({"mix_blocks", {cu / 2, cu, 2 * cu}, &ctx->mix_blocks});
    double best = 0.0;
    if ((st = trial(&best)) == MNC_OK) {
        char line[160];
        snprintf(line, sizeof line, "start %.4f ms/step\n", best);
        rep += line;
        for (auto &kb : knobs) {   // coordinate descent, one pass
            const int keep = *kb.slot;
            int arg = keep;
            // the network is extra work: a gate that consults it must beat the
            // gate that switches it off by more than the trials' noise (1%)
            const bool gate = std::strcmp(kb.key, "learned_gate_log10") == 0;
            double ms_off = (gate && keep == kGateOff) ? best : 0.0;
            for (int v : kb.vals) {
                if (v == keep || (v < 1 && std::strstr(kb.key, "_blocks") != nullptr)) continue;
                *kb.slot = v;
                ++ctx->epoch;
                double ms = 0.0;
                if ((st = trial(&ms))) break;
                snprintf(line, sizeof line, "%s=%d %.4f ms/step\n", kb.key, v, ms);
                rep += line;
                if (gate && v == kGateOff) ms_off = ms;
                if (ms < best) { best = ms; arg = v; }
            }
            if (gate && !st && arg != kGateOff && ms_off > 0.0 && ms_off <= 1.01 * best) {
                arg = kGateOff;
                best = ms_off;
            }
            *kb.slot = arg;
            ++ctx->epoch;
            if (st) break;
        }
    }
    const int st2 = restore();
    (void)hipFree(bk);
    ++ctx->epoch;
    ctx->timing = timing;
    if (report && report_len > 0) {
        snprintf(report, size_t(report_len), "%s", rep.c_str());
    }
    return st ? st : st2;
}

int mnc_mlp_num_params(void) { return mnc::mlp_param_count() + mnc::kMlpStats; }

int mnc_mlp_init(mnc_ctx *ctx, unsigned long long seed) {
    if (!ctx) return MNC_ERR_ARG;
    int st = mlp_check(ctx, false);
    if (st) return st;
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    if ((st = mlp_alloc(ctx))) return st;
    const int np = mnc::mlp_param_count();
    std::vector<float> h(size_t(np) + mnc::kMlpStats, 0.0f);
    // SplitMix64 stream -> U(-1, 1); weights U(-b, b), b = sqrt(6 / (fan_in + fan_out)); biases 0
    unsigned long long x = seed;
    auto uni = [&x]() {
        unsigned long long z = (x += 0x9e3779b97f4a7c15ull);
        z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
        z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
        z ^= z >> 31;
        return 2.0 * (double(z >> 11) * (1.0 / 9007199254740992.0)) - 1.0;
    };
    const int dims[5] = {15, 128, 128, 128, 15};
    size_t off = 0;
    for (int l = 0; l < 4; ++l) {
        const double bnd = std::sqrt(6.0 / double(dims[l] + dims[l + 1]));
        for (int i = 0; i < dims[l] * dims[l + 1]; ++i) h[off++] = float(bnd * uni());
        off += dims[l + 1];   // bias
    }
    for (int k = 0; k < 15; ++k) { h[np + 15 + k] = 1.0f; h[np + 45 + k] = 1.0f; }   // identity standardisation
    const size_t nall = h.size();
    MNC_HIP_CHECK(hipMemcpyAsync(ctx->d_mlp, h.data(), nall * sizeof(float), hipMemcpyHostToDevice, ctx->stream));
    MNC_HIP_CHECK(hipMemsetAsync(ctx->d_mlp + 2 * nall, 0, 2 * nall * sizeof(float), ctx->stream));   // Adam m, v
    mnc::mlp_pack(mlp_buffers(ctx), ctx->stream);
    MNC_HIP_CHECK(hipGetLastError());
    MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    ctx->mlp_ready = true;
    ctx->mlp_stats_set = false;
    ctx->mlp_step = 0;
    return MNC_OK;
}

int mnc_mlp_train(mnc_ctx *ctx, long long npairs, const double *u_scaled, const double *alpha_scaled, int steps,
                  int batch, double lr, unsigned long long seed, float *loss_out) {
    if (!ctx) return MNC_ERR_ARG;
    int st = mlp_check(ctx, true);
    if (st) return st;
    if (npairs < 1 || !u_scaled || !alpha_scaled || steps < 0 || batch < 1 || batch > (1 << 20) || !(lr > 0.0))
        return ctx_fail(ctx, MNC_ERR_ARG, "bad training arguments");
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    if ((st = mlp_train_alloc(ctx, batch, size_t(std::max(steps, 1)))) || (st = mlp_io(ctx, size_t(npairs) * 30))) return st;
    const size_t n15 = size_t(npairs) * 15;
    MNC_HIP_CHECK(hipMemcpyAsync(ctx->d_mlp_io, u_scaled, n15 * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    MNC_HIP_CHECK(hipMemcpyAsync(ctx->d_mlp_io + n15, alpha_scaled, n15 * sizeof(double), hipMemcpyHostToDevice,
                                 ctx->stream));
    const int np = mnc::mlp_param_count();
    if (!ctx->mlp_stats_set) {   // standardisation from this data
        float stats[mnc::kMlpStats];
        for (int part = 0; part < 2; ++part) {
            const double *src = part == 0 ? u_scaled : alpha_scaled;
            for (int k = 0; k < 15; ++k) {
                double m = 0.0, q = 0.0;
                for (long long i = 0; i < npairs; ++i) m += src[i * 15 + k];
                m /= double(npairs);
                for (long long i = 0; i < npairs; ++i) q += (src[i * 15 + k] - m) * (src[i * 15 + k] - m);
                const double sd = std::sqrt(q / double(npairs));
                stats[30 * part + k] = float(m);
                stats[30 * part + 15 + k] = float(sd > 1e-6 ? sd : 1.0);
            }
        }
        MNC_HIP_CHECK(hipMemcpyAsync(ctx->d_mlp + np, stats, sizeof stats, hipMemcpyHostToDevice, ctx->stream));
        MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
        ctx->mlp_stats_set = true;
    }
    const auto b0 = mlp_buffers(ctx);
    {
        Timed tm(ctx, MNC_KCLASS_MLP);
        for (int k = 0; k < steps; ++k) {
            auto b = b0;
            b.loss = ctx->d_mlp_loss + k;
            const int step = ++ctx->mlp_step;
            const unsigned long long sk = (seed * 0x9e3779b97f4a7c15ull) ^ (unsigned long long)(step) ^ 0x5bd1e995ull;
            mnc::mlp_train_step(b, ctx->d_mlp_io, ctx->d_mlp_io + n15, npairs, batch, sk | 1ull, float(lr), step,
                                ctx->stream);
        }
    }
    MNC_HIP_CHECK(hipGetLastError());
    if (loss_out && steps > 0)
        MNC_HIP_CHECK(hipMemcpyAsync(loss_out, ctx->d_mlp_loss, size_t(steps) * sizeof(float), hipMemcpyDeviceToHost,
                                     ctx->stream));
    MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    return MNC_OK;
}

int mnc_mlp_predict(mnc_ctx *ctx, int n, const double *u_scaled, double *alpha_scaled) {
    if (!ctx) return MNC_ERR_ARG;
    int st = mlp_check(ctx, true);
    if (st) return st;
    if (n < 0 || (n > 0 && (!u_scaled || !alpha_scaled))) return ctx_fail(ctx, MNC_ERR_ARG, "bad predict arguments");
    if (n == 0) return MNC_OK;
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    if ((st = mlp_io(ctx, size_t(n) * 30))) return st;
    const size_t n15 = size_t(n) * 15;
    MNC_HIP_CHECK(hipMemcpyAsync(ctx->d_mlp_io, u_scaled, n15 * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    {
        Timed tm(ctx, MNC_KCLASS_MLP);
        mnc::mlp_predict(mlp_buffers(ctx), ctx->d_mlp_io, n, ctx->d_mlp_io + n15, ctx->stream);
    }
    MNC_HIP_CHECK(hipGetLastError());
    MNC_HIP_CHECK(hipMemcpyAsync(alpha_scaled, ctx->d_mlp_io + n15, n15 * sizeof(double), hipMemcpyDeviceToHost,
                                 ctx->stream));
    MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    return MNC_OK;
}

int mnc_mlp_get_params(mnc_ctx *ctx, float *params) {
    if (!ctx || !params) return MNC_ERR_ARG;
    int st = mlp_check(ctx, true);
    if (st) return st;
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    MNC_HIP_CHECK(hipMemcpyAsync(params, ctx->d_mlp, size_t(mnc_mlp_num_params()) * sizeof(float),
                                 hipMemcpyDeviceToHost, ctx->stream));
    MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    return MNC_OK;
}

int mnc_mlp_set_params(mnc_ctx *ctx, const float *params) {
    if (!ctx || !params) return MNC_ERR_ARG;
    int st = mlp_check(ctx, false);
    if (st) return st;
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    if ((st = mlp_alloc(ctx))) return st;
    const size_t nall = size_t(mnc_mlp_num_params());
    MNC_HIP_CHECK(hipMemcpyAsync(ctx->d_mlp, params, nall * sizeof(float), hipMemcpyHostToDevice, ctx->stream));
    MNC_HIP_CHECK(hipMemsetAsync(ctx->d_mlp + 2 * nall, 0, 2 * nall * sizeof(float), ctx->stream));
    mnc::mlp_pack(mlp_buffers(ctx), ctx->stream);
    MNC_HIP_CHECK(hipGetLastError());
    MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    ctx->mlp_ready = true;
    ctx->mlp_stats_set = true;
    ctx->mlp_step = 0;
    return MNC_OK;
}

int mnc_mlp_gradient(mnc_ctx *ctx, int rows, const double *u_scaled, const double *alpha_scaled, float *grad,
                     float *loss) {
    if (!ctx) return MNC_ERR_ARG;
    int st = mlp_check(ctx, true);
    if (st) return st;
    if (rows < 1 || rows > (1 << 20) || !u_scaled || !alpha_scaled || !grad || !loss)
        return ctx_fail(ctx, MNC_ERR_ARG, "bad gradient arguments");
    MNC_HIP_CHECK(hipSetDevice(ctx->device));
    if ((st = mlp_train_alloc(ctx, rows, 1)) || (st = mlp_io(ctx, size_t(rows) * 30))) return st;
    const size_t n15 = size_t(rows) * 15;
    MNC_HIP_CHECK(hipMemcpyAsync(ctx->d_mlp_io, u_scaled, n15 * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    MNC_HIP_CHECK(hipMemcpyAsync(ctx->d_mlp_io + n15, alpha_scaled, n15 * sizeof(double), hipMemcpyHostToDevice,
                                 ctx->stream));
    const auto b = mlp_buffers(ctx);
    mnc::mlp_gradient(b, ctx->d_mlp_io, ctx->d_mlp_io + n15, rows, ctx->stream);
    MNC_HIP_CHECK(hipGetLastError());
    MNC_HIP_CHECK(hipMemcpyAsync(grad, b.grad, size_t(mnc::mlp_param_count()) * sizeof(float), hipMemcpyDeviceToHost,
                                 ctx->stream));
    MNC_HIP_CHECK(hipMemcpyAsync(loss, ctx->d_mlp_loss, sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
    MNC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    return MNC_OK;
}

}  // extern "C"
