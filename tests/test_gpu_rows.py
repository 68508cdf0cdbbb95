"""The FP64 solve with a row of lanes per cell (csrc/mnc_rows.hip), which takes
every closure of an FP64 solve whose decisions do not rest on the reference line
search's rounding: batches around its launch rules (one wave per cell up to 8
per CU, four cells per wave above, partly filled waves and blocks) against the
CPU oracle and the known multipliers, for both Hessian forms and both closures,
at quadratures whose orbits fill and do not fill a tile of 16 or a group of 64."""
import numpy as np
import pytest

from helpers import config2_batch, isotropic_start, load_pkg, oracle


def _mn_batch(o, order, Q, gaunt, n, seed):
    tab = o.Tables(order, Q, gaunt)
    u, astar, _ = config2_batch(tab.w, tab.p, tab.xi, tab.eta, tab.nm, n, np.random.default_rng(seed),
                                near_boundary_frac=0.0)
    return tab, u, astar


@pytest.mark.gpu
@pytest.mark.parametrize("order,Q,gaunt", [(0, 8, False), (1, 8, False), (2, 12, False), (2, 14, True), (3, 20, True),
                                           (3, 30, False), (4, 16, False), (4, 18, False), (4, 16, True)])
@pytest.mark.parametrize("n", [1, 6, 2048, 2049, 4101])
def test_rows_match_oracle(order, Q, gaunt, n):
    """Smooth closures, robust line search: the oracle's iteration counts, its
    answers to rounding (a quadratically converging Newton path amplifies the
    sums' rounding, ~1e-15, by the Hessian's condition number, below 1e4 for
    these multipliers: 1e-10 with a margin of ten), u_0 kept exactly."""
    mnc, o = load_pkg("mnc"), oracle()
    print("case rows N=%d Q=%d gaunt=%d n=%d" % (order, Q, gaunt, n), flush=True)
    tab, u, astar = _mn_batch(o, order, Q, gaunt, n, 17 * order + n)
    a0 = isotropic_start(u)
    tol = 1e-6 if gaunt else 1e-8
    ctx = mnc.Context(order, Q, use_gaunt=gaunt)
    opt = mnc.options(tol=tol, line_search=mnc.LS_ROBUST)
    st, ug, ag, itg, rg, ng = ctx.opt_batch_host(u, a0, opt)
    s = ctx.stats()
    ctx.close()
    m = min(n, 600)
    sto, uo, ao, ito, ro, _ = tab.opt_batch(u[-m:], a0[-m:], tol=tol, nthreads=8, line_search=1)
    assert st == sto == 0 and np.all(rg == 0.0)
    same = itg[-m:] == ito
    assert same.mean() >= 0.99
    assert np.abs(ug[-m:][same] - uo[same]).max() <= 1e-10 * np.abs(uo).max()
    assert np.abs(ag[-m:][same] - ao[same]).max() <= 1e-10 * (1.0 + np.abs(ao).max())
    assert np.array_equal(ug[:, 0], u[:, 0])
    assert np.all(ng <= tol * np.linalg.norm(u / u[:, :1], axis=1))
    assert s.num_dual_solves == n and s.iter_sum == itg.sum() and s.hist_reg[0] == n


@pytest.mark.gpu
@pytest.mark.parametrize("order,Q,gaunt", [(2, 12, False), (3, 14, True), (4, 16, False)])
@pytest.mark.parametrize("n", [5, 2051])
def test_rows_ppn_recover_multipliers(order, Q, gaunt, n):
    """PPn closures of known multipliers: alpha* to the tolerance times the
    condition number (below 1e3), u unchanged bit for bit up to u_0's scaling."""
    mnc, o = load_pkg("mnc"), oracle()
    print("case rows PPn N=%d Q=%d gaunt=%d n=%d" % (order, Q, gaunt, n), flush=True)
    tab = o.Tables(order, Q, gaunt)
    rng = np.random.default_rng(n + order)
    nm, delta = tab.nm, 1e-10
    alpha = 0.3 * rng.normal(size=(n, nm)) / (1.0 + np.arange(nm))
    alpha[:, 0] = rng.uniform(4.0, 8.0, n)
    z = alpha @ tab.p[:, :nm].T
    u = (0.5 * z + np.sqrt(0.25 * z * z + delta)) @ (tab.w[:, None] * tab.p[:, :nm])
    a0 = np.zeros_like(u)
    a0[:, 0] = u[:, 0] - 4.0 * np.pi * delta / u[:, 0]
    ctx = mnc.Context(order, Q, use_gaunt=gaunt, moment_type=mnc.MOMENT_PPN)
    st, ug, ag, it, r, _ = ctx.opt_batch_host(u, a0, mnc.options(tol=1e-8, line_search=mnc.LS_ROBUST, delta_ppn=delta))
    ctx.close()
    assert st == 0 and np.all(r == 0.0)
    assert np.abs(ag - alpha).max() <= 1e-5 * np.abs(alpha).max()
    assert np.abs(ug - u).max() <= 4e-16 * np.abs(u).max()


@pytest.mark.gpu
def test_rows_bad_cells_and_lists():
    """u_0 <= 0 cells are flagged and skipped, the others solved; the same cells
    through lockstep rounds first (the kernel then takes what is left on the
    lists) end at the same answers to rounding."""
    mnc, o = load_pkg("mnc"), oracle()
    print("case rows bad cells", flush=True)
    tab, u, _ = _mn_batch(o, 4, 16, False, 2500, 5)
    a0 = isotropic_start(u)
    opt = mnc.options(tol=1e-8, line_search=mnc.LS_ROBUST)
    ctx = mnc.Context(4, 16)
    bad = u.copy()
    bad[[0, 77, 2499], 0] = [-1.0, 0.0, np.nan]
    st, ub, ab, itb, _, _ = ctx.opt_batch_host(bad, a0, opt, allow_status=(mnc.ERR_U0,))
    assert st == mnc.ERR_U0 and np.all(itb[[0, 77, 2499]] == -1)
    st, ug, ag, itg, _, _ = ctx.opt_batch_host(u, a0, opt)
    ok = np.ones(2500, dtype=bool)
    ok[[0, 77, 2499]] = False
    assert np.array_equal(ab[ok], ag[ok]) and np.array_equal(ub[ok], ug[ok]) and np.array_equal(itb[ok], itg[ok])
    for rounds in (1, 5, 7):
        ctx.tune("rounds", rounds)
        st, ul, al, itl, _, _ = ctx.opt_batch_host(u, a0, opt)
        assert np.array_equal(itl, itg)
        assert np.abs(al - ag).max() <= 1e-10 * (1.0 + np.abs(ag).max())
    ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("order,Q,n,ppn", [(2, 12, 60, False), (4, 16, 2048, False), (4, 16, 2500, False), (2, 12, 70, True)])
def test_reference_line_search_takes_seven_rounds(order, Q, n, ppn):
    """Below TOL 1e-6 the reference's line search goes by the rounding of f, so an
    untouched context runs seven lockstep rounds, no more (each costs a small batch a
    lane's walk over the quadrature), before this kernel takes what is left: the same
    bits and counts as with the rounds set, for batches that one cell per wave
    covers and that it does not."""
    mnc, o = load_pkg("mnc"), oracle()
    print("case reference rounds N=%d n=%d ppn=%d" % (order, n, ppn), flush=True)
    tab, u, _ = _mn_batch(o, order, Q, False, n, 40 + n)
    a0 = isotropic_start(u)
    if ppn:
        a0[:, 0] = u[:, 0] - 4.0 * np.pi * 1e-10 / u[:, 0]
    res = []
    for rounds in (None, 7):
        ctx = mnc.Context(order, Q, moment_type=mnc.MOMENT_PPN if ppn else mnc.MOMENT_MN)
        if rounds is not None:
            ctx.tune("rounds", rounds)
        opt = mnc.options(tol=1e-8, line_search=mnc.LS_REFERENCE, delta_ppn=1e-10 if ppn else 0.0)
        out = ctx.opt_batch_host(u, a0, opt, allow_status=(mnc.OK, mnc.ERR_MAXREG))
        s = ctx.stats()
        res.append((out, (s.iter_sum, s.trial_sum, s.tail_cells, s.tail_iter_sum)))
        ctx.close()
    assert res[0][0][0] == res[1][0][0] and res[0][1] == res[1][1]
    for a, b in zip(res[0][0][1:], res[1][0][1:]):
        assert np.array_equal(a, b)
    if not ppn:
        _, _, _, ito, ro, _ = tab.opt_batch(u, a0, tol=1e-8, nthreads=8)
        assert ((res[0][0][3] == ito) & (res[0][0][4] == ro)).mean() >= 0.95


@pytest.mark.gpu
@pytest.mark.parametrize("order,Q,gaunt", [(1, 82, False), (4, 34, False), (4, 36, True)])
@pytest.mark.parametrize("n", [3, 2053])
def test_rows_with_the_table_in_l2(order, Q, gaunt, n):
    """Quadratures whose orbit table does not fit in LDS beside the waves' words (the
    smallest such at M1 and M4): the oracle's iterations and, with the bound of
    test_rows_match_oracle, its answers."""
    mnc, o = load_pkg("mnc"), oracle()
    print("case rows L2 N=%d Q=%d gaunt=%d n=%d" % (order, Q, gaunt, n), flush=True)
    tab, u, _ = _mn_batch(o, order, Q, gaunt, n, Q + n)
    a0 = isotropic_start(u)
    tol = 1e-6 if gaunt else 1e-8
    ctx = mnc.Context(order, Q, use_gaunt=gaunt)
    st, ug, ag, itg, rg, _ = ctx.opt_batch_host(u, a0, mnc.options(tol=tol, line_search=mnc.LS_ROBUST))
    ctx.close()
    m = min(n, 200)
    sto, uo, ao, ito, _, _ = tab.opt_batch(u[-m:], a0[-m:], tol=tol, nthreads=8, line_search=1)
    assert st == sto == 0 and np.all(rg == 0.0)
    same = itg[-m:] == ito
    assert same.mean() >= 0.99
    assert np.abs(ug[-m:][same] - uo[same]).max() <= 1e-10 * np.abs(uo).max()
    assert np.abs(ag[-m:][same] - ao[same]).max() <= 1e-10 * (1.0 + np.abs(ao).max())


@pytest.mark.gpu
@pytest.mark.parametrize("order,Q,gaunt,ppn", [(2, 12, False, False), (4, 16, False, False), (4, 16, True, False),
                                               (3, 12, False, True)])
@pytest.mark.parametrize("n", [5, 2100])
def test_rows_supplementary_stop(order, Q, gaunt, ppn, n):
    """tol_gamma holds cells back that pass the gradient test: the oracle's iterations
    (Mn: more of them than without it) and its answers (a further quadratic step
    leaves them at rounding, 1e-10 as above)."""
    mnc, o = load_pkg("mnc"), oracle()
    print("case rows tol_gamma N=%d gaunt=%d ppn=%d n=%d" % (order, gaunt, ppn, n), flush=True)
    tab = o.Tables(order, Q, gaunt)
    rng = np.random.default_rng(7 * order + n)
    nm, delta = tab.nm, 1e-10 if ppn else 0.0
    if ppn:
        alpha = 0.3 * rng.normal(size=(n, nm)) / (1.0 + np.arange(nm))
        alpha[:, 0] = rng.uniform(4.0, 8.0, n)
        z = alpha @ tab.p[:, :nm].T
        u = (0.5 * z + np.sqrt(0.25 * z * z + delta)) @ (tab.w[:, None] * tab.p[:, :nm])
        a0 = np.zeros_like(u)
        a0[:, 0] = u[:, 0] - 4.0 * np.pi * delta / u[:, 0]
    else:
        tab, u, _ = _mn_batch(o, order, Q, gaunt, n, 7 * order + n)
        a0 = isotropic_start(u)
    ctx = mnc.Context(order, Q, use_gaunt=gaunt, moment_type=mnc.MOMENT_PPN if ppn else mnc.MOMENT_MN)
    kw = dict(tol=1e-2, line_search=mnc.LS_ROBUST, delta_ppn=delta)
    it0 = ctx.opt_batch_host(u, a0, mnc.options(**kw))[3]
    st, ug, ag, itg, rg, _ = ctx.opt_batch_host(u, a0, mnc.options(tol_gamma=1.1, **kw))
    ctx.close()
    m = min(n, 600)
    sto, uo, ao, ito, _, _ = tab.opt_batch(u[-m:], a0[-m:], tol=1e-2, nthreads=8, line_search=1, delta_ppn=delta,
                                           moment_type=o.MOMENT_PPN if ppn else o.MOMENT_MN, tol_gamma=1.1)
    assert st == sto == 0 and np.all(rg == 0.0)
    same = itg[-m:] == ito
    assert same.mean() >= 0.99
    assert np.all(itg >= it0) and (ppn or itg.sum() > it0.sum())   # PPn's quadratic steps need none
    assert np.abs(ug[-m:][same] - uo[same]).max() <= 1e-10 * np.abs(uo).max()
    assert np.abs(ag[-m:][same] - ao[same]).max() <= 1e-10 * (1.0 + np.abs(ao).max())


@pytest.mark.gpu
@pytest.mark.parametrize("order,Q,gaunt", [(2, 12, False), (4, 16, False), (4, 16, True)])
def test_rows_agree_across_the_launch_rule(order, Q, gaunt):
    """One cell per wave up to four per CU, four cells per wave above: on both sides of
    the line (on a card of 256 CUs) the same cells take the same iterations and end
    at the same answers to rounding (1e-10 as above), and a repeated call at the
    same bits."""
    mnc, o = load_pkg("mnc"), oracle()
    print("case rows launch rule N=%d gaunt=%d" % (order, gaunt), flush=True)
    tab, u, _ = _mn_batch(o, order, Q, gaunt, 1025, 300 + order)
    a0 = isotropic_start(u)
    opt = mnc.options(tol=1e-6 if gaunt else 1e-8, line_search=mnc.LS_ROBUST)
    ctx = mnc.Context(order, Q, use_gaunt=gaunt)
    wide, four = ctx.opt_batch_host(u[:1024], a0[:1024], opt), ctx.opt_batch_host(u, a0, opt)
    again = ctx.opt_batch_host(u, a0, opt)
    ctx.close()
    assert wide[0] == four[0] == 0
    same = wide[3] == four[3][:1024]
    assert same.mean() >= 0.99
    for k in (1, 2):
        assert np.abs(wide[k][same] - four[k][:1024][same]).max() <= 1e-10 * (1.0 + np.abs(four[k]).max())
        assert np.array_equal(four[k], again[k])
