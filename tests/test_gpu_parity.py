"""GPU parity: libcintx_hip.so (HIP kernels on the MI355X) against the oracle
on the same seeded inputs.  FP64 bar: the reference's own element criterion
|got - ref| <= 1e-12 + 1e-12 |ref| (UNIFIED_ATOL/UNIFIED_RTOL and the pass rule
of crates/cintx-oracle/src/compare.rs:21-22, 256-259) for every family,
derivatives included, with `ref` from the oracle's long-double build (the
judge: the exact integrals of the FP64 inputs, pinned in
test_oracle_judge.py).  The oracle's FP64 build restates libcint's rounding
as well as its algorithm, and that rounding alone breaks the criterion on
ill-conditioned quartets (up to 1e-10 on (g d|g g) of the s..g molecule, ~1e-11
on cfg-1 nabla integrals), so it is not the reference value here."""
import ctypes
import sys

import numpy as np
import pytest

from cintx_amd import capi
from cintx_amd import molecule as M

pytestmark = pytest.mark.gpu
ATOL = 1e-12
RTOL = 1e-12


def assert_parity(got, ref):
    err = np.abs(got - ref)
    tol = ATOL + RTOL * np.abs(ref)
    bad = err > tol
    say(f"  max abs err {err.max():.3e}  max |ref| {np.abs(ref).max():.3e}  "
        f"max rel(>1e-6) {np.max(err[np.abs(ref) > 1e-6] / np.abs(ref[np.abs(ref) > 1e-6]), initial=0):.3e}")
    assert not bad.any(), (int(bad.sum()), float(err.max()))


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def oracle_blocks(O, name, tuples, mol):
    """The judge's blocks (long-double oracle) of the tuples, libcint layout."""
    out, offs, sizes = O.eval_list(name, tuples, mol.atm, mol.bas, mol.env, ext=True)
    return out, offs, sizes


def check_plan(O, name, tuples, mol, variant=None):
    say(f"plan {name} ntuples={len(tuples)} variant={variant}")
    p = capi.Plan(name, mol.atm, mol.bas, mol.env, tuples)
    if variant is not None:
        p.set_variant(variant)
    p.execute()
    p.sync()
    got = p.output()
    ref, offs, sizes = oracle_blocks(O, name, tuples, mol)
    t, o = p.tuples()
    assert np.array_equal(o, offs)
    assert_parity(got, ref)
    p.close()
    return got


def test_device_rys_rule_matches_oracle(oracle):
    """The device rule against the oracle's, and against the host evaluation
    of the same table (which test_rys_table_moment_equations pins to the
    moment equations with mpmath alone, independently of the oracle)."""
    L = capi.lib()
    L.cintx_rys_eval_device.argtypes = [ctypes.c_int, capi.DP, ctypes.c_int64, capi.DP, capi.DP]
    L.cintx_rys_eval_host.argtypes = [ctypes.c_int, capi.DP, ctypes.c_int64, capi.DP, capi.DP]
    for n in range(1, 15):
        xs = np.concatenate([np.linspace(0.0, 40.0 + 5 * n, 301), [1e-12, 3e-7, 1e4]])
        u = np.zeros(len(xs) * n)
        w = np.zeros(len(xs) * n)
        assert L.cintx_rys_eval_device(n, capi._dp(xs), len(xs), capi._dp(u), capi._dp(w)) == 0
        uh = np.zeros(len(xs) * n)
        wh = np.zeros(len(xs) * n)
        assert L.cintx_rys_eval_host(n, capi._dp(xs), len(xs), capi._dp(uh), capi._dp(wh)) == 0
        assert np.max(np.abs(u - uh) / uh) < 4e-14 and np.max(np.abs(w - wh) / wh) < 4e-14, n
        u, w = u.reshape(-1, n), w.reshape(-1, n)
        for k, x in enumerate(xs):
            uo, wo = oracle.rys_roots(n, x)
            tol = 1e-13 if x >= 35.0 + 5 * n else 2e-14
            assert np.max(np.abs(u[k] - uo) / uo) < tol
            assert np.max(np.abs(w[k] - wo) / wo) < tol


@pytest.mark.parametrize("n", [1, 2, 3, 4, 9, 14])
def test_device_rys_rule_at_interval_edges(n):
    """The device rule where its table changes interval and where the
    asymptotic rule takes over, by the moments sum_r w_r s_r^m = F_m(x)
    (mpmath, 40 digits).  Tolerance: s and w within two units in the last
    place and u = s/(1-s) one more, so (m + 2) 5e-16 of the moment.  Past
    1e300 s and w vanish."""
    import mpmath as mp
    mp.mp.dps = 40
    top = 35.0 + 5 * n
    edges = np.array([0.5, 1.0, 7.5, 20.0, top - 0.5, top])
    xs = np.concatenate([[0.0, 1e-300, 0.25], np.nextafter(edges, 0), edges,
                         np.nextafter(edges, 1e3), [0.75 * top, top + 0.5, 1e300, 1e308, np.inf]])
    L = capi.lib()
    L.cintx_rys_eval_device.argtypes = [ctypes.c_int, capi.DP, ctypes.c_int64, capi.DP, capi.DP]
    u = np.zeros(len(xs) * n)
    w = np.zeros(len(xs) * n)
    assert L.cintx_rys_eval_device(n, capi._dp(xs), len(xs), capi._dp(u), capi._dp(w)) == 0
    u, w = u.reshape(-1, n), w.reshape(-1, n)
    for k, x in enumerate(xs):
        if x >= 1e300:
            assert np.all((u[k] >= 0) & (u[k] < 1e-297) & (w[k] >= 0) & (w[k] < 1e-149)), x
            continue
        if x >= top:  # the asymptotic rule itself is good to 1e-13
            continue
        s = [mp.mpf(v) / (1 + mp.mpf(v)) for v in u[k]]
        for m in range(2 * n):
            a, y = m + mp.mpf(1) / 2, mp.mpf(x)
            ref = 1 / (2 * a) if x < 1e-200 else mp.gammainc(a, 0, y) / (2 * y ** a)
            got = mp.fsum(mp.mpf(float(w[k][r])) * s[r] ** m for r in range(n))
            assert abs(got / ref - 1) < 5e-16 * (m + 2), (x, m)
    far = xs[(xs >= top) & (xs < 1e300)]
    uh = np.zeros(len(far) * n)
    wh = np.zeros(len(far) * n)
    L.cintx_rys_eval_host.argtypes = [ctypes.c_int, capi.DP, ctypes.c_int64, capi.DP, capi.DP]
    assert L.cintx_rys_eval_host(n, capi._dp(far), len(far), capi._dp(uh), capi._dp(wh)) == 0
    sel = (xs >= top) & (xs < 1e300)
    assert np.allclose(u[sel].ravel(), uh, rtol=1e-15, atol=0)
    assert np.allclose(w[sel].ravel(), wh, rtol=1e-15, atol=0)


def test_int2e_sph_cfg1_full_tensor(oracle):
    mol = M.config(1)
    n = mol.nbas
    tuples = [(i, j, k, l) for l in range(n) for k in range(n) for j in range(n) for i in range(n)]
    check_plan(oracle, "int2e_sph", tuples, mol)


def test_int2e_sph_cfg2_sampled(oracle):
    mol = M.config(2)
    rng = np.random.default_rng(2)
    tuples = [tuple(int(s) for s in rng.integers(0, mol.nbas, 4)) for _ in range(3000)]
    check_plan(oracle, "int2e_sph", tuples, mol)


def test_int2e_ip1_sph_cfg1(oracle):
    mol = M.config(1)
    rng = np.random.default_rng(3)
    tuples = [tuple(int(s) for s in rng.integers(0, mol.nbas, 4)) for _ in range(2000)]
    check_plan(oracle, "int2e_ip1_sph", tuples, mol)


def test_int3c2e_sph_cfg4_sampled(oracle):
    mol = M.config(4)
    rng = np.random.default_rng(4)
    tuples = [(int(rng.integers(0, mol.aux_start)), int(rng.integers(0, mol.aux_start)),
               int(rng.integers(mol.aux_start, mol.nbas))) for _ in range(3000)]
    check_plan(oracle, "int3c2e_sph", tuples, mol)


def test_int3c2e_ip1_sph_cfg4_sampled(oracle):
    mol = M.config(4)
    rng = np.random.default_rng(5)
    tuples = [(int(rng.integers(0, mol.aux_start)), int(rng.integers(0, mol.aux_start)),
               int(rng.integers(mol.aux_start, mol.nbas))) for _ in range(1500)]
    check_plan(oracle, "int3c2e_ip1_sph", tuples, mol)


def test_int2e_ip2_sph_cfg1(oracle):
    mol = M.config(1)
    rng = np.random.default_rng(13)
    tuples = [tuple(int(s) for s in rng.integers(0, mol.nbas, 4)) for _ in range(2000)]
    check_plan(oracle, "int2e_ip2_sph", tuples, mol)


def test_int3c2e_ip2_sph_cfg4_sampled(oracle):
    mol = M.config(4)
    rng = np.random.default_rng(14)
    tuples = [(int(rng.integers(0, mol.aux_start)), int(rng.integers(0, mol.aux_start)),
               int(rng.integers(mol.aux_start, mol.nbas))) for _ in range(1500)]
    check_plan(oracle, "int3c2e_ip2_sph", tuples, mol)


def test_cart_families(oracle):
    mol = M.config(1)
    n = mol.nbas
    full = [(i, j, k, l) for l in range(n) for k in range(n) for j in range(n) for i in range(n)]
    check_plan(oracle, "int2e_cart", full, mol)
    aux = M.config(4)
    rng = np.random.default_rng(17)
    t3 = [(int(rng.integers(0, aux.aux_start)), int(rng.integers(0, aux.aux_start)),
           int(rng.integers(aux.aux_start, aux.nbas))) for _ in range(3000)]
    check_plan(oracle, "int3c2e_cart", t3, aux)
    gc = M.general_contraction_h2()
    low = [s for s in range(gc.nbas) if gc.bas[s][1] <= 2]
    for _ in range(10):
        sh = [int(low[i]) for i in rng.integers(0, len(low), 4)]
        dims = [d + 1 for d in capi.natural_dims("int2e_cart", sh, gc.bas)]
        got, not0 = capi.raw_call("int2e_cart", sh, gc.atm, gc.bas, gc.env, dims)
        ref, rnot0 = oracle.eval_tuple("int2e_cart", sh, gc.atm, gc.bas, gc.env, dims=dims, ext=True)
        assert not0 == rnot0
        assert_parity(got, ref)
        got, not0 = capi.raw_call("int3c2e_cart", sh[:3], gc.atm, gc.bas, gc.env)
        ref, rnot0 = oracle.eval_tuple("int3c2e_cart", sh[:3], gc.atm, gc.bas, gc.env, ext=True)
        assert not0 == rnot0
        assert_parity(got, ref)
    with pytest.raises(capi.CintxError):
        capi.Plan("int2e_cart", mol.atm, mol.bas, mol.env, full[:10], precision=capi.PREC_MIXED,
                  mixed_threshold=1.0)


def test_int2c2e_sph_cfg4_aux_metric(oracle):
    # every (P|Q) of the cfg-4 auxiliary basis (s..g on 64 centres)
    mol = M.config(4)
    aux = np.arange(mol.aux_start, mol.nbas)
    rng = np.random.default_rng(9)
    tuples = [(int(i), int(k)) for i in aux for k in aux]
    tuples = [tuples[j] for j in rng.permutation(len(tuples))[:20000]]
    check_plan(oracle, "int2c2e_sph", tuples, mol)
    gc = M.general_contraction_h2()
    check_plan(oracle, "int2c2e_sph", [(i, k) for i in range(gc.nbas) for k in range(gc.nbas)],
               gc)


def test_raw_signature_dims_and_general_contraction(oracle):
    mol = M.general_contraction_h2()
    low = [s for s in range(mol.nbas) if mol.bas[s][1] <= 2]
    rng = np.random.default_rng(6)
    for _ in range(25):
        shls = [int(low[i]) for i in rng.integers(0, len(low), 4)]
        got, not0 = capi.int2e_sph(shls, mol.atm, mol.bas, mol.env)
        ref, rnot0 = oracle.eval_tuple("int2e_sph", shls, mol.atm, mol.bas, mol.env, ext=True)
        assert not0 == rnot0
        assert_parity(got, ref)
        d0 = capi.natural_dims("int2e_sph", shls, mol.bas)
        dims = [d + 1 for d in d0]
        gd, _ = capi.int2e_sph(shls, mol.atm, mol.bas, mol.env, dims=dims)
        rd, _ = oracle.eval_tuple("int2e_sph", shls, mol.atm, mol.bas, mol.env, dims=dims,
                                  ext=True)
        assert_parity(gd, rd)
    shls = [int(low[0]), int(low[1]), int(low[2])]
    for name in ("int2e_ip1_sph", "int3c2e_sph", "int3c2e_ip1_sph", "int2c2e_sph",
                 "int2e_ip2_sph", "int3c2e_ip2_sph"):
        sh = shls + [int(low[3])] if name.startswith("int2e") else shls
        sh = sh[:capi.arity(name)]
        got, not0 = capi.raw_call(name, sh, mol.atm, mol.bas, mol.env)
        ref, rnot0 = oracle.eval_tuple(name, sh, mol.atm, mol.bas, mol.env, ext=True)
        assert not0 == rnot0
        assert_parity(got, ref)
    for _ in range(10):
        sh = [int(low[i]) for i in rng.integers(0, len(low), 2)]
        dims = [d + 2 for d in capi.natural_dims("int2c2e_sph", sh, mol.bas)]
        gd, not0 = capi.int2c2e_sph(sh, mol.atm, mol.bas, mol.env, dims=dims)
        rd, rnot0 = oracle.eval_tuple("int2c2e_sph", sh, mol.atm, mol.bas, mol.env, dims=dims,
                                       ext=True)
        assert not0 == rnot0
        assert_parity(gd, rd)


def test_raw_calls_with_optimizers_from_four_threads(oracle):
    """Four host threads call the libcint-signature entry points at once,
    sharing one device-resident optimizer per family (the role of CINTOpt's
    pair data, libcint-master/src/optimizer.c:344-425), with some calls
    passing none; the calls take no lock and every block equals the judge."""
    import threading
    m1 = M.config(1)
    gc = M.general_contraction_h2()
    n = m1.nbas
    rng = np.random.default_rng(31)
    uniq = [(i, j, k, l) for i in range(n) for j in range(i + 1) for k in range(i + 1)
            for l in range(k + 1)]
    opts = {("int2e_sph", 1): capi.Optimizer("int2e_sph", m1.atm, m1.bas, m1.env),
            ("int2e_ip1_sph", 1): capi.Optimizer("int2e_ip1_sph", m1.atm, m1.bas, m1.env),
            ("int2e_sph", 0): capi.Optimizer("int2e_sph", gc.atm, gc.bas, gc.env),
            ("int3c2e_sph", 0): capi.Optimizer("int3c2e_sph", gc.atm, gc.bas, gc.env)}
    mols = {1: m1, 0: gc}
    jobs = [("int2e_sph", 1, t, True) for t in uniq]
    jobs += [("int2e_ip1_sph", 1, tuple(int(v) for v in rng.integers(0, n, 4)), True)
             for _ in range(800)]
    jobs += [("int2e_sph", 1, tuple(int(v) for v in rng.integers(0, n, 4)), False)
             for _ in range(400)]
    jobs += [("int2e_sph", 0, tuple(int(v) for v in rng.integers(0, gc.nbas, 4)), True)
             for _ in range(150)]
    jobs += [("int3c2e_sph", 0, tuple(int(v) for v in rng.integers(0, gc.nbas, 3)), True)
             for _ in range(150)]
    order = rng.permutation(len(jobs))
    jobs = [jobs[i] for i in order]
    results = [None] * len(jobs)
    errors = []

    def worker(t):
        try:
            for i in range(t, len(jobs), 4):
                fam, mk, sh, use = jobs[i]
                mol = mols[mk]
                results[i] = capi.raw_call(fam, sh, mol.atm, mol.bas, mol.env,
                                           opt=opts[(fam, mk)] if use else None)
        except Exception as e:  # reported below
            errors.append(repr(e))

    threads = [threading.Thread(target=worker, args=(t,)) for t in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not errors, errors[:3]
    say(f"  {len(jobs)} raw calls from 4 threads")
    for fam in ("int2e_sph", "int2e_ip1_sph", "int3c2e_sph"):
        for mk, mol in mols.items():
            idx = [i for i, j in enumerate(jobs) if j[0] == fam and j[1] == mk]
            if not idx:
                continue
            ref, offs, sizes = oracle.eval_list(fam, [jobs[i][2] for i in idx], mol.atm, mol.bas,
                                                mol.env, ext=True)
            got = np.concatenate([results[i][0] for i in idx])
            say(f"  {fam} on {'cfg1' if mk else 'gc basis'}: {len(idx)} calls")
            assert_parity(got, ref)
    for o in opts.values():
        o.close()


def test_cintrs_eval_on_device(oracle):
    mol = M.config(1)
    shls = [5, 3, 4, 8]
    req = int(np.prod(capi.natural_dims("int2e_sph", shls, mol.bas)))
    out = np.zeros(req)
    s = capi.eval_raw(capi.INT2E_SPH, out, None, shls, mol.atm, mol.bas, mol.env)
    ref, not0 = oracle.eval_tuple("int2e_sph", shls, mol.atm, mol.bas, mol.env, ext=True)
    assert s["not0"] == not0 and s["bytes_written"] == req * 8
    assert_parity(out, ref)
    # api 9 (int2e_cart): Cartesian extents
    req = int(np.prod(capi.natural_dims("int2e_cart", shls, mol.bas)))
    out = np.zeros(req)
    s = capi.eval_raw(capi.INT2E_CART, out, None, shls, mol.atm, mol.bas, mol.env)
    ref, not0 = oracle.eval_tuple("int2e_cart", shls, mol.atm, mol.bas, mol.env, ext=True)
    assert s["not0"] == not0 and s["bytes_written"] == req * 8
    assert_parity(out, ref)


def test_graph_replay_equals_eager(oracle):
    mol = M.config(1)
    n = mol.nbas
    tuples = [(i, j, k, l) for i in range(n) for j in range(i + 1) for k in range(n)
              for l in range(k + 1)]
    p = capi.Plan("int2e_sph", mol.atm, mol.bas, mol.env, tuples)
    p.execute()
    p.sync()
    eager = p.output()
    assert not np.isnan(eager).any()
    for rep in range(4):
        # poison the buffer first: a bin the graph left out would stay NaN
        p.fill_output(np.nan)
        p.execute(graph=True)
        p.sync()
        again = p.output()
        assert np.array_equal(eager, again), rep
        p.fill_output(np.nan)
        p.execute()
        p.sync()
        assert np.array_equal(eager, p.output()), rep
    p.close()


def test_graph_chains_with_runtime_class_bins(oracle):
    """The captured graph runs the bins as concurrent chains and gives the
    runtime-class bins of different chains their own workspace slices: many
    f/g classes replayed several times must equal the one-bin-at-a-time
    execution bit for bit, and the oracle."""
    mol = M.config(5)
    rng = np.random.default_rng(21)
    hi = [s for s in range(mol.nbas) if mol.bas[s][1] >= 3]
    tuples = [(int(hi[i]), int(hi[j]), int(rng.integers(0, mol.nbas)), int(rng.integers(0, mol.nbas)))
              for i, j in rng.integers(0, len(hi), (120, 2))]
    say(f"plan int2e_sph cfg5 ntuples={len(tuples)} (graph chains)")
    p = capi.Plan("int2e_sph", mol.atm, mol.bas, mol.env, tuples)
    assert sum(b["generic"] for b in p.bin_stats()) >= 8
    p.execute()
    p.sync()
    eager = p.output()
    assert not np.isnan(eager).any()
    for rep in range(3):
        p.fill_output(np.nan)
        p.execute(graph=True)
        p.sync()
        assert np.array_equal(eager, p.output()), rep
        p.fill_output(np.nan)
        p.execute()
        p.sync()
    ref, offs, sizes = oracle_blocks(oracle, "int2e_sph", tuples, mol)
    assert_parity(eager, ref)
    p.close()


def test_screened_plan_cfg2(oracle):
    mol = M.config(2)
    say("screened plan cfg2")
    p = capi.Plan("int2e_sph", mol.atm, mol.bas, mol.env, screened=(1e-12, 97))
    p.execute()
    p.sync()
    got = p.output()
    t, offs = p.tuples()
    say(f"  tuples {p.ntuples}")
    assert p.ntuples > 1000
    rng = np.random.default_rng(7)
    pick = rng.choice(p.ntuples, size=min(2000, p.ntuples), replace=False)
    sub = [tuple(int(v) for v in t[q]) for q in pick]
    ref, roffs, sizes = oracle.eval_list("int2e_sph", sub, mol.atm, mol.bas, mol.env, ext=True)
    blk = np.concatenate([got[offs[q]:offs[q] + sizes[k]] for k, q in enumerate(pick)])
    assert_parity(blk, ref)
    p.close()


def test_screened_enumeration_complete_and_unique(oracle):
    """The screened plan holds each unordered quartet of shells at most once
    (i >= j, k >= l, ij >= kl in the pair order), and exactly the quartets
    whose Schwarz product sqrt(max|(ij|ij)|) sqrt(max|(kl|kl)|) reaches the
    threshold, with bra pairs restricted to every stride-th pair: the set is
    recomputed here from the judge's diagonal integrals (pairs within 1e-6
    relative of the threshold, where the device's and the judge's rounding
    may decide differently, are left out of the comparison)."""
    mol = M.config(2)
    thr, stride = 1e-12, 37
    p = capi.Plan("int2e_sph", mol.atm, mol.bas, mol.env, screened=(thr, stride))
    t, _ = p.tuples()
    p.close()
    n = mol.nbas
    ls = mol.bas[:, 1]
    pid = {}
    diag = []
    for i in range(n):
        for j in range(i + 1):
            pid[(i, j)] = len(diag)
            diag.append((i, j, i, j))
    ref, offs, sizes = oracle.eval_list("int2e_sph", diag, mol.atm, mol.bas, mol.env, ext=True)
    q = np.sqrt([np.abs(ref[a:a + k]).max() for a, k in zip(offs, sizes)])
    qmax = q.max()

    def key(a, b):
        return pid[(max(a, b), min(a, b))]

    got = {}
    for a, b, c, d in t:
        ka, kb = key(a, b), key(c, d)
        assert ls[a] >= ls[b] and ls[c] >= ls[d]
        assert ka >= kb
        k = (ka, kb)
        assert k not in got, k
        got[k] = True
    say(f"  screened cfg2 stride {stride}: {len(got)} unique quartets")
    live = np.where(q * qmax >= thr)[0]
    border = 0
    want = set()
    for ka in live:
        if ka % stride:
            continue
        for kb in live[live <= ka]:
            v = q[ka] * q[kb]
            if abs(v - thr) <= 1e-6 * thr:
                border += 1
                got.pop((int(ka), int(kb)), None)
                continue
            if v >= thr:
                want.add((int(ka), int(kb)))
    assert want == set(got), (len(want - set(got)), len(set(got) - want), border)


def test_high_l_against_judge_sg_sample(oracle):
    """The f/g classes of the 32-atom s..g molecule (runtime-class kernel):
    the benchmark's own sample (300 tuples, seed 5, of the screened plan with
    bra stride 64, and of its every-8th-tuple int2e_ip1_sph plan), the
    (g d|g g) tuple on which libcint's FP64 route loses 1e-10, and 1500
    random tuples with an f or g shell, all at the element rule against the
    judge."""
    mol = M.config(5)
    p5 = capi.Plan("int2e_sph", mol.atm, mol.bas, mol.env, screened=(1e-12, 64))
    t5, _ = p5.tuples()
    p5.execute()
    p5.sync()
    rng = np.random.default_rng(5)
    pick = np.sort(rng.choice(len(t5), size=min(300, len(t5)), replace=False))
    got, _, _ = p5.output_tuples(pick)
    ref, _, _ = oracle.eval_list("int2e_sph", [tuple(int(v) for v in t5[q]) for q in pick],
                                 mol.atm, mol.bas, mol.env, ext=True)
    say(f"plan int2e_sph s..g screened sample {len(pick)} of {len(t5)}")
    assert_parity(got, ref)
    p5.close()
    t8 = np.array(t5[::8], dtype=np.int32)
    pi = capi.Plan("int2e_ip1_sph", mol.atm, mol.bas, mol.env, t8)
    pi.execute()
    pi.sync()
    rng = np.random.default_rng(5)
    pick = np.sort(rng.choice(len(t8), size=min(300, len(t8)), replace=False))
    got, _, _ = pi.output_tuples(pick)
    ref, _, _ = oracle.eval_list("int2e_ip1_sph", [tuple(int(v) for v in t8[q]) for q in pick],
                                 mol.atm, mol.bas, mol.env, ext=True)
    say(f"plan int2e_ip1_sph s..g sample {len(pick)}")
    assert_parity(got, ref)
    pi.close()
    ls = mol.bas[:, 1]
    rng = np.random.default_rng(23)
    hl = [(215, 140, 79, 71)]
    while len(hl) < 1500:
        sh = tuple(int(s) for s in rng.integers(0, mol.nbas, 4))
        if max(ls[list(sh)]) >= 3:
            hl.append(sh)
    check_plan(oracle, "int2e_sph", hl, mol)
    check_plan(oracle, "int2e_ip1_sph", hl[:600], mol)


def test_high_l_generic_kernel_cfg5(oracle):
    # (ff|..) and (gg|gg) classes run the runtime-class kernel
    mol = M.config(5)
    rng = np.random.default_rng(8)
    ls = mol.bas[:, 1]
    hi = [s for s in range(mol.nbas) if ls[s] >= 3]
    tuples = [tuple(int(s) for s in rng.integers(0, mol.nbas, 4)) for _ in range(150)]
    tuples += [(int(hi[i]), int(hi[j]), int(hi[k]), int(hi[l])) for i, j, k, l in
               rng.integers(0, len(hi), (40, 4))]
    check_plan(oracle, "int2e_sph", tuples, mol)


def test_high_l_ip1_cfg5(oracle):
    mol = M.config(5)
    rng = np.random.default_rng(9)
    tuples = [tuple(int(s) for s in rng.integers(0, mol.nbas, 4)) for _ in range(120)]
    check_plan(oracle, "int2e_ip1_sph", tuples, mol)


@pytest.mark.parametrize("variant", range(capi.NVARIANTS))
def test_high_l_template_classes_every_variant(oracle, variant):
    """The int2e_sph classes with an f or g shell that run as template
    kernels (at most 3500 Cartesian elements and 135 values per chain; cintx_amd.build.high_l_classes):
    on the s..g molecule, eight tuples of every such class, shells taken from
    two neighbouring atoms (so the blocks are not screened to zero) and put
    in a random one of the eight orders of the quartet's symmetry, in every
    compiled launch shape, against the judge."""
    from cintx_amd import build as B
    mol = M.config(5)
    ls, at = mol.bas[:, 1], mol.bas[:, 0]
    natm = int(at.max()) + 1
    rng = np.random.default_rng(40 + variant)
    tuples = []
    for cls in B.high_l_classes():
        for _ in range(8):
            a = int(rng.integers(0, natm))
            near = (at == a) | (at == (a + 1) % natm)
            sh = [int(rng.choice(np.where(near & (ls == l))[0])) for l in cls]
            i, j, k, l = sh
            orders = [(i, j, k, l), (j, i, k, l), (i, j, l, k), (j, i, l, k),
                      (k, l, i, j), (l, k, i, j), (k, l, j, i), (l, k, j, i)]
            tuples.append(orders[int(rng.integers(0, 8))])
    check_plan(oracle, "int2e_sph", tuples, mol, variant)


@pytest.mark.parametrize("variant", range(capi.NVARIANTS))
def test_high_l_nabla_templates_every_variant(oracle, variant):
    """The nabla_i template classes with an f or g shell i and an s shell j
    (cintx_amd.build.high_l_nabla_classes): int2e_ip1_sph (f s|..) and
    (g s|..) tuples of neighbouring atoms on the s..g molecule, and
    int3c2e_ip2_sph triples whose aux shell is f or g (nabla on it), in
    every compiled launch shape, against the judge."""
    from cintx_amd import build as B
    rng = np.random.default_rng(60 + variant)
    mol = M.config(5)
    ls, at = mol.bas[:, 1], mol.bas[:, 0]
    natm = int(at.max()) + 1
    tuples = []
    for cls in B.high_l_nabla_classes():
        for _ in range(10):
            a = int(rng.integers(0, natm))
            near = (at == a) | (at == (a + 1) % natm)
            i, j, k, l = [int(rng.choice(np.where(near & (ls == v))[0])) for v in cls]
            tuples.append((i, j, k, l) if rng.integers(0, 2) else (i, j, l, k))
    check_plan(oracle, "int2e_ip1_sph", tuples, mol, variant)
    aux = M.config(4)
    ls, at = aux.bas[:, 1], aux.bas[:, 0]
    natm = int(at.max()) + 1
    orb = np.arange(aux.nbas) < aux.aux_start
    triples = []
    for lk in (3, 4):
        for li in range(3):
            for lj in range(3):
                for _ in range(6):
                    a = int(rng.integers(0, natm))
                    near = (at == a) | (at == (a + 1) % natm)
                    pick = [np.where(near & orb & (ls == li))[0],
                            np.where(near & orb & (ls == lj))[0],
                            np.where(near & ~orb & (ls == lk))[0]]
                    if all(len(c) for c in pick):
                        triples.append(tuple(int(rng.choice(c)) for c in pick))
    check_plan(oracle, "int3c2e_ip2_sph", triples, aux, variant)


def test_high_l_ip1_neighbouring_atoms(oracle):
    """int2e_ip1_sph f/g classes on tuples of neighbouring atoms of the s..g
    molecule, where the integrals are large and libcint's FP64 route loses
    most (measured against the judge: up to 1e4 times the 1e-12 bar on
    (f g|d s), 2e3 on (g g|s s), 110 on (s p|g g)): the device, whose
    transfers start from the centre of the larger exponent per primitive
    pair, stays within the bar."""
    mol = M.config(5)
    ls, at = mol.bas[:, 1], mol.bas[:, 0]
    natm = int(at.max()) + 1
    rng = np.random.default_rng(7)
    tuples = []
    for c in ("3030", "4130", "1131", "3032", "1300", "3420", "0144", "2311", "4400",
              "3300", "1311"):
        for _ in range(40):
            a = int(rng.integers(0, natm))
            near = (at == a) | (at == (a + 1) % natm) | (at == (a + 8) % natm)
            tuples.append(tuple(int(rng.choice(np.where(near & (ls == int(l)))[0])) for l in c))
    check_plan(oracle, "int2e_ip1_sph", tuples, mol)


def test_general_contraction_all_classes(oracle):
    mol = M.general_contraction_h2()
    rng = np.random.default_rng(10)
    tuples = [tuple(int(s) for s in rng.integers(0, mol.nbas, 4)) for _ in range(200)]
    check_plan(oracle, "int2e_sph", tuples, mol)
    check_plan(oracle, "int3c2e_sph", [t[:3] for t in tuples[:100]], mol)


def test_jk_build_cfg1(oracle):
    # J/K from the screened unique-quartet plan (screen off) against an
    # einsum over the oracle's full cfg-1 tensor
    mol = M.config(1)
    eri = oracle.full_tensor_int2e(mol.atm, mol.bas, mol.env, ext=True)
    nao = eri.shape[0]
    rng = np.random.default_rng(11)
    D = rng.normal(size=(nao, nao)) / nao
    D = D + D.T
    Jr = np.einsum("pqrs,rs->pq", eri, D)
    Kr = np.einsum("pqrs,qs->pr", eri, D)
    p = capi.Plan("int2e_sph", mol.atm, mol.bas, mol.env, screened=(1e-300, 1))
    n = mol.nbas
    # every unique quartet except those with a zero Schwarz factor (a pair
    # whose primitives libcint's screen drops entirely)
    assert 0 < p.ntuples <= (n * (n + 1) // 2) * (n * (n + 1) // 2 + 1) // 2
    J, K = p.jk(D)
    say(f"  J err {np.abs(J - Jr).max():.3e}  K err {np.abs(K - Kr).max():.3e}  "
        f"|J| {np.abs(Jr).max():.3e}")
    assert np.abs(J - Jr).max() <= 1e-11 * max(1.0, np.abs(Jr).max())
    assert np.abs(K - Kr).max() <= 1e-11 * max(1.0, np.abs(Kr).max())
    p.close()


def _jk_reference(eri, nao, seed):
    rng = np.random.default_rng(seed)
    D = rng.normal(size=(nao, nao)) / nao
    D = D + D.T
    return D, np.einsum("pqrs,rs->pq", eri, D), np.einsum("pqrs,qs->pr", eri, D)


def test_jk_fused_every_launch_variant(oracle):
    """The fused J/K epilogues (one-lane kernels: blocks staged in LDS per
    chunk and digested by their lane; wide kernels: the staged spherical
    block digested by the tuple's lanes) in every compiled launch shape,
    against an einsum over the oracle's full cfg-1 tensor."""
    mol = M.config(1)
    eri = oracle.full_tensor_int2e(mol.atm, mol.bas, mol.env, ext=True)
    D, Jr, Kr = _jk_reference(eri, eri.shape[0], 12)
    p = capi.Plan("int2e_sph", mol.atm, mol.bas, mol.env, screened=(1e-300, 1))
    for v in range(capi.NVARIANTS):
        p.set_variant(v)
        J, K = p.jk(D)
        say(f"variant {v}: J err {np.abs(J - Jr).max():.3e}  K err {np.abs(K - Kr).max():.3e}")
        assert np.abs(J - Jr).max() <= 1e-11 * max(1.0, np.abs(Jr).max())
        assert np.abs(K - Kr).max() <= 1e-11 * max(1.0, np.abs(Kr).max())
    p.close()


def test_jk_with_runtime_class_bins(oracle):
    """J/K over s..g shells on two centres: the f and g classes run the
    runtime-class kernel (blocks written, then the digest kernel), the rest
    the fused class kernels; against an einsum over the oracle tensor."""
    mol = M.Molecule()
    a0 = mol.add_atom(8, (0.0, 0.0, 0.0))
    a1 = mol.add_atom(8, (0.3, -0.4, 1.9))
    rng = np.random.default_rng(21)
    for atom in (a0, a1):
        for l in range(5):
            e = sorted(rng.uniform(0.3, 6.0, 2), reverse=True)
            mol.add_shell(atom, l, e, [[M.gto_norm(l, x) * c for x, c in zip(e, (0.6, 0.5))]])
    mol.build()
    eri = oracle.full_tensor_int2e(mol.atm, mol.bas, mol.env)
    D, Jr, Kr = _jk_reference(eri, eri.shape[0], 13)
    p = capi.Plan("int2e_sph", mol.atm, mol.bas, mol.env, screened=(1e-300, 1))
    J, K = p.jk(D)
    say(f"s..g: J err {np.abs(J - Jr).max():.3e}  K err {np.abs(K - Kr).max():.3e}  "
        f"|J| {np.abs(Jr).max():.3e}")
    assert np.abs(J - Jr).max() <= 1e-11 * max(1.0, np.abs(Jr).max())
    assert np.abs(K - Kr).max() <= 1e-11 * max(1.0, np.abs(Kr).max())
    p.close()


@pytest.mark.parametrize("variant", range(capi.NVARIANTS))
def test_every_launch_variant(oracle, variant):
    """Every compiled launch shape (lanes per tuple, primitive tuples per
    step) of every class meets the same parity bar; classes with fewer
    variants fall back to their default."""
    mol = M.config(1)
    n = mol.nbas
    rng = np.random.default_rng(20 + variant)
    full = [(i, j, k, l) for l in range(n) for k in range(n) for j in range(n) for i in range(n)]
    check_plan(oracle, "int2e_sph", full, mol, variant)
    check_plan(oracle, "int2e_ip1_sph",
               [tuple(int(s) for s in rng.integers(0, n, 4)) for _ in range(1500)], mol, variant)
    aux = M.config(4)
    t3 = [(int(rng.integers(0, aux.aux_start)), int(rng.integers(0, aux.aux_start)),
           int(rng.integers(aux.aux_start, aux.nbas))) for _ in range(1500)]
    check_plan(oracle, "int3c2e_sph", t3, aux, variant)
    check_plan(oracle, "int3c2e_ip1_sph", t3[:700], aux, variant)
    check_plan(oracle, "int2e_cart", full[::7], mol, variant)
    check_plan(oracle, "int3c2e_cart", t3[:700], aux, variant)
    # FP32 instantiations: every tuple of a mixed plan with a huge threshold
    p = capi.Plan("int2e_sph", mol.atm, mol.bas, mol.env, full, precision=capi.PREC_MIXED,
                  mixed_threshold=1e300)
    assert p.ntuples_fp32 == p.ntuples
    p.set_variant(variant)
    p.execute()
    p.sync()
    got = p.output()
    ref, offs, sizes = oracle_blocks(oracle, "int2e_sph", full, mol)
    # FP32 rounding is relative to the terms summed, not to the (possibly
    # cancelled) result: bound it by the tuple's Schwarz factor
    # sqrt(max|(ij|ij)|) sqrt(max|(kl|kl)|)
    diag = [(i, j, i, j) for i in range(n) for j in range(n)]
    dref, doffs, dsizes = oracle_blocks(oracle, "int2e_sph", diag, mol)
    qf = np.sqrt([np.abs(dref[a:a + k]).max() for a, k in zip(doffs, dsizes)]).reshape(n, n)
    scale = np.repeat([qf[i, j] * qf[k, l] for i, j, k, l in full], sizes)
    err = np.abs(got - ref)
    ratio = err[scale > 0] / scale[scale > 0]
    # a pair whose (ij|ij) libcint's screen drops entirely (e^-cce beyond
    # the cutoff twice) can still meet a compact ket pair: its integrals are
    # then below e^-30 or so
    assert np.all(err[scale == 0] <= 1e-11)
    worst = np.argsort(err / np.maximum(scale, 1e-300))[-3:]
    say(f"  fp32 variant {variant}: max err {err.max():.3e}, err/Schwarz bound "
        f"max {ratio.max():.3e} p99.9 {np.quantile(ratio, 0.999):.3e}; worst "
        + ", ".join(f"{got[w]:.6e} vs {ref[w]:.6e} (bound {scale[w]:.2e})" for w in worst))
    # FP32 recurrences: rounding relative to the bound, amplified by the HRR
    # cancellation of distant pairs (measured up to ~3e-4 of the bound on this
    # basis); an indexing error would be O(1) here
    assert ratio.max() <= 1e-2
    assert np.quantile(ratio, 0.999) <= 1e-4
    p.close()


def test_mixed_plan_error_bound_cfg2(oracle):
    """The mixed path (FP32 recurrences for tuples whose Schwarz bound is
    below 1e-9) stays within 1e-10 absolute of the oracle."""
    mol = M.config(2)
    p = capi.Plan("int2e_sph", mol.atm, mol.bas, mol.env, screened=(1e-12, 97),
                  precision=capi.PREC_MIXED, mixed_threshold=1e-9)
    assert p.ntuples_fp32 > 0
    p.execute()
    p.sync()
    t, _ = p.tuples()
    rng = np.random.default_rng(11)
    first32 = p.ntuples - p.ntuples_fp32
    pick = np.sort(first32 + rng.choice(p.ntuples_fp32, size=min(3000, p.ntuples_fp32),
                                        replace=False))
    got, _, _ = p.output_tuples(pick)
    ref, _, _ = oracle.eval_list("int2e_sph", [tuple(int(v) for v in t[q]) for q in pick],
                                 mol.atm, mol.bas, mol.env, ext=True)
    err = float(np.abs(got - ref).max())
    say(f"  mixed cfg2: {p.ntuples_fp32}/{p.ntuples} tuples in FP32, max abs err {err:.3e}")
    assert err <= 1e-10
    p.close()


def test_mixed_plan_cfg3_256_atoms(oracle):
    """The 256-atom lattice (the headline molecule) in the mixed mode at the
    bench's thresholds, every 16384th bra pair: tuples sampled from the FP32
    and FP64 bins within 1e-10 of the judge, and the plan's J/K against the CPU
    J/K of the same unique quartets (every distinct 8-fold image added, an
    independent digestion)."""
    mol = M.config(3)
    p = capi.Plan("int2e_sph", mol.atm, mol.bas, mol.env, screened=(1e-12, 16384),
                  precision=capi.PREC_MIXED, mixed_threshold=1e-9)
    say(f"  cfg3 mixed: {p.ntuples} quartets, {p.ntuples_fp32} in FP32")
    assert p.ntuples_fp32 > 0
    p.execute()
    p.sync()
    t, _ = p.tuples()
    rng = np.random.default_rng(12)
    first32 = p.ntuples - p.ntuples_fp32
    pick = np.sort(np.concatenate([rng.choice(first32, size=min(1000, first32), replace=False),
                                   first32 + rng.choice(p.ntuples_fp32,
                                                        size=min(1000, p.ntuples_fp32),
                                                        replace=False)]))
    got, _, _ = p.output_tuples(pick)
    ref, _, _ = oracle.eval_list("int2e_sph", [tuple(int(v) for v in t[q]) for q in pick],
                                 mol.atm, mol.bas, mol.env, ext=True)
    err = float(np.abs(got - ref).max())
    say(f"  sampled max abs err vs judge {err:.3e}")
    assert err <= 1e-10
    nao = mol.nao()
    D = rng.normal(size=(nao, nao)) / nao
    D = D + D.T
    J, K = p.jk(D)
    Jc, Kc = oracle.cpu_baseline_jk(t, mol.atm, mol.bas, mol.env, D, nthreads=16)
    ej, ek = float(np.abs(J - Jc).max()), float(np.abs(K - Kc).max())
    say(f"  J/K vs CPU: {ej:.3e} {ek:.3e} (|J| {np.abs(Jc).max():.3e})")
    assert ej <= 1e-10 and ek <= 1e-10
    p.close()


def test_int3c2e_mixed_cfg4(oracle):
    """int3c2e_sph in the mixed mode on the 64-atom lattice with the
    6s5p4d3f1g auxiliary basis: a triple takes the FP32 recurrences when
    sqrt((ij|ij)) sqrt((P|P)) over the absolute coefficients is below 1e-9;
    every triple within 1e-10 of the judge."""
    mol = M.config(4)
    rng = np.random.default_rng(41)
    a0 = mol.aux_start
    tuples = [(int(rng.integers(0, a0)), int(rng.integers(0, a0)),
               int(rng.integers(a0, mol.nbas))) for _ in range(4000)]
    p = capi.Plan("int3c2e_sph", mol.atm, mol.bas, mol.env, tuples, precision=capi.PREC_MIXED,
                  mixed_threshold=1e-9)
    say(f"  int3c2e mixed: {p.ntuples_fp32} of {p.ntuples} triples in FP32")
    assert 0 < p.ntuples_fp32 < p.ntuples
    p.execute()
    p.sync()
    got = p.output()
    ref, _, _ = oracle.eval_list("int3c2e_sph", tuples, mol.atm, mol.bas, mol.env, ext=True)
    err = float(np.abs(got - ref).max())
    say(f"  max abs err vs judge {err:.3e}")
    assert err <= 1e-10
    p.close()


@pytest.mark.parametrize("kind", ["tight_diffuse_d", "contracted", "screened", "int3c2e"])
def test_mixed_plan_error_of_distant_pairs(oracle, kind):
    """Pairs of a tight and a distant diffuse shell, whose transfer cancels in
    FP32 (the error of a (d d|d d) quartet was up to 220 times its Schwarz
    bound): what a mixed plan puts in FP32 stays within a tenth of its
    threshold (1e-3 here, where an error of the order of the bound shows)."""
    rng = np.random.default_rng({"tight_diffuse_d": 1, "contracted": 2, "screened": 3,
                                 "int3c2e": 4}[kind])
    thr, nfp32, worst = 1e-3, 0, 0.0
    for _ in range(3):
        mol = M.Molecule()
        r = float(rng.uniform(3.0, 7.0))
        for x in (0.0, r):
            for _ in range(2):
                mol.add_atom(1, [x + 0.4 * rng.normal(), 0.4 * rng.normal(), 0.4 * rng.normal()])
        for a in range(4):
            for l in range(3):
                if kind == "tight_diffuse_d":
                    for lo, hi in ((200.0, 5000.0), (0.1, 1.5)):
                        e = float(np.exp(rng.uniform(np.log(lo), np.log(hi))))
                        mol.add_shell(a, l, [e], [[M.gto_norm(l, e)]])
                else:
                    n = int(rng.integers(1, 5))
                    e = np.sort(np.exp(rng.uniform(np.log(0.1), np.log(5000.0), n)))[::-1]
                    mol.add_shell(a, l, e, [[rng.normal() * M.gto_norm(l, v) for v in e]])
        mol.build()
        name = "int3c2e_sph" if kind == "int3c2e" else "int2e_sph"
        arity = 3 if kind == "int3c2e" else 4
        if kind == "screened":
            p = capi.Plan(name, mol.atm, mol.bas, mol.env, screened=(1e-9, 1),
                          precision=capi.PREC_MIXED, mixed_threshold=thr)
        else:
            ls = mol.bas[:, 1]
            d = np.nonzero(ls == 2)[0] if kind == "tight_diffuse_d" else np.nonzero(ls >= 1)[0]
            tuples = [tuple(int(s) for s in rng.choice(d, arity)) for _ in range(1500)]
            p = capi.Plan(name, mol.atm, mol.bas, mol.env, tuples, precision=capi.PREC_MIXED,
                          mixed_threshold=thr)
        p.execute()
        p.sync()
        got = p.output()
        t, _ = p.tuples()
        ref, _, _ = oracle.eval_list(name, [tuple(int(v) for v in q[:arity]) for q in t], mol.atm,
                                     mol.bas, mol.env, ext=True)
        nfp32 += p.ntuples_fp32
        worst = max(worst, float(np.abs(got - ref).max()))
        p.close()
    say(f"  {kind}: {nfp32} tuples in FP32, max abs err {worst:.3e}")
    assert nfp32 > 0
    assert worst <= thr / 10


def test_autotune_keeps_results(oracle):
    mol = M.config(1)
    n = mol.nbas
    tuples = [(i, j, k, l) for i in range(n) for j in range(i + 1) for k in range(n)
              for l in range(k + 1)]
    p = capi.Plan("int2e_sph", mol.atm, mol.bas, mol.env, tuples)
    p.execute()
    p.sync()
    before = p.output()
    p.autotune(reps=2)
    info = p.bin_variants()
    say("  variants " + " ".join(f"{b['variant']}/{b['nvariants']}:T{b['lanes']}P{b['prims']}"
                                 for b in info))
    assert all(0 <= b["variant"] < b["nvariants"] for b in info)
    p.fill_output(np.nan)
    p.execute(graph=True)
    p.sync()
    after = p.output()
    scale = np.abs(before).max()
    assert np.abs(after - before).max() <= 1e-13 * scale
    p.close()


def test_mixed_jk_with_runtime_class_bins(oracle):
    """J/K of a mixed plan whose bins digest in fused kernels and from blocks
    of the runtime-class kernel, against the CPU J/K of the same quartets."""
    rng = M.SplitMix64(5)
    mol = M.Molecule()
    atoms = [mol.add_atom(8, r) for r in M._lattice(rng, 2, 2, 2, 2.8, 0.3)]
    M._orbital_basis(mol, rng, atoms, [True] * len(atoms), 0.1, 5000.0)
    mol.build()
    p = capi.Plan("int2e_sph", mol.atm, mol.bas, mol.env, screened=(1e-12, 4),
                  precision=capi.PREC_MIXED, mixed_threshold=1e-9)
    kinds = {(b["precision"], b["generic"]) for b in p.bin_stats()}
    say(f"  {p.ntuples} quartets, {p.ntuples_fp32} in FP32, bins {sorted(kinds)}")
    assert p.ntuples_fp32 > 0 and {True, False} == {g for _, g in kinds}
    nao = mol.nao()
    D = np.random.default_rng(8).normal(size=(nao, nao)) / nao
    D = D + D.T
    t, _ = p.tuples()
    Jc, Kc = oracle.cpu_baseline_jk(t, mol.atm, mol.bas, mol.env, D, nthreads=16)
    for _ in range(2):
        J, K = p.jk(D)
        ej, ek = float(np.abs(J - Jc).max()), float(np.abs(K - Kc).max())
        say(f"  J/K vs CPU: {ej:.3e} {ek:.3e} (|J| {np.abs(Jc).max():.3e})")
        assert ej <= 1e-10 and ek <= 1e-10
    p.close()


def _two_site_shells(l, nprim, r):
    """One shell of momentum l with nprim primitives on each of two sites."""
    mol = M.Molecule()
    for x in (0.0, r):
        a = mol.add_atom(1, (x, 0.1 * x, 0.0))
        e = [0.7 * 1.2 ** k for k in range(nprim)]
        mol.add_shell(a, l, e, [[M.gto_norm(l, v) for v in e]])
    return mol.build()


def test_bin_variants_report_the_runtime_class_kernel():
    """The primitive tuples of a step of the runtime-class kernel: several
    where the tuples have several and their g tensors fit, never more than
    the tuples have."""
    for nprim, want in ((1, (1, 1)), (2, (2, 16)), (4, (2, 16))):
        mol = _two_site_shells(3, nprim, 1.0)
        p = capi.Plan("int2e_ip1_sph", mol.atm, mol.bas, mol.env, [(0, 1, 0, 1), (1, 0, 1, 1)])
        for b, v in zip(p.bin_stats(), p.bin_variants()):
            assert b["generic"] and v["variant"] == -1 and v["lanes"] == 256
            assert want[0] <= v["prims"] <= want[1], (nprim, v)
        p.close()


def test_runtime_class_blocks_finish_several_slabs_at_a_time(oracle):
    """Blocks finished by the workgroup that made them, with one slab, with
    all slabs in one pass and with a remainder; and nabla_i (s s|g g), 15
    slabs, in about the time of (g g|s s), one slab of as many elements (it
    took 3.3 times as long slab by slab; 2 at most)."""
    mol = M.Molecule()
    for r in ((0, 0, 0), (0.9, 0.3, 0)):
        a = mol.add_atom(1, r)
        for l in range(5):
            e = 0.5 + 0.2 * l
            mol.add_shell(a, l, [e], [[M.gto_norm(l, e)]])
    mol.build()
    for ls in ((4, 4, 0, 0), (0, 0, 4, 4), (2, 4, 1, 4), (2, 4, 4, 3), (4, 3, 4, 4), (0, 4, 2, 2)):
        t = (ls[0], ls[1] + 5, ls[2], ls[3] + 5)
        check_plan(oracle, "int2e_ip1_sph", [t, t], mol)

    def best(ls):
        p = capi.Plan("int2e_ip1_sph", mol.atm, mol.bas, mol.env,
                      [(ls[0], ls[1] + 5, ls[2], ls[3] + 5)] * 5000)
        ms = []
        for _ in range(8):
            assert capi.lib().cintx_plan_execute_timed(p.h, None) == 0
            ms.append(p.bin_stats()[0]["ms"])
        p.close()
        return min(ms)

    many, one = best((0, 0, 4, 4)), best((4, 4, 0, 0))
    say(f"  15 slabs {many:.3f} ms, one slab {one:.3f} ms")
    assert many <= 2 * one


def test_default_shape_of_short_lists(oracle):
    """Short lists of short contracted tuples of classes whose wide kernels
    would keep one lane busy, or of few registers, run the one-lane kernel;
    uncontracted pairs of several rows the wide one."""
    mol = M.Molecule()
    rng = np.random.default_rng(17)
    for r in ((0, 0, 0), (1.0, 0.3, 0.2)):
        a = mol.add_atom(1, r)
        for l in range(3):
            e = [4.0, 1.1, 0.4]
            mol.add_shell(a, l, e, [[rng.normal() * M.gto_norm(l, v) for v in e]])
            mol.add_shell(a, l, [0.7], [[M.gto_norm(l, 0.7)]])
    mol.build()
    s, p, d, p1, d1 = 0, 2, 4, 3, 5  # contracted s, p, d; uncontracted p, d
    for name, t, one in (("int3c2e_sph", (d, d + 6, s), True),
                         ("int3c2e_sph", (p, s + 6, d), True),
                         ("int2c2e_sph", (p1, d1), False)):
        plan = capi.Plan(name, mol.atm, mol.bas, mol.env, [t] * 100)
        assert (plan.bin_variants()[0]["lanes"] == 1) == one, (name, t)
        plan.close()
        check_plan(oracle, name, [t] * 3, mol)


def test_list_of_one_class_has_the_lines_of_a_launch_alone(oracle):
    """240 nabla_i (s d|d d) tuples of 54 to 81 primitive tuples, 13,000 to
    19,440 in all: the compiled kernel when the list has no other class, the
    runtime-class kernel beside another."""
    mol = M.Molecule()
    for r in ((0, 0, 0), (0.8, 0.3, 0.2)):
        a = mol.add_atom(1, r)
        for l in (0, 2):
            e = [2.0, 0.9, 0.4]
            mol.add_shell(a, l, e, [[M.gto_norm(l, v) for v in e]])
    mol.build()
    t = [(0, 1, 3, 1), (2, 3, 1, 3), (0, 3, 1, 1)] * 80
    for tuples, generic in ((t, False), (t + [(0, 0, 0, 2)], True)):
        p = capi.Plan("int2e_ip1_sph", mol.atm, mol.bas, mol.env, tuples)
        got = {b["class"]: b["generic"] for b in p.bin_stats()}
        p.close()
        assert got[(0, 2, 2, 2)] == generic, got
    check_plan(oracle, "int2e_ip1_sph", t, mol)


def test_three_row_chunks_leave_long_tuples_to_the_wide_kernel(oracle):
    """nabla_i (p d|d s), whose one-lane kernel works in three row chunks:
    1,200 tuples of 54 or 81 primitive tuples run the wide kernel, (p p|d s),
    of two chunks, the one-lane kernel."""
    mol = M.Molecule()
    for r in ((0, 0, 0), (0.8, 0.3, 0.2)):
        a = mol.add_atom(1, r)
        for l in range(3):
            e = [2.0, 0.9, 0.4]
            mol.add_shell(a, l, e, [[M.gto_norm(l, v) for v in e]])
    mol.build()
    s, p, d = 0, 1, 2
    for j, one in ((d, False), (p, True)):
        t = [(p, j + 3, d, s), (p + 3, j, d, s + 3), (p, j, d + 3, s)] * 400
        plan = capi.Plan("int2e_ip1_sph", mol.atm, mol.bas, mol.env, t)
        assert plan.nbins == 1 and not plan.bin_stats()[0]["generic"]
        assert (plan.bin_variants()[0]["lanes"] == 1) == one, j
        plan.close()
        check_plan(oracle, "int2e_ip1_sph", t[:60], mol)


def test_autotuned_shapes_stay_with_their_size():
    """Autotuning a long list of a class leaves the launch shapes of a short
    list of long tuples of that class as they are."""
    mol = M.Molecule()
    for r in ((0, 0, 0), (1.1, 0.2, 0), (0.1, 1.3, 0.4)):
        a = mol.add_atom(1, r)
        for e in ([3.0, 0.9, 0.3], [1.4, 0.5]):
            mol.add_shell(a, 2, e, [[M.gto_norm(2, v) for v in e]])
    mol.build()
    rng = np.random.default_rng(3)

    def plan(shells, count):
        return capi.Plan("int2e_sph", mol.atm, mol.bas, mol.env,
                         [tuple(int(s) for s in rng.choice(shells, 4)) for _ in range(count)])

    def shapes():  # 3 tuples of 81 primitive tuples
        p = plan([0, 2, 4], 3)
        got = [(b["generic"], v["variant"], v["lanes"], v["prims"])
               for b, v in zip(p.bin_stats(), p.bin_variants())]
        p.close()
        return got

    before = shapes()
    p = plan([1, 3, 5], 6000)  # of 16 each
    p.autotune(reps=1)
    say(f"  short list {before}, long list {p.bin_variants()}")
    p.close()
    assert shapes() == before


@pytest.mark.parametrize("variant", range(capi.NVARIANTS))
def test_work_counters_match_oracle_model(oracle, variant):
    """The device work counters (surviving primitive tuples after libcint's
    screen, algorithmic FLOPs) equal the oracle's count for every launch
    shape."""
    mol = M.config(1)
    n = mol.nbas
    tuples = [(i, j, k, l) for i in range(n) for j in range(i + 1) for k in range(n)
              for l in range(k + 1)]
    p = capi.Plan("int2e_sph", mol.atm, mol.bas, mol.env, tuples)
    p.set_variant(variant)
    prim, roots, flops = p.work()
    ref = np.sum([oracle.work_model("int2e_sph", t, mol.atm, mol.bas, mol.env) for t in tuples],
                 axis=0)
    say(f"  variant {variant}: prim {prim:.0f} vs {ref[0]:.0f}, flops {flops:.4e} vs {ref[2]:.4e}")
    assert prim == ref[0]
    assert roots == ref[1]
    # the device transforms cart->sph in the canonical shell order of its
    # class, the oracle in the caller's: the c2s FLOPs differ by the axis order
    assert abs(flops - ref[2]) <= 1e-3 * ref[2]
    p.close()


@pytest.mark.parametrize("count", [1, 3, 65, 700])
def test_lanes_shared_by_a_tuple(oracle, count):
    """Lists of few and many long contractions, whose tuples take 64 and fewer
    lanes of the one-lane kernels: odd counts (the last wavefront partly
    filled), screened-out tuples among them, every output form, and the J/K
    build that digests split tuples."""
    mol = M.config(2)
    rng = np.random.default_rng(90 + count)
    prims = mol.bas[:, 2]
    long = np.nonzero(prims >= 4)[0]
    assert set(int(v) for v in mol.bas[long, 1]) == {0, 1, 2}
    pick = [tuple(int(s) for s in rng.choice(long, 4)) for _ in range(count)]
    near = [(t[0], t[0], t[2], t[2]) for t in pick]  # nothing screened: up to 1296 of them
    for name in ("int2e_sph", "int2e_cart", "int2e_ip1_sph"):
        check_plan(oracle, name, pick + near, mol)
    if count == 65:
        small = M.config(1)
        p = capi.Plan("int2e_sph", small.atm, small.bas, small.env, screened=(0.0, 1))
        n = small.nao()
        D = rng.normal(size=(n, n))
        D = D + D.T
        J, K = p.jk(D)
        shells = range(small.nbas)
        full = [(i, j, k, l) for l in shells for k in shells for j in shells for i in shells]
        ref, offs, _ = oracle_blocks(oracle, "int2e_sph", full, small)
        width = 2 * small.bas[:, 1] + 1
        off = np.cumsum(width) - width
        eri = np.zeros((n, n, n, n))
        for t, o in zip(full, offs):
            w = [int(width[s]) for s in t]
            sl = tuple(slice(int(off[s]), int(off[s]) + v) for s, v in zip(t, w))
            eri[sl] = ref[o:o + int(np.prod(w))].reshape(w[::-1]).transpose(3, 2, 1, 0)
        Jr = np.einsum("pqrs,rs->pq", eri, D)
        Kr = np.einsum("pqrs,qs->pr", eri, D)
        # each of the n^2 terms of an element is within 1e-12 (1 + |eri|)
        tol = 1e-12 * (1 + np.abs(eri).max()) * np.abs(D).sum()
        assert np.abs(J - Jr).max() <= tol and np.abs(K - Kr).max() <= tol
        p.close()


@pytest.mark.parametrize("count", [1, 255, 257])
def test_one_primitive_tuple_per_lane(oracle, count):
    """Lists of uncontracted shells, whose one-lane kernels read the Rys table
    from memory: every output form, 1 to 3 roots and more, arguments from 0
    to beyond the table, a last workgroup of one lane; and beside contracted
    shells on the other side of the rule."""
    mol = M.Molecule()
    rng = np.random.default_rng(60 + count)
    for r in ((0, 0, 0), (0.7, 0.2, 0.1), (0.3, 9.0, 2.0)):
        a = mol.add_atom(1, r)
        for l in range(3):
            for e in (0.3, 1.7, 900.0):
                mol.add_shell(a, l, [e], [[M.gto_norm(l, e)]])
    contracted = mol.add_atom(1, (1.0, 0.4, 0.3))
    for l in range(2):
        e = [20.0, 4.0, 1.0, 0.4]
        mol.add_shell(contracted, l, e, [[M.gto_norm(l, v) for v in e]])
    mol.build()
    n = 27
    one = [s for s in range(n) if mol.bas[s, 1] < 2]
    t4 = [tuple(int(v) for v in rng.choice(one, 4)) for _ in range(count)]
    t3 = [tuple(int(v) for v in rng.integers(0, n, 3)) for _ in range(count)]
    t2 = [t[:2] for t in t3]
    for name, t in (("int2e_sph", t4), ("int2e_cart", t4), ("int2e_ip1_sph", t4),
                    ("int3c2e_sph", t3), ("int3c2e_ip1_sph", t3), ("int2c2e_sph", t2),
                    ("int2e_sph", t4 + [(n, n + 1, n, n)] * 40)):
        check_plan(oracle, name, t, mol)


@pytest.mark.parametrize("count", [1, 7, 300])
def test_small_launches_of_the_runtime_class_kernel(oracle, count):
    """Classes with compiled kernels whose small launches take the
    runtime-class kernel, a tuple on several workgroups: one tuple, odd
    counts, blocks of one and of several row chunks, tuples without a
    surviving primitive tuple among them, and the nabla_i and Cartesian
    forms; the same as a graph."""
    mol = M.config(5)
    rng = np.random.default_rng(120 + count)
    ls = mol.bas[:, 1]
    long = np.nonzero(mol.bas[:, 2] >= 3)[0]
    by_l = {l: [int(s) for s in long if ls[s] == l] for l in range(5)}
    pairs = [(2, 2, 2, 2), (2, 2, 2, 1), (4, 4, 1, 0), (3, 1, 2, 2), (4, 2, 3, 1)]
    tuples = []
    for cls in pairs:
        for _ in range(max(1, count // len(pairs))):
            a = [by_l[l][int(rng.integers(0, 3))] for l in cls]  # near: little is screened
            tuples.append(tuple(a))
    far = (by_l[2][0], by_l[2][-1], by_l[2][1], by_l[2][-2])
    tuples.append(far)
    p = capi.Plan("int2e_sph", mol.atm, mol.bas, mol.env, tuples)
    assert any(b["generic"] for b in p.bin_stats())
    p.execute(graph=True)
    p.sync()
    p.fill_output(np.nan)
    p.execute(graph=True)
    p.sync()
    ref, _, _ = oracle_blocks(oracle, "int2e_sph", tuples, mol)
    assert_parity(p.output(), ref)
    p.close()
    check_plan(oracle, "int2e_sph", tuples, mol)
    check_plan(oracle, "int2e_ip1_sph", tuples[:40], mol)
    check_plan(oracle, "int2e_cart", tuples[:40], mol)


def test_wide_shapes_list_tuples_by_primitive_counts():
    """nabla_i (p p|p p) tuples of 36 surviving primitive tuples each, 36 x 1
    and 1 x 36 of them in turn.  A wide shape loops to the largest counts of
    its workgroup's tuples, so a workgroup of both kinds runs 1296 steps
    instead of 36: the mixed list has to take about as long as both halves
    (three times as long at most)."""
    mol = M.Molecule()
    at = [mol.add_atom(1, r) for r in ((0, 0, 0), (0.3, 0.2, 0), (0, 0.4, 0.1), (0.2, 0, 0.3))]
    for a in at:
        for e in ([0.3, 0.4, 0.5, 0.7, 0.9, 1.2], [0.6]):
            mol.add_shell(a, 1, e, [[M.gto_norm(1, v) for v in e]])
    mol.build()
    long, short = [0, 2, 4, 6], [1, 3, 5, 7]
    rng = np.random.default_rng(7)
    halves = [[(*(int(v) for v in rng.choice(b, 2)), *(int(v) for v in rng.choice(k, 2)))
               for _ in range(8000)] for b, k in ((long, short), (short, long))]

    def best(tuples, v):
        p = capi.Plan("int2e_ip1_sph", mol.atm, mol.bas, mol.env, tuples)
        p.set_variant(v)
        lanes = p.bin_variants()[0]["lanes"]
        ms = []
        for _ in range(6):
            assert capi.lib().cintx_plan_execute_timed(p.h, None) == 0
            ms.append(p.bin_stats()[0]["ms"])
        p.close()
        return lanes, min(ms)

    seen = 0
    for v in range(capi.NVARIANTS):
        lanes, mixed = best([t for pair in zip(*halves) for t in pair], v)
        if lanes == 1:
            continue
        seen += 1
        parts = [best(h, v)[1] for h in halves]
        say(f"  {lanes} lanes: {mixed:.3f} ms, halves {parts[0]:.3f} + {parts[1]:.3f}")
        assert mixed <= 3 * sum(parts)
    assert seen >= 2
