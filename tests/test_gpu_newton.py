"""GPU parity of the HIP Newton-step path against the CPU oracle, through the
C ABI (libsgipc.so).  Inputs are the seeded synthetic cube scenes."""
import ctypes as C

import numpy as np
import pytest

from conftest import oracle_system, dense_from_bcoo

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch


def make_system(sc, precond=None):
    from sgipc import capi
    from sgipc.system import NewtonSystem
    return NewtonSystem(sc, "cuda:0", precond=capi.PRECOND_MAS if precond is None else precond)


@pytest.mark.parametrize("name", ["cube4", "cube10"])
def test_fem_assembly_matches_oracle(torch_cuda, oracle, request, name):
    sc = request.getfixturevalue(name)
    print("case: fem assembly", name, "n", sc.n, "T", sc.T, flush=True)
    ref = oracle_system(oracle, sc)
    sys_ = make_system(sc)
    sys_.assemble()
    R, Cc, V = sys_.triplets()
    Ro, Co, Vo = ref["trip"]
    assert np.array_equal(R, Ro) and np.array_equal(Cc, Co)          # bit-exact indices
    scale = np.abs(Vo).max()
    assert np.abs(V - Vo).max() <= 1e-12 * scale                      # FP64 values
    g = sys_.shape.cpu().numpy().reshape(-1, 3)
    assert np.abs(g - ref["shape"]).max() <= 1e-12 * np.abs(ref["shape"]).max()
    b = sys_.b.cpu().numpy()
    assert np.abs(b - ref["b"]).max() <= 1e-12 * np.abs(ref["b"]).max()


@pytest.mark.parametrize("name", ["cube4", "cube10"])
def test_convert_matches_oracle(torch_cuda, oracle, request, name):
    sc = request.getfixturevalue(name)
    print("case: convert", name, flush=True)
    ref = oracle_system(oracle, sc)
    sys_ = make_system(sc)
    sys_.assemble()
    K = sys_.convert()
    kr, kc, kv = sys_.bcoo()
    orow, ocol, oval = ref["bcoo"]
    assert K == len(orow)
    assert np.array_equal(kr, orow) and np.array_equal(kc, ocol)     # bit-exact BCOO index set and order
    assert np.abs(kv - oval).max() <= 1e-12 * np.abs(oval).max()


def test_convert_on_oracle_triplets_is_bitexact(torch_cuda, oracle, cube4):
    """Fed the oracle's own triplets, the GPU convert reproduces the oracle's
    BCOO bit for bit (same per-block summation order)."""
    import torch
    print("case: convert bit-exact on oracle triplets", flush=True)
    ref = oracle_system(oracle, cube4)
    sys_ = make_system(cube4)
    R, Cc, V = ref["trip"]
    nt = len(R)
    sys_.tr[:nt] = torch.tensor(R, dtype=torch.int32, device=sys_.dev)
    sys_.tc[:nt] = torch.tensor(Cc, dtype=torch.int32, device=sys_.dev)
    sys_.tv[:9 * nt] = torch.tensor(V.reshape(-1), dtype=torch.float64, device=sys_.dev)
    sys_.nt = nt
    sys_.convert()
    kr, kc, kv = sys_.bcoo()
    orow, ocol, oval = ref["bcoo"]
    assert np.array_equal(kr, orow) and np.array_equal(kc, ocol)
    assert np.array_equal(kv, oval)


def test_spmv_matches_dense(torch_cuda, oracle, cube10):
    print("case: spmv cube10", flush=True)
    sys_ = make_system(cube10)
    sys_.assemble(); sys_.convert()
    kr, kc, kv = sys_.bcoo()
    A = dense_from_bcoo(kr, kc, kv, cube10.n)
    rng = np.random.default_rng(3)
    x = rng.normal(size=3 * cube10.n); y0 = rng.normal(size=3 * cube10.n)
    y = sys_.spmv(x, a=0.7, b=-0.3, y=y0)
    ref = 0.7 * A @ x - 0.3 * y0
    assert np.abs(y - ref).max() <= 1e-12 * np.abs(ref).max()


def test_mas_tables_bitexact(torch_cuda, oracle, cube10):
    print("case: mas tables cube10", flush=True)
    ref = oracle_system(oracle, cube10)
    sys_ = make_system(cube10)
    sys_.assemble(); sys_.convert(); sys_.build_precond()
    t = sys_.mas_tables()
    kr, kc, kv = ref["bcoo"]
    mas = oracle.Mas(cube10.n, sys_.part_map, sys_.real_map, sys_.ns, sys_.nn, sys_.nl, cube10.bank)
    tot = mas.build(kr, kc, kv)
    to = mas.tables()
    assert t["levelnum"] == mas.levelnum and t["total"] == tot
    assert np.array_equal(t["level_size"], to["level_size"])
    assert np.array_equal(t["coarse_space"], to["coarse_space"])
    assert np.array_equal(t["coarse_table"][:, :mas.levelnum - 1], to["coarse_table"][:, :mas.levelnum - 1])
    assert np.array_equal(t["fine_mask"], to["fine_mask"])
    assert np.array_equal(t["prefix0"], to["prefix0"])


@pytest.mark.parametrize("fp32", [False, True])
def test_mas_apply_matches_oracle(torch_cuda, oracle, cube10, fp32):
    from sgipc import capi
    print("case: mas apply fp32=%s" % fp32, flush=True)
    ref = oracle_system(oracle, cube10)
    sys_ = make_system(cube10, capi.PRECOND_MAS_FP32 if fp32 else capi.PRECOND_MAS)
    sys_.assemble(); sys_.convert(); sys_.build_precond()
    kr, kc, kv = ref["bcoo"]
    mas = oracle.Mas(cube10.n, sys_.part_map, sys_.real_map, sys_.ns, sys_.nn, sys_.nl, cube10.bank)
    mas.build(kr, kc, kv)
    r = np.random.default_rng(5).normal(size=3 * cube10.n)
    z = sys_.precond_apply(r)
    zo = mas.apply(r, fp32=False)
    tol = 1e-5 if fp32 else 1e-11
    assert np.abs(z - zo).max() <= tol * np.abs(zo).max()
    b0 = sys_.bank_inverse(0)
    _, Ainv = mas.bank_matrix(0)
    assert np.abs(b0 - Ainv).max() <= 1e-10 * np.abs(Ainv).max()


@pytest.mark.parametrize("precond", [0, 1, 2])
def test_pcg_matches_oracle(torch_cuda, oracle, cube10, precond):
    print("case: pcg precond=%d" % precond, flush=True)
    ref = oracle_system(oracle, cube10)
    sys_ = make_system(cube10, precond)
    sys_.assemble(); sys_.convert(); sys_.build_precond()
    kr, kc, kv = ref["bcoo"]
    mas = None
    if precond == 2:
        mas = oracle.Mas(cube10.n, sys_.part_map, sys_.real_map, sys_.ns, sys_.nn, sys_.nl, cube10.bank)
        mas.build(kr, kc, kv)
    # reference stopping rule: identical iteration count, direction within 1e-10
    st = sys_.solve(tol=1e-4, stop_rule=0)
    xo, ito, _ = oracle.pcg(kr, kc, kv, cube10.n, ref["b"], precond=precond, mas=mas, tol=1e-4, rule=0)
    x = sys_.dx.cpu().numpy()
    assert st.iterations == ito
    assert np.linalg.norm(x - xo) <= 1e-10 * np.linalg.norm(xo)
    # true relative residual 1e-6 against a direct solve
    st = sys_.solve(tol=1e-6, stop_rule=1, max_iter=5000)
    x = sys_.dx.cpu().numpy()
    A = dense_from_bcoo(kr, kc, kv, cube10.n)
    xs = np.linalg.solve(A, ref["b"])
    assert st.converged and st.rel_residual <= 1.5e-6
    assert np.linalg.norm(A @ x - ref["b"]) <= 1.5e-6 * np.linalg.norm(ref["b"])
    assert np.linalg.norm(x - xs) <= 1e-3 * np.linalg.norm(xs)


@pytest.mark.parametrize("budget", [6, 7, 1, 2])
def test_pcg_iteration_budget_matches_oracle(torch_cuda, oracle, cube10, budget):
    # an unreachable tolerance: both stop at the budget with the same iterate
    # (graphs hold two iterations: odd budgets stop inside one; a budget of
    # one runs no iteration)
    print("case: pcg budget max_iter=%d" % budget, flush=True)
    ref = oracle_system(oracle, cube10)
    sys_ = make_system(cube10)
    sys_.assemble(); sys_.convert(); sys_.build_precond()
    kr, kc, kv = ref["bcoo"]
    mas = oracle.Mas(cube10.n, sys_.part_map, sys_.real_map, sys_.ns, sys_.nn, sys_.nl, cube10.bank)
    mas.build(kr, kc, kv)
    st = sys_.solve(tol=1e-30, stop_rule=0, max_iter=budget)
    xo, ito, _ = oracle.pcg(kr, kc, kv, cube10.n, ref["b"], precond=2, mas=mas, tol=1e-30, rule=0, max_iter=budget)
    assert st.iterations == ito and not st.converged
    x = sys_.dx.cpu().numpy()
    assert np.linalg.norm(x - xo) <= 1e-10 * max(np.linalg.norm(xo), 1e-300)


def test_pcg_graph_replays_match_eager(torch_cuda, cube10):
    # captured iteration graphs (profiling off) against the eager launch
    # sequence (profiling on), replayed over several solves with other
    # device work in between; results must be bit-identical
    import torch
    from sgipc import capi
    print("case: pcg graph replay vs eager", flush=True)
    sys_ = make_system(cube10)
    sys_.assemble(); sys_.convert(); sys_.build_precond()
    b0 = sys_.b.clone()
    xs = []
    for rep in range(3):
        sys_.b.copy_(b0 * (1.0 + rep))
        st = sys_.solve(tol=1e-6, stop_rule=1, max_iter=5000)
        xs.append((st.iterations, sys_.dx.clone()))
        torch.cuda.synchronize()
        _ = (sys_.b * 2.0).sum().item()  # unrelated eager work between replays
    sys_.ctx.call("sgipc_profile_enable", 1)
    try:
        for rep in range(3):
            sys_.b.copy_(b0 * (1.0 + rep))
            st = sys_.solve(tol=1e-6, stop_rule=1, max_iter=5000)
            it, xg = xs[rep]
            assert st.iterations == it
            assert torch.equal(sys_.dx, xg)
    finally:
        sys_.ctx.call("sgipc_profile_enable", 0)
    sys_.b.copy_(b0)


@pytest.mark.parametrize("mode", ["mas_fp32", "mixed_mas", "mixed_diag", "mixed_none"])
def test_reduced_precision_solves(torch_cuda, oracle, cube10, mode):
    # FP32 preconditioner storage and the mixed FP32/FP64 solve reach the
    # same FP64 true relative residual as the FP64 solve
    from sgipc import capi
    print("case: reduced precision %s" % mode, flush=True)
    ref = oracle_system(oracle, cube10)
    kind = {"mas_fp32": capi.PRECOND_MAS_FP32, "mixed_mas": capi.PRECOND_MAS, "mixed_diag": capi.PRECOND_DIAG,
            "mixed_none": capi.PRECOND_NONE}[mode]
    prec = capi.PRECISION_FP64 if mode == "mas_fp32" else capi.PRECISION_MIXED
    sys_ = make_system(cube10, kind)
    sys_.assemble(); sys_.convert(); sys_.build_precond()
    kr, kc, kv = ref["bcoo"]
    A = dense_from_bcoo(kr, kc, kv, cube10.n)
    xs = np.linalg.solve(A, ref["b"])
    st64 = sys_.solve(tol=1e-6, stop_rule=1, max_iter=20000)
    st = sys_.solve(tol=1e-6, stop_rule=1, max_iter=20000, precision=prec)
    x = sys_.dx.cpu().numpy()
    assert st.converged and st.rel_residual <= 1e-6
    assert np.linalg.norm(A @ x - ref["b"]) <= 1.5e-6 * np.linalg.norm(ref["b"])
    assert np.linalg.norm(x - xs) <= 1e-3 * np.linalg.norm(xs)
    # reduced precision costs at most a modest number of extra iterations
    assert st.iterations <= 1.5 * st64.iterations + 10
    if prec == capi.PRECISION_MIXED:
        assert st.refinements >= 1


def test_convert_long_rows_bitexact(torch_cuda, oracle, cube4):
    """Rows of every length class (one wavefront up to 256 triplets, one
    workgroup's bitonic sort up to 4096, and the device radix-sort path above
    that, which the rows of affine bodies reach), at and either side of each
    class boundary, convert bit for bit as the oracle does."""
    import torch
    print("case: convert long rows", flush=True)
    rng = np.random.default_rng(21)
    n = cube4.n
    lens = {0: 9000, 1: 5000, 2: 3000, 3: 200, 4: 257, 5: 4096, 6: 256}
    R, Cc = [], []
    for r, L in lens.items():
        R.append(np.full(L, r)); Cc.append(rng.integers(r, n, L))
    for r in range(len(lens), n):
        L = int(rng.integers(0, 12))
        R.append(np.full(L, r)); Cc.append(rng.integers(r, n, L))
    R = np.concatenate(R).astype(np.int32); Cc = np.concatenate(Cc).astype(np.int32)
    perm = rng.permutation(len(R))                     # rows interleaved in the store
    R, Cc = R[perm], Cc[perm]
    V = rng.normal(size=(len(R), 9))
    sys_ = make_system(cube4)
    nt = len(R)
    sys_._set_capacity(nt)
    sys_.tr[:nt] = torch.tensor(R, dtype=torch.int32, device=sys_.dev)
    sys_.tc[:nt] = torch.tensor(Cc, dtype=torch.int32, device=sys_.dev)
    sys_.tv[:9 * nt] = torch.tensor(V.reshape(-1), dtype=torch.float64, device=sys_.dev)
    sys_.nt = nt
    K = sys_.convert()
    kr, kc, kv = sys_.bcoo()
    orow, ocol, oval = oracle.convert(R, Cc, V)
    assert K == len(orow)
    assert np.array_equal(kr, orow) and np.array_equal(kc, ocol)
    assert np.array_equal(kv, oval)


@pytest.mark.parametrize("mode", ["fp64", "fp32_apply", "mixed", "diag"])
def test_zero_rhs_returns_zero(torch_cuda, cube10, mode):
    """A zero right-hand side stops the loop before its first iteration (the
    device sees rz0 = 0 itself): x = 0, no iterations, converged, and a
    following solve of a real right-hand side is unaffected."""
    from sgipc import capi
    print("case: zero rhs", mode, flush=True)
    kind = {"fp64": capi.PRECOND_MAS, "fp32_apply": capi.PRECOND_MAS_FP32, "mixed": capi.PRECOND_MAS,
            "diag": capi.PRECOND_DIAG}[mode]
    prec = capi.PRECISION_MIXED if mode == "mixed" else capi.PRECISION_FP64
    sys_ = make_system(cube10, kind)
    sys_.assemble(); sys_.convert(); sys_.build_precond()
    b0 = sys_.b.clone()
    ref = sys_.solve(tol=1e-6, stop_rule=1, max_iter=5000, precision=prec)
    x_ref = sys_.dx.clone()
    sys_.dx.fill_(1.0)
    sys_.b.zero_()
    st = sys_.solve(tol=1e-6, stop_rule=1, max_iter=5000, precision=prec)
    assert st.iterations == 0 and st.converged and st.rz0 == 0.0
    assert not torch_cuda.any(sys_.dx != 0)
    sys_.b.copy_(b0)
    st2 = sys_.solve(tol=1e-6, stop_rule=1, max_iter=5000, precision=prec)
    assert st2.converged and st2.iterations == ref.iterations
    assert torch_cuda.equal(sys_.dx, x_ref)


@pytest.mark.parametrize("cells,hub,mixed", [(1, 7, False), (3, 60, False), (4, 100, True), (10, 1300, False),
                                             (10, 1300, True), (16, 4500, True), (16, 4500, False)])
def test_solve_with_rows_of_thousands_of_entries(torch_cuda, cells, hub, mixed):
    """The SpMV by entries: rows that cross chunk groups of 64 entries and LDS
    batches of 1024, next to rows with only their diagonal, in systems of one
    chunk and of many.  A strictly diagonally dominant arrow matrix (dominance
    2, so the error is at most about the relative residual): solved to 1e-9
    (FP64) or 1e-6 (FP32 inner solves), compared at ten times that."""
    import scipy.sparse as sp
    import scipy.sparse.linalg as spla
    from sgipc import capi, scene
    print("case: arrow matrix", cells, hub, mixed, flush=True)
    sc = scene.cube_scene(cells, seed=2)
    s = make_system(sc, capi.PRECOND_MAS_FP32 if mixed else capi.PRECOND_MAS)
    s.assemble()
    n, rng = sc.n, np.random.default_rng(cells)
    nt = 10 * s.T + s.n
    hubs = [0, n // 2] if n > 100 else [0]                     # rows with `hub` couplings each
    off = {}
    for h in hubs:
        for v in rng.choice(n, size=min(hub, n - 1), replace=False):
            if v != h and len(off) < nt - n:
                off[(min(h, v), max(h, v))] = 0.5 * rng.normal(size=(3, 3)) / 3
    A = sp.lil_matrix((3 * n, 3 * n))
    sums = np.zeros(n)
    for (i, j), M in off.items():
        A[3 * i:3 * i + 3, 3 * j:3 * j + 3] = M; A[3 * j:3 * j + 3, 3 * i:3 * i + 3] = M.T
        w = np.abs(M).sum(); sums[i] += w; sums[j] += w
    R = [i for i, _ in off] + list(range(n)); Cc = [j for _, j in off] + list(range(n))
    V = [M.T.reshape(-1) for M in off.values()] + [((1 + 2 * sums[v]) * np.eye(3)).reshape(-1) for v in range(n)]
    for v in range(n):
        A[3 * v:3 * v + 3, 3 * v:3 * v + 3] = (1 + 2 * sums[v]) * np.eye(3)
    k = len(R)
    R += [0] * (nt - k); Cc += [0] * (nt - k); V += [np.zeros(9)] * (nt - k)    # (the store's count is fixed)
    dev = s.tr.device
    s.tr[:nt] = torch_cuda.tensor(np.array(R, np.int32), device=dev)
    s.tc[:nt] = torch_cuda.tensor(np.array(Cc, np.int32), device=dev)
    s.tv[:9 * nt] = torch_cuda.tensor(np.array(V).reshape(-1), device=dev)
    s.convert(); s.build_precond()
    b = s.b.cpu().numpy()
    tol = 1e-6 if mixed else 1e-9
    st = s.solve(tol=tol, stop_rule=capi.STOP_TRUE_REL, max_iter=2000,
                 precision=capi.PRECISION_MIXED if mixed else capi.PRECISION_FP64)
    x = s.dx.cpu().numpy()
    A = A.tocsc()
    assert st.converged and np.linalg.norm(b - A @ x) <= 1.5 * tol * np.linalg.norm(b)
    d = A.diagonal()
    xs = spla.spsolve(A, b)
    assert np.abs(d * (x - xs)).max() <= 10 * tol * np.linalg.norm(b)


@pytest.mark.parametrize("kind", [0, 1, 2, 3])
def test_fp64_solve_follows_values_edited_in_place(torch_cuda, cube4, kind):
    """The converted values live in the caller's store: a diagonal shift or a
    scaling written there between two solves is the matrix of the next one,
    without another convert.  Every solve reaches 1e-9 of the matrix as it then
    is, by the reported residual (half a digit of slack for the recurrence's
    own drift) and by numpy's."""
    print("case: values edited in place, precond", kind, flush=True)
    s = make_system(cube4, kind)
    s.assemble(); s.convert(); s.build_precond()
    kr, kc, kv = s.bcoo()
    diag = torch_cuda.tensor(np.flatnonzero(kr == kc), device=s.dev)
    v = s.tv[:9 * s.K].view(s.K, 9)
    shift = float(np.abs(kv[kr == kc][:, [0, 4, 8]]).mean())
    b = s.b.cpu().numpy()
    for step in range(4):
        if step == 3:
            v *= 0.5
        elif step:
            for e in (0, 4, 8):
                v[diag, e] += shift * step
        st = s.solve(tol=1e-9, stop_rule=1, max_iter=5000)
        A = dense_from_bcoo(*s.bcoo(), cube4.n)
        x = s.dx.cpu().numpy()
        res = np.linalg.norm(A @ x - b) / np.linalg.norm(b)
        assert st.converged and res <= 3e-9 and st.rel_residual <= 3e-9, (step, res, st.rel_residual)


_TRAILING = [[125, 126, 127, 128], list(range(125, 136)), list(range(125, 145))]
_AMONG = [list(range(64, 88)), [0, 1, 2, 3, 4, 5, 6, 7, 140]]


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("kind,empty", [(k, e) for k in (0, 1) for e in _TRAILING + _AMONG] +
                         [(2, e) for e in _TRAILING])
def test_solve_with_rows_without_triplets(torch_cuda, oracle, cube4, kind, mixed, empty):
    """Block rows that no triplet names, at the end of the system (so that the
    SpMV's last chunk of eight rows has no entry, one alone or several rows), in
    whole chunks of the middle and at the front: they stay zero and the others
    solve the system without them.  (MAS covers the leading rows only, so it is
    run where the empty ones follow.)"""
    from sgipc import capi
    from sgipc.system import _p
    print("case: rows without triplets", kind, mixed, len(empty), empty[0], flush=True)
    n = cube4.n
    ref = oracle_system(oracle, cube4)
    nb = max(n + len(empty), empty[-1] + 1)
    rows = np.array([r for r in range(nb) if r not in set(empty)])[:n]      # new row of each old one
    s = make_system(cube4, kind)
    R, Cc, V = ref["trip"]
    nt = len(R)
    s.tr[:nt] = torch_cuda.tensor(rows[R].astype(np.int32), device=s.dev)
    s.tc[:nt] = torch_cuda.tensor(rows[Cc].astype(np.int32), device=s.dev)
    s.tv[:9 * nt] = torch_cuda.tensor(V.reshape(-1), dtype=torch_cuda.float64, device=s.dev)
    K = C.c_int(0)
    s.ctx.call("sgipc_convert", nt, nb, C.byref(K))
    kr, kc, kv = ref["bcoo"]
    entries = 2 * K.value - n                                               # every old row has its diagonal
    assert K.value == len(kr) and entries % 64 != 0
    s.ctx.call("sgipc_precond_build", kind, 0, n if kind == 2 else nb, None, 0)
    b = np.zeros((nb, 3))
    b[rows] = ref["b"].reshape(n, 3)
    bt = torch_cuda.tensor(b.reshape(-1), device=s.dev)
    xt = torch_cuda.full_like(bt, 7.0)
    tol = 1e-6 if mixed else 1e-9
    o = capi.SolveOpts(capi.PRECISION_MIXED if mixed else capi.PRECISION_FP64, capi.STOP_TRUE_REL, tol, 0.3, 5000, 8)
    st = capi.SolveStats()
    s.ctx.call("sgipc_solve", _p(bt), _p(xt), C.byref(o), C.byref(st))
    x = xt.cpu().numpy().reshape(nb, 3)
    assert not np.any(np.delete(x, rows, axis=0))
    A = dense_from_bcoo(kr, kc, kv, n)
    res = np.linalg.norm(A @ x[rows].reshape(-1) - ref["b"]) / np.linalg.norm(ref["b"])
    # the FP64 recurrence's residual drifts from the true one by rounding (half a digit of slack)
    assert st.converged and res <= 3 * tol and st.rel_residual <= 3 * tol, (res, st.rel_residual)


@pytest.mark.parametrize("kind,group", [(0, 8), (1, 4), (2, 4), (2, 8), (2, 16), (3, 16)])
def test_fp64_solve_on_the_upper_blocks(torch_cuda, monkeypatch, cube10, kind, group):
    """Where the entry-order copy does not fit the device (or is switched off) the
    FP64 solve reads the converted upper blocks in place: the iteration count and
    iterate of the solve on the copy, but for the order of the row sums (1e-10,
    as against the oracle above)."""
    print("case: upper-BCOO FP64 solve, precond", kind, "group", group, flush=True)
    monkeypatch.setenv("SGIPC_SPMV_FULL64", "1")
    ref = make_system(cube10, kind)
    monkeypatch.setenv("SGIPC_SPMV_FULL64", "0")
    s = make_system(cube10, kind)
    s.ctx.call("sgipc_set_schedule", group, 4)
    for q in (ref, s):
        q.ctx.call("sgipc_set_deterministic", 1)
        q.assemble(); q.convert(); q.build_precond()
    for tol, rule in ((1e-4, 0), (1e-30, 0)):
        st, so = (q.solve(tol=tol, stop_rule=rule, max_iter=12 if tol < 1e-9 else 5000) for q in (s, ref))
        assert st.iterations == so.iterations and st.converged == so.converged
        x, xo = s.dx.cpu().numpy(), ref.dx.cpu().numpy()
        assert np.linalg.norm(x - xo) <= 1e-10 * np.linalg.norm(xo)
        assert abs(st.rel_residual - so.rel_residual) <= 1e-6 * so.rel_residual


def test_fp64_solve_where_the_copy_leaves_the_cache(torch_cuda, monkeypatch):
    """300,763 rows under block Jacobi, where the solve chooses the blocks in
    place: twenty iterations are those on the copy and in place when either is
    forced, up to the order of the row sums."""
    from sgipc import scene
    print("case: FP64 solve at 300,763 rows", flush=True)
    sc = scene.cube_scene(66, seed=1)
    xs = []
    for force in ("1", "0", None):
        if force is None:
            monkeypatch.delenv("SGIPC_SPMV_FULL64")
        else:
            monkeypatch.setenv("SGIPC_SPMV_FULL64", force)
        s = make_system(sc, 1)
        s.assemble(); s.convert(); s.build_precond()
        st = s.solve(tol=1e-30, stop_rule=1, max_iter=21)
        assert st.iterations == 21
        xs.append(s.dx.cpu().numpy().copy())
        del s
    assert np.linalg.norm(xs[1] - xs[0]) <= 1e-10 * np.linalg.norm(xs[0])
    assert np.array_equal(xs[2], xs[1])
