"""MAS restriction fused into the PCG update, on a partition whose level-0
banks split into many components of varying count.

Level-1 nodes are the components of the level-0 banks, numbered bank by
bank, so a level-0 bank whose components run over a multiple of the bank
size has coarse nodes in two level-1 banks (it "straddles" them) and is
visited by the two workgroups that own those level-1 banks.  Here every
level-0 bank holds 10-16 vertices drawn at random from the mesh, so most
vertices are singleton components, straddling banks are everywhere and
there are more level-1 banks than the fused update launches workgroups for
them (its grid-stride loop runs).  PCG iterates after a fixed budget depend
on the restriction of each updated residual, so they are compared with the
oracle's PCG (its own MAS apply of the same residual) at 1e-10.
"""
import numpy as np
import pytest

from conftest import oracle_system

pytestmark = pytest.mark.gpu

# workgroups the fused x/r update launches for level-1 banks (one partial
# slot each; the library's partial-sum width)
FUSED_UPDATE_WORKGROUPS = 1024


def scrambled_scene(cells=26, seed=11, min_size=10, bank=16):
    """cube_scene with its vertices regrouped into parts of min_size..bank
    randomly drawn vertices (numbering part-contiguous again)."""
    from sgipc import scene
    sc = scene.cube_scene(cells, seed=1)
    rng = np.random.default_rng(seed)
    n = sc.n
    order = rng.permutation(n)
    sizes = []
    tot = 0
    while tot < n:
        s = int(rng.integers(min_size, bank + 1))
        s = min(s, n - tot)
        sizes.append(s)
        tot += s
    part_of = np.empty(n, np.int32)
    part_of[order] = np.repeat(np.arange(len(sizes), dtype=np.int32), sizes)
    perm, inv, part_sorted = scene.renumber_by_part(part_of)
    tets = inv[sc.tets.astype(np.int64)].astype(np.uint32)
    return scene.Scene("scrambled%d" % cells, sc.x_rest[perm], sc.x[perm], sc.x_tilde[perm], tets,
                       part_sorted.astype(np.int32), sc.btype[perm], sc.DmInv, sc.vol, sc.mass[perm], sc.mu,
                       sc.lam, sc.dt, bank=bank, meta=dict(sc.meta, scrambled_seed=seed))


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch


@pytest.fixture(scope="module")
def scrambled():
    return scrambled_scene()


@pytest.fixture(scope="module")
def scrambled_system(torch_cuda, oracle, scrambled):
    from sgipc import capi
    from sgipc.system import NewtonSystem
    ref = oracle_system(oracle, scrambled)
    sys_ = NewtonSystem(scrambled, "cuda:0", precond=capi.PRECOND_MAS)
    sys_.assemble(); sys_.convert(); sys_.build_precond()
    kr, kc, kv = ref["bcoo"]
    mas = oracle.Mas(scrambled.n, sys_.part_map, sys_.real_map, sys_.ns, sys_.nn, sys_.nl, scrambled.bank)
    mas.build(kr, kc, kv)
    return sys_, ref, mas


def test_scrambled_partition_exercises_straddling_banks(scrambled_system):
    sys_, _, _ = scrambled_system
    t = sys_.mas_tables()
    B = sys_.sc.bank
    ls = t["level_size"]
    n1 = int(ls[1, 0])
    nb1 = (n1 + B - 1) // B
    print("case: scrambled partition levels", t["levelnum"], "level-1 nodes", n1, "level-1 banks", nb1, flush=True)
    assert nb1 > FUSED_UPDATE_WORKGROUPS           # grid-stride loop over level-1 banks runs
    # level-0 banks whose coarse nodes fall in two level-1 banks
    p0 = t["prefix0"].astype(np.int64)
    psum = np.concatenate([[0], np.cumsum(p0)[:-1]])
    nz = p0 > 0
    straddle = ((psum[nz] // B) != ((psum[nz] + p0[nz] - 1) // B)).sum()
    assert straddle > 100


@pytest.mark.parametrize("budget", [2, 3, 7])
def test_pcg_budget_matches_oracle_on_straddling_banks(scrambled_system, oracle, budget):
    sys_, ref, mas = scrambled_system
    print("case: scrambled pcg budget", budget, flush=True)
    kr, kc, kv = ref["bcoo"]
    st = sys_.solve(tol=1e-30, stop_rule=0, max_iter=budget)
    xo, ito, _ = oracle.pcg(kr, kc, kv, sys_.sc.n, ref["b"], precond=2, mas=mas, tol=1e-30, rule=0,
                            max_iter=budget)
    assert st.iterations == ito
    x = sys_.dx.cpu().numpy()
    assert np.linalg.norm(x - xo) <= 1e-10 * np.linalg.norm(xo)


def test_solves_repeat_bitwise_on_straddling_banks(scrambled_system):
    from sgipc import capi
    sys_, _, _ = scrambled_system
    print("case: scrambled repeat", flush=True)
    for prec in (capi.PRECISION_FP64, capi.PRECISION_MIXED):
        xs = []
        for _ in range(3):
            sys_.solve(tol=1e-6, stop_rule=capi.STOP_TRUE_REL, precision=prec, max_iter=2000)
            xs.append(sys_.dx.cpu().numpy().copy())
        assert np.array_equal(xs[0], xs[1]) and np.array_equal(xs[0], xs[2])


@pytest.mark.parametrize("cells,boxes,bank", [(1, 1, 16), (2, 1, 32), (11, 1, 16), (11, 1, 32), (12, 1, 16),
                                              (9, 2, 16), (9, 2, 32), (10, 2, 16)])
def test_tables_and_apply_on_both_sides_of_the_one_workgroup_limit(torch_cuda, oracle, cells, boxes, bank):
    """Up to 2048 vertices one workgroup numbers the whole hierarchy, above it
    a few launches per level do: the integer tables equal the oracle's bit for
    bit and the FP64 apply agrees to rounding (a 96-term bank product and its
    inverse; 1e-11 is what the other apply tests hold), with and without
    contacts, for the smallest meshes and just below and above the limit."""
    from sgipc import capi, scene
    from sgipc.system import NewtonSystem
    print("case: mas tables", cells, boxes, bank, flush=True)
    sc = (scene.cube_scene if boxes == 1 else scene.two_box_scene)(cells, seed=3, bank=bank)
    s = NewtonSystem(sc, "cuda:0", precond=capi.PRECOND_MAS)
    pairs = None
    if boxes == 2:
        s.setup_contacts(*scene.facing_contact_candidates(sc))
        pairs = s.pairs.cpu().numpy().reshape(-1, 4)
        assert 0 < len(pairs) <= 4096
    s.assemble(); s.convert(); s.build_precond()
    mas = oracle.Mas(sc.n, s.part_map, s.real_map, s.ns, s.nn, s.nl, sc.bank)
    mas.build(*s.bcoo(), pairs=pairs)
    t, to = s.mas_tables(), mas.tables()
    for key in ("level_size", "coarse_space", "fine_mask", "prefix0"):
        assert np.array_equal(t[key], to[key]), key
    k = mas.levelnum - 1
    assert np.array_equal(t["coarse_table"][:, :k], to["coarse_table"][:, :k])
    r = np.random.default_rng(4).normal(size=3 * sc.n)
    z, zo = s.precond_apply(r), mas.apply(r, fp32=False)
    assert np.abs(z - zo).max() <= 1e-11 * np.abs(zo).max()


def _two_hierarchies():
    """Two neighbour lists over 512 vertices in 32 banks of two components: 64
    level-1 nodes each, then 40 and 10 nodes (banks: 3 + 1) or 32 and 32 (2 + 2),
    so the same number of banks, another first bank of level 3."""
    def lists(joins):
        nb = [set() for _ in range(512)]
        def join(a, b):
            nb[a].add(b); nb[b].add(a)
        for v in range(512):
            if v % 8:
                join(v - 1, v)                      # level-1 node v // 8
        for a, b in joins:
            join(8 * a, 8 * b)
        num = np.array([len(q) for q in nb], np.uint32)
        start = np.concatenate([[0], np.cumsum(num)[:-1]]).astype(np.uint32)
        return start, num, np.array([u for q in nb for u in sorted(q)], np.uint32)
    wide = [(i, i + 2) for i in range(64) if i % 4 < 2]
    narrow = [(16 * k, 16 * k + j) for k in range(4) for j in (2, 4, 6, 8, 10, 12)]
    left = [0, 1, 3, 5, 7, 9, 11, 13, 14, 15]       # a level-1 bank's nodes after these joins, by lowest member
    node2 = lambda q: 16 * (q // 10) + left[q % 10]
    pairs2 = [(10, q) for q in range(10)] + [(0, q) for q in range(11, 16)]
    pairs2 += [(16, q) for q in list(range(20, 30)) + [30, 31]] + [(20, q) for q in (17, 18, 19)]
    return lists(narrow + [(node2(a), node2(b)) for a, b in pairs2]), lists(wide)


@pytest.mark.parametrize("batched", [False, True])
def test_graphs_follow_the_split_of_the_upper_levels(torch_cuda, batched):
    """The fused bank solves are captured with the first bank of level 3.  A
    hierarchy with as many banks in all, but another such bank, is solved on a
    context that holds the graph of the other one: the iterates are bit for bit
    those of a context of its own."""
    import ctypes as C
    from sgipc import capi, scene
    from sgipc.system import NewtonSystem, _p
    print("case: graphs and level splits, batched", batched, flush=True)
    sc = scene.cube_scene(7, seed=4)
    ident = np.arange(512, dtype=np.int32)
    topos = _two_hierarchies()

    def system():
        s = NewtonSystem(sc, "cuda:0", precond=capi.PRECOND_MAS)
        s.ctx.call("sgipc_set_deterministic", 1)
        s.assemble(); s.convert()
        return s

    def solve(s, topo, precision):
        ns, nn, nl = topo
        s.ctx.call("sgipc_set_mas_topology", 512, 0, ns.ctypes.data, nn.ctypes.data, nl.ctypes.data, len(nl),
                   ident.ctypes.data, 512, ident.ctypes.data, 16)
        s.build_precond()
        if batched:
            st = (capi.SolveStats * 1)()
            o = capi.SolveOpts(precision, 1, 1e-6, 0.3, 2000, 8)
            rs = np.array([0, 512], np.int32)
            s.ctx.call("sgipc_solve_batched", 1, rs.ctypes.data, _p(s.b), _p(s.dx), C.byref(o), st)
            st = st[0]
        else:
            st = s.solve(tol=1e-6, stop_rule=1, precision=precision, max_iter=2000)
        L, tot = C.c_int(0), C.c_int(0)
        ls = np.zeros(16, np.int32)
        s.ctx.call("sgipc_mas_info", C.byref(L), C.byref(tot), ls.ctypes.data)
        return st.iterations, s.dx.cpu().numpy().copy(), (L.value, tot.value, (ls[2] + 15) // 16), ls[7]

    for precision in (capi.PRECISION_FP64, capi.PRECISION_MIXED):
        own = [solve(system(), t, precision) for t in topos]
        assert own[0][2] == own[1][2] == (4, 640, 4) and own[0][3] != own[1][3]
        assert own[0][0] > 3 and own[1][0] > 3
        one = system()
        for k in (0, 1, 0, 1, 1):
            it, x, _, _ = solve(one, topos[k], precision)
            assert it == own[k][0] and np.array_equal(x, own[k][1])


@pytest.mark.parametrize("cells,bank", [(4, 16), (11, 32), (12, 16), (13, 16)])
def test_padded_neighbour_lists_give_the_same_tables(torch_cuda, cells, bank):
    """Neighbour ids of 2^31 and above are padding: lists with such ids before,
    between and after the neighbours (and vertices with nothing else) give the
    tables of the lists without them, bit for bit, on both sides of the
    one-workgroup limit; any other id outside the range is refused."""
    from sgipc import capi, scene
    from sgipc.capi import SgipcError
    from sgipc.system import NewtonSystem
    print("case: padded neighbour lists", cells, bank, flush=True)
    sc = scene.cube_scene(cells, seed=3, bank=bank)
    s = NewtonSystem(sc, "cuda:0", precond=capi.PRECOND_MAS)
    s.assemble(); s.convert()
    lists = [list(s.nl[a:a + k]) for a, k in zip(s.ns.astype(int), s.nn.astype(int))]
    lists[sc.n // 2] = []

    def tables(padding, bad=None):
        rng, out, num = np.random.default_rng(6), [], []
        for q in lists:
            q = list(q)
            if padding:
                for pad in rng.choice([0xFFFFFFFF, 0x80000000, 0x80000005], size=int(rng.integers(1, 4))):
                    q.insert(int(rng.integers(0, len(q) + 1)), int(pad))
            num.append(len(q)); out += q
        if bad is not None:
            out[len(out) // 2] = bad
        num = np.array(num, np.uint32); out = np.array(out, np.uint32)
        start = np.concatenate([[0], np.cumsum(num)[:-1]]).astype(np.uint32)
        s.ctx.call("sgipc_set_mas_topology", sc.n, 0, start.ctypes.data, num.ctypes.data, out.ctypes.data, len(out),
                   s.part_map.ctypes.data, len(s.part_map), s.real_map.ctypes.data, bank)
        s.build_precond()
        return s.mas_tables()

    t, p = tables(False), tables(True)
    assert t["levelnum"] == p["levelnum"] and t["total"] == p["total"]
    for key in ("level_size", "coarse_space", "fine_mask", "prefix0", "going_next"):
        assert np.array_equal(t[key], p[key]), key
    k = t["levelnum"] - 1
    assert np.array_equal(t["coarse_table"][:, :k], p["coarse_table"][:, :k])
    for bad in (sc.n, 0x7FFFFFFF):
        with pytest.raises(SgipcError, match="neighbour index out of range"):
            tables(False, bad)
