"""Sizes at which a kernel's tiling or dispatch changes: node counts around
the slices of 64 and the one-workgroup kernel's limits, nodes with more links
than an out-link record (4 lanes, 6 slots) or an in-link slice (16 rows)
holds, link counts around a workgroup of the line search.  Labels equal the
oracle's bit for bit; volumes, costs and step sizes of two paths are equal
bit for bit (integer demand, so every partial sum is exact)."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import pred_reaches_origin, pred_tie_check, random_demand

pytestmark = pytest.mark.gpu


def small_network(seed, N, Z, ft, extra, kind, hub=0):
    """A two-way ring of the through nodes, every zone joined to one of them,
    `extra` random links (self-loops and parallel links among them) and
    `hub` links out of and into one through node."""
    from traffic_assignment_amd import synth
    rng = np.random.default_rng(seed)
    thru = np.arange(ft, N + 1)
    z = np.arange(1, ft)
    t = rng.integers(ft, N + 1, z.size)
    a = [thru, np.roll(thru, -1), z, t, rng.integers(1, N + 1, extra)]
    b = [np.roll(thru, -1), thru, t, z, rng.integers(1, N + 1, extra)]
    if hub:
        h = rng.integers(ft, N + 1, hub)
        c = np.full(hub, ft + (N - ft) // 2)
        a += [c, h]
        b += [h, c]
    init, term = np.concatenate(a), np.concatenate(b)
    order = np.lexsort((term, init))
    init, term = init[order].astype(np.int64), term[order].astype(np.int64)
    E = init.size
    if kind == "ints":
        cost = rng.integers(0, 4, E).astype(np.float64)
    else:
        cost = rng.uniform(0.01, 5.0, E)
    net = synth.Network(num_zones=Z, num_nodes=N, first_thru_node=ft, init=init, term=term,
                        capacity=rng.uniform(20.0, 200.0, E), length=np.ones(E), fftime=cost,
                        B=np.full(E, 0.15), power=np.full(E, 4.0), speed=np.zeros(E),
                        toll=np.zeros(E), ltype=np.ones(E, np.int16))
    return net, rng


@pytest.mark.parametrize("N,ft,hub", [(63, 1, 0), (64, 20, 5), (65, 1, 6), (128, 65, 7), (129, 64, 16),
                                      (300, 1, 17), (1000, 90, 60), (4097, 300, 700)])
@pytest.mark.parametrize("kind", ["cont", "ints"])
def test_lds_kernel_records_and_slices(engine_mod, oracle_lib, N, ft, hub, kind):
    import oracle
    print(f"case lds edges N={N} ft={ft} hub={hub} {kind}", flush=True)
    Z = min(max(ft - 1, 12), 40)
    net, rng = small_network(N + hub, N, Z, ft, N, kind, hub)
    dem = random_demand(net, rng)
    origins = np.arange(1, Z + 1)
    od, op = oracle.sssp_all(net, net.fftime)
    with engine_mod.TapEngine(net, dem) as eng:
        eng.set_strategy("lds")
        d, p = eng.sssp(origins)
        assert np.array_equal(d[1:].view(np.int64), od[1:].view(np.int64))
        bad, _ = pred_tie_check(net, net.fftime, d, p, op, origins)
        assert bad == 0
        pred_reaches_origin(net, d, p, origins)
        ys = []
        for q in (-1, 0, 1, 16):                       # queue sizes: scan rounds and mixed rounds
            eng.set_origin_queue(q)
            ys.append(eng.aon())
        eng.set_strategy("hbm")
        ys.append(eng.aon())
    for y in ys[1:]:
        assert np.array_equal(y, ys[0])


def _run(engine_mod, net, dem, graphs, chunks, window=0, **kw):
    with engine_mod.TapEngine(net, dem, **kw) as eng:
        eng.set_graphs(graphs)
        eng.set_link_passes(0, window)
        eng.fw_init()
        out = [eng.flows(v) for v in range(eng.V)]
        for n in chunks:
            eng.fw_run(max_iters=n)
            out += [eng.flows(v) for v in range(eng.V)]
        return out, [eng.trace(v) for v in range(eng.V)]


def _same(a, b):
    for (xa, ca), (xb, cb) in zip(a[0], b[0]):
        assert np.array_equal(xa, xb) and np.array_equal(ca, cb)
    for ta, tb in zip(a[1], b[1]):
        assert np.array_equal(ta["lambda_"], tb["lambda_"])
        # compensated sums in another order: a few units in the last place
        for k in ("objective", "vht"):
            assert np.allclose(ta[k], tb[k], rtol=1e-14, atol=0.0)


@pytest.mark.parametrize("N,Z,ft", [(2, 2, 1), (24, 24, 1), (31, 8, 9), (32, 32, 1), (33, 10, 11), (64, 16, 1),
                                    (65, 30, 31), (128, 17, 1), (129, 40, 41), (192, 64, 65), (193, 20, 1)])
@pytest.mark.parametrize("kind", ["cont", "ints"])
def test_one_workgroup_iterations(engine_mod, N, Z, ft, kind):
    """Iterations inside one kernel (up to 192 nodes, 64 zones) against the
    same iterations launch by launch: the wavefront's and half wavefront's
    origins, two and three nodes a lane, nodes with more in-links than its
    registers hold, zero-cost links and their level ties."""
    print(f"case one-workgroup N={N} Z={Z} ft={ft} {kind}", flush=True)
    net, rng = small_network(N, N, Z, ft, 2 * N, kind, hub=min(9, N // 4))
    dem = random_demand(net, rng)
    _same(_run(engine_mod, net, dem, 1, (5, 12)), _run(engine_mod, net, dem, 0, (5, 12)))


def test_one_workgroup_batch_and_windows(engine_mod):
    """Three variants with their own capacities, presence and stopping
    iteration; line-search windows of two step sizes; a launch's 256
    iterations passed; deep steps on a converged network."""
    print("case one-workgroup batch", flush=True)
    net, rng = small_network(7, 40, 12, 1, 60, "cont")
    dem = random_demand(net, rng)
    E = net.num_links
    ring = np.isin(np.arange(E), rng.choice(E, E // 3, replace=False))
    thru = np.abs(net.init - net.term) % (net.num_nodes - 2) <= 1        # the ring's own links stay
    present = np.stack([np.ones(E, bool), ~ring | thru, np.ones(E, bool)]).astype(np.uint8)
    cap = np.stack([net.capacity, net.capacity, 0.7 * net.capacity])
    kw = dict(num_variants=3, present=present, capacity=cap)
    for window in (0, 2):
        _same(_run(engine_mod, net, dem, 1, (3, 300), window, **kw),
              _run(engine_mod, net, dem, 0, (3, 300), window, **kw))
    with engine_mod.TapEngine(net, dem) as a, engine_mod.TapEngine(net, dem) as b:
        b.set_graphs(0)
        for eng in (a, b):
            eng.fw_init()
        ra, rb = a.fw_run(3000, 1e-3)[0], b.fw_run(3000, 1e-3)[0]
        assert ra["iterations"] == rb["iterations"] and ra["converged"] == rb["converged"]
        assert np.array_equal(a.flows()[0], b.flows()[0])


def test_one_workgroup_no_path(engine_mod):
    """Demand between disconnected zones is an error in the one-workgroup
    kernel too, and the engine works on afterwards."""
    from traffic_assignment_amd import synth
    net, rng = small_network(3, 20, 6, 7, 10, "cont")
    keep = net.term != 4                                # nothing reaches zone 4
    import dataclasses
    f = {k: getattr(net, k)[keep] for k in ("init", "term", "capacity", "length", "fftime", "B", "power",
                                            "speed", "toll", "ltype")}
    cut = dataclasses.replace(net, **f)
    dem = synth.Demand(6, np.array([0, 1, 1, 1, 1, 1, 1]), np.array([4]), np.array([5.0]))
    with engine_mod.TapEngine(cut, dem) as eng:
        with pytest.raises(engine_mod.NoPathError):
            eng.fw_init()
        d, _ = eng.sssp([1])
        assert d[4, 0] > 1.7e308


@pytest.mark.parametrize("E", [255, 256, 257, 511, 512, 513, 1025])
def test_line_search_blocks(engine_mod, E):
    """Link counts around a workgroup of the line search: one workgroup per
    variant against many."""
    print(f"case line search E={E}", flush=True)
    net, rng = small_network(E, 80, 10, 1, E - 160, "cont")
    assert net.num_links == E
    dem = random_demand(net, rng)
    res = []
    for mode in (1, 2):
        with engine_mod.TapEngine(net, dem) as eng:
            eng.set_link_passes(mode)
            eng.fw_init()
            eng.fw_run(max_iters=20)
            res.append(([eng.flows()], [eng.trace()]))
    _same(*res)


@pytest.mark.parametrize("M", [2, 17, 512, 513, 514, 1500])
def test_gradient_rows_of_parallel_routes(engine_mod, M):
    """M equal-time routes from a hub: M - 1 cycles, all through the tree's
    route, so two links' rows have M - 1 entries (512 is the longest that
    takes lanes, longer ones a workgroup).  Volumes of half the capacity are
    the equilibrium in exact arithmetic.  Tolerance as for the other
    comparisons with the dense solve; a repeat gives the same bits."""
    from oracle import gradient as G
    from traffic_assignment_amd import synth
    print(f"case gradient rows M={M}", flush=True)
    rng = np.random.default_rng(M)
    mid = np.arange(4, 4 + M)
    cap = 2.0 * rng.integers(5, 40, M)
    init = np.concatenate([[1], np.full(M, 3), mid])
    term = np.concatenate([[3], mid, np.full(M, 2)])
    E = init.size
    capacity = np.concatenate([[cap.sum()], cap, cap])
    net = synth.Network(num_zones=2, num_nodes=3 + M, first_thru_node=3, init=init, term=term,
                        capacity=capacity, length=np.ones(E), fftime=np.ones(E), B=np.full(E, 0.15),
                        power=np.full(E, 4.0), speed=np.zeros(E), toll=np.zeros(E),
                        ltype=np.ones(E, np.int16))
    x = capacity / 2
    dem = synth.Demand(2, np.array([0, 1, 1]), np.array([2]), np.array([x[0]]))
    links = np.stack([np.zeros(M, np.int64), 1 + np.arange(M), 1 + M + np.arange(M)], 1)
    ref = G.reference_gradient(net, x, dict(od=np.zeros(M, np.int64), flow=cap / 2,
                                            off=3 * np.arange(M + 1), links=links.ravel()))
    assert ref["rank"] == M - 1
    with engine_mod.TapEngine(net, dem) as eng:
        eng.fw_init(x)
        g = eng.gradient(eps=1e-9, cg_tol=1e-13)
        h = eng.gradient(eps=1e-9, cg_tol=1e-13)
    assert g["info"]["cg_status"] == 1 and g["info"]["cycles"] == M - 1
    for k in ("dobj_dt0", "dobj_dcap"):
        np.testing.assert_allclose(g[k], ref[k], rtol=1e-12, atol=1e-300)
    for k in ("dvht_dcap", "dvht_dt0"):
        np.testing.assert_allclose(g[k], ref[k], rtol=1e-7, atol=1e-9 * np.abs(ref[k]).max())
        assert np.array_equal(g[k].view(np.int64), h[k].view(np.int64))


@pytest.mark.parametrize("N,starts,strategy", [(300, 582, "lds"), (300, 583, "lds"), (1100, 400, "hbm"),
                                               (4097, 45, "lds"), (4097, 1060, "lds")])
def test_shortest_paths_in_slabs(engine_mod, N, starts, strategy):
    """Results of one copy, of several slabs placed by the caller and of
    slabs placed by threads, with more starts than a launch takes: the
    columns equal calls of 40 starts (one copy each), in both layouts and
    with either array left out."""
    import ctypes as C
    from conftest import empty_demand
    print(f"case slabs N={N} starts={starts} {strategy}", flush=True)
    net, rng = small_network(N + starts, N, 20, 21, 2 * N, "cont", 30)
    s = rng.integers(1, N + 1, starts).astype(np.int64)
    with engine_mod.TapEngine(net, empty_demand(20)) as eng:
        eng.set_strategy(strategy)
        d, p = eng.sssp(s)
        for j in range(0, starts, 40):
            dj, pj = eng.sssp(s[j:j + 40])
            assert np.array_equal(d[:, j:j + 40].view(np.int64), dj.view(np.int64))
            assert np.array_equal(p[:, j:j + 40], pj)
        L = engine_mod.lib()
        vp = C.c_void_p
        ld = starts + 3
        d2, p2 = np.full((N + 1, ld), 7.0), np.full((N + 1, ld), 7, np.int64)
        assert L.tapgpu_sssp(eng._h, 0, vp(s.ctypes.data), starts, vp(d2.ctypes.data), None, ld, 2) == 0
        assert L.tapgpu_sssp(eng._h, 0, vp(s.ctypes.data), starts, None, vp(p2.ctypes.data), ld, 2) == 0
    assert np.array_equal(d2[:, 2:-1], d) and np.array_equal(p2[:, 2:-1], p)
    assert (d2[:, [0, 1, -1]] == 7).all() and (p2[:, [0, 1, -1]] == 7).all()


@pytest.mark.parametrize("threads", [512, 1024])
def test_lds_rounds_of_several_workgroups_per_cu(engine_mod, threads):
    """Workgroups that share a CU and its LDS, 24 x 397 searches: equal
    labels and trees every time."""
    from conftest import network
    print(f"case lds shared CU {threads}", flush=True)
    net, dem = network("metro", 0.63)
    origins = np.tile(np.arange(1, net.num_zones + 1), 4)
    with engine_mod.TapEngine(net, dem) as eng:
        eng.set_strategy("hbm")
        d0, p0 = eng.sssp(origins[:net.num_zones])
        eng.set_strategy("lds")
        eng.set_origin_block(threads)
        for q in (-1, 1024, 256) * 2:
            eng.set_origin_queue(q)
            eng.set_origin_block(threads)
            d, p = eng.sssp(origins)
            assert np.array_equal(d.view(np.int64), np.tile(d0.view(np.int64), 4))
            assert np.array_equal(p, np.tile(p0, 4))


@pytest.mark.parametrize("N,ft,hub", [(63, 1, 5), (129, 64, 16), (1000, 90, 60), (4097, 300, 700)])
@pytest.mark.parametrize("kind", ["cont", "ints"])
def test_hbm_kernel_queues_and_records(engine_mod, N, ft, hub, kind):
    """Nodes with more links than a record or an in-link slice holds, queues
    of 64 entries (they overflow) to the largest, bucket widths from one
    bucket per label to all in one: labels, trees and loads equal the LDS
    kernel's."""
    print(f"case hbm edges N={N} ft={ft} hub={hub} {kind}", flush=True)
    Z = min(max(ft - 1, 12), 40)
    net, rng = small_network(3 * N + hub, N, Z, ft, N, kind, hub)
    dem = random_demand(net, rng)
    starts = rng.integers(1, N + 1, 50)
    with engine_mod.TapEngine(net, dem) as eng:
        eng.set_strategy("lds")
        d0, p0 = eng.sssp(starts)
        y0 = eng.aon()
        eng.set_strategy("hbm")
        for q in (0, 64, 200, -1):
            for width in (0.0, 1e-3, 1.0, 1e6):
                eng.set_origin_queue(q)
                eng.set_origin_delta(width)
                d, p = eng.sssp(starts)
                assert np.array_equal(d.view(np.int64), d0.view(np.int64)), (q, width)
                assert np.array_equal(p, p0), (q, width)
                assert np.array_equal(eng.aon().view(np.int64), y0.view(np.int64)), (q, width)


def test_lds_kernel_looks_at_a_link_once(engine_mod, oracle_lib):
    """Nodes with more links than a record holds: an expansion relaxes each
    of the node's eight links once."""
    import oracle
    print("case lds links once", flush=True)
    from traffic_assignment_amd import synth
    rng = np.random.default_rng(8)
    N, Z, degree = 2000, 30, 8
    init = np.repeat(np.arange(1, N + 1), degree)
    term = rng.integers(1, N + 1, init.size)
    term[::degree] = np.roll(np.arange(1, N + 1), -1)
    order = np.lexsort((term, init))
    E = init.size
    net = synth.Network(num_zones=Z, num_nodes=N, first_thru_node=1, init=init[order], term=term[order],
                        capacity=np.full(E, 100.0), length=np.ones(E), fftime=rng.uniform(0.5, 3.0, E),
                        B=np.full(E, 0.15), power=np.full(E, 4.0), speed=np.zeros(E), toll=np.zeros(E),
                        ltype=np.ones(E, np.int16))
    origins = np.arange(1, Z + 1)
    od, _ = oracle.sssp_all(net, net.fftime)
    with engine_mod.TapEngine(net, random_demand(net, rng)) as eng:
        eng.set_strategy("lds")
        eng.aon()
        a = eng.stats()
        eng.aon()
        b = eng.stats()
        d, _ = eng.sssp(origins)
    assert np.array_equal(d[1:].view(np.int64), od[1:].view(np.int64))
    n = {k: b[k] - a[k] for k in ("origin_scanned", "origin_expansions")}
    assert 0 < n["origin_scanned"] <= degree * n["origin_expansions"]


def grid_network(rows, cols, Z, diagonals, power=4.0):
    """A grid of through nodes whose first Z are zones, with both diagonals of
    every square or none: up to 4 or 8 links into a node."""
    from traffic_assignment_amd import synth
    rng = np.random.default_rng(rows * cols + Z)
    i = 1 + np.arange(rows * cols).reshape(rows, cols)
    pairs = [(i[:, :-1], i[:, 1:]), (i[:-1], i[1:])]
    if diagonals:
        pairs += [(i[:-1, :-1], i[1:, 1:]), (i[:-1, 1:], i[1:, :-1])]
    a = np.concatenate([p.ravel() for p, _ in pairs])
    b = np.concatenate([q.ravel() for _, q in pairs])
    init, term = np.concatenate([a, b]), np.concatenate([b, a])
    order = np.lexsort((term, init))
    E = init.size
    pw = np.full(E, 4.0)
    pw[0] = power
    net = synth.Network(num_zones=Z, num_nodes=rows * cols, first_thru_node=1, init=init[order],
                        term=term[order], capacity=rng.uniform(20.0, 200.0, E), length=np.ones(E),
                        fftime=rng.uniform(0.5, 3.0, E), B=np.full(E, 0.15), power=pw, speed=np.zeros(E),
                        toll=np.zeros(E), ltype=np.ones(E, np.int16))
    return net, rng


@pytest.mark.parametrize("rows,cols,Z,diagonals,V,power,one", [
    (4, 6, 24, 0, 1, 4.0, True), (4, 8, 32, 1, 1, 4.0, True), (8, 8, 64, 0, 1, 4.0, True),
    (8, 8, 16, 1, 1, 4.0, True), (9, 11, 16, 0, 1, 4.0, True), (13, 14, 16, 0, 1, 4.0, True),
    (13, 14, 64, 0, 64, 4.0, True), (9, 11, 48, 1, 64, 4.0, True),
    (13, 14, 64, 0, 1, 4.0, False), (9, 11, 16, 1, 1, 4.0, False), (8, 8, 48, 1, 1, 4.0, False),
    (12, 12, 60, 1, 1, 4.0, False), (9, 11, 48, 1, 4, 4.0, False), (14, 14, 8, 0, 1, 4.0, False),
    (4, 6, 24, 0, 1, 3.0, False), (4, 6, 24, 0, 3, 2.5, False)])
def test_one_workgroup_kernel_where_it_pays(engine_mod, rows, cols, Z, diagonals, V, power, one):
    """Which form the iterations take (replays of a graph are counted, the
    one kernel's launches are not), and that both give the same."""
    print(f"case one-workgroup choice {rows}x{cols} Z={Z} diag={diagonals} V={V} p={power}", flush=True)
    net, rng = grid_network(rows, cols, Z, diagonals, power)
    dem = random_demand(net, rng)
    kw = {}
    if V > 1:
        kw = dict(num_variants=V, capacity=net.capacity * rng.uniform(0.8, 1.25, (V, net.num_links)))
    out = []
    for graphs in (1, 0):
        with engine_mod.TapEngine(net, dem, **kw) as eng:
            eng.set_graphs(graphs)
            eng.fw_init()
            eng.fw_run(max_iters=12)
            n = eng.stats()["graph_launches"]
            assert (n == 0) == (one or not graphs), n
            out.append(([eng.flows(v) for v in range(V)], [eng.trace(v) for v in range(V)]))
    _same(*out)


@pytest.mark.parametrize("N,Z,ft,extra", [(31, 8, 9, 31), (33, 10, 11, 33), (64, 16, 1, 64), (65, 30, 31, 30),
                                          (128, 17, 1, 60), (129, 40, 41, 50), (192, 32, 33, 60)])
@pytest.mark.parametrize("kind", ["cont", "ints"])
def test_one_workgroup_batches(engine_mod, N, Z, ft, extra, kind):
    """64 variants, for which the one kernel is the faster form with more
    nodes and in-links too: zones that are no through nodes, level ties, one
    to three nodes a lane and several origins a wavefront."""
    print(f"case one-workgroup batch N={N} Z={Z} ft={ft} {kind}", flush=True)
    net, rng = small_network(5 * N, N, Z, ft, extra, kind)
    dem = random_demand(net, rng)
    V = 64
    cap = net.capacity * rng.uniform(0.8, 1.25, (V, net.num_links))
    out = []
    for graphs in (1, 0):
        with engine_mod.TapEngine(net, dem, num_variants=V, capacity=cap) as eng:
            eng.set_graphs(graphs)
            eng.fw_init()
            x = [eng.flows(v) for v in range(V)]
            eng.fw_run(max_iters=6)
            if graphs:                                 # (every other form replays graphs)
                assert eng.stats()["graph_launches"] == 0
            out.append((x + [eng.flows(v) for v in range(V)], [eng.trace(v) for v in range(V)]))
    _same(*out)


@pytest.mark.parametrize("form", ["plain", "one by one", "batch", "lanes", "hbm"])
def test_further_windows_over_many_workgroups(engine_mod, oracle_lib, form):
    """A twentieth of the links with a millionth of their capacity: some steps
    are far below the first window's 2^-15.  On a network of 28,084 links each
    further window is a pass over many workgroups, counted with the others;
    steps and volumes are the oracle's, whichever form the iterations take,
    and a batch's other variant is not held up."""
    import oracle
    print(f"case further windows {form}", flush=True)
    base, rng = grid_network(60, 60, 12, 1)
    dem = random_demand(base, rng)
    net = base.copy()
    narrow = np.random.default_rng(5).random(net.num_links) < 0.05
    net.capacity = np.where(narrow, 1e-6, 1.0) * net.capacity
    iters = 60
    ref = []
    oracle.lib().ora_set_pow_mode(1)
    try:
        for n in (net, base):
            ref.append(oracle.fw_solve(n, dem, max_iters=iters))
    finally:
        oracle.lib().ora_set_pow_mode(0)
    deep = int((ref[0]["trace"]["lambda_"] < 2.0 ** -15).sum())
    assert deep >= 5 and (ref[1]["trace"]["lambda_"] >= 2.0 ** -15).all()
    kw = {}
    if form in ("batch", "lanes"):
        kw = dict(num_variants=2, capacity=np.stack([net.capacity, base.capacity]))
    with engine_mod.TapEngine(net, dem, **kw) as eng:
        if form == "one by one":
            eng.set_graphs(0)
        if form == "lanes":
            eng.set_lanes(1)
        if form == "hbm":
            eng.set_strategy("hbm")
        eng.fw_init()
        eng.fw_run(max_iters=iters)
        assert eng.stats()["link_passes"] >= iters + deep
        for v in range(eng.V):
            assert np.array_equal(eng.trace(v)["lambda_"], ref[v]["trace"]["lambda_"])
            assert np.array_equal(eng.flows(v)[0], ref[v]["x"])


def test_one_workgroup_failed_loading_changes_nothing(engine_mod):
    """A loading without a path leaves volumes and costs as the launches do:
    fw_init the volumes it found and free-flow costs, an iteration both."""
    import dataclasses
    from traffic_assignment_amd import synth
    print("case one-workgroup failed loading", flush=True)
    net, rng = small_network(3, 20, 6, 7, 10, "cont")
    dem = random_demand(net, rng)
    closed = np.where(net.term == 4, np.inf, net.fftime)                 # nothing reaches zone 4
    states = []
    for graphs in (1, 0):
        with engine_mod.TapEngine(net, dem) as eng:
            eng.set_graphs(graphs)
            eng.fw_init()
            eng.fw_run(max_iters=3)
            s = [eng.flows()]
            eng.set_links(fftime=closed)
            with pytest.raises(engine_mod.NoPathError):
                eng.fw_init()
            s.append(eng.flows())
            eng.set_links(fftime=net.fftime)
            eng.fw_init()
            s.append(eng.flows())
        cut = synth.Demand(6, np.array([0, 1, 1, 1, 1, 1, 1]), np.array([4]), np.array([5.0]))
        with engine_mod.TapEngine(dataclasses.replace(net, fftime=closed), cut) as eng:
            eng.set_graphs(graphs)
            x = rng.uniform(0.0, 5.0, net.num_links) if graphs else x
            eng.fw_init(x)                                               # (a warm start loads nothing)
            s.append(eng.flows())
            with pytest.raises(engine_mod.NoPathError):
                eng.fw_run(max_iters=3)
            s.append(eng.flows())
            assert np.array_equal(s[-1][0], s[-2][0])
        states.append(s)
    for a, b in zip(*states):
        assert np.array_equal(a[0], b[0])
        assert np.array_equal(a[1], b[1], equal_nan=True)


def test_one_workgroup_statistics(engine_mod):
    """What the one kernel counts is what the launches count under that name;
    what it does not count is 0."""
    print("case one-workgroup statistics", flush=True)
    net, rng = grid_network(6, 7, 20, 0)
    dem = random_demand(net, rng)
    st = []
    for graphs in (1, 0):
        with engine_mod.TapEngine(net, dem) as eng:
            eng.set_graphs(graphs)
            eng.fw_init()
            eng.fw_run(max_iters=9)
            st.append(eng.stats())
    one, launches = st
    for k in ("origin_blocks", "origin_walk_steps", "link_passes"):
        assert one[k] == launches[k] > 0, k
    assert one["origin_relax_rounds"] > 0
    for k in ("origin_loaded", "origin_expansions", "origin_scanned", "origin_updates"):
        assert one[k] == 0 < launches[k], k


@pytest.mark.parametrize("form,power", [("tiny", 4.0), ("lds", 2.0), ("lanes", 2.0), ("passes", 2.0)])
def test_more_variants_than_a_grid_dimension(engine_mod, form, power):
    """66,000 variants, above the 65,535 of a launch in the grid's second
    dimension: those on both sides of the cut are what a context of their own
    gives, whichever kernels load them and take their steps."""
    print(f"case 66,000 variants {form}", flush=True)
    net, rng = grid_network(3, 3, 3, 0, power)
    dem = random_demand(net, rng)
    V = 66000
    cap = net.capacity * rng.uniform(0.8, 1.25, (V, net.num_links))

    def solve(**kw):
        with engine_mod.TapEngine(net, dem, **kw) as eng:
            if form != "tiny":
                eng.set_graphs(0)
            if form == "passes":
                eng.set_link_passes(2)
            if kw.get("num_variants", 1) > 1 and form != "tiny":
                eng.set_lanes(1 if form == "lanes" else 0)
            eng.fw_init()
            eng.fw_run(max_iters=3)
            at = watched if "num_variants" in kw else [0]
            return [eng.flows(v) for v in at], [eng.trace(v) for v in at], [eng.totals(v) for v in at]
    watched = [0, 65534, 65535, V - 1]
    many = solve(num_variants=V, capacity=cap)
    alone = [solve(capacity=cap[v:v + 1]) for v in watched]
    _same(many, [[one[k][0] for one in alone] for k in range(3)])
    np.testing.assert_allclose(many[2], [one[2][0] for one in alone], rtol=1e-14, atol=0.0)


@pytest.mark.parametrize("kind", ["cont", "ints", "zeros"])
def test_lds_kernel_nodes_of_many_in_links(engine_mod, kind):
    """Nodes with 15 to 900 in-links (a slice holds 16, a wavefront looks at
    64 at a time), some of them parallel: the tree link is the tight one with
    the smallest tail label, then tail, then link, and the labels-in-HBM
    kernel chooses the same, equal labels included."""
    from traffic_assignment_amd import synth
    print(f"case LDS kernel, nodes of many in-links, {kind}", flush=True)
    rng = np.random.default_rng(5)
    N, Z, ft = 1200, 20, 11                            # (zones 11..20 are through nodes)
    ring, zones = np.arange(ft, N + 1), np.arange(1, ft)
    at = rng.choice(ring, zones.size, replace=False)
    init = [ring, np.roll(ring, -1), zones, at]
    term = [np.roll(ring, -1), ring, at, zones]
    for v, n in zip(rng.choice(np.arange(ft, N + 1), 9, replace=False), (15, 16, 17, 63, 64, 65, 128, 300, 900)):
        t = rng.integers(1, N + 1, n)
        t[t == v] = ft if v == N else v + 1
        init += [t, np.full(n, v)]
        term += [np.full(n, v), t]
    init, term = np.concatenate(init), np.concatenate(term)
    order = np.lexsort((term, init))
    E = init.size
    cost = {"cont": rng.uniform(0.5, 3.0, E), "ints": rng.integers(1, 4, E).astype(float),
            "zeros": rng.integers(0, 2, E).astype(float)}[kind]
    net = synth.Network(num_zones=Z, num_nodes=N, first_thru_node=ft, init=init[order], term=term[order],
                        capacity=np.full(E, 100.0), length=np.ones(E), fftime=cost, B=np.full(E, 0.15),
                        power=np.full(E, 4.0), speed=np.zeros(E), toll=np.zeros(E), ltype=np.ones(E, np.int16))
    dem = random_demand(net, rng)
    starts = np.arange(1, 60)
    got = {}
    for strategy in ("lds", "hbm"):
        with engine_mod.TapEngine(net, dem) as eng:
            eng.set_strategy(strategy)
            eng.set_costs(cost)
            d, p = eng.sssp(starts)
            got[strategy] = (d, p, eng.aon())
    for a, b in zip(got["lds"], got["hbm"]):
        np.testing.assert_array_equal(a, b)
    d, p, _ = got["lds"]
    tail, head = net.init, net.term
    for j, s in enumerate(starts):
        dist, pred = d[1:, j], p[1:, j]
        du, dv = dist[tail - 1], dist[head - 1]
        tight = (du + cost == dv) & (du < dv) & ((tail >= ft) | (tail == s)) & (tail != head)
        k = np.flatnonzero(tight)
        k = k[np.lexsort((k, tail[k], du[k], head[k]))]
        first = np.r_[True, head[k][1:] != head[k][:-1]] if k.size else np.zeros(0, bool)
        np.testing.assert_array_equal(pred[head[k[first]] - 1], k[first])
