"""Searches of the labels-in-HBM kernel whose fronts or far nodes exceed its
queues.  Labels, trees and volumes equal the LDS kernel's bit for bit, and the
work stays in proportion: counts of expansions and rounds, not times."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import network, random_demand

pytestmark = pytest.mark.gpu


def random_graph(N, degree, Z, seed):
    """A ring and `degree` links from every node to random ones: a search's
    front is a large part of the nodes."""
    from traffic_assignment_amd import synth
    rng = np.random.default_rng(seed)
    node = np.arange(1, N + 1)
    init = np.concatenate([np.repeat(node, degree), node])
    term = np.concatenate([rng.integers(1, N + 1, N * degree), np.roll(node, -1)])
    order = np.lexsort((term, init))
    E = init.size
    net = synth.Network(num_zones=Z, num_nodes=N, first_thru_node=1, init=init[order].astype(np.int64),
                        term=term[order].astype(np.int64), capacity=rng.uniform(20.0, 200.0, E),
                        length=np.ones(E), fftime=rng.uniform(0.5, 3.0, E), B=np.full(E, 0.15),
                        power=np.full(E, 4.0), speed=np.zeros(E), toll=np.zeros(E),
                        ltype=np.ones(E, np.int16))
    return net, rng


def _both(eng, costs, starts):
    """Equal results of both kernels; the labels-in-HBM kernel's counts."""
    eng.set_costs(costs)
    eng.set_strategy("lds")
    d0, p0 = eng.sssp(starts)
    y0 = eng.aon()
    eng.set_strategy("hbm")
    d, p = eng.sssp(starts)
    a = eng.stats()
    y = eng.aon()
    b = eng.stats()
    assert np.array_equal(d.view(np.int64), d0.view(np.int64))
    assert np.array_equal(p, p0)
    assert np.array_equal(y.view(np.int64), y0.view(np.int64))
    return {k: b[k] - a[k] for k in ("origin_expansions", "origin_relax_rounds")}


@pytest.mark.parametrize("N,degree", [(10000, 4), (8000, 6)])      # (fewer than 65,535 links)
def test_hbm_fronts_beyond_the_queues(engine_mod, N, degree):
    """Thousands of nodes in a round.  A node is expanded once more for each
    time its label falls after an expansion, less than twice on average here,
    whatever the queues hold."""
    print(f"case hbm wide front N={N} degree={degree}", flush=True)
    Z = 40
    net, rng = random_graph(N, degree, Z, degree)
    dem = random_demand(net, rng)
    with engine_mod.TapEngine(net, dem) as eng:
        eng.set_strategy("hbm")
        eng.aon()                                   # (the bucket width is tuned)
        for q in (-1, 200, 64):
            eng.set_origin_queue(q)
            n = _both(eng, net.fftime, rng.integers(1, net.num_nodes + 1, 20))
            assert n["origin_expansions"] <= 2.0 * N * Z, q


def test_hbm_few_expensive_links(engine_mod):
    """One link in twenty at a million times its cost: what such links gave
    nodes long reached otherwise costs no rounds."""
    print("case hbm expensive links", flush=True)
    net, dem = network("metro", 0.9)
    rng = np.random.default_rng(5)
    dear = net.fftime * np.where(rng.random(net.num_links) < 0.05, 1e6, 1.0)
    starts = rng.integers(1, net.num_nodes + 1, 20)
    with engine_mod.TapEngine(net, dem) as eng:
        eng.set_strategy("hbm")
        eng.aon()
        plain = _both(eng, net.fftime, starts)["origin_relax_rounds"]
        assert _both(eng, dear, starts)["origin_relax_rounds"] <= 1.5 * plain


@pytest.mark.parametrize("degree", [5, 6, 10, 11, 15, 16, 31])
def test_hbm_nodes_beyond_a_record(engine_mod, degree):
    """Every node has `degree` links (a record holds five), one has 2,000:
    rows of further records of every shape, with queues that hold them and
    with the smallest."""
    from traffic_assignment_amd import synth
    print(f"case hbm records degree={degree}", flush=True)
    N, Z = 1900, 30
    net, rng = random_graph(N, degree - 1, Z, 100 + degree)
    hub = np.full(2000, 700)
    init = np.concatenate([net.init, hub])
    term = np.concatenate([net.term, rng.integers(1, N + 1, hub.size)])
    order = np.lexsort((term, init))
    E = init.size
    net = synth.Network(num_zones=Z, num_nodes=N, first_thru_node=1, init=init[order], term=term[order],
                        capacity=np.full(E, 100.0), length=np.ones(E), fftime=rng.uniform(0.5, 3.0, E),
                        B=np.full(E, 0.15), power=np.full(E, 4.0), speed=np.zeros(E), toll=np.zeros(E),
                        ltype=np.ones(E, np.int16))
    dem = random_demand(net, rng)
    starts = rng.integers(1, N + 1, 40)
    starts[0] = 700
    with engine_mod.TapEngine(net, dem) as eng:
        for q in (-1, 200, 64):
            eng.set_origin_queue(q)
            for width in (0.25, 2.0):
                eng.set_origin_delta(width)
                _both(eng, net.fftime, starts)
                _both(eng, np.floor(net.fftime * 2.0), starts)           # level ties


def test_hbm_batch_memory_and_parts(engine_mod):
    """A batch beyond LDS: creation holds the mirrors of one variant (its
    loadings usually run on the lanes kernel); loadings by the labels-in-HBM
    kernel of more variants than 512 MiB of mirrors hold go by parts, and the
    free-flow volumes of variants on both sides of a part's end are those of
    the variant alone."""
    import torch
    from traffic_assignment_amd import synth
    print("case hbm batch parts", flush=True)
    N, Z, V = 60000, 4, 115
    net, rng = random_graph(N, 1, Z, 3)                  # 4.8 MB of mirrors a variant: 111 in a part
    st = np.arange(Z + 1) * (Z - 1)
    dest = np.concatenate([[d for d in range(1, Z + 1) if d != o] for o in range(1, Z + 1)])
    dem = synth.Demand(Z, st, dest, np.arange(1.0, dest.size + 1.0))
    E = net.num_links
    t0 = rng.uniform(0.5, 3.0, (V, E))

    def used():
        torch.cuda.synchronize()
        free, total = torch.cuda.mem_get_info()
        return total - free

    before = used()
    with engine_mod.TapEngine(net, dem, num_variants=V, fftime=t0) as eng:
        # nine arrays of doubles and one of bytes per link and variant, sums of the line search
        assert used() - before <= 1.05 * V * (73 * E + 65536) + (64 << 20)
        eng.set_lanes(0)
        eng.fw_init()
        x = {v: eng.flows(v)[0] for v in (0, 57, 109, 110, 111, 112, 114)}
        eng.fw_run(max_iters=2)                          # (captured, in parts)
        x2 = {v: eng.flows(v)[0] for v in x}
    for v in x:
        with engine_mod.TapEngine(net, dem, num_variants=1, fftime=t0[v:v + 1]) as one:
            one.fw_init()
            assert np.array_equal(one.flows()[0], x[v]), v
            one.fw_run(max_iters=2)
            assert np.array_equal(one.flows()[0], x2[v]), v


def test_hbm_queue_size_is_the_one_asked_for(engine_mod):
    """With no queue, or one entry, a search goes on with bitmaps at once:
    few nodes wait in a queue for a later bucket.  The results are those of
    full queues."""
    print("case hbm queue sizes", flush=True)
    net, dem = network("metro", 0.3)
    out = []
    with engine_mod.TapEngine(net, dem) as eng:
        eng.set_strategy("hbm")
        eng.set_origin_delta(1.0)
        waited = []
        for q in (-1, 0, 1, 2, 16, 65):
            eng.set_origin_queue(q)
            a = eng.stats()["origin_deferred"]
            out.append(eng.aon())
            waited.append(eng.stats()["origin_deferred"] - a)
            assert eng.origin_queue == q or q < 0
    assert 10 * max(waited[1], waited[2]) < waited[0]
    for y in out[1:]:
        assert np.array_equal(y, out[0])
