"""Lists that do not follow the lattice: a run has to stop where it finds
that, as the oracle does, and must not write there.

local_smart: in the oracle's state.  lat_int: at the oracle's step with a
stop status (the deletion of an entry that is not registered is undefined in
the reference, and the engine applies a step's deletions after its writes)."""
import numpy as np
import pytest

from kmos_amd import workloads as W
from kmos_amd.compiler import compile_model
from paritylib import compare_state, oracle_replica
from test_fused_records import Records

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("way", ["touchup", "run_proc_nr"])
@pytest.mark.parametrize("backend", ["local_smart", "lat_int"])
def test_new_lattice_of_a_stopped_replica(engine, oracle, backend, way):
    """A stopped replica keeps its lists when set_config replaces its lattice;
    touchup and run_proc_nr let it go on."""
    pt = W.zgb_project()
    cm = compile_model(pt, backend)
    sid = pt.species_ids()
    sizes = [(12, 16), (9, 18)]
    seeds = np.array([5, 6], np.uint32)
    rates = np.tile([5.0, 1.0, 1.0, 1.0, 1.0, 0.5, 0.5], (2, 1))
    b = engine.Batch(engine.Model(cm), [s + (1,) for s in sizes])
    b.init(seeds)
    b.set_rates(rates)
    orcs = [oracle_replica(oracle, cm, s, int(seeds[r]), 0, rates[r]) for r, s in enumerate(sizes)]
    b.run(40)
    b.set_rates(0.0 * rates)
    b.run(1)
    for o in orcs:
        o.run(40)
        o.set_rates(0.0 * rates[0])
        o.run(1)
    assert list(b.scalars_all()[2]) == [1, 1] and all(o.status == 1 for o in orcs)
    # other species in the lower rows, the upper ones as they are
    g = np.random.default_rng(2)
    before = [b.avail(r) for r in range(2)]
    configs = []
    for r, (X, Y) in enumerate(sizes):
        lat = b.lattice(r).copy()
        lat[:X * (Y // 2)] = g.integers(0, cm.nr_of_species, X * (Y // 2))
        configs.append(lat)
    b.set_config(configs)
    b.set_rates(rates)
    for r, o in enumerate(orcs):
        st = o.get_state(rates[r])
        st["lattice"] = configs[r]
        o.set_state(st)
        for got, kept in zip(b.avail(r), before[r]):
            np.testing.assert_array_equal(got, kept)
        X, Y = sizes[r]
        if way == "touchup":
            b.touchup(r, 1, Y - 4, 0, 1)
            o.touchup(1, Y - 4, 0, 1)
        else:
            # CO adsorbs on an empty site far from the rows that changed
            x = int(np.nonzero(configs[r].reshape(Y, X)[Y - 4] == sid["empty"])[0][0])
            proc = cm.process_names.index("CO_adsorption") + 1
            b.run_proc_nr(r, proc, (Y - 4) * X + x + 1)
            o.run_proc_nr(proc, (Y - 4) * X + x + 1)
        compare_state(b, r, o, where="%s replica %d" % (way, r))
        assert o.status == 0
    b.run(300)
    for r, o in enumerate(orcs):
        o.run(300)
        assert o.status != 0
        if backend == "local_smart":
            compare_state(b, r, o, where="%s replica %d after its stop" % (way, r))
        else:
            _, _, ks, ctr, st = b.scalars(r)
            assert st in (2, 3) and ks == o.kmc_step and ctr == o.rng_ctr, (st, ks, o.kmc_step)
    b.close()


def test_entries_listed_twice(engine, oracle):
    """A step on a database that replace_species left stale adds entries that
    are listed already.  set_config takes one of the two away, as the oracle
    does; the run then stops where a step finds that the other does not
    hold."""
    pt = W.zgb_project()
    cm = compile_model(pt, "local_smart")
    sid = pt.species_ids()
    X, Y = 12, 10
    rates = np.array([[0.5, 1.0, 1.0, 1.0, 1.0, 5.0, 5.0]])
    g = np.random.default_rng(4)
    lat = g.choice([sid["O"], sid["empty"]], size=X * Y).astype(np.int8)
    rows = lat.reshape(Y, X)
    rows[3, 2:6] = [sid["empty"], sid["empty"], sid["O"], sid["empty"]]
    rows[2, 3] = rows[4, 3] = sid["empty"]
    b = engine.Batch(engine.Model(cm), [(X, Y, 1)])
    b.init([5], [0])
    b.set_rates(rates)
    b.set_config([lat])
    o = oracle_replica(oracle, cm, (X, Y), 5, 0, rates[0], lat)
    site, proc = 3 * X + 3 + 1, cm.process_names.index("CO_oxidation1") + 1
    b.replace_species(0, site, sid["empty"], sid["CO"])
    oracle.lib().orc_replace_species(o.h, site, sid["empty"], sid["CO"])
    b.run_proc_nr(0, proc, site)
    o.run_proc_nr(proc, site)
    compare_state(b, 0, o, where="after the step")
    sites, _ = o.avail()
    listed = [s[:n] for s, n in zip(sites, o.nr_of_sites())]
    assert any(np.unique(s).size < s.size for s in listed)
    new = g.integers(0, cm.nr_of_species, X * Y).astype(np.int8)
    b.set_config([new])
    o.set_config(new)
    compare_state(b, 0, o, where="after set_config")
    b.run(400)
    o.run(400)
    assert o.status == 2
    compare_state(b, 0, o, where="after the run")
    b.close()


def test_restored_entries_of_another_site_type(engine, oracle):
    """set_state takes lists as they are given, a site of a type that the
    process never runs on among them; set_config leaves what the oracle's
    touchups leave."""
    pt = W.ruo2_project()
    cm = compile_model(pt, "local_smart")
    g = np.random.default_rng(8)
    size = (7, 6)
    rates = 10.0 ** g.uniform(-1, 3, (1, cm.nr_of_proc))
    b = engine.Batch(engine.Model(cm), [size + (1,)])
    b.init([5], [0])
    b.set_rates(rates)
    b.run(60)
    o = oracle_replica(oracle, cm, size, 5, 0, rates[0])
    o.run(60)
    st = o.get_state(rates[0])
    p = int(np.argmax(st["nr_of_sites"]))
    k = int(st["nr_of_sites"][p])
    other = int(st["avail_sites"][p, 0]) + (1 if st["avail_sites"][p, 0] % 2 else -1)
    st["avail_sites"][p, k] = other
    st["avail_sites_back"][p, other - 1] = k + 1
    st["nr_of_sites"][p] = k + 1
    b.set_state(0, st)
    o.set_state(st)
    compare_state(b, 0, o, where="restored")
    new = g.integers(0, cm.nr_of_species, int(b.volumes[0])).astype(np.int8)
    b.set_config([new])
    o.set_config(new)
    compare_state(b, 0, o, where="after set_config")
    b.run(200)
    o.run(200)
    compare_state(b, 0, o, where="after the run")
    b.close()


@pytest.mark.parametrize("backend", ["local_smart", "lat_int"])
def test_stopped_replica_among_others(engine, oracle, backend):
    """A stopped replica takes no step, so its lists keep no other replica
    from the fused loop; let go on by a touchup, they do."""
    pt = W.zgb_project()
    cm = compile_model(pt, backend)
    form = Records(cm).form
    g = np.random.default_rng(12)
    sizes = [(9, 8), (12, 10), (7, 11)]
    rates = 10.0 ** g.uniform(-1, 1, (3, cm.nr_of_proc))
    b = engine.Batch(engine.Model(cm), [s + (1,) for s in sizes])
    b.init([5, 6, 7])
    b.set_rates(rates)
    b.set_rates(0.0 * rates[:1], r0=1)
    b.run(20)
    orcs = [oracle_replica(oracle, cm, s, 5 + r, 0, rates[r]) for r, s in enumerate(sizes)]
    orcs[1].set_rates(0.0 * rates[1])
    configs = [g.integers(0, cm.nr_of_species, int(v)).astype(np.int8) for v in b.volumes]
    b.set_config(configs)
    b.set_rates(rates)
    b.run(100)
    assert b.last_form() == form
    for r, o in enumerate(orcs):
        o.run(20)
        if r != 1:
            o.set_config(configs[r])
            o.run(100)
            compare_state(b, r, o, where="replica %d" % r)
    assert b.scalars(1)[4] == 1 and b.scalars(1)[2] == 0
    np.testing.assert_array_equal(b.lattice(1), configs[1])
    b.touchup(1, 0, 0, 0, 1)
    assert b.scalars(1)[4] == 0
    b.run(1)
    assert b.last_form() == 0
    b.set_config(configs[:1])
    b.run(1, [0, 2])
    assert b.last_form() == form
    b.close()


@pytest.mark.parametrize("backend", ["local_smart", "lat_int"])
def test_process_that_stops_halfway(engine, oracle, backend):
    """run_proc_nr of a process whose action finds another species stops the
    replica, in lat_int with its deletions done: the lists are not taken for
    the lattice's when a touchup elsewhere lets it go on."""
    pt = W.zgb_project()
    cm = compile_model(pt, backend)
    sid = pt.species_ids()
    X, Y = 10, 12
    rates = np.array([[5.0, 1.0, 1.0, 1.0, 1.0, 0.5, 0.5]])
    b = engine.Batch(engine.Model(cm), [(X, Y, 1)])
    b.init([5])
    b.set_rates(rates)
    b.run(30)
    assert b.last_form() == Records(cm).form
    o = oracle_replica(oracle, cm, (X, Y), 5, 0, rates[0])
    o.run(30)
    site = int(np.nonzero(o.lattice() == sid["CO"])[0][0]) + 1
    proc = cm.process_names.index("CO_adsorption") + 1
    b.run_proc_nr(0, proc, site)
    o.run_proc_nr(proc, site)
    assert b.scalars(0)[4] in (2, 3) and o.status == 2
    b.touchup(0, (site - 1 + X // 2) % X, ((site - 1) // X + Y // 2) % Y, 0, 1)
    assert b.scalars(0)[4] == 0
    b.run(200)
    assert b.last_form() == 0
    if backend == "local_smart":
        o.set_state(o.get_state(rates[0]))
        o.touchup((site - 1 + X // 2) % X, ((site - 1) // X + Y // 2) % Y, 0, 1)
        o.run(200)
        compare_state(b, 0, o, where="after the touchup")
    b.close()
