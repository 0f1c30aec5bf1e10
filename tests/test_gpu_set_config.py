"""kmcg_set_config (the database rebuilt list by list) against the oracle's
touchups one after the other: lists left by earlier steps and an earlier
configuration, every backend, one and several layers, two and three
dimensions, lattices whose lists fit LDS (up to 127 KiB of it) and lattices
whose lists do not."""
import os

import numpy as np
import pytest

from kmos_amd import workloads as W
from kmos_amd.compiler import compile_model
from kmos_amd.model import Process, load_project
from paritylib import GOLDEN, compare_state, oracle_replica, pdopd_project, random_config

pytestmark = pytest.mark.gpu

SMALL = [(8, 8), (9, 13), (16, 17), (31, 11)]


def zgb_3d():
    pt = W.zgb_project()
    pt.model_dimension = 3
    s = lambda sp, off=(0, 0, 0): W._c(sp, "site", off, "sc")  # noqa: E731
    pt.processes.append(Process("O2_adsorption3", "1.", [s("empty"), s("empty", (0, 0, 1))],
                                [s("O"), s("O", (0, 0, 1))]))
    pt.validate()
    return pt


CASES = [
    ("quickstart", W.quickstart_project, "local_smart", [(1, 1), (5, 3), (215, 211)]),
    # lists of 64 KiB and more in LDS
    ("quickstart_lds", W.quickstart_project, "local_smart", [(127, 128), (128, 128), (129, 128), (180, 180)]),
    ("ruo2_lds", W.ruo2_project, "local_smart", [(128, 128)]),
    ("zgb_3d", zgb_3d, "local_smart", [(5, 6, 7), (8, 5, 5)]),
    ("zgb_3d_li", zgb_3d, "lat_int", [(5, 6, 7), (8, 5, 5)]),
    ("zgb", W.zgb_project, "local_smart", SMALL), ("zgb_li", W.zgb_project, "lat_int", SMALL),
    ("ruo2", W.ruo2_project, "local_smart", SMALL), ("ruo2_li", W.ruo2_project, "lat_int", SMALL),
    ("pairwise", W.pairwise_project, "local_smart", SMALL), ("pairwise_li", W.pairwise_project, "lat_int", SMALL),
    ("grid", lambda: load_project(os.path.join(GOLDEN, "2d_grid.xml")), "local_smart", SMALL),
    ("pdopd", pdopd_project, "local_smart", [(4, 4), (8, 5)]), ("pdopd_li", pdopd_project, "lat_int", [(4, 4), (8, 5)]),
]


@pytest.mark.parametrize("name,factory,backend,sizes", CASES, ids=[c[0] for c in CASES])
def test_set_config_matches_oracle(engine, oracle, name, factory, backend, sizes):
    pt = factory()
    cm = compile_model(pt, backend)
    g = np.random.default_rng(23)
    n = len(sizes)
    rates = 10.0 ** g.uniform(-1, 3, (n, cm.nr_of_proc))
    seeds = g.integers(1 << 31, size=n).astype(np.uint32)
    b = engine.Batch(engine.Model(cm), [(s + (1,))[:3] for s in sizes])
    b.init(seeds, np.zeros(n, np.uint32))
    b.set_rates(rates)
    orcs = [oracle_replica(oracle, cm, s, int(seeds[i]), 0, rates[i]) for i, s in enumerate(sizes)]
    for rnd, steps in enumerate((200, 300, 50)):
        configs = [random_config(pt, int(v), g) for v in b.volumes]
        b.set_config(configs)
        for i, o in enumerate(orcs):
            o.set_config(configs[i])
            compare_state(b, i, o, where="%s %s configuration %d" % (name, sizes[i], rnd))
        b.run(steps)
        for i, o in enumerate(orcs):
            o.run(steps)
            compare_state(b, i, o, where="%s %s steps %d" % (name, sizes[i], rnd))
    b.close()


@pytest.mark.parametrize("name,factory,backend,sizes", [
    ("quickstart", W.quickstart_project, "local_smart", [(5, 3), (16, 17), (215, 211)]),
    ("ruo2", W.ruo2_project, "local_smart", [(9, 13), (16, 17)]),
    ("zgb_li", W.zgb_project, "lat_int", [(9, 13), (16, 17)]),
], ids=["quickstart", "ruo2", "zgb_li"])
def test_set_config_before_init(engine, oracle, name, factory, backend, sizes):
    """Replicas that were never initialised have empty lists, whatever the
    memory they lie in held: a configuration builds the lists from nothing."""
    pt = factory()
    cm = compile_model(pt, backend)
    g = np.random.default_rng(29)
    b = engine.Batch(engine.Model(cm), [s + (1,) for s in sizes])
    configs = [random_config(pt, int(v), g) for v in b.volumes]
    b.set_config(configs)
    for i, s in enumerate(sizes):
        o = oracle.Oracle(cm.to_blob(), s)
        o.set_config(configs[i])
        assert b.scalars(i)[4] == 0
        np.testing.assert_array_equal(b.lattice(i), o.lattice())
        np.testing.assert_array_equal(b.nr_of_sites(i), o.nr_of_sites())
        for got, want in zip(b.avail(i), o.avail()):
            np.testing.assert_array_equal(got, want)
    assert (b.check_lists() == 0).all()
    b.close()


def test_set_config_fills_and_empties_lists(engine, oracle):
    """Every cell in one list, none, every one again: an addition to a list
    one short of full, with the list in LDS and in memory."""
    pt = W.quickstart_project()
    cm = compile_model(pt, "local_smart")
    ids = pt.species_ids()
    sizes = [(1, 1), (5, 3), (16, 16), (215, 211)]
    rates = np.full((len(sizes), 2), 3.0)
    b = engine.Batch(engine.Model(cm), [s + (1,) for s in sizes])
    b.init(np.arange(len(sizes), dtype=np.uint32))
    b.set_rates(rates)
    orcs = [oracle_replica(oracle, cm, s, i, 0, rates[i]) for i, s in enumerate(sizes)]
    for species in ("CO", "empty", "CO", "CO", "empty"):
        configs = [np.full(int(v), ids[species], np.int8) for v in b.volumes]
        b.set_config(configs)
        b.run(1)
        for i, o in enumerate(orcs):
            o.set_config(configs[i])
            o.run(1)
            compare_state(b, i, o, where="%s %s" % (species, sizes[i]))
    b.close()
