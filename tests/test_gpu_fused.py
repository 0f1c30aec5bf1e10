"""The fused step loop against the oracle where its rules have edges: the
smallest extents it takes and the largest it leaves to the generic loop, one
and several chunks of records per process, the refill of the uniforms after
64 steps, a stopped replica in the launch."""
import os

import numpy as np
import pytest

from kmos_amd import workloads as W
from kmos_amd.acf import displacement_table
from kmos_amd.compiler import compile_model
from kmos_amd.model import load_project
from paritylib import compare_state, four_species_project, oracle_replica, pdopd_project, random_config
from test_fused_records import FORM_M, GOLDEN, Records

pytestmark = pytest.mark.gpu



def one_dimension(pt):
    """The processes of a model that lie in a row."""
    pt.model_dimension = 1
    pt.processes = [p for p in pt.processes if not any(c.coord.offset[1] for c in p.conditions + p.actions)]
    pt.validate()
    return pt


CASES = [
    # one chunk of one-condition records, several chunks of wide ones, lat_int
    ("quickstart", W.quickstart_project, "local_smart"), ("zgb", W.zgb_project, "local_smart"),
    ("ruo2", W.ruo2_project, "local_smart"), ("pairwise", W.pairwise_project, "local_smart"),
    ("ab_ini", lambda: load_project(os.path.join(GOLDEN, "ab_model.ini")), "local_smart"),
    ("pdopd", pdopd_project, "local_smart"),        # several layers
    ("zgb_li", W.zgb_project, "lat_int"), ("ruo2_li", W.ruo2_project, "lat_int"),
    ("pairwise_li", W.pairwise_project, "lat_int"),
    # a byte per site on one layer
    ("four", four_species_project, "local_smart"), ("four_li", four_species_project, "lat_int"),
    ("four_wide", lambda: four_species_project(True), "local_smart"),
    ("one_dimension", lambda: one_dimension(W.zgb_project()), "local_smart"),
    ("one_dimension_li", lambda: one_dimension(W.zgb_project()), "lat_int"),
]
# each with the fused loop, with one lattice below its extents (where the
# model runs on such a one) and with the generic loop asked for
WAYS = [c + (way,) for c in CASES for way in ("fused", "below_the_extent", "generic")
        if way != "below_the_extent" or c[0] != "pdopd"]


def least_extent(cm, R):
    """The smallest lattice side the fused loop takes: no two offsets of the
    records meet, and a row has more than one site."""
    return max(2 * R.reach + 1, 1 if cm.spuck > 1 else 2)


@pytest.mark.parametrize("name,factory,backend,way", WAYS, ids=["%s-%s" % (c[0], c[3]) for c in WAYS])
def test_edges_match_oracle(engine, oracle, name, factory, backend, way):
    pt = factory()
    cm = compile_model(pt, backend)
    R = Records(cm)
    assert R.have
    m = least_extent(cm, R)
    sizes = [(m, m), (m, m + 3), (m + 4, m), (31, 17), (64, 33)]
    if way == "below_the_extent":
        sizes.append((m - 1, m + 2))       # the whole launch runs the generic loop
    g = np.random.default_rng(17)
    n = len(sizes)
    rates = 10.0 ** g.uniform(-1, 3, (n, cm.nr_of_proc))
    rates[0] = 0.0                          # no process possible: stops at once
    seeds = g.integers(1 << 31, size=n).astype(np.uint32)
    b = engine.Batch(engine.Model(cm), [s + (1,) for s in sizes])
    b.init(seeds, np.arange(n, dtype=np.uint32))
    b.set_rates(rates)
    if way == "generic":
        b.set_overlap(0)
    configs = [random_config(pt, int(v), g) for v in b.volumes]
    b.set_config(configs)
    orcs = [oracle_replica(oracle, cm, s, int(seeds[i]), i, rates[i], configs[i]) for i, s in enumerate(sizes)]
    for steps in (1, 2, 61, 1, 140, 795):
        b.run(steps)
        assert b.last_form() == (R.form if way == "fused" else 0)
        for i, o in enumerate(orcs):
            o.run(steps)
            compare_state(b, i, o, where="%s %s" % (name, sizes[i]))
    assert b.scalars(0)[4] == 1
    ok = b.scalars_all()[2] <= 1
    assert (b.check_lists()[ok] == 0).all()
    b.close()


def test_layers_stop_where_the_oracle_stops(engine, oracle):
    """Several layers on lattices of any species anywhere: steps whose write
    finds another species are left to the generic loop, which stops there."""
    pt = pdopd_project()
    cm = compile_model(pt, "local_smart")
    g = np.random.default_rng(5)
    n = 30
    sizes = [(6, 5) if i % 2 else (7, 9) for i in range(n)]
    rates = 10.0 ** g.uniform(-1, 3, (n, cm.nr_of_proc))
    b = engine.Batch(engine.Model(cm), [s + (1,) for s in sizes])
    b.init(np.arange(n, dtype=np.uint32), np.zeros(n, np.uint32))
    b.set_rates(rates)
    configs = [g.integers(0, cm.nr_of_species + 1, int(v)).astype(np.int8) for v in b.volumes]
    b.set_config(configs)
    orcs = [oracle_replica(oracle, cm, s, i, 0, rates[i], configs[i]) for i, s in enumerate(sizes)]
    for steps, limits in ((100, None), (400, 150 + 10 * np.arange(n)), (900, None)):
        left = b.run(steps, budget=limits)
        assert b.last_form() == FORM_M
        for i, o in enumerate(orcs):
            before = o.kmc_step
            o.run(steps if limits is None else int(min(steps, limits[i])))
            compare_state(b, i, o, where="replica %d" % i)
            if limits is not None and o.status == 0:
                assert left[i] == limits[i] - (o.kmc_step - before)
    stops = b.scalars_all()[2]
    assert (stops == 2).any() and (stops == 0).any()
    b.close()


@pytest.mark.parametrize("overlap", [-1, 0], ids=["fused", "generic"])
@pytest.mark.parametrize("backend", ["local_smart", "lat_int"])
@pytest.mark.parametrize("factory,species", [(W.pairwise_project, "A"), (four_species_project, "N")],
                         ids=["pairwise", "four"])
def test_moves_match_oracle(engine, oracle, factory, species, backend, overlap):
    """Particle moves, written one step after their hop: launches that end
    on a hop, particles without a number (adsorbed after the start), a
    trajectory that fills up inside a launch, a stopped replica."""
    pt = factory()
    cm = compile_model(pt, backend)
    hops, disp = displacement_table(cm)
    R = Records(cm)
    assert R.have
    m = 2 * R.reach + 1
    sizes = [(m, m), (m, m + 3), (31, 17), (64, 33)]
    g = np.random.default_rng(23)
    n = len(sizes)
    rates = 10.0 ** g.uniform(-1, 3, (n, cm.nr_of_proc))
    rates[0] = 0.0
    ids = pt.species_ids()
    seeds = g.integers(1 << 31, size=n).astype(np.uint32)
    b = engine.Batch(engine.Model(cm), [s + (1,) for s in sizes])
    b.init(seeds, np.arange(n, dtype=np.uint32))
    b.set_rates(rates)
    configs = [np.where(g.random(int(v)) < 0.4, ids[species], ids["empty"]).astype(np.int8) for v in b.volumes]
    b.set_config(configs)
    b.msd_init(ids[species], hops, disp)
    b.msd_trajectory(300)
    b.set_overlap(overlap)
    orcs = []
    for i, s in enumerate(sizes):
        o = oracle_replica(oracle, cm, s, int(seeds[i]), i, rates[i], configs[i])
        o.msd_init(ids[species], hops, disp)
        o.msd_trajectory(300)
        orcs.append(o)
    for steps in (1, 2, 61, 1, 140, 395):
        b.run_displacement(steps, traj_on=True)
        assert b.last_form() == (0 if overlap == 0 else R.form)
        for i, o in enumerate(orcs):
            o.run_displacement(steps, traj_on=True)
            got, want = b.msd_state(i), o.msd_state()
            for key in ("nr_of_ions", "site_arr", "id_arr", "displacement", "events"):
                np.testing.assert_array_equal(got[key], want[key], err_msg="%s %s" % (sizes[i], key))
            compare_state(b, i, o, where="%s %s" % (backend, sizes[i]))
    assert b.scalars(0)[4] == 1
    b.close()
