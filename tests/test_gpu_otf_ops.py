"""The otf step loop with one lane per list operation against the oracle at
the edges of its rule: the smallest extents on which no two offsets of the
operations meet, lists whose ends lie on and beside a checkpoint block of 16,
and batches in which one smaller lattice sends every replica through the
general loop."""
import numpy as np
import pytest

from test_gpu_otf import _compare, _intzgb, _ruo2, otf_engine, otf_oracle  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("small", [False, True], ids=["ops", "general"])
@pytest.mark.parametrize("model", ["ruo2", "intzgb"])
def test_otf_edges_match_oracle(otf_engine, otf_oracle, model, small):  # noqa: F811
    cm, base = _ruo2() if model == "ruo2" else _intzgb()
    x, y = (2 * max(abs(op.off[d]) for ops in cm.otf_programs for op in ops) + 1 for d in range(2))
    sizes = [(x, y), (x, y + 3), (16, y), (16, 16), (31, 11), (33, 16)] + ([(x - 1, y + 1)] if small else [])
    n, P = len(sizes), cm.nr_of_proc
    g = np.random.default_rng(41)
    rates = base[None, :] * 10.0 ** g.uniform(-0.5, 0.5, (n, P))
    userpar = g.uniform(0.6, 1.6, (n, len(cm.param_names)))
    seeds = g.integers(1 << 31, size=n).astype(np.uint32)
    b = otf_engine.OtfBatch(otf_engine.OtfModel(cm), sizes)
    b.set_params(rates, userpar)
    b.init(seeds, np.arange(n, dtype=np.uint32))
    orcs = []
    for r, s in enumerate(sizes):
        o = otf_oracle.OtfOracle(cm.to_blob(), s)
        o.init(int(seeds[r]), r)
        o.set_params(rates[r], userpar[r])
        if r % 2:
            cfg = g.integers(0, cm.nr_of_species, int(b.volumes[r])).astype(np.int8)
            b.set_config([cfg], r0=r)
            assert o.set_config(cfg) == 0
        orcs.append(o)
    for steps in (1, 62, 2, 700):
        b.run(steps)
        assert b.last_form() == (0 if small else 1)
        for r, o in enumerate(orcs):
            o.run(steps)
            _compare(b, r, o, "%s %s" % (model, sizes[r]))
    b.close()
