"""The fused step loop's records (kmcg_model_fused) against the oracle.

Per process, the records are its routines' list updates folded into one list,
with the conditions the process's own conditions decide resolved when the
model is loaded.  Here every step the oracle takes is taken once more from
the records alone, on the lattice and lists before the step: the conditions
evaluated, the updates of each process applied in order, the writes done.
Lists, back-indices and lattice must equal the oracle's after the step, and
every update must find its entry.
"""
import ctypes
import os

import numpy as np
import pytest

from kmos_amd import _lib, workloads as W
from kmos_amd.compiler import compile_model
from kmos_amd.model import load_project
from paritylib import pdopd_project, random_config

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def fused_records(cm):
    """(records [P][chunks][64][words] or None, condition words, reach)"""
    lib = _lib.load()
    blob = np.ascontiguousarray(cm.to_blob(), dtype=np.int32)
    h = ctypes.c_void_p()
    assert lib.kmcg_model_load(blob.ctypes.data_as(ctypes.c_void_p), blob.size, ctypes.byref(h)) == 0
    info = np.zeros(4, np.int32)
    assert lib.kmcg_model_fused(h, info.ctypes.data_as(ctypes.c_void_p), None) == 0
    words = np.zeros(max(int(info[0]), 1), np.int32)
    lib.kmcg_model_fused(h, info.ctypes.data_as(ctypes.c_void_p), words.ctypes.data_as(ctypes.c_void_p))
    lib.kmcg_model_free(h)
    if not info[0]:
        return None, 0, 0
    rw = 4 if info[1] == 1 else 8
    return words.reshape(cm.nr_of_proc, int(info[2]), 64, rw), int(info[1]), int(info[3])


def field(w, off, n, signed=False):
    v = (int(w) >> off) & ((1 << n) - 1)
    return v - (1 << n) if signed and v >> (n - 1) else v


def site_of(w, cell, size, spuck):
    x, y, z = ((cell[k] + field(w, 7 * k, 7, True)) % size[k] for k in range(3))
    return spuck * (x + size[0] * (y + size[1] * z)) + field(w, 21, 5)


def step_from_records(rec, proc, site, lat, lists, size, spuck, code):
    s0 = site - 1
    c = s0 // spuck
    cell = (c % size[0], c // size[0] % size[1], c // (size[0] * size[1]))
    chunks = field(rec[proc - 1, 0, 0, 0], 27, 5)
    for ch in range(chunks):
        blk = rec[proc - 1, ch]
        ups = []
        for q in blk:
            hold = bool(field(q[0], 7, 1)) and all(
                lat[site_of(q[2 + k], cell, size, spuck)] + code == field(q[2 + k], 26, 6)
                for k in range(field(q[0], 24, 3)))
            ups.append((hold, field(q[0], 0, 6), field(q[0], 6, 1), site_of(q[1], cell, size, spuck) + 1))
        covered = 0
        for p, lst in enumerate(lists):
            a, n = field(blk[p][0], 8, 6), field(blk[p][0], 16, 6)
            covered += n
            for hold, q, dele, s in ups[a:a + n]:
                assert q == p
                if not hold:
                    continue
                if dele:
                    at = lst.index(s)          # registered, as its conditions hold
                    lst[at] = lst[-1]
                    lst.pop()
                else:
                    lst.append(s)
        assert covered == sum(field(q[0], 7, 1) for q in blk)
    for q in rec[proc - 1, 0]:
        old, new = field(q[-1], 26, 3), field(q[-1], 29, 3)
        if old != new:
            s = site_of(q[-1], cell, size, spuck)
            assert lat[s] == old
            lat[s] = new


MODELS = [
    ("quickstart", W.quickstart_project, [(1, 1), (5, 4)]),
    ("zgb", W.zgb_project, [(5, 5), (6, 9)]),
    ("zgb_ini", lambda: load_project(os.path.join(GOLDEN, "zgb_model.ini")), [(5, 5), (7, 6)]),
    ("ab_ini", lambda: load_project(os.path.join(GOLDEN, "ab_model.ini")), [(7, 7), (8, 11)]),
    ("ruo2", W.ruo2_project, [(5, 5), (9, 6)]),
    ("grid", lambda: load_project(os.path.join(GOLDEN, "2d_grid.xml")), [(3, 3), (5, 4)]),
    ("pairwise", W.pairwise_project, [(7, 7), (9, 8)]),
]


@pytest.mark.parametrize("name,factory,sizes", MODELS, ids=[m[0] for m in MODELS])
def test_records_take_the_oracles_steps(oracle, name, factory, sizes):
    pt = factory()
    cm = compile_model(pt, "local_smart")
    rec, _, reach = fused_records(cm)
    assert rec is not None
    code = 1 if cm.nr_of_species + 1 <= 4 else 0
    g = np.random.default_rng(3)
    for xy in sizes:
        size = (xy[0], xy[1] if cm.dimension >= 2 else 1, 1)
        assert min(size[:cm.dimension]) >= 2 * reach + 1
        o = oracle.Oracle(cm.to_blob(), size)
        o.init(int(g.integers(1 << 30)), 0, random_config(pt, size[0] * size[1] * cm.spuck, g))
        o.set_rates(10.0 ** g.uniform(-1, 3, cm.nr_of_proc))
        for _ in range(150):
            lat = o.lattice().copy()
            sites, back = o.avail()
            lists = [[int(s) for s in row[:n]] for row, n in zip(sites, o.nr_of_sites())]
            _, procs, at, _ = o.run(1, trace=True)
            if o.status:
                break
            step_from_records(rec, int(procs[0]), int(at[0]), lat, lists, size, cm.spuck, code)
            np.testing.assert_array_equal(lat, o.lattice())
            after, back = o.avail()
            for p, lst in enumerate(lists):
                assert lst == [int(s) for s in after[p][:len(lst)]] and len(lst) == o.nr_of_sites()[p]
                assert all(back[p][s - 1] == k + 1 for k, s in enumerate(lst))


def test_models_without_records():
    # several layers, more than 64 processes' routines, process groups
    for pt, backend in ((pdopd_project(), "local_smart"), (W.ruo2_project(), "lat_int")):
        assert fused_records(compile_model(pt, backend))[0] is None
