"""The fused step loop's records (kmcg_model_fused) against the oracle.

Per process, the records are its routines' list updates folded into one list,
with the conditions the process's own conditions decide resolved when the
model is loaded.  Here every step the oracle takes is taken once more from
the records alone, on the lattice and lists before the step: the conditions
evaluated (lat_int: the tables looked up before and after the writes), the
updates of each process applied in order, the writes done.  Lists,
back-indices and lattice must equal the oracle's after the step, and every
deletion must find its entry.
"""
import ctypes
import os

import numpy as np
import pytest

from kmos_amd import _lib, workloads as W
from kmos_amd.compiler import compile_model
from kmos_amd.model import load_project
from paritylib import four_species_project, pdopd_project, random_config

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
FORM_1, FORM_LI, FORM_M, FORM_4 = 1, 2, 3, 4


class Records:
    def __init__(self, cm):
        lib = _lib.load()
        vp = ctypes.c_void_p
        blob = np.ascontiguousarray(cm.to_blob(), dtype=np.int32)
        h = vp()
        assert lib.kmcg_model_load(blob.ctypes.data_as(vp), blob.size, ctypes.byref(h)) == 0
        info = np.zeros(6, np.int32)
        assert lib.kmcg_model_fused(h, info.ctypes.data_as(vp), None) == 0
        words = np.zeros(max(int(info[0]), 1), np.int32)
        lib.kmcg_model_fused(h, info.ctypes.data_as(vp), words.ctypes.data_as(vp))
        lib.kmcg_model_free(h)
        self.have = bool(info[0])
        self.form, chunks, self.reach = int(info[1]), int(info[2]), int(info[3])
        if not self.have:
            return
        self.P, self.spuck = cm.nr_of_proc, cm.spuck
        n = int(info[4]) if self.form == FORM_LI else words.size
        self.rec = words[:n].reshape(self.P, chunks, 64, 4 if self.form == FORM_1 else 8)
        self.tab = words[n:].view(np.uint8)
        assert self.form != FORM_LI or self.tab.size == info[5]


def field(w, off, n, signed=False):
    v = (int(w) >> off) & ((1 << n) - 1)
    return v - (1 << n) if signed and v >> (n - 1) else v


class Cell:
    """The picked site and its row, offsets wrapped as the step loop does."""

    def __init__(self, site, size, spuck):
        self.X, self.Y, self.spuck = size[0] * spuck, size[1], spuck
        self.y, self.rem = divmod(site - 1, self.X)

    def at(self, lo, dy):
        return (self.rem + lo) % self.X + self.X * ((self.y + dy) % self.Y)

    def word(self, w):
        return self.at(field(w, 0, 16, True), field(w, 16, 16, True))


def updates_local(R, blk, cell, lat, code):
    """Per lane: process, deletes, site, takes place; per process its lanes."""
    out = []
    for q in blk:
        if R.form == FORM_1:
            conds = [(field(q[0], 18, 4), q[2])]
            at = q[1]
        else:
            conds = [(field(q[1], 4 * c, 4), q[3 + c]) for c in range(4)]
            at = q[2]
        hold = all(lat[cell.word(w)] + code == want for want, w in conds)
        out.append((field(q[0], 0, 7) - R.P, field(q[0], 31, 1), cell.word(at) + 1, hold))
    runs = []
    for p in range(R.P):
        a, n = field(blk[p][0], 7, 6), field(blk[p][0], 13, 5)
        assert all(u[0] == p for u in out[a:a + n])
        runs.append([(u[1], u[2]) for u in out[a:a + n] if u[3]])
    assert sum(len(r) for r in runs) == sum(u[3] for u in out)
    return runs


def updates_lat_int(R, blk, cell, lat, code):
    dels, adds = [[] for _ in range(R.P)], [[] for _ in range(R.P)]
    for lane, q in enumerate(blk):
        idx = sum((int(lat[cell.at(field(w, 0, 12, True), field(w, 12, 7, True))]) + code) * field(w, 19, 13)
                  for w in q[3:7])
        site = cell.word(q[1]) + 1
        place = field(q[0], 13, 4)
        for var, lst in ((int(R.tab[field(q[2], 0, 16) + idx]), dels), (int(R.tab[field(q[2], 16, 16) + idx]), adds)):
            if var:
                assert field(blk[var - 1][0], 7, 6) + place == lane
                lst[var - 1].append((place, site))
    return [[(1, s) for _, s in sorted(d)] + [(0, s) for _, s in sorted(a)] for d, a in zip(dels, adds)]


def step_from_records(R, proc, site, lat, lists, size, code):
    cell = Cell(site, size, R.spuck)
    chunks = field(R.rec[proc - 1, 0, 0, 1], 16, 5) if R.form in (FORM_M, FORM_4) else 1
    for ch in range(chunks):
        blk = R.rec[proc - 1, ch]
        for p, ups in enumerate((updates_lat_int if R.form == FORM_LI else updates_local)(R, blk, cell, lat, code)):
            for dele, s in ups:
                if dele and R.form == FORM_M and s not in lists[p]:
                    continue                   # several layers: it need not be
                if dele:
                    at = lists[p].index(s)     # registered, as its conditions hold
                    lists[p][at] = lists[p][-1]
                    lists[p].pop()
                else:
                    lists[p].append(s)
        for q in blk:
            old, new = field(q[0], 22, 4), field(q[0], 26, 4)
            if old != new:
                s = cell.word(q[-1])
                assert lat[s] == old and (R.form == FORM_M or not field(q[0], 30, 1))
                lat[s] = new


def _golden(name):
    return lambda: load_project(os.path.join(GOLDEN, name))


MODELS = [
    ("quickstart", W.quickstart_project, "local_smart", FORM_1), ("zgb", W.zgb_project, "local_smart", FORM_1),
    ("zgb_ini", _golden("zgb_model.ini"), "local_smart", FORM_1),
    ("ab_ini", _golden("ab_model.ini"), "local_smart", FORM_1), ("ruo2", W.ruo2_project, "local_smart", FORM_1),
    ("grid", _golden("2d_grid.xml"), "local_smart", FORM_1), ("pairwise", W.pairwise_project, "local_smart", FORM_4),
    ("quickstart_li", W.quickstart_project, "lat_int", FORM_LI), ("zgb_li", W.zgb_project, "lat_int", FORM_LI),
    ("ab_ini_li", _golden("ab_model.ini"), "lat_int", FORM_LI), ("ruo2_li", W.ruo2_project, "lat_int", FORM_LI),
    ("grid_li", _golden("2d_grid.xml"), "lat_int", FORM_LI), ("pdopd", pdopd_project, "local_smart", FORM_M),
    ("pairwise_li", W.pairwise_project, "lat_int", FORM_LI),
    # a byte per site on one layer
    ("four", four_species_project, "local_smart", FORM_1), ("four_li", four_species_project, "lat_int", FORM_LI),
    ("four_wide", lambda: four_species_project(True), "local_smart", FORM_4),
]


@pytest.mark.parametrize("name,factory,backend,form", MODELS, ids=[m[0] for m in MODELS])
def test_records_take_the_oracles_steps(oracle, name, factory, backend, form):
    pt = factory()
    cm = compile_model(pt, backend)
    R = Records(cm)
    assert R.have and R.form == form
    # (the null species of several layers is one more value)
    code = 1 if cm.nr_of_species + (2 if cm.null_species >= 0 else 1) <= 4 else 0
    g = np.random.default_rng(3)
    m = 2 * R.reach + 1
    for size in ((m, m, 1), (m + 2, m + 5, 1)):
        o = oracle.Oracle(cm.to_blob(), size)
        o.init(int(g.integers(1 << 30)), 0, random_config(pt, size[0] * size[1] * cm.spuck, g))
        o.set_rates(10.0 ** g.uniform(-1, 3, cm.nr_of_proc))
        for _ in range(120):
            lat = o.lattice().copy()
            sites, _ = o.avail()
            lists = [[int(s) for s in row[:n]] for row, n in zip(sites, o.nr_of_sites())]
            _, procs, at, _ = o.run(1, trace=True)
            if o.status:
                break
            step_from_records(R, int(procs[0]), int(at[0]), lat, lists, size, code)
            np.testing.assert_array_equal(lat, o.lattice())
            after, back = o.avail()
            assert [len(lst) for lst in lists] == list(o.nr_of_sites())
            for p, lst in enumerate(lists):
                assert lst == [int(s) for s in after[p][:len(lst)]]
                assert all(back[p][s - 1] == k + 1 for k, s in enumerate(lst))


def test_models_without_records():
    # a variant's table entries leave what its writes replace open
    assert not Records(compile_model(pdopd_project(), "lat_int")).have
