"""Performance cases: the work a user has this engine do, through its public
entry points, over the sizes its workloads, tests and configurations use.

listed()            the named cases
draw(rng)           one more case of the same ranges
prepare(case, seed) models, batches and lattices a program holds before a call
run(state)          one pass through the public entry points and its outputs
work(case)          bytes and FP64 operations one pass cannot do without
exact(case, seed)   run()'s outputs in plain numpy, where that is feasible

A pass continues its trajectories, as a program that samples a run does, but
for "serve" and "config", which start from given lattices each time.
"""
import os
import tempfile

import numpy as np

from kmos_amd import acf, workloads
from kmos_amd.compiler import compile_model
from kmos_amd.engine import Batch, Model
from kmos_amd.export import export_source
from kmos_amd.model import load_project
from kmos_amd.otf_engine import OtfBatch, OtfModel
from kmos_amd.run import KMC_Model

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# bytes of avail_sites / back-index entries the step algorithm itself reads
# and writes per kMC step (4 per int32 entry, counted on the CPU
# restatement of the algorithm once the lattice is populated)
STEP_BYTES = {
    ("quickstart", "local_smart"): 36, ("zgb", "local_smart"): 115, ("zgb", "lat_int"): 98,
    ("ruo2", "local_smart"): 317, ("ruo2", "lat_int"): 250,
    ("pairwise", "local_smart"): 1416, ("pairwise", "lat_int"): 521,
    ("pdopd", "local_smart"): 49, ("pdopd", "lat_int"): 59,
    ("ruo2", "otf"): 580,
}
NPROC = {"quickstart": 2, "zgb": 7, "ruo2": 36, "pairwise": 49, "pdopd": 46, "intzgb": 10}
SPUCK = {"quickstart": 1, "zgb": 1, "ruo2": 2, "pairwise": 1, "pdopd": 25, "intzgb": 1}
# share of the sites that hold each species at the start, per model; the
# rest is empty
COVERAGE = {"ruo2": {"co": 0.3, "oxygen": 0.3}, "pairwise": {"A": 0.4}}


def _case(name, kind, model, backend, replicas, sides, steps):
    return {"name": name, "kind": kind, "model": model, "backend": backend, "replicas": replicas,
            "sides": sides, "steps": steps}


def listed():
    return [
        # the smallest call: a short run of one small lattice, then its
        # sample record (the `kmos benchmark` model and size)
        _case("quickstart_100_steps", "batch", "quickstart", "local_smart", 1, "20", 100),
        # one RuO2 trajectory through the KMC_Model front end, read as
        # get_atoms reads it: what an interactive user waits for
        _case("ruo2_front_end", "front", "ruo2", "local_smart", 1, "64", 2000),
        # the throughput workloads: full chip, ordinary lattices
        _case("zgb_4096", "batch", "zgb", "local_smart", 4096, "128", 1000),
        # ... 2048 replicas of three sizes, 36 processes with stiff rates
        _case("ruo2_mix_2048", "batch", "ruo2", "local_smart", 2048, "20,64,64,128", 1000),
        # ... lateral interactions as lat_int process groups, large lattices
        _case("pairwise_512", "batch", "pairwise", "lat_int", 512, "256", 1000),
        # lat_int without lateral interactions, a part-filled chip, odd sizes
        _case("ruo2_lat_int_odd", "batch", "ruo2", "lat_int", 300, "17x23,31x9,45x64,101x63", 1000),
        # two layers, 25 sites per cell: one byte per site, small lattices
        _case("pdopd_layers", "batch", "pdopd", "local_smart", 256, "8,12x20,20", 1000),
        # rates from each site's surroundings, full chip
        _case("intzgb_otf_2048", "otf", "intzgb", "otf", 2048, "64", 4000),
        # one otf trajectory through the KMC_Model front end
        _case("ruo2_otf_front_end", "front", "ruo2", "otf", 1, "20", 1000),
        # particle tracking for mean squared displacements
        _case("pairwise_tracking", "track", "pairwise", "local_smart", 32, "128", 4000),
        # a server's tick: new requests start from their lattices and run
        # four sampling intervals in one launch, sizes mixed
        _case("serve_mix", "serve", "zgb", "local_smart", 200, "20,64,128,256", 2000),
        # load a configuration: the database rebuilt for a given lattice
        _case("ruo2_set_config", "config", "ruo2", "local_smart", 1, "64", 0),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _side(rng, lo, hi):
    """One lattice size: square or not, odd ones among them."""
    x = _log_int(rng, lo, hi)
    return "%d" % x if rng.random() < 0.4 else "%dx%d" % (x, _log_int(rng, lo, hi))


def draw(rng):
    kind = rng.choice(["batch", "batch", "batch", "otf", "front", "track", "serve", "config"])
    if kind == "batch":
        model = rng.choice(["quickstart", "zgb", "ruo2", "pairwise", "pdopd"])
        backend = rng.choice(["local_smart", "lat_int"]) if model != "quickstart" else "local_smart"
        big = {"quickstart": 4096, "zgb": 4096, "ruo2": 1500, "pairwise": 512, "pdopd": 256}[model]
        lo, hi = {"pairwise": (20, 200), "pdopd": (6, 20)}.get(model, (12, 128))
        sides = ",".join(_side(rng, lo, hi) for _ in range(rng.randint(1, 4)))
        return {k: v for k, v in _case("", kind, model, backend, _log_int(rng, 1, big), sides,
                                       _log_int(rng, 50, 1000)).items() if k != "name"}
    if kind == "otf":
        c = _case("", kind, "intzgb", "otf", _log_int(rng, 8, 2048),
                  ",".join(_side(rng, 12, 64) for _ in range(rng.randint(1, 3))), _log_int(rng, 200, 4000))
    elif kind == "front":
        model, backend = rng.choice([("ruo2", "local_smart"), ("ruo2", "lat_int"), ("ruo2", "otf"),
                                     ("intzgb", "otf"), ("zgb", "local_smart")])
        c = _case("", kind, model, backend, 1, _side(rng, 12, 64), _log_int(rng, 50, 4000))
    elif kind == "track":
        c = _case("", kind, "pairwise", rng.choice(["local_smart", "lat_int"]), _log_int(rng, 1, 32),
                  _side(rng, 20, 128), _log_int(rng, 200, 4000))
    elif kind == "serve":
        c = _case("", kind, rng.choice(["zgb", "ruo2", "quickstart"]), "local_smart", _log_int(rng, 1, 200),
                  ",".join(_side(rng, 20, 200) for _ in range(rng.randint(1, 4))), 4 * _log_int(rng, 50, 1000))
    else:
        c = _case("", kind, rng.choice(["ruo2", "zgb", "pairwise"]), rng.choice(["local_smart", "lat_int"]),
                  rng.randint(1, 8), _side(rng, 12, 64), 0)
    return {k: v for k, v in c.items() if k != "name"}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

_projects = {}
_compiled = {}
_exports = {}


def _project(model):
    if model not in _projects:
        _projects[model] = {
            "quickstart": workloads.quickstart_project, "zgb": workloads.zgb_project,
            "ruo2": workloads.ruo2_project, "pairwise": workloads.pairwise_project,
            "intzgb": workloads.intzgb_otf_project,
            "pdopd": lambda: load_project(os.path.join(ROOT, "tests", "golden", "pdopd.xml")),
        }[model]()
    return _projects[model]


def _compile(model, backend):
    if (model, backend) not in _compiled:
        _compiled[model, backend] = compile_model(_project(model), backend)
    return _compiled[model, backend]


def _export(model, backend):
    """The model's export directory, written once as a user's program does."""
    if (model, backend) not in _exports:
        d = tempfile.mkdtemp(prefix="kmc_export_")
        _exports[model, backend] = export_source(_project(model), d, backend)
    return _exports[model, backend]


def _sizes(case):
    sides = []
    for s in case["sides"].split(","):
        x, _, y = s.partition("x")
        sides.append((int(x), int(y or x), 1))
    return [sides[i] for i in np.sort(np.arange(case["replicas"]) % len(sides))]


def _gen(seed):
    return np.random.Generator(np.random.Philox(key=int(seed)))


def _rates(case, g):
    n, model = case["replicas"], case["model"]
    pt = _project(model)
    P = len(pt.processes)
    if model == "quickstart":
        return np.full((n, P), 100.0)
    if model == "zgb":
        # inside the reactive window, so that no replica poisons
        y = g.uniform(0.41, 0.51, n)
        out = np.full((n, P), 1e10)
        for i, p in enumerate(pt.processes):
            if p.name == "CO_adsorption":
                out[:, i] = y
            elif p.name.startswith("O2_adsorption"):
                out[:, i] = (1.0 - y) / 2.0
        return out
    if model == "ruo2":
        return 10.0 ** g.uniform(-2.0, 9.0 if case["backend"] != "otf" else 6.0, (n, P))
    if model == "pairwise":
        return np.stack([workloads.pairwise_rates(pt, e) for e in g.uniform(-0.2, 0.2, n)])
    if model == "pdopd":
        return 10.0 ** g.uniform(-2.0, 4.0, (n, P))
    raise ValueError(model)


def _lattices(case, sizes, g):
    """Random lattices at the model's coverage, or None (default species)."""
    cov = COVERAGE.get(case["model"])
    if cov is None:
        return None
    ids = _project(case["model"]).species_ids()
    V = np.array([x * y * SPUCK[case["model"]] for x, y, _ in sizes])
    u = g.random(int(V.sum()), dtype=np.float32)
    flat = np.full(u.size, ids["empty"], np.int8)
    lo = 0.0
    for sp, c in cov.items():
        flat[(u >= lo) & (u < lo + c)] = ids[sp]
        lo += c
    return np.split(flat, np.cumsum(V)[:-1])


def _steps_before(case, sizes):
    """Steps run before the first pass, past the first transient."""
    if case["model"] == "quickstart":
        return 0
    if case["model"] == "zgb":
        return 2 * max(x * y for x, y, _ in sizes) if len(sizes) * max(x * y for x, y, _ in sizes) > 1 << 20 else 20000
    return 2000


def _front(case, seed):
    x, y, _ = _sizes(case)[0]
    m = KMC_Model(export_dir=_export(case["model"], case["backend"]), size=[x, y], random_seed=int(seed) % (1 << 31))
    g = _gen(seed)
    if case["model"] in ("zgb", "ruo2"):
        for name, k in zip(m.compiled.process_names, _rates(case, g)[0]):
            m.rate_constants.set(name, float(k))
        if case["backend"] == "otf":
            m.proclist.recalculate_rates_matrix()
    elif case["model"] == "intzgb":
        m.parameters.yCO = float(g.uniform(0.41, 0.51))
    cfg = _lattices(case, [(x, y, 1)], g)
    if cfg is not None:
        m._set_configuration(cfg[0].reshape(1, y, x, -1).transpose(2, 1, 0, 3))
    m.do_steps(1000)
    m.get_atoms(geometry=False)
    return {"kind": "front", "model": m, "steps": case["steps"]}


def _otf(case, seed):
    sizes = _sizes(case)
    n = case["replicas"]
    wl = workloads.intzgb_otf(n, seed=int(seed))
    b = OtfBatch(OtfModel(_compile("intzgb", "otf")), sizes)
    b.set_params(wl.rates, wl.userpar)
    b.init(np.full(n, seed % (1 << 32), np.uint32), np.arange(n, dtype=np.uint32))
    b.run(2000)
    return {"kind": "otf", "batch": b, "steps": case["steps"]}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "front":
        return _front(case, seed)
    if kind == "otf":
        return _otf(case, seed)
    g = _gen(seed)
    sizes = _sizes(case)
    n = case["replicas"]
    cm = _compile(case["model"], case["backend"])
    b = Batch(Model(cm), sizes)
    seeds, streams = np.full(n, seed % (1 << 32), np.uint32), np.arange(n, dtype=np.uint32)
    rates = _rates(case, g)
    lattices = _lattices(case, sizes, g)
    state = {"kind": kind, "batch": b, "steps": case["steps"], "ids": np.arange(n, dtype=np.int32)}
    if kind == "serve":
        if lattices is None:
            # requests of the absorbing models start from a run's lattice
            b.init(seeds, streams + np.uint32(n))
            b.set_rates(rates)
            b.run(5000)
            lattices = [b.lattice(r) for r in range(n)]
        state.update(seeds=seeds, streams=streams, rates=rates, lattices=lattices,
                     budget=np.full(n, case["steps"], np.int64))
        return state
    b.init(seeds, streams, configs=None if kind == "config" else lattices)
    b.set_rates(rates)
    if kind == "config":
        if lattices is None:
            b.run(3000)
            lattices = [b.lattice(r) for r in range(n)]
        state["lattices"] = lattices
        return state
    before = _steps_before(case, sizes)
    if before:
        b.run(before)
    if kind == "track":
        hops, disp = acf.displacement_table(cm)
        b.msd_init(_project(case["model"]).species_ids()["A"], hops, disp)
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(state):
    kind = state["kind"]
    if kind == "front":
        m = state["model"]
        m.do_steps(state["steps"])
        a = m.get_atoms(geometry=False)
        return {"kmc_time": a.kmc_time, "kmc_step": a.kmc_step, "procstat": a.procstat,
                "occupation": np.asarray(a.occupation), "integ_rates": a.integ_rates, "tof": a.tof_integ}
    b = state["batch"]
    if kind == "otf":
        b.run(state["steps"])
        c = [b.counters(r) for r in range(b.n)]
        s = [b.scalars_full(r) for r in range(b.n)]
        out = {k: np.stack([x[k] for x in c]) for k in c[0]}
        out["kmc_time"] = np.array([x[0] for x in s])
        out["kmc_step"] = np.array([x[2] for x in s])
        return out
    ids = state["ids"]
    if kind == "batch":
        b.run(state["steps"])
        return b.sample(ids)
    if kind == "track":
        b.run_displacement(state["steps"])
        out = b.sample(ids)
        msd = [b.msd_state(r) for r in range(b.n)]
        out["displacement"] = np.concatenate([x["displacement"] for x in msd])
        out["site_arr"] = np.concatenate([x["site_arr"] for x in msd])
        return out
    if kind == "serve":
        b.init(state["seeds"], state["streams"], configs=state["lattices"])
        b.set_rates(state["rates"])
        every = state["steps"] // 4
        left, recs = b.run_recorded(state["steps"], ids, state["budget"], every, 4)()
        return {"left": left, **{k: np.concatenate([r[k] for r in recs]) for k in recs[0]}}
    # the database of each replica rebuilt for its lattice
    b.set_config(state["lattices"])
    out = {"nr_of_sites": np.stack([b.nr_of_sites(r) for r in range(b.n)])}
    av = [b.avail(r) for r in range(b.n)]
    out["sites"] = np.concatenate([s.reshape(-1) for s, _ in av])
    out["back"] = np.concatenate([k.reshape(-1) for _, k in av])
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    n, P, steps = case["replicas"], NPROC[case["model"]], case["steps"]
    cells = [x * y for x, y, _ in _sizes(case)]
    sites = sum(cells) * SPUCK[case["model"]]
    if case["kind"] == "config":
        # the lattice in (one byte per site), both tables out
        return {"bytes": sites + 8.0 * P * sites, "flops": 0.0}
    if case["model"] == "intzgb":
        # running sums from the first changed entry on (0.39 entries per
        # cell and step), 8 bytes in and 8 out, plus some 330 bytes of list
        # operations and search
        per = [330.0 + 16 * 0.39 * c for c in cells]
        return {"bytes": steps * sum(per), "flops": steps * sum(0.39 * c + 4 * P for c in cells)}
    moved = float(n) * steps * STEP_BYTES[case["model"], case["backend"]]
    if case["kind"] == "track":
        moved += sum(32.0 * c for c in cells)
    if case["kind"] == "serve":
        moved += sites
    return {"bytes": moved, "flops": 4.0 * P * n * steps}


# ---------------------------------------------------------------------------
# the quickstart model in plain numpy
# ---------------------------------------------------------------------------

def _philox(c0, c1, c2, k0, k1):
    """Philox4x32-10 of the counters (c0, c1, c2, 0) (Salmon et al. 2011)."""
    M = np.uint64(0xFFFFFFFF)
    c = [np.asarray(v, np.uint64) for v in (c0, c1, c2, np.zeros_like(np.asarray(c0)))]
    k0, k1 = int(k0), int(k1)
    for _ in range(10):
        a, b = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(b >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), b & M,
             (a >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), a & M]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return c


def _u52(lo, hi):
    return (((hi << np.uint64(32)) | lo) >> np.uint64(12)).astype(np.float64) * 2.0 ** -52 + 2.0 ** -53


def exact(case, seed):
    """Adsorption and desorption on one site per cell: two lists of sites,
    the last entry moved into a freed place."""
    n, steps = case["replicas"], case["steps"]
    if case["kind"] != "batch" or case["model"] != "quickstart" or n * steps > 400000:
        return None
    sizes = _sizes(case)
    rates = np.full(2, 100.0)
    order = [p.name for p in _project("quickstart").processes]
    ads, des = order.index("CO_adsorption"), order.index("CO_desorption")
    ids = _project("quickstart").species_ids()
    S = len(ids)
    out = {k: [] for k in ("kmc_time", "kmc_time_step", "occupation", "integ_rates")}
    for r in range(n):
        V = sizes[r][0] * sizes[r][1]
        k = np.arange(steps, dtype=np.uint64)
        o = _philox(k, k >> np.uint64(32), np.zeros_like(k), seed % (1 << 32), r)
        o2 = _philox(k, k >> np.uint64(32), np.ones_like(k), seed % (1 << 32), r)
        u = np.stack([_u52(o[0], o[1]), _u52(o[2], o[3]), _u52(o2[0], o2[1])], axis=1)
        lists = [[], []]
        lists[ads] = list(range(V))
        t, dt, integ = 0.0, 0.0, np.zeros(2)
        for i in range(steps):
            c = np.array([len(lists[0]) * rates[0], len(lists[1]) * rates[1]])
            acc = [c[0], c[0] + c[1]]
            dt = -np.log(u[i, 0]) / acc[1]
            t += dt
            integ += c * dt
            p = 0 if u[i, 1] * acc[1] < acc[0] else 1
            at = min(int(1.0 + u[i, 2] * len(lists[p])), len(lists[p])) - 1
            s = lists[p][at]
            lists[p][at] = lists[p][-1]
            lists[p].pop()
            lists[1 - p].append(s)
        occ = np.zeros((S, 1))
        occ[ids["CO"]] = len(lists[des]) / V
        occ[ids["empty"]] = len(lists[ads]) / V
        for key, v in (("kmc_time", t), ("kmc_time_step", dt), ("occupation", occ), ("integ_rates", integ)):
            out[key].append(v)
    res = {key: np.array(v) for key, v in out.items()}
    res.update(kmc_step=None, status=None, procstat=None)
    return res
