"""Timed cases of the simplifier: what a solver, a batch job or a model
checker has this library do, from formulas of a thousand clauses to the
40M-clause one, through the public Python binding (parafrost_amd.simplifier).

A case is a dict of plain values:
  family   uniform3 | circuit | heavytail | equiv | bmc | batch
  size     variables (uniform3, heavytail, equiv), gates (circuit), frames
           (bmc) or formulas (batch)
  op       what one pass does:
    round    the formula is resident in HBM (its device copy is restored),
             one simplify call, the result taken back
    handoff  a host solver's call: its clause database uploaded, simplified,
             taken back, and the variables renumbered
    ingest   DIMACS text parsed on the device, simplified, taken back
    els      resident formula: equivalent literals substituted, simplified,
             taken back
    session  a BMC session from its first frame: per request the next frames'
             clauses appended, the assumed variables replaced, simplified;
             the state taken back after the last request
    batch    many resident formulas simplified by the native batch executor
  options  simplifier options, "name=value ..." ("" for the defaults)
  learnt   percentage of the clauses handed over as learnt (handoff)

A pass ends with what the host takes back (pfs_download_*, include/pfsimp.h)
in buffers that it keeps from call to call, as a solver keeps its clause
database: clauses, new units, variable states, eliminated-variable stack,
proof, and the counts of each round.  Everything is whole numbers, so every
output has to be equal, and there are no values to compute in 64 bits.
"""
import ctypes
import os
import tempfile

import numpy as np
import torch

from parafrost_amd import bmc, gen
from parafrost_amd.simplifier import Simplifier, batch_simplify
from parafrost_amd.simplifier import _RoundStats as ROUND_STATS

ROUND = "phases=1 bce=1"  # one full round: SUB, BVE, BCE, then the stopping round's ERE


def _case(name, family, size, op, options=ROUND, learnt=0):
    return {"name": name, "family": family, "size": size, "op": op, "options": options, "learnt": learnt}


def listed():
    return [
        # the smallest calls: launches, host reads and latency are all there is
        _case("uniform-301", "uniform3", 301, "round", ""),
        # the small configuration of the benchmark: uniform random 3-SAT at the threshold
        _case("uniform-20k", "uniform3", 20000, "round"),
        # a small circuit through all five default phases (VE, SUB, ERE, no BCE), with its DRAT proof
        _case("circuit-4999-proof", "circuit", 4999, "round", "proof=1"),
        # incremental model checking: ten requests of ten frames on one session
        _case("bmc-100", "bmc", 100, "session"),
        # batch preprocessing of mixed circuits and heavy-tailed formulas of 1k-200k clauses
        _case("batch-24", "batch", 24, "batch"),
        # inprocessing call of a running solver: a third of a million clauses, some of them learnt
        _case("handoff-100k", "circuit", 100003, "handoff", "", 20),
        # preprocessing from a file's text
        _case("ingest-300k", "circuit", 300000, "ingest"),
        # an odd size, every technique on, three phases
        _case("uniform-77777-all", "uniform3", 77777, "round", "all=1 phases=3"),
        # equivalent-literal substitution before the rounds
        _case("els-500k", "equiv", 500000, "els"),
        # the benchmark's circuit: 2M gates, 6.8M clauses
        _case("circuit-2m", "circuit", 2000000, "round"),
        # heavy-tailed, elimination and subsumption off: BCE, ERE and collection at size
        _case("heavy-2500k-bce", "heavytail", 2500000, "round", "phases=1 bce=1 ve=0 sub=0 ve+=0"),
        # the benchmark's headline: 10M variables, 40M clauses (its strengthening refutes it)
        _case("heavy-10m", "heavytail", 10000000, "round"),
    ]


def _logsize(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """One more case of the same uses; sizes over their logarithm, mostly odd ones."""
    kind = rng.randrange(9)
    opts = rng.choice([ROUND, "", "all=1 phases=2", "phases=2 bce=1 mupos=16 muneg=16"])
    if kind == 0:
        c = _case("", "uniform3", _logsize(rng, 200, 200000), "round", opts)
    elif kind == 1:
        c = _case("", "circuit", _logsize(rng, 300, 1500000), "round", opts)
    elif kind == 2:
        c = _case("", "heavytail", _logsize(rng, 1000, 6000000), "round", ROUND)
    elif kind == 3:
        c = _case("", "heavytail", _logsize(rng, 1000, 1500000), "round",
                  rng.choice(["phases=1 bce=1 ve=0 sub=0 ve+=0", "phases=1 bce=1 sub=0 ve+=0"]))
    elif kind == 4:
        c = _case("", "circuit", _logsize(rng, 500, 400000), "handoff", opts, rng.choice([0, 10, 20, 30]))
    elif kind == 5:
        c = _case("", "circuit", _logsize(rng, 500, 600000), "ingest", opts)
    elif kind == 6:
        c = _case("", "equiv", _logsize(rng, 2000, 700000), "els", opts)
    elif kind == 7:
        c = _case("", "bmc", rng.randrange(11, 130), "session")
    else:
        c = _case("", "batch", rng.randrange(5, 29), "batch")
    del c["name"]
    return c


# ---------------------------------------------------------------- inputs
def _heavytail(nvars, nclauses, seed):
    """The heavy-tailed k-SAT family of parafrost_amd.gen (lengths 2 +
    Geometric(1/2) capped at 30, variable weights rank^(-2/3) over a random
    numbering, repeated variables dropped), drawn on the GPU: the generator's
    sequential draw of 40M clauses takes 12 s."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    g = torch.Generator(device=dev).manual_seed(seed)
    n = nclauses + nclauses // 8 + 64  # some are left with fewer than two literals and dropped
    u = torch.rand(n, generator=g, device=dev)
    lens = 2 + torch.clamp(torch.floor(-torch.log2(1.0 - u)), 0, 28).to(torch.int64)
    cid = torch.repeat_interleave(torch.arange(n, device=dev), lens)
    top = (nvars + 1.0) ** (1.0 / 3.0) - 1.0
    x = 1.0 + top * torch.rand(cid.shape[0], generator=g, device=dev, dtype=torch.float64)
    rank = torch.clamp((x * x * x).to(torch.int64), 1, nvars) - 1
    del x
    var = torch.randperm(nvars, generator=g, device=dev)[rank] + 1
    lit = 2 * var + torch.randint(0, 2, (cid.shape[0],), generator=g, device=dev)
    del rank, var
    key = torch.sort((cid << 32) | lit).values
    del cid, lit
    vkey = key >> 1
    first = torch.ones(key.shape[0], dtype=torch.bool, device=dev)
    first[1:] = vkey[1:] != vkey[:-1]
    key = key[first]
    del vkey, first
    cid = key >> 32
    size = torch.bincount(cid, minlength=n)
    ids = torch.nonzero(size >= 2).flatten()[:nclauses]
    if ids.shape[0] < nclauses:
        raise RuntimeError("too few clauses drawn")
    keep = torch.zeros(n, dtype=torch.bool, device=dev)
    keep[ids] = True
    lits = (key[keep[cid]] & 0xFFFFFFFF).to(torch.int32).cpu().numpy().view(np.uint32)
    off = np.zeros(nclauses + 1, np.uint64)
    off[1:] = torch.cumsum(size[ids], 0).cpu().numpy().astype(np.uint64)
    return gen.Cnf(nvars, off, lits)


def _circuit(gates, seed):
    """A random circuit with satisfiable outputs, in proportion to the
    2M-gate workload, root-propagated as a host solver hands it over."""
    cnf, refuted = gen.prepare(gen.tseitin(gates, max(10, gates // 400), max(1, gates // 2000), seed,
                                           sat_outputs=True))
    if refuted:
        raise RuntimeError("circuit refuted at the root")
    return cnf


def _formula(family, size, seed):
    if family == "uniform3":
        return gen.uniform_ksat(size, int(round(4.26 * size)), 3, seed)
    if family == "circuit":
        return _circuit(size, seed)
    if family == "heavytail":
        return _heavytail(size, 4 * size, seed)
    return gen.equivalences(size, 3 * size, size // 10, 5, seed=seed, chords=0.4)


def _options(text):
    return {k: int(v) for k, v in (kv.split("=") for kv in text.split())}


def prepare(case, seed):
    opts = _options(case["options"])
    op, size = case["op"], case["size"]
    st = {"op": op, "res": _Result(case)}
    if op == "session":
        st["s"] = _Host(0, **opts)
        st["requests"] = bmc.session_requests(seed, size)
        return st
    if op == "batch":
        st["ctx"] = []
        for cnf in gen.batch(size, seed=seed, cmax=2e5):
            s = _Host(0, keep_input=True, **opts)
            s.upload(cnf.maxvar, cnf.offsets, cnf.lits, trail=cnf.trail)
            st["ctx"].append(s)
        return st
    if op == "ingest":
        # the text as a user's file has it: the circuit with its output units
        raw = gen.tseitin(size, max(10, size // 400), max(1, size // 2000), seed, sat_outputs=True)
        with tempfile.TemporaryDirectory() as d:
            path = os.path.join(d, "f.cnf")
            gen.write_dimacs(raw, path)
            with open(path, "rb") as f:
                st["text"] = f.read()
        st["s"] = _Host(0, **opts)
        return st
    cnf = _formula(case["family"], size, seed)
    if op == "handoff":
        rng = np.random.default_rng(seed)
        learnt = rng.random(cnf.nclauses) * 100 < case["learnt"]
        st["cnf"] = cnf
        st["flags"] = (learnt | (rng.integers(0, 3, cnf.nclauses) << 4) * learnt).astype(np.uint8)
        st["lbd"] = (rng.integers(1, 9, cnf.nclauses) * learnt).astype(np.uint32)
        st["s"] = _Host(0, **opts)
        return st
    s = st["s"] = _Host(0, keep_input=True, **opts)
    s.upload(cnf.maxvar, cnf.offsets, cnf.lits, trail=cnf.trail)
    return st


# ---------------------------------------------------------------- what the host takes back
COUNTS = ("elected", "eliminated", "units", "resolvents", "clauses_after", "literals_after")
ROUNDS = 8


class _Result:
    """The host's buffers for 'case', sized from the family's expected
    counts, and the downloads into them; formulas of a batch follow one
    another in the same buffers."""

    def __init__(self, case):
        v, c, l, _ = _expected(case)
        cap_c, cap_l = int(1.05 * c) + 4096, int(1.1 * l) + 16384
        self.out = {"offsets": np.zeros(cap_c, np.int64), "lits": np.zeros(cap_l, np.int32),
                    "flags": np.zeros(cap_c, np.uint8), "lbd": np.zeros(cap_c, np.int32),
                    "units": np.zeros(int(1.05 * v) + 1024, np.int32),
                    "stack": np.zeros(int(1.3 * (c + l)) + 16384, np.int32),
                    "vstate": np.zeros(int(1.05 * v) + 1024, np.uint8),
                    "counts": np.zeros(case["size"] * ROUNDS * 6 if case["op"] == "batch" else ROUNDS * 6, np.int64)}
        if "proof=1" in case["options"]:
            self.out["proof"] = np.zeros(64 * cap_c, np.uint8)
        if case["op"] == "handoff":
            self.out["map"] = np.zeros(int(1.05 * v) + 1024, np.int32)
        self.begin()

    def begin(self):
        self.at = dict.fromkeys(self.out, 0)

    def _room(self, name, n):
        """n values of a buffer and their address."""
        i = self.at[name]
        self.at[name] = i + n
        if i + n > self.out[name].shape[0]:
            raise RuntimeError("the result does not fit the host's " + name)
        part = self.out[name][i:i + n]
        return part, part.ctypes.data


class _Host(Simplifier):
    """A context with the host's side of the downloads."""

    def take(self, res, status):
        L, h = self._L, self._h
        nc, nl, nu, ns, npf = (ctypes.c_uint64() for _ in range(5))
        nr = ctypes.c_uint32()
        by = ctypes.byref
        self._check(L.pfs_result_sizes(h, by(nc), by(nl), by(nu), by(ns), by(nr)), "pfs_result_sizes")
        self._check(L.pfs_proof_size(h, by(npf)), "pfs_proof_size")
        counts, _ = res._room("counts", ROUNDS * 6)
        rs = (ROUND_STATS * max(nr.value, 1))()
        n = ctypes.c_uint32()
        self._check(L.pfs_round_stats_get(h, rs, nr.value, by(n)), "pfs_round_stats_get")
        for i in range(min(n.value, ROUNDS)):
            counts[6 * i:6 * i + 6] = [getattr(rs[i], k) for k in COUNTS]
        # the order of the units that one propagation derives is left open
        # by the library: the host puts them in its trail in any order
        units, p = res._room("units", nu.value)
        self._check(L.pfs_download_units(h, p), "pfs_download_units")
        units.sort()
        if npf.value and "proof" in res.out:
            _, p = res._room("proof", npf.value)
            self._check(L.pfs_download_proof(h, p), "pfs_download_proof")
        if status == 0:  # refuted: there are no clauses to go on with
            return
        # offsets: one more than there are clauses
        _, po = res._room("offsets", nc.value + 1)
        _, pl = res._room("lits", nl.value)
        _, pf = res._room("flags", nc.value)
        _, pb = res._room("lbd", nc.value)
        self._check(L.pfs_download_cnf(h, po, pl, pf, pb), "pfs_download_cnf")
        _, p = res._room("stack", ns.value)
        self._check(L.pfs_download_stack(h, p), "pfs_download_stack")
        _, p = res._room("vstate", self.maxvar + 1)
        self._check(L.pfs_download_vstate(h, p), "pfs_download_vstate")


# ---------------------------------------------------------------- one pass
def run(st):
    op, res = st["op"], st["res"]
    res.begin()
    if op == "batch":
        for s in st["ctx"]:
            s.rewind()
        status, _ = batch_simplify(st["ctx"], 8)
        for s, x in zip(st["ctx"], status):
            s.take(res, x)
        return dict(res.out, status=np.array(status, np.int32))
    s = st["s"]
    if op == "session":
        s.upload(0, np.zeros(1, np.uint64), np.zeros(0, np.uint32))
        status = []
        for rq in st["requests"]:
            s.append(rq.maxvar, rq.offsets, rq.lits)
            s.assume(rq.assumed)
            status.append(s.simplify())
        s.take(res, status[-1])
        return dict(res.out, status=np.array(status, np.int32))
    if op == "handoff":
        c = st["cnf"]
        s.upload(c.maxvar, c.offsets, c.lits, flags=st["flags"], lbd=st["lbd"], trail=c.trail)
        status = s.simplify()
        s.take(res, status)
        if status:
            old = s.map(force=True)["old_maxvar"]
            _, p = res._room("map", old + 1)
            s._check(s._L.pfs_download_map(s._h, p), "pfs_download_map")
        return dict(res.out, status=status)
    if op == "ingest":
        s.parse_dimacs(st["text"])
    else:
        s.rewind()
    got = {}
    if op == "els":
        info = s.decompose()
        got = {"substituted": info["substituted"], "els_units": info["units"]}
    status = s.simplify()
    s.take(res, status)
    return dict(res.out, status=status, **got)


# ---------------------------------------------------------------- what a pass cannot do without
def _expected(case):
    """Variables, clauses and literals of the family at this size, and the
    share of the clauses that remains: of a circuit about two thirds, of the
    other families nearly all; a refuted formula (the heavy-tailed ones with
    SUB or BVE on, at size) leaves nothing."""
    n, family = case["size"], case["family"]
    if family == "uniform3":
        return n + 1, 4.26 * n, 12.78 * n, 1.0
    if family == "circuit":
        return n + max(10, n // 400) + 1, 3.4 * n, 9.0 * n, 0.65
    if family == "heavytail":
        return n + 1, 4.0 * n, 12.0 * n, 1.0 if "ve=0" in case["options"] else 0.0
    if family == "equiv":
        return n + 1, 3.7 * n, 10.4 * n, 0.9
    if family == "bmc":
        return 64 + 2032 * n + 1, 6667.0 * n, 17333.0 * n, 0.5
    # clause counts log-uniform in [1e3, 2e5]: mean 37,560, standard
    # deviation 48,600; this is room for nearly every batch of n
    c = 37560.0 * n + 4.5 * 48600.0 * n ** 0.5
    return 0.5 * c, c, 2.8 * c, 0.8


def work(case):
    """Every clause of the input read once and every clause of the result
    written once: four bytes per literal and four per clause (text: 22 bytes
    per clause)."""
    _, c, l, left = _expected(case)
    if case["op"] == "batch":
        c, l = 37560.0 * case["size"], 2.8 * 37560.0 * case["size"]
    size = 4.0 * (c + l)
    read = 22.0 * c if case["op"] == "ingest" else size
    return {"bytes": float(read + left * size), "flops": 0.0}
