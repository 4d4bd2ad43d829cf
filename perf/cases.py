"""Workloads of the table-commitment path, through the library's entry points.

Every case is one step of a prover that keeps its tables on the GPU: commits of
whole tables, their parts where a prover calls these by themselves, and the
rounds of the transcript.  Heights and widths are those of the prover's tables
(main 379 columns, 88 extension-field columns = 264 limbs, a 156-column table),
expansion 4 or 8, 98 randomizer coefficients per column, coset offset 7.
Field elements are uniform 64-bit values below p = 2^64 - 2^32 + 1, held in
int64 tensors; every output is a whole number and compares bit for bit.
"""
from __future__ import annotations

import importlib.util
import os
import sys

import numpy as np
import torch

ROOT = os.getcwd()
P = 0xFFFFFFFF00000001
OFFSET = 7
EPS = (1 << 32) - 1
LEVEL_ORDER, HEAP = 0, 1

# libtvh has to share the HIP runtime of this process's torch: two runtimes
# would neither see each other's memory nor wait for each other's work.
os.environ.setdefault("TVH_HIP_RUNTIME",
                      os.path.join(os.path.dirname(torch.__file__), "lib", "libamdhip64.so"))


def _binding():
    if "tvh" in sys.modules:
        return sys.modules["tvh"]
    path = os.path.join(ROOT, "triton-vm-prover_amd", "tvh.py")
    spec = importlib.util.spec_from_file_location("tvh", path)
    mod = importlib.util.module_from_spec(spec)
    sys.modules["tvh"] = mod
    spec.loader.exec_module(mod)
    return mod


_LIB = None


def _library():
    """The loaded library, with device 0 set up."""
    global _LIB
    if _LIB is None:
        torch.zeros(1, device="cuda")
        lib = _binding().load()
        if lib.tvh_init(0):
            raise RuntimeError("tvh_init: " + lib.last_error())
        _LIB = lib
    return _LIB


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # The smallest plain commit: the reference's own CPU-sized table.  A few
        # short kernels, so launches and single-hash latency count.
        dict(name="commit_2p10x379", kind="commit", log_n=10, cols=379, log_e=2, rand=0),
        # An ordinary table of a mixed batch, committed by itself, randomized.
        dict(name="commit_2p16x156", kind="commit", log_n=16, cols=156, log_e=2, rand=98),
        # The prover's main table at full height: the headline commit.
        dict(name="commit_2p20x379", kind="commit", log_n=20, cols=379, log_e=2, rand=0),
        # The auxiliary table: extension-field columns as limbs, extension-field
        # randomizers, its row hash and its tree.
        dict(name="aux_2p18x88", kind="aux", log_n=18, cols=88, log_e=2, rand=98),
        # A commit that streams its columns instead of keeping the codewords.
        dict(name="frugal_2p18x379", kind="frugal", log_n=18, cols=379, log_e=2, rand=0, chunk=32),
        # The two-phase prover: one of 8 cosets evaluated from the coefficients,
        # hashed, and its digests put in the leaves' order.
        dict(name="coset_2p19x379", kind="coset", log_n=19, cols=379, log_e=3, rand=98),
        # ... and the phase before it, on a ragged width.
        dict(name="coeffs_2p17x251", kind="coeffs", log_n=17, cols=251),
        # Batched transforms by themselves, as a polynomial library calls them:
        # a few columns of odd log2 length, on a copy of coefficients kept.
        dict(name="ntt_2p13x41", kind="ntt", log_n=13, cols=41, inverse=False),
        # A whole tree over row digests that are there already (heap layout).
        dict(name="merkle_2p21", kind="merkle", log_n=21, heap=True),
        # One late FRI round: a short codeword's tree, its root into the
        # transcript (with what else the round sends), the next challenge out.
        dict(name="fri_round_2p11", kind="fri", log_n=11, sent=0),
        # Many tables of different heights in one plan, replayed as a graph.
        dict(name="batch_24_tables", kind="batch", tables=24, min_log=10, max_log=16, shape_seed=7),
        # The drop-in for host callers: a table in pageable memory, its digests
        # and root back.
        dict(name="host_2p12x379", kind="host", log_n=12, cols=379, log_e=2),
    ]


def draw(rng):
    kind = rng.choice(["commit", "commit", "commit", "aux", "frugal", "coset", "coeffs", "ntt",
                       "ntt", "merkle", "fri", "batch", "host"])
    cols = max(1, min(400, round(2 ** rng.uniform(0, 8.65))))
    if kind == "commit":
        log_e = rng.choice([1, 2, 2, 2, 3])
        return dict(kind=kind, log_n=rng.randint(6, 21 - log_e), cols=cols, log_e=log_e,
                    rand=rng.choice([0, 0, 37, 98]))
    if kind == "aux":
        return dict(kind=kind, log_n=rng.randint(8, 18), cols=rng.randint(1, 100), log_e=2,
                    rand=rng.choice([0, 61, 98]))
    if kind == "frugal":
        return dict(kind=kind, log_n=rng.randint(9, 18), cols=rng.randint(20, 400), log_e=2,
                    rand=rng.choice([0, 98]), chunk=rng.randint(7, 64))
    if kind == "coset":
        return dict(kind=kind, log_n=rng.randint(8, 20), cols=cols, log_e=3,
                    rand=rng.choice([0, 41, 98]))
    if kind == "coeffs":
        return dict(kind=kind, log_n=rng.randint(6, 20), cols=cols)
    if kind == "ntt":
        return dict(kind=kind, log_n=rng.randint(3, 20), cols=cols, inverse=rng.random() < 0.5)
    if kind == "merkle":
        return dict(kind=kind, log_n=rng.randint(4, 22), heap=rng.random() < 0.5)
    if kind == "fri":
        return dict(kind=kind, log_n=rng.randint(4, 20), sent=rng.randint(1, 200))
    if kind == "batch":
        top = rng.randint(12, 17)
        return dict(kind=kind, tables=rng.randint(3, 32), min_log=rng.randint(8, top - 2),
                    max_log=top, shape_seed=rng.randint(0, 1 << 30))
    return dict(kind=kind, log_n=rng.randint(6, 14), cols=cols, log_e=2)


def _table_shapes(case):
    """[(log2 height, width)] of a batch."""
    g = np.random.RandomState(case["shape_seed"])
    return [(int(g.randint(case["min_log"], case["max_log"] + 1)),
             int(g.choice([264, 156, 379]))) for _ in range(case["tables"])]


# ---------------------------------------------------------------- inputs
def _field(gen, count):
    """count uniform field elements (int64 bit patterns of values below p)."""
    x = torch.randint(-(1 << 63), (1 << 63) - 1, (count,), dtype=torch.int64, device="cuda",
                      generator=gen)
    # p .. 2^64 - 1 are the int64 values -(2^32 - 1) .. -1: lowered by p
    return torch.where((x < 0) & (x >= -EPS), x + EPS, x)


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _out(count):
    return torch.zeros(count, dtype=torch.int64, device="cuda")


class _Plan:
    """A batch plan, freed with the state that holds it."""

    def __init__(self, lib, descs):
        self.lib, self.handle = lib, lib.batch_plan(descs)

    def __del__(self):
        torch.cuda.synchronize()
        self.lib.batch_destroy(self.handle)


def prepare(case, seed):
    lib = _library()
    gen = _generator(seed)
    kind = case["kind"]
    s = dict(case, lib=lib)
    if kind == "batch":
        tables, descs = [], []
        for log_n, cols in _table_shapes(case):
            n, m = 1 << log_n, 4 << log_n
            t = dict(trace=_field(gen, n * cols), codewords=_out(m * cols), tree=_out(5 * (2 * m - 1)))
            descs.append(lib.table_desc(t["trace"], cols, n, m, t["codewords"], t["tree"]))
            tables.append(t)
        s.update(tables=tables, plan=_Plan(lib, descs), stream=_binding().hip_rt.Stream())
        torch.cuda.synchronize()  # the tables are filled on the null stream
        return s
    n = 1 << case["log_n"]
    if kind == "merkle":
        s.update(leaves=_field(gen, 5 * n), tree=_out(5 * 2 * n))
    elif kind == "fri":
        s.update(xfe=_field(gen, 3 * n), tree=_out(5 * (2 * n - 1)), sponge=_out(16),
                 item=torch.cat([_out(6), _field(gen, case["sent"])]),
                 challenge=_out(10))
    elif kind == "ntt":
        s.update(coeffs=_field(gen, n * case["cols"]), data=_out(n * case["cols"]))
    elif kind == "coeffs":
        s.update(trace=_field(gen, n * case["cols"]), coeffs=_out(n * case["cols"]))
    elif kind == "host":
        m = n << case["log_e"]
        lib.lde_prepare(n, m, 1, OFFSET)
        trace = _field(gen, n * case["cols"]).cpu().numpy().view(np.uint64)
        s.update(trace=trace, digests=np.zeros(5 * m, np.uint64), root=np.zeros(5, np.uint64))
    else:
        limbs = 3 if kind == "aux" else 1
        cols, m = limbs * case["cols"], n << case["log_e"]
        k = min(case["rand"], n)
        rand = _field(gen, k * cols) if k else None
        if kind == "coset":
            s.update(coeffs=_field(gen, n * cols), rand=rand, k=k, evals=_out(n * cols),
                     digests=_out(5 * n), leaves=_out(5 * m))
            return s
        lib.lde_prepare(n, m, 1, OFFSET)
        s.update(trace=_field(gen, n * cols), rand=rand, k=k, tree=_out(5 * (2 * m - 1)))
        if kind == "frugal":
            s["work"] = _out(lib.frugal_workspace_elems(cols, n, m, case["chunk"]))
        else:
            s["codewords"] = _out(m * cols)
    return s


# ---------------------------------------------------------------- one pass
def run(s):
    lib, kind = s["lib"], s["kind"]
    if kind == "batch":
        lib.batch_launch_graph(s["plan"].handle, s["stream"])
        return [t["tree"] for t in s["tables"]]
    n = 1 << s["log_n"]
    if kind == "merkle":
        lib.merkle_tree(s["leaves"], s["tree"], n, HEAP if s["heap"] else LEVEL_ORDER)
        return s["tree"][5:] if s["heap"] else s["tree"][:-5]  # a heap has no node 0
    if kind == "fri":
        lib.fri_commit(s["xfe"], n, s["tree"])
        s["item"][1:6].copy_(s["tree"][-5:])  # the transcript's root item: [0, root]
        lib.sponge_init(s["sponge"])
        lib.sponge_absorb(s["sponge"], s["item"], 6 + s["sent"])
        lib.sponge_squeeze(s["sponge"], s["challenge"])
        return dict(tree=s["tree"], sponge=s["sponge"], challenge=s["challenge"])
    if kind == "ntt":
        s["data"].copy_(s["coeffs"])
        (lib.ntt_inverse_batched if s["inverse"] else lib.ntt_forward_batched)(s["data"], n, s["cols"])
        return s["data"]
    if kind == "coeffs":
        lib.trace_coefficients(s["trace"], s["cols"], n, 1, s["coeffs"])
        return s["coeffs"]
    m = n << s["log_e"]
    if kind == "host":
        lib.commit_host(s["trace"], s["cols"], n, m, 1, OFFSET, digests=s["digests"], root=s["root"])
        return dict(digests=s["digests"].view(np.int64), root=s["root"].view(np.int64))
    if kind == "coset":
        index = 3
        lib.evaluate_coset(s["coeffs"], s["cols"], n, s["rand"], s["k"], 1,
                           _coset_offset(s["log_n"] + s["log_e"], index), s["evals"])
        lib.hash_bfield_rows(s["evals"], n, s["cols"], s["digests"])
        lib.scatter_digests(s["digests"], s["leaves"], n, index, m // n)
        return dict(evals=s["evals"], leaves=s["leaves"])
    if kind == "frugal":
        lib.commit_frugal(s["trace"], s["cols"], n, s["rand"], s["k"], 1, OFFSET, m, s["chunk"],
                          s["work"], s["tree"])
        return s["tree"]
    if kind == "aux":
        lib.lde_xfe_limbs(s["trace"], s["cols"], n, s["rand"], s["k"], 1, OFFSET, m, s["codewords"], 1)
        lib.hash_xfield_rows(s["codewords"], m, s["cols"], s["tree"])
        lib.merkle_tree(s["tree"], s["tree"], m)
    else:
        lib.commit(s["trace"], s["cols"], n, s["rand"], s["k"], 1, OFFSET, m, s["codewords"], s["tree"])
    return dict(codewords=s["codewords"], tree=s["tree"])


def _coset_offset(log_m, index):
    """OFFSET * w^index, w the primitive 2^log_m-th root of unity 7^((p-1) / 2^log_m)."""
    return OFFSET * pow(pow(7, (P - 1) >> log_m, P), index, P) % P


# ---------------------------------------------------------------- work
def work(case):
    """Bytes of each input read and each output written once.  The arithmetic is
    whole-number (field products and Tip5 permutations), so there are no flops."""
    kind = case["kind"]
    if kind == "batch":
        words = sum((w << lg) * 5 + 10 * (4 << lg) for lg, w in _table_shapes(case))
        return {"bytes": 8.0 * words, "flops": 0.0}
    n = 1 << case["log_n"]
    if kind == "merkle":
        words = 5 * n + 10 * n
    elif kind == "fri":
        words = 3 * n + 10 * n + case["sent"] + 32
    elif kind in ("ntt", "coeffs"):
        words = 2 * n * case["cols"]
    else:
        cols = case["cols"] * (3 if kind == "aux" else 1)
        m = n << case["log_e"]
        rand = min(case.get("rand", 0), n) * cols
        if kind == "host":
            words = n * cols + 5 * m
        elif kind == "coset":
            words = 2 * n * cols + rand + 5 * n
        elif kind == "frugal":
            words = n * cols + rand + 10 * m
        else:
            words = n * cols + rand + m * cols + 10 * m
    return {"bytes": 8.0 * words, "flops": 0.0}


# ---------------------------------------------------------------- 64-bit answers
def _mul(a, b):
    """a * b mod p on uint64 arrays (schoolbook on 32-bit halves, 2^64 = 2^32 - 1)."""
    e, u = np.uint64(EPS), np.uint64
    a0, a1, b0, b1 = a & e, a >> u(32), b & e, b >> u(32)
    ll, hh, x, y = a0 * b0, a1 * b1, a1 * b0, a0 * b1
    mid = x + (ll >> u(32))
    mid2 = (mid & e) + y
    lo = (mid2 << u(32)) | (ll & e)
    hi = hh + (mid >> u(32)) + (mid2 >> u(32))
    h1, h0 = hi >> u(32), hi & e
    t = lo - h1
    t = np.where(lo < h1, t - e, t)
    w = h0 * e
    r = t + w
    r = np.where(r < w, r + e, r)
    return np.where(r >= u(P), r - u(P), r)


def _add(a, b):
    s = a + b
    s = np.where(s < a, s + np.uint64(EPS), s)
    return np.where(s >= np.uint64(P), s - np.uint64(P), s)


def _sub(a, b):
    d = a - b
    return np.where(a < b, d - np.uint64(EPS), d)


def _transform(x, inverse):
    """Transform of every row of x (rows x n), natural order in and out."""
    n = x.shape[1]
    log_n = n.bit_length() - 1
    rev = np.zeros(n, np.int64)
    for i in range(log_n):
        rev |= ((np.arange(n) >> i) & 1) << (log_n - 1 - i)
    x = x[:, rev]
    root = pow(7, (P - 1) >> log_n, P) if log_n else 1
    root = pow(root, P - 2, P) if inverse else root
    half = 1
    while half < n:
        step, tw = pow(root, n // (2 * half), P), [1]
        for _ in range(half - 1):
            tw.append(tw[-1] * step % P)
        v = x.reshape(x.shape[0], -1, 2, half)
        t = _mul(v[:, :, 1], np.array(tw, np.uint64))
        x = np.stack([_add(v[:, :, 0], t), _sub(v[:, :, 0], t)], axis=2).reshape(x.shape)
        half *= 2
    return _mul(x, np.uint64(pow(n, P - 2, P))) if inverse else x


def exact(case, seed):
    """The transforms by themselves, where they are small; the hashes of the
    other cases are whole numbers that compare bit for bit."""
    if case["kind"] not in ("ntt", "coeffs") or (case["cols"] << case["log_n"]) > 1 << 22:
        return None
    n, cols = 1 << case["log_n"], case["cols"]
    x = _field(_generator(seed), n * cols).cpu().numpy().view(np.uint64).reshape(cols, n)
    with np.errstate(over="ignore"):
        y = _transform(x, case["kind"] == "coeffs" or case["inverse"])
    return y.reshape(-1).view(np.int64)
