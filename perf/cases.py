"""Performance cases of the commit pipeline, each one pass through public entry points.

Kinds (the `kind` of a case; `draw` takes any of them at other sizes):

  prove        Prover.prove: a Fibonacci proof from (a, b), KRAK bytes on the host
  prove_device Prover.prove_device: the trace is resident, the proof stays in HBM
  prove_batch  Prover.prove_batch_async: many proofs of one size per launch sequence
  prove_once   vortexstark_amd.prove: one proof by a program that keeps no prover
  serve        Server: a list of jobs of mixed sizes submitted, served and collected
  wide         WideCommit: stwo-basis LDE, lifted tree and FRI over columns of mixed sizes
  deep         DeepQuotient: the fused DEEP quotient over the LDE columns
  native_lde   the kernel ABI as the Rust prover calls it: interpolate, zero pad, evaluate
               (one column, or the batch calls for several)
  native_fri   the kernel ABI as the Rust prover calls it after the LDE: trace tree,
               quotient and its tree, fold twiddles, folds and their trees
  stwo         the kernel ABI as the stwo backend calls it: transforms, lifted leaves and
               their tree, DEEP numerators and combine, folds

Every output is whole numbers (M31 words or hash words), computed exactly, so there
is no rounding to price: `exact` has no value to give.
"""

import ctypes as C
import math

import numpy as np
import torch

import vortexstark_amd as vx

P = (1 << 31) - 1
MASK64 = (1 << 64) - 1
DEV = "cuda"
COMPRESSION_OPS = 968  # int32 operations of one Blake2s compression
BUTTERFLY_OPS = 12  # int32 operations of one M31 butterfly


def listed():
    return [
        # the smallest proof in use: a latency-bound call, as an interactive prover makes it
        {"name": "prove_2p10", "kind": "prove", "log_n": 10, "queries": 80, "last": 3},
        # the size the CPU baseline is quoted on (2^16 rows, 64 queries, last layer 2^4)
        {"name": "prove_2p16", "kind": "prove", "log_n": 16, "queries": 64, "last": 4},
        # the headline workload of bench.py: 2^24 rows, 100 queries, trace resident in HBM
        {"name": "prove_2p24", "kind": "prove_device", "log_n": 24, "queries": 100, "last": 4},
        # one batch of small proofs, as a server of many small jobs runs it
        {"name": "batch_64x2p12", "kind": "prove_batch", "log_n": 12, "count": 64, "queries": 80, "last": 3},
        # a program that proves once: set-up (memory, twiddles) is part of the call
        {"name": "once_2p18", "kind": "prove_once", "log_n": 18, "queries": 80, "last": 3},
        # a burst of small jobs of mixed sizes through the proof server
        {"name": "served_mix", "kind": "serve", "log_min": 10, "log_max": 14, "jobs": 14, "cols_max": 4},
        # the wide commitment of bench.py: 34 columns (4 x 2^14, 10 x 2^18, 20 x 2^20), blowup 4
        {"name": "wide_34", "kind": "wide", "sizes": "14x4,18x10,20x20", "blowup": 2, "last": 4},
        # a narrow table with ragged small columns
        {"name": "wide_ragged", "kind": "wide", "sizes": "7x1,9x3,10x2,12x5,13x2", "blowup": 2, "last": 3},
        # the DEEP quotient of the wide shape's LDE columns at two sample points
        {"name": "deep_34", "kind": "deep", "sizes": "16x4,20x10,22x20", "points": 2},
        # one column's LDE by the Rust prover's calls (2^22 rows onto 2^24 points)
        {"name": "native_lde_2p22", "kind": "native_lde", "log_n": 22, "cols": 1},
        # the same prover's commitments and FRI on an evaluation domain of 2^20 points
        {"name": "native_fri_2p20", "kind": "native_fri", "log_e": 20},
        # the stwo backend's calls for a trace of 15 columns of three sizes
        {"name": "stwo_15", "kind": "stwo", "sizes": "11x3,14x4,17x8", "points": 2},
    ]


def draw(rng):
    """One more case of the same ranges, sizes spread over their logarithm."""
    known = [{k: v for k, v in c.items() if k != "name"} for c in listed()]
    while True:
        case = draw_any(rng)
        if case not in known:
            return case


def draw_any(rng):
    kind = rng.choice(["prove", "prove", "prove_device", "prove_batch", "prove_once", "serve", "wide", "wide", "deep",
                       "native_lde", "native_lde", "native_fri", "native_fri", "stwo", "stwo"])
    queries, last = rng.choice([64, 80, 100]), rng.randint(3, 5)
    if kind == "prove":
        return {"kind": kind, "log_n": rng.randint(10, 21), "queries": queries, "last": last}
    if kind == "prove_device":
        return {"kind": kind, "log_n": rng.randint(14, 23), "queries": queries, "last": last}
    if kind == "prove_batch":
        log_n = rng.randint(10, 16)
        return {"kind": kind, "log_n": log_n, "count": max(2, round(2 ** rng.uniform(1, min(7, 20 - log_n)))),
                "queries": queries, "last": last}
    if kind == "prove_once":
        return {"kind": kind, "log_n": rng.randint(10, 20), "queries": queries, "last": last}
    if kind == "serve":
        lo = rng.randint(10, 12)
        return {"kind": kind, "log_min": lo, "log_max": lo + rng.randint(1, 3), "jobs": rng.randint(4, 16),
                "cols_max": rng.randint(1, 5)}
    if kind in ("wide", "deep", "stwo"):
        top = rng.randint(10, 19) if kind == "wide" else rng.randint(12, 21) if kind == "deep" else rng.randint(9, 16)
        logs = sorted({top} | {max(5, top - rng.randint(1, 7)) for _ in range(rng.randint(0, 2))})
        sizes = ",".join("%dx%d" % (k, rng.randint(1, 12)) for k in logs)
        if kind == "wide":
            return {"kind": kind, "sizes": sizes, "blowup": rng.choice([1, 2, 2, 2, 3]), "last": last}
        return {"kind": kind, "sizes": sizes, "points": rng.randint(1, 3) if kind == "deep" else rng.randint(1, 2)}
    if kind == "native_lde":
        log_n = rng.randint(9, 22)
        return {"kind": kind, "log_n": log_n, "cols": rng.choice([1, 1, rng.randint(2, 9)]) if log_n <= 19 else 1}
    return {"kind": kind, "log_e": rng.randint(12, 22)}


# ---------------------------------------------------------------- inputs
def parse_sizes(text):
    """"14x4,18x10": four columns of 2^14 rows, ten of 2^18 (ascending)."""
    out = []
    for part in text.split(","):
        log, count = part.split("x")
        out += [int(log)] * int(count)
    return out


def mix64(x):
    z = (x + 0x9E3779B97F4A7C15) & MASK64
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & MASK64
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & MASK64
    return z ^ (z >> 31)


class Numbers:
    """Uniform M31 values from the seed: on the host one by one, on the GPU as tensors."""

    def __init__(self, seed):
        self.state = mix64(seed & MASK64)
        self.gen = torch.Generator(device=DEV)
        self.gen.manual_seed(self.state & ((1 << 62) - 1))

    def one(self):
        self.state = mix64(self.state)
        return self.state % P

    def below(self, n):
        self.state = mix64(self.state)
        return self.state % n

    def column(self, n):
        return torch.randint(0, P, (n,), generator=self.gen, device=DEV, dtype=torch.int32)


class DeviceWords:
    """Device memory of a library object, for torch.as_tensor: the tensor keeps this, and this the object."""

    def __init__(self, owner, addr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<i4", "data": (addr, False), "version": 2}


def view(owner, addr, n):
    return torch.as_tensor(DeviceWords(owner, addr, (n,)), device=DEV)


def ptrs(tensors):
    """Device array of device pointers."""
    return torch.tensor([t.data_ptr() for t in tensors], dtype=torch.int64, device=DEV)


def h32(values):
    return (C.c_uint32 * len(values))(*[int(v) for v in values])


def words(n):
    return torch.empty(n, dtype=torch.int32, device=DEV)


# circle group of the M31 field: cosets as (initial, step) points
def pmul(a, b):
    return ((a[0] * b[0] - a[1] * b[1]) % P, (a[0] * b[1] + a[1] * b[0]) % P)


def gen_pow2(n):
    """The generator of the group of order 2^31, doubled n times."""
    g = (2, 1268011823)
    for _ in range(n):
        g = pmul(g, g)
    return g


def half_coset(k):
    return gen_pow2(30 - k), gen_pow2(31 - k)


def half_odds(k):
    return gen_pow2(29 - k), gen_pow2(31 - k)


class NativeTwiddles:
    """The twiddle tables a Rust prover keeps for one transform size, built by the kernel ABI."""

    def __init__(self, log_n, inverse):
        n = 1 << log_n
        (ix, iy), (sx, sy) = half_coset(log_n)
        xs, ys = words(n), words(n)
        line, circle = torch.zeros(max(1, n - 1), dtype=torch.int32, device=DEV), words(n // 2)
        vx.lib.cuda_compute_coset_points(ix, iy, sx, sy, xs.data_ptr(), ys.data_ptr(), n)
        circle.copy_(ys[: n // 2])
        self.n_line, offs, sizes, at, cur = log_n - 1, [], [], 0, xs
        for layer in range(self.n_line):
            half = (n >> layer) // 2
            nxt = words(half)
            vx.lib.cuda_extract_and_squash(cur.data_ptr(), line.data_ptr() + 4 * at, nxt.data_ptr(), half)
            offs.append(at)
            sizes.append(half)
            at, cur = at + half, nxt
        self.offs, self.sizes = h32(offs), h32(sizes)
        if inverse:
            iline, icircle = words(line.numel()), words(n // 2)
            vx.lib.cuda_batch_inverse_m31(line.data_ptr(), iline.data_ptr(), line.numel())
            vx.lib.cuda_batch_inverse_m31(circle.data_ptr(), icircle.data_ptr(), n // 2)
            line, circle = iline, icircle
        self.line, self.circle = line, circle
        torch.cuda.synchronize()


# ---------------------------------------------------------------- prepare
def prepare(case, seed):
    num = Numbers(seed)
    return globals()["prepare_" + case["kind"]](case, num)


def run(state):
    return state["run"](state)


def prepare_prove(case, num):
    prover = vx.Prover(case["log_n"], case["queries"], case["last"])
    return {"run": run_prove, "prover": prover, "a": num.one(), "b": num.one()}


def run_prove(s):
    return np.frombuffer(s["prover"].prove(s["a"], s["b"]), dtype=np.int32)


def prepare_prove_device(case, num):
    prover = vx.Prover(case["log_n"], case["queries"], case["last"])
    a, b = num.one(), num.one()
    trace = vx.fibonacci_trace_device(a, b, case["log_n"])
    proof = view(prover, vx.lib.vx_prover_proof_device(prover.handle), prover.proof_size // 4)
    return {"run": run_prove_device, "prover": prover, "a": a, "b": b, "trace": trace, "proof": proof}


def run_prove_device(s):
    s["prover"].prove_device(s["trace"].addr, s["a"], s["b"])
    return s["proof"]


def prepare_prove_batch(case, num):
    n = case["count"]
    prover = vx.Prover(case["log_n"], case["queries"], case["last"], capacity=n)
    ab = [(num.one(), num.one()) for _ in range(n)]
    addr = [vx.lib.vx_prover_proof_device_at(prover.handle, i) for i in range(n)]
    # proofs of a batch lie equally far apart: one strided view of all of them
    size, step = prover.proof_size // 4, ((addr[1] - addr[0]) // 4 if n > 1 else 0)
    whole = view(prover, addr[0], step * (n - 1) + size)
    return {"run": run_prove_batch, "prover": prover, "ab": ab, "proofs": torch.as_strided(whole, (n, size), (max(step, size), 1))}


def run_prove_batch(s):
    s["prover"].prove_batch_async(s["ab"])
    return s["proofs"]


def prepare_prove_once(case, num):
    return {"run": run_prove_once, "args": (num.one(), num.one(), case["log_n"], case["queries"], case["last"])}


def run_prove_once(s):
    return np.frombuffer(vx.prove(*s["args"]), dtype=np.int32)


def job_list(case):
    """Sizes and column counts of a served list: fixed by the case, so that every seed serves the same work."""
    num, jobs = mix64(case["jobs"]), []
    span = case["log_max"] - case["log_min"] + 1
    for _ in range(case["jobs"]):
        num = mix64(num)
        jobs.append((case["log_min"] + num % span, 1 + (num >> 20) % case["cols_max"]))
    return jobs


def prepare_serve(case, num):
    server = vx.Server(budget_bytes=40 << 30, result_bytes=256 << 20)
    server.set_graphs(True)
    jobs = [(log_n, [(num.one(), num.one()) for _ in range(cols)]) for log_n, cols in job_list(case)]
    for log_n in sorted({j[0] for j in jobs}):
        server.prewarm(log_n, 1)
    size = {j[0]: int(vx.lib.vx_krak_proof_size(j[0], server.n_queries, server.log_last_layer)) for j in jobs}
    out = np.zeros(sum(size[log_n] * len(ab) for log_n, ab in jobs), dtype=np.uint8)
    torch.cuda.synchronize()
    return {"run": run_serve, "server": server, "jobs": jobs, "size": size, "out": out}


def run_serve(s):
    server, at, base = s["server"], 0, s["out"].ctypes.data
    ids = [server.submit(log_n, ab) for log_n, ab in s["jobs"]]
    server.wait_all()
    for job, (log_n, ab) in zip(ids, s["jobs"]):
        size = s["size"][log_n]
        for col in range(len(ab)):
            vx.lib.vx_server_proof_copy(server.handle, job, col, base + at, size)
            at += size
        server.release(job)
    return s["out"]


def prepare_wide(case, num):
    logs = parse_sizes(case["sizes"])
    wide = vx.WideCommit(logs, case["blowup"], case["last"])
    cols = [num.column(1 << k) for k in logs]
    lde = [view(wide, vx.lib.vx_wide_lde_device(wide.handle, c), 1 << (k + case["blowup"])) for c, k in enumerate(logs)]
    return {"run": run_wide, "wide": wide, "cols": cols, "addrs": [c.data_ptr() for c in cols], "lde": lde}


def run_wide(s):
    s["wide"].commit_device(s["addrs"])
    return {"results": [r.view(np.int32) for r in s["wide"].results()], "lde": s["lde"]}


def prepare_deep(case, num):
    logs = parse_sizes(case["sizes"])
    top, n_points = logs[-1], case["points"]
    cols = [num.column(1 << k) for k in logs]
    xs, ys = vx.circle_domain_points(top)
    points = np.array([num.one() for _ in range(8 * n_points)], np.uint32).reshape(n_points, 8)
    coeffs = np.array([num.one() for _ in range(12 * n_points * len(logs))], np.uint32)
    return {"run": run_deep, "deep": vx.DeepQuotient(len(logs), n_points), "cols": cols,
            "addrs": [c.data_ptr() for c in cols], "logs": logs, "points": points,
            "coeffs": coeffs.reshape(n_points, len(logs), 12), "top": top, "xs": xs, "ys": ys,
            "out": [words(1 << top) for _ in range(4)]}


def run_deep(s):
    s["deep"].quotient(s["addrs"], s["logs"], s["points"], s["coeffs"], s["top"], s["xs"].addr, s["ys"].addr,
                       [o.data_ptr() for o in s["out"]])
    return s["out"]


def prepare_native_lde(case, num):
    log_n, cols = case["log_n"], case["cols"]
    trace = []
    for _ in range(cols):
        t = words(1 << log_n)
        vx.lib.vx_fibonacci_trace(num.one(), num.one(), log_n, t.data_ptr(), None)
        trace.append(t)
    coeffs, evals = [words(1 << log_n) for _ in range(cols)], [words(4 << log_n) for _ in range(cols)]
    return {"run": run_native_lde, "n": 1 << log_n, "trace": trace, "coeffs": coeffs, "evals": evals,
            "inv": NativeTwiddles(log_n, True), "fwd": NativeTwiddles(log_n + 2, False),
            "coeff_ptrs": ptrs(coeffs), "eval_ptrs": ptrs(evals)}


def run_native_lde(s):
    lib, n, inv, fwd, cols = vx.lib, s["n"], s["inv"], s["fwd"], len(s["trace"])
    ti = (inv.line.data_ptr(), inv.circle.data_ptr(), inv.offs, inv.sizes, inv.n_line, n)
    te = (fwd.line.data_ptr(), fwd.circle.data_ptr(), fwd.offs, fwd.sizes, fwd.n_line, 4 * n)
    for t, c in zip(s["trace"], s["coeffs"]):  # the transforms work in place
        c.copy_(t)
    if cols == 1:
        lib.cuda_circle_ntt_interpolate(s["coeffs"][0].data_ptr(), *ti)
    else:
        lib.cuda_circle_ntt_interpolate_batch(s["coeff_ptrs"].data_ptr(), *ti, cols)
    for c, e in zip(s["coeffs"], s["evals"]):
        lib.cuda_zero_pad(c.data_ptr(), e.data_ptr(), n, 4 * n)
    if cols == 1:
        lib.cuda_circle_ntt_evaluate(s["evals"][0].data_ptr(), *te)
    else:
        lib.cuda_circle_ntt_evaluate_batch(s["eval_ptrs"].data_ptr(), *te, cols)
    return [s["coeffs"], s["evals"]]


def native_layers(log_e):
    """log2 of the layers folded on the GPU: the circle fold's, then line folds down to 2^10."""
    return list(range(log_e - 1, 9, -1))


def prepare_native_fri(case, num):
    log_e = case["log_e"]
    E = 1 << log_e
    layers = [[words(1 << k) for _ in range(4)] for k in native_layers(log_e)]
    # the evaluation column is any M31 column: the commitments and folds do not depend on its degree
    evals = num.column(E)
    alphas = [h32([num.one() for _ in range(4)]) for _ in range(2 + 2 * len(layers))]
    nodes = [words(8 * max(1, E >> 10)), words(8 * max(1, E >> 11))]
    return {"run": run_native_fri, "log_e": log_e, "eval": evals, "eval_ptr": ptrs([evals]),
            "quotient": [words(E) for _ in range(4)], "layers": layers, "alphas": alphas, "nodes": nodes,
            "sources": words(E // 2), "twiddles": words(E // 2),
            "roots": torch.zeros(8 * (2 + len(layers)), dtype=torch.int32, device=DEV)}


def native_root(s, n_nodes, root):
    """Subtree roots to the tree's root, level by level while one workgroup cannot take them."""
    a, b = s["nodes"]
    while n_nodes > 1024:
        n_nodes //= 2
        vx.lib.cuda_merkle_hash_nodes(a.data_ptr(), b.data_ptr(), n_nodes)
        a, b = b, a
    vx.lib.cuda_merkle_reduce_to_root(a.data_ptr(), root, n_nodes)


def native_tree_soa4(s, cols, n, root):
    p = [c.data_ptr() for c in cols]
    if n <= 2048:
        vx.lib.cuda_merkle_commit_small_soa4(*p, root, n)
    else:
        vx.lib.cuda_merkle_tiled_soa4(*p, s["nodes"][0].data_ptr(), n)
        native_root(s, n // 1024, root)


def run_native_fri(s):
    lib, log_e = vx.lib, s["log_e"]
    E, root = 1 << log_e, s["roots"].data_ptr()
    lib.cuda_merkle_tiled_generic(s["eval_ptr"].data_ptr(), s["nodes"][0].data_ptr(), 1, E)
    native_root(s, E // 1024, root)
    q = [c.data_ptr() for c in s["quotient"]]
    lib.cuda_fibonacci_quotient(s["eval"].data_ptr(), *q, s["alphas"][0], E)
    native_tree_soa4(s, s["quotient"], E, root + 32)
    prev = q
    for j, cols in enumerate(s["layers"]):
        k, out = log_e - j, [c.data_ptr() for c in cols]
        (ix, iy), (sx, sy) = half_coset(k) if j == 0 else half_odds(k)
        half = 1 << (k - 1)
        lib.cuda_compute_fold_twiddle_sources(ix, iy, sx, sy, s["sources"].data_ptr(), 2 * half, k, 1 if j == 0 else 0)
        lib.cuda_batch_inverse_m31(s["sources"].data_ptr(), s["twiddles"].data_ptr(), half)
        if j == 0:
            for c in cols:
                c.zero_()
            lib.cuda_fold_circle_into_line_soa(*out, *prev, s["twiddles"].data_ptr(), s["alphas"][1], s["alphas"][2], half)
        else:
            lib.cuda_fold_line_soa(*prev, s["twiddles"].data_ptr(), *out, s["alphas"][2 + j], half)
        native_tree_soa4(s, cols, half, root + 64 + 32 * j)
        prev = out
    return {"roots": s["roots"], "quotient": s["quotient"], "first": s["layers"][0], "last": s["layers"][-1]}


def prepare_stwo(case, num):
    trace_logs = parse_sizes(case["sizes"])
    logs = [k + 2 for k in trace_logs]
    S, n_cols, n_points = logs[-1], len(logs), case["points"]
    fwd, inv = vx.stwo_twiddles_device(S)  # a smaller domain's buffer is a suffix of the largest's
    xs, ys = vx.circle_domain_points(S)
    trace = [num.column(1 << k) for k in trace_logs]
    coeffs, evals = [words(1 << k) for k in trace_logs], [words(1 << k) for k in logs]
    chunks, at = [], 0
    for k in sorted(set(logs)):
        group = [c for c in range(n_cols) if logs[c] == k]
        for i in range(0, len(group), 16):
            part = group[i: i + 16]
            chunks.append(part + [0] * (16 - len(part)) + [len(part), k])
    accs = [(p, k) for p in range(n_points) for k in sorted(set(logs))]
    numers = [[words(1 << k) for _ in range(4)] for _, k in accs]
    folds = []
    for k in range(S, max(S - 4, 4), -1):  # the circle fold and the first line folds
        d, half = half_odds(k - 1) if k == S else half_odds(k), 1 << (k - 1)
        src, tw = words(half), words(half)
        if k == S:
            src.copy_(view(ys, ys.addr, 1 << S)[0::2])
        else:
            vx.lib.cuda_compute_fold_twiddle_sources(*d[0], *d[1], src.data_ptr(), 2 * half, k, 0)
        vx.lib.cuda_batch_inverse_m31(src.data_ptr(), tw.data_ptr(), half)
        folds.append((tw, [torch.zeros(half, dtype=torch.int32, device=DEV) for _ in range(4)], h32([num.one() for _ in range(4)])))
    s = {"run": run_stwo, "logs": logs, "S": S, "n_points": n_points, "fwd": fwd, "inv": inv, "xs": xs, "ys": ys,
         "trace": trace, "coeffs": coeffs, "evals": evals, "eval_ptrs": ptrs(evals), "n_chunks": len(chunks),
         "schedule": torch.tensor(chunks, dtype=torch.int32, device=DEV), "accs": accs, "numers": numers,
         "tree": [words(8 << k) for k in range(S, -1, -1)],
         "indices": [torch.tensor([c for c in range(n_cols) if logs[c] == k], dtype=torch.int32, device=DEV) for _, k in accs],
         "b": [num.column(4 * n_cols) for _ in accs], "c": [num.column(4 * n_cols) for _ in accs],
         "px": num.column(4 * len(accs)), "py": num.column(4 * len(accs)), "fla": num.column(4 * len(accs)),
         "acc_logs": torch.tensor([k for _, k in accs], dtype=torch.int32, device=DEV),
         "numer_ptrs": [ptrs([n[i] for n in numers]) for i in range(4)],
         "quotient": [words(1 << S) for _ in range(4)], "folds": folds}
    torch.cuda.synchronize()
    return s


def run_stwo(s):
    lib, S, logs = vx.lib, s["S"], s["logs"]
    tc = 1 << (S - 1)
    for t, c, e, k in zip(s["trace"], s["coeffs"], s["evals"], logs):
        c.copy_(t)  # the transforms work in place
        lib.cuda_stwo_ntt_interpolate(c.data_ptr(), s["inv"].addr + 4 * (tc - (1 << (k - 3))), 1 << (k - 2))
        lib.cuda_zero_pad(c.data_ptr(), e.data_ptr(), 1 << (k - 2), 1 << k)
        lib.cuda_stwo_ntt_evaluate(e.data_ptr(), s["fwd"].addr + 4 * (tc - (1 << (k - 1))), 1 << k)
    tree = s["tree"]
    lib.cuda_build_leaves_lifted(s["eval_ptrs"].data_ptr(), s["schedule"].data_ptr(), s["n_chunks"], S, tree[0].data_ptr(), 1 << S)
    for k in range(S):
        lib.cuda_merkle_hash_nodes(tree[k].data_ptr(), tree[k + 1].data_ptr(), 1 << (S - 1 - k))
    for i, (_, k) in enumerate(s["accs"]):
        lib.cuda_accumulate_numerators(s["eval_ptrs"].data_ptr(), s["indices"][i].data_ptr(), s["b"][i].data_ptr(),
                                       s["c"][i].data_ptr(), s["indices"][i].numel(), 1 << k,
                                       *[o.data_ptr() for o in s["numers"][i]])
    q = [o.data_ptr() for o in s["quotient"]]
    lib.cuda_compute_quotients_combine(s["px"].data_ptr(), s["py"].data_ptr(), s["fla"].data_ptr(),
                                       *[p.data_ptr() for p in s["numer_ptrs"]], s["acc_logs"].data_ptr(), len(s["accs"]),
                                       s["xs"].addr, s["ys"].addr, S, 1 << S, *q)
    prev, zero = q, h32([0, 0, 0, 0])
    for j, (tw, cols, alpha) in enumerate(s["folds"]):
        out, half = [c.data_ptr() for c in cols], tw.numel()
        if j == 0:  # onto what the layer held, times zero: the layer starts empty
            lib.cuda_fold_circle_into_line_soa(*out, *prev, tw.data_ptr(), alpha, zero, half)
        else:
            lib.cuda_fold_line_soa(*prev, tw.data_ptr(), *out, alpha, half)
        prev = out
    return {"evals": s["evals"], "leaves": tree[0], "root": tree[-1], "quotient": s["quotient"],
            "folded": [c for _, cols, _ in s["folds"][-1:] for c in cols]}


# ---------------------------------------------------------------- work
def ntt_ops(log_n):
    return BUTTERFLY_OPS * log_n * (1 << log_n) / 2


def proof_work(log_n, queries, last):
    """One proof: interpolation and evaluation (whose top two layers only copy), 6 E compressions
    (trace and quotient trees of E leaves, FRI trees of E / 2 and less); the trace read, the proof written."""
    E, log_e = 4 << log_n, log_n + 2
    depth = sum(range(last + 1, log_e)) + 2 * log_e
    proof = 8 * queries * (depth * 8 + 5 * (log_e - last + 2))
    return 4 * (1 << log_n) + proof, COMPRESSION_OPS * 6 * E + ntt_ops(log_n) + BUTTERFLY_OPS * log_n * E / 2


def work(case):
    kind = case["kind"]
    if kind in ("prove", "prove_device", "prove_once", "prove_batch"):
        nbytes, ops = proof_work(case["log_n"], case["queries"], case["last"])
        n = case.get("count", 1)
        return {"bytes": n * nbytes, "flops": n * ops}
    if kind == "serve":
        each = [(proof_work(log_n, 80, 3), cols) for log_n, cols in job_list(case)]
        return {"bytes": sum(w[0] * c for w, c in each), "flops": sum(w[1] * c for w, c in each)}
    if kind in ("wide", "deep", "stwo"):
        logs = parse_sizes(case["sizes"])
        n = len(logs)
        if kind == "deep":
            rows = 1 << logs[-1]
            return {"bytes": 4 * sum(1 << k for k in logs) + 8 * rows + 16 * rows,
                    "flops": rows * case["points"] * (8 * n + 250)}
        B = case.get("blowup", 2)
        leaves = 1 << (logs[-1] + B)
        lde = sum(ntt_ops(k) + BUTTERFLY_OPS * k * (1 << (k + B)) / 2 for k in logs)
        tree = COMPRESSION_OPS * leaves * (math.ceil(n / 16) + 1)
        cols = 4 * sum((1 << k) + (1 << (k + B)) for k in logs)
        if kind == "wide":
            return {"bytes": cols, "flops": lde + tree + COMPRESSION_OPS * 2 * leaves}
        accs = case["points"] * len(set(logs))
        return {"bytes": cols + 4 * sum(4 << k for k in logs) * case["points"] + 2 * 32 * leaves + 16 * leaves * (accs + 2) + 8 * leaves,
                "flops": lde + tree + leaves * accs * 259}
    if kind == "native_lde":
        n, k = 1 << case["log_n"], case["log_n"]
        return {"bytes": case["cols"] * 4 * (n + n + 4 * n), "flops": case["cols"] * (ntt_ops(k) + BUTTERFLY_OPS * k * 4 * n / 2)}
    E = 1 << case["log_e"]
    return {"bytes": 4 * E + 16 * E + 16 * E, "flops": COMPRESSION_OPS * 6 * E}


def exact(case, seed):
    """Every output is whole numbers, which have to be equal: there is no rounding to measure."""
    return None
