"""Performance cases of the framework: what a user's program has it do,
through the public entry points of gpumemefficient_amd.

Kinds of case (the "kind" field):

  dropin   the reference's signatures LCS(), ED(), SW(): host symbols in,
           bottom-right cell out (symbol encoding, upload, launch, result),
           `calls` pairs one call after another;
  align    Context.align: one pair a call, score and (SW) maximum out, `calls`
           pairs one call after another;
  plan     Plan.run + Plan.results: pairs resident in HBM, run again and again;
  batch    Context.align_batch: many uneven pairs of host symbols in one call;
  serve    Server (stream slots): a backlog of requests submitted and drained;
  stencil  Context.stencil_device: one in-place SAT or 2D-SOR sweep of a table
           in HBM.

Symbols are int32 host arrays, as the reference's arr1 / arr2.  `related` is
the share of positions in which the second sequence of a pair differs from
(a copy of) the first, 0 for independent sequences, which is what the
reference's generator writes; SW pairs also hold a planted homologous
segment.
"""
from __future__ import annotations

import numpy as np
import torch

from gpumemefficient_amd import Context, ED, Job, LCS, SW, Tile, datagen
from gpumemefficient_amd.server import Server

DROPIN = {"LCS": LCS, "ED": ED, "SW": SW}


def listed():
    return [
        # The smallest pair the reference's generator writes (2^8 symbols),
        # through the reference's signature: the latency of a call.
        {"name": "lcs_256", "kind": "dropin", "problem": "LCS", "n1": 256, "n2": 256, "alphabet": 4, "related": 0.0,
         "calls": 8},
        # Ordinary requests: two related strings of uneven, odd lengths.
        {"name": "ed_1500", "kind": "align", "problem": "ED", "n1": 1531, "n2": 1187, "alphabet": 20, "related": 0.15,
         "textbook": True, "calls": 4},
        # Protein local alignment: 20 letters (row tables do not fit bytes),
        # score and maximum.
        {"name": "sw_protein", "kind": "align", "problem": "SW", "n1": 7013, "n2": 3001, "alphabet": 20,
         "related": 0.0, "no_max": False, "calls": 1},
        # The workload the reference publishes a time for.
        {"name": "lcs_32768", "kind": "dropin", "problem": "LCS", "n1": 32768, "n2": 32768, "alphabet": 4,
         "related": 0.0, "calls": 1},
        # The large edit-distance pair of bench.py, resident.
        {"name": "ed_65536", "kind": "plan", "problem": "ED", "n1": 65536, "n2": 65536, "alphabet": 20,
         "related": 0.0, "textbook": False},
        # A large local alignment with the maximum (the library's own output).
        {"name": "sw_32768_max", "kind": "align", "problem": "SW", "n1": 32768, "n2": 32768, "alphabet": 4,
         "related": 0.0, "no_max": False, "calls": 1},
        # bench.py's headline pair: the reference's output of SW() only.
        {"name": "sw_131072", "kind": "plan", "problem": "SW", "n1": 131072, "n2": 131072, "alphabet": 4,
         "related": 0.0, "no_max": True},
        # bench.py's batch: thousands of uneven pairs in one persistent launch.
        {"name": "sw_batch_4096", "kind": "plan", "problem": "SW", "count": 4096, "lo": 64, "hi": 4096,
         "alphabet": 4, "no_max": True},
        # A batch of host strings, compared once (encoding and upload count).
        {"name": "ed_batch_2048", "kind": "batch", "problem": "ED", "count": 2048, "lo": 64, "hi": 4096,
         "alphabet": 20, "textbook": True},
        # A backlog of the serving mix (ED and SW of 100 to 131072 symbols).
        {"name": "serve_200", "kind": "serve", "count": 200},
        # The table sweeps at bench.py's size, and one of odd sizes.
        {"name": "sat_32768", "kind": "stencil", "op": "SAT", "n1": 32768, "n2": 32768},
        {"name": "sor_9001", "kind": "stencil", "op": "SOR", "n1": 9001, "n2": 7043},
    ]


def _log(rng, lo, hi):
    return int(round(np.exp(rng.uniform(np.log(lo), np.log(hi)))))


def draw(rng):
    kind = rng.choice(["dropin", "align", "align", "plan", "plan", "batch", "batch", "serve", "stencil", "stencil"])
    if kind == "serve":
        return {"kind": kind, "count": _log(rng, 20, 150)}
    if kind == "stencil":
        return {"kind": kind, "op": rng.choice(["SAT", "SOR"]), "n1": _log(rng, 256, 24576),
                "n2": _log(rng, 256, 24576)}
    problem = rng.choice(["LCS", "ED", "SW"])
    case = {"kind": kind, "problem": problem,
            "alphabet": 4 if problem == "LCS" or (problem == "SW" and kind == "dropin") else rng.choice([4, 20])}
    if problem == "ED":
        case["textbook"] = rng.random() < 0.5 if kind != "dropin" else False
    if problem == "SW" and kind != "dropin":
        # Over 20 letters the last cell alone is 0 for most pairs: nobody asks for it without the maximum.
        case["no_max"] = case["alphabet"] == 4 and rng.random() < 0.5
    if kind == "batch" or (kind == "plan" and rng.random() < 0.4):
        lo = _log(rng, 32, 512)
        return {**case, "count": _log(rng, 8, 3000), "lo": lo, "hi": lo * rng.choice([1, 4, 8])}
    n1 = _log(rng, 128, 98304)
    n2 = min(98304, max(128, int(n1 * np.exp(rng.uniform(-1.5, 1.5)))))
    # A few calls a pass where a call is short.
    return {**case, "n1": n1, "n2": n2, "related": rng.choice([0.0, 0.0, 0.02, 0.15]),
            "calls": 1 if kind == "plan" or n1 * n2 > 5e7 else 4}


# ---------------------------------------------------------------- inputs

def _pair(rng, case, n1, n2):
    """One pair: independent letters, or the second a copy of the first with
    `related` of its letters replaced (and the lengths' difference appended);
    SW pairs get a homologous segment at an offset of each sequence."""
    k = case["alphabet"]
    a = rng.integers(0, k, n1, dtype=np.int32)
    b = rng.integers(0, k, n2, dtype=np.int32)
    rel = case.get("related", 0.0)
    m = min(n1, n2)
    if rel > 0.0:
        keep = rng.random(m) >= rel
        b[:m][keep] = a[:m][keep]
    elif case["problem"] == "SW":
        seg = m // 8
        if seg:
            oa, ob = int(rng.integers(0, n1 - seg + 1)), int(rng.integers(0, n2 - seg + 1))
            keep = rng.random(seg) >= 0.1
            b[ob:ob + seg][keep] = a[oa:oa + seg][keep]
    return a, b


def _pairs(case, seed):
    rng = np.random.default_rng([seed, 11])
    if "count" not in case:
        return [_pair(rng, case, case["n1"], case["n2"]) for _ in range(case.get("calls", 1))]
    n1 = datagen.loguniform_lengths(rng, case["count"], case["lo"], case["hi"])
    n2 = datagen.loguniform_lengths(rng, case["count"], case["lo"], case["hi"])
    return [_pair(rng, case, int(x), int(y)) for x, y in zip(n1, n2)]


def _jobs(case, seed):
    return [Job(case["problem"], a, b, ed_textbook=case.get("textbook", False), no_max=case.get("no_max", False))
            for a, b in _pairs(case, seed)]


def _requests(case, seed):
    return [Job(r.problem, r.a, r.b) for r in datagen.serving_requests(5e4, case["count"], seed=seed + 100)]


def _ld(n1):
    return (n1 + 3 + 3) // 4 * 4


def _table(case, seed):
    """An (n2 + 2) x (n1 + 3) table of small values, as the reference's
    generator writes, in rows of a pitch divisible by 4."""
    gen = torch.Generator(device="cuda").manual_seed(seed * 7919 + 5)
    return torch.randint(0, 100, (case["n2"] + 2, _ld(case["n1"])), dtype=torch.int32, device="cuda", generator=gen)


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    if kind == "serve":
        # The budget keeps three servers on one GPU.
        state["server"] = Server(0, hbm_budget=16 << 30)
        state["jobs"] = _requests(case, seed)
        return state
    if kind == "dropin":
        state["pairs"] = _pairs(case, seed)
        return state
    state["ctx"] = Context(0)
    if kind == "stencil":
        state["table"] = _table(case, seed)
    elif kind == "align":
        state["pairs"] = _pairs(case, seed)
        state["tile"] = Tile(no_max=True) if case.get("no_max") else None
    elif kind == "batch":
        state["jobs"] = _jobs(case, seed)
    else:
        state["plan"] = state["ctx"].plan(_jobs(case, seed))
    return state


# ---------------------------------------------------------------- one pass

def _scores(results):
    return {"last": np.array([r.last for r in results], dtype=np.int32),
            "max": np.array([r.max_score for r in results], dtype=np.int32)}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "dropin":
        f = DROPIN[case["problem"]]
        return [f(a.size, b.size, a, b, 3, 1, None, 32, 256) for a, b in state["pairs"]]
    if kind == "align":
        return _scores([state["ctx"].align(case["problem"], a, b, tile=state["tile"],
                                           ed_textbook=case.get("textbook", False)) for a, b in state["pairs"]])
    if kind == "plan":
        state["plan"].run()
        return _scores(state["plan"].results())
    if kind == "batch":
        return _scores(state["ctx"].align_batch(state["jobs"]))
    if kind == "serve":
        srv = state["server"]
        tickets = [srv.submit(j) for j in state["jobs"]]
        srv.wait_idle()
        done = {c.ticket: c for c in srv.poll()}
        return _scores([done[t] for t in tickets])
    t = state["table"]
    state["ctx"].stencil_device(case["op"], t.data_ptr(), case["n1"], case["n2"], t.shape[1])
    return t[:, :case["n1"] + 3]


# ---------------------------------------------------------------- work

# Integer operations of one cell of the reference's recurrences.
OPS = {"LCS": 4, "ED": 7, "SW": 8, "SAT": 3, "SOR": 5}


def work(case):
    if case["kind"] == "stencil":
        cells = case["n1"] * case["n2"]
        return {"bytes": 8 * cells, "flops": OPS[case["op"]] * cells}
    if case["kind"] == "serve":
        pairs = [(r.problem, r.a.size, r.b.size) for r in datagen.serving_requests(5e4, case["count"], seed=100)]
    elif "count" in case:
        # The mean of log-uniform lengths.
        lo, hi = case["lo"], case["hi"]
        mean = (hi - lo) / np.log(hi / lo) if hi > lo else lo
        return {"bytes": 8 * case["count"] * mean + 8 * case["count"],
                "flops": OPS[case["problem"]] * case["count"] * mean * mean}
    else:
        pairs = [(case["problem"], case["n1"], case["n2"])] * case.get("calls", 1)
    return {"bytes": sum(4 * (x + y) + 8 for _, x, y in pairs), "flops": sum(OPS[p] * x * y for p, x, y in pairs)}


# ---------------------------------------------------------------- exact results

def _dp(problem, a, b, textbook):
    """(bottom-right cell, maximum) of one pair, by anti-diagonals: cells
    (y, d - y) of one diagonal together, in 64 bits."""
    a, b = a.astype(np.int64), b.astype(np.int64)
    n1, n2 = a.size, b.size

    def edge_row(x):  # row 0
        return 0 if problem != "ED" else x if textbook else max(0, x - 1)

    prev2 = np.zeros(n2 + 1, dtype=np.int64)  # indexed by y
    prev = np.zeros(n2 + 1, dtype=np.int64)
    best = 0
    prev[0] = edge_row(1)
    if n2 >= 1:
        prev[1] = 1 if problem == "ED" else 0
    for d in range(2, n1 + n2 + 1):
        cur = np.zeros(n2 + 1, dtype=np.int64)
        y0, y1 = max(1, d - n1), min(n2, d - 1)
        y = slice(y0, y1 + 1)
        up, left, diag = prev[y0 - 1:y1], prev[y], prev2[y0 - 1:y1]
        eq = b[y0 - 1:y1] == a[d - y1 - 1:d - y0][::-1]
        if problem == "LCS":
            cur[y] = np.where(eq, diag + 1, np.maximum(left, up))
        elif problem == "ED":
            cur[y] = np.where(eq, diag, 1 + np.minimum(np.minimum(up, left), diag))
        else:
            cur[y] = np.maximum(np.maximum(np.maximum(left - 2, up - 2), diag + np.where(eq, 3, -3)), 0)
            best = max(best, int(cur[y].max()))
        if d <= n1:
            cur[0] = edge_row(d)
        if d <= n2 and problem == "ED":
            cur[d] = d
        prev2, prev = prev, cur
    return int(prev[n2]), best


def _sor(t, n1, n2):
    """One Gauss-Seidel sweep, by anti-diagonals of the flat table."""
    ld = t.shape[1]
    f = np.ascontiguousarray(t.cpu().numpy()).astype(np.int64).reshape(-1)
    for d in range(2, n1 + n2 + 1):
        y0, y1 = max(1, d - n1), min(n2, d - 1)
        start, count = y0 * ld + d - y0, y1 - y0 + 1
        step = ld - 1

        def at(off):
            s = start + off
            return f[s:s + (count - 1) * step + 1:step]

        s = at(-1) + at(-ld) + at(0) + at(1) + at(ld)
        at(0)[:] = np.sign(s) * (np.abs(s) // 5)  # C division truncates
    return f.reshape(-1, ld)[:, :n1 + 3]


def exact(case, seed):
    kind = case["kind"]
    if kind == "stencil":
        n1, n2 = case["n1"], case["n2"]
        t = _table(case, seed)
        if case["op"] == "SOR":
            return _sor(t, n1, n2) if n1 * n2 <= 1e8 else None
        if n1 * n2 > 2e9:
            return None
        # T(y, x) = T(0, x) + T(y, 0) - T(0, 0) + the sum of the interior up to (y, x).
        out = t[:, :n1 + 3].to(torch.int64)
        inner = out[1:n2 + 1, 1:n1 + 1].cumsum(0).cumsum(1)
        inner += out[0, 1:n1 + 1] + out[1:n2 + 1, :1] - out[0, 0]
        out[1:n2 + 1, 1:n1 + 1] = (inner + 2 ** 31) % 2 ** 32 - 2 ** 31
        return out
    if kind in ("batch", "serve") or "count" in case or case["n1"] * case["n2"] * case.get("calls", 1) > 1e8:
        return None
    got = [_dp(case["problem"], a, b, case.get("textbook", False)) for a, b in _pairs(case, seed)]
    if kind == "dropin":
        return [last for last, _ in got]
    mx = None if case.get("no_max") else np.array([best for _, best in got])
    return {"last": np.array([last for last, _ in got]), "max": mx}
