"""Workloads of the library's public entry points: seed matching over 2 to 8
genomes, the batched inter-anchor DP (full, banded, wildcard letters), the band
network, and the whole pairwise path.

A case is a dict of plain values with a "kind":

  match     sorted mer lists of 2 to 4 genomes + PairwiseMatchFinder
  unique    sorted mer lists of 5 to 8 genomes + UniqueMatchFinder
  dp        one batch of full DP jobs, some with wildcard letters
  band      gap features, network and banded DP with its fallback
  net       network output, loss and gradient of a batch of feature rows
  path      align_pair: two genomes in, alignment rows and index LUT out

Genomes and DP operands are made on the GPU from the seed alone.  Results whose
size depends on the inputs (match lists, paths, rows) go into buffers that the
program holds, sized by the case; what lies past the result stays zero.
"""
import ctypes as C
import os
import shutil
import sys
import tempfile
import weakref

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "mauve-py_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import mauvehip  # noqa: E402
from mauvehip import band, pipeline  # noqa: E402

CODING = mauvehip.CODING_SEED
X, OTHER = 4, 5                   # wildcard operand codes (mh_dp_job)


def listed():
    return [
        {"name": "match_pair_20kb", "kind": "match", "genomes": 2, "length": 20_000, "weight": 15, "rank": CODING},
        {"name": "match_pair_200kb_spaced", "kind": "match", "genomes": 2, "length": 200_003, "weight": 13, "rank": 0},
        {"name": "match_pair_4600kb", "kind": "match", "genomes": 2, "length": 4_600_000, "weight": 17,
         "rank": CODING},
        {"name": "match_four_1mb", "kind": "match", "genomes": 4, "length": 1_000_000, "weight": 17, "rank": CODING},
        {"name": "unique_eight_5mb", "kind": "unique", "genomes": 8, "length": 5_000_000, "weight": 19, "rank": 0},
        {"name": "dp_one_90", "kind": "dp", "jobs": 1, "shortest": 90, "longest": 90, "wild": 0.0},
        {"name": "dp_gaps_20k", "kind": "dp", "jobs": 20_000, "shortest": 5, "longest": 500, "wild": 0.0},
        {"name": "dp_long_4k", "kind": "dp", "jobs": 4_000, "shortest": 10, "longest": 20_000, "wild": 0.0},
        {"name": "dp_letters_2k", "kind": "dp", "jobs": 2_000, "shortest": 10, "longest": 1_000, "wild": 0.05},
        {"name": "band_gaps_6k", "kind": "band", "jobs": 6_000, "shortest": 10, "longest": 20_000},
        {"name": "net_rows_4096", "kind": "net", "rows": 4_096},
        {"name": "path_4600kb", "kind": "path", "length": 4_600_000, "weight": 17},
    ]


def _log_size(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["match", "match", "unique", "dp", "dp", "dp", "band", "net", "path"])
    if kind == "match":
        k = rng.choice([2, 2, 2, 3, 4])
        length = _log_size(rng, 3_000, 4_600_000 if k == 2 else 1_200_000)
        least = mauvehip.get_default_seed_weight(length) | 1
        return {"kind": kind, "genomes": k, "length": length, "weight": min(21, least + 2 * rng.randrange(2)),
                "rank": rng.choice([0, CODING])}
    if kind == "unique":
        k = rng.randrange(5, 9)
        length = _log_size(rng, 20_000, 5_000_000)
        least = mauvehip.get_default_seed_weight(length) | 1
        return {"kind": kind, "genomes": k, "length": length, "weight": max(11, min(19, least + 2 * rng.randrange(2))),
                "rank": rng.choice([0, CODING])}
    if kind == "dp":
        longest = _log_size(rng, 30, 20_000)
        # the batch's cells stay below those of the listed long batch
        jobs = min(40_000, max(1, int(4_000 * (20_000 / longest) ** 2 * rng.random())))
        jobs = _log_size(rng, 1, jobs) if rng.random() < 0.5 else jobs
        return {"kind": kind, "jobs": jobs, "shortest": rng.randrange(1, min(longest, 40)), "longest": longest,
                "wild": rng.choice([0.0, 0.0, 0.02, 0.1]) if longest <= 1_500 else 0.0}
    if kind == "band":
        longest = _log_size(rng, 500, 20_000)
        return {"kind": kind, "jobs": _log_size(rng, 50, 6_000), "shortest": rng.randrange(5, 40), "longest": longest}
    if kind == "net":
        return {"kind": kind, "rows": _log_size(rng, 100, 16_000)}
    length = _log_size(rng, 20_000, 4_600_000)
    return {"kind": kind, "length": length, "weight": rng.choice([15, 17])}


# ---- inputs ------------------------------------------------------------------

_shared = {}


def _context():
    if "ctx" not in _shared:
        _shared["ctx"] = mauvehip.Context(0)
    return _shared["ctx"]


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _derive(codes, lens, rate, indel_share, g):
    """Mutated copies of concatenated sequences: per base an event with
    probability rate (a value per sequence), a share of the events insertions
    or deletions of geometric length, the others substitutions.  No copy is
    left empty.  Returns (codes, lens)."""
    n = codes.numel()
    owner = torch.repeat_interleave(torch.arange(lens.numel(), device="cuda"), lens)
    event = torch.rand(n, device="cuda", generator=g) < rate[owner]
    kind = torch.rand(n, device="cuda", generator=g)
    ins, dele = event & (kind < indel_share / 2), event & (kind >= indel_share / 2) & (kind < indel_share)
    sub = event & (kind >= indel_share)
    shift = torch.randint(1, 4, (n,), device="cuda", generator=g, dtype=torch.uint8)
    out = torch.where(sub, (codes + shift) & 3, codes)
    size = 1 + torch.floor(torch.log(torch.rand(n, device="cuda", generator=g).clamp_min(1e-7)) / np.log(0.7)).long()
    start = torch.cumsum(lens, 0) - lens
    at = torch.arange(n, device="cuda")
    last = (start + lens)[owner]
    edge = torch.zeros(n + 1, dtype=torch.long, device="cuda")
    d = dele.nonzero().squeeze(1)
    edge.index_add_(0, d, torch.ones_like(d))
    edge.index_add_(0, torch.minimum(d + size[d], last[d]), -torch.ones_like(d))
    keep = torch.cumsum(edge[:n], 0) == 0
    keep |= at == start[owner]
    reps = keep.long() + torch.where(ins, size, torch.zeros_like(size))
    made = torch.repeat_interleave(out, reps)
    first = (torch.cumsum(reps, 0) - reps)[keep]
    new = torch.randint(0, 4, (made.numel(),), device="cuda", generator=g, dtype=torch.uint8)
    new[first] = made[first]
    total = torch.zeros_like(lens).index_add_(0, owner, reps)
    return new, total


def _genome(length, g):
    """Random bases with a few repeated stretches."""
    codes = torch.randint(0, 4, (length,), device="cuda", generator=g, dtype=torch.uint8)
    for _ in range(4):
        span = max(1, min(2_500, length // 50))
        a, b = (int(v) for v in torch.randint(0, length - span, (2,), generator=g, device="cuda"))
        codes[b:b + span] = codes[a:a + span].clone()
    return codes


def _relative(codes, rate, g):
    """A relative of a genome, of the same length: substitutions, indels and
    one inversion."""
    n = codes.numel()
    lens = torch.tensor([n], device="cuda")
    out, _ = _derive(codes, lens, torch.tensor([rate], device="cuda"), 0.05, g)
    tail = torch.randint(0, 4, (max(0, n - out.numel()),), device="cuda", generator=g, dtype=torch.uint8)
    out = torch.cat([out[:n], tail])
    span = max(2, min(30_000, n // 20))
    at = int(torch.randint(0, n - span, (1,), generator=g, device="cuda"))
    out[at:at + span] = 3 - out[at:at + span].flip(0)
    return out


_ASCII = torch.tensor(list(b"ACGT"), dtype=torch.uint8)


def _ascii(codes):
    return _ASCII.cuda()[codes.long()].contiguous()


def _family(k, length, g):
    """k genomes along a random binary tree from one ancestor."""
    leaves = [_genome(length, g)]
    while len(leaves) < k:
        parent = leaves.pop(int(torch.randint(0, len(leaves), (1,), generator=g, device="cuda")))
        leaves += [_relative(parent, 0.01 + 0.03 * float(torch.rand(1, generator=g, device="cuda")), g)
                   for _ in range(2)]
    return leaves


def _jobs(case, g):
    """DP jobs: A's length log-uniform, B derived from A at a divergence of
    2-30%; a share of the jobs hold a few wildcard letters."""
    n, lo, hi = case["jobs"], case["shortest"], case["longest"]
    # one length from each n-th of the range: the batch's total hardly varies
    u = (torch.randperm(n, device="cuda", generator=g)
         + torch.rand(n, device="cuda", generator=g, dtype=torch.float64)) / n
    la = torch.clamp((lo * torch.pow(torch.tensor((hi + 1) / lo, dtype=torch.float64, device="cuda"), u)).long(), 1, hi)
    rate = 0.02 + 0.28 * torch.rand(n, device="cuda", generator=g)
    a = torch.randint(0, 4, (int(la.sum()),), device="cuda", generator=g, dtype=torch.uint8)
    b, lb = _derive(a, la, rate, 0.1, g)
    a_off, b_off = torch.cumsum(la, 0) - la, torch.cumsum(lb, 0) - lb
    wild = case.get("wild", 0.0)
    if wild:
        pick = (torch.rand(n, device="cuda", generator=g) < wild).nonzero().squeeze(1)
        for codes, off, ln in ((a, a_off, la), (b, b_off, lb)):
            for letter in (OTHER, OTHER, X):
                at = off[pick] + (torch.rand(len(pick), device="cuda", generator=g) * ln[pick]).long()
                codes[at] = letter
    jobs = mauvehip.make_jobs(a_off.cpu().numpy(), la.cpu().numpy(), b_off.cpu().numpy(), lb.cpu().numpy())
    slots = int(2.3 * float(np.floor(lo * ((hi + 1) / lo) ** (np.arange(1, n + 1) / n)).sum())) + 64 * n
    assert int((la + lb).sum()) <= slots
    return {"a": a, "b": b, "jobs": jobs, "paths": torch.zeros(slots, dtype=torch.uint8, device="cuda"),
            "results": torch.zeros(n, 4, dtype=torch.int32, device="cuda")}


def _model():
    path = os.path.join(PKG, "mauvehip", "band_model.npz")
    return band.load_model(path)


def prepare(case, seed):
    ctx = _context()
    g = _generator(seed)
    kind = case["kind"]
    s = {"kind": kind, "ctx": ctx}
    if kind in ("match", "unique"):
        k, length = case["genomes"], case["length"]
        if kind == "match":
            base = _genome(length, g)
            codes = [base] + [_relative(base, 0.015, g) for _ in range(k - 1)]
        else:
            codes = _family(k, length, g)
        s["seqs"] = [_ascii(c) for c in codes]
        s["seed"] = mauvehip.get_seed(case["weight"], case["rank"])
        if kind == "match":
            s["matches"] = np.zeros(k * length // 8 + 1000, dtype=mauvehip.MATCH_DTYPE)
        else:
            s["starts"] = np.zeros((length // 2 + 1000, k), dtype=np.int64)
            s["lengths"] = np.zeros(len(s["starts"]), dtype=np.int64)
    elif kind == "dp":
        s.update(_jobs(case, g))
    elif kind == "band":
        s.update(_jobs(case, g))
        n = case["jobs"]
        s["features"] = torch.zeros(n, mauvehip.MLP_IN, dtype=torch.float32, device="cuda")
        s["dev"] = torch.zeros(n, dtype=torch.int32, device="cuda")
        params, s["delta"], s["min_band"] = _model()
        s["net"] = mauvehip.Mlp(ctx, params=params)
    elif kind == "net":
        rows = case["rows"]
        d = _jobs({"jobs": rows, "shortest": 10, "longest": 400}, g)
        s["x"] = torch.zeros(rows, mauvehip.MLP_IN, dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        mauvehip.gap_features_device(ctx, d["a"].data_ptr(), d["b"].data_ptr(), d["jobs"], s["x"].data_ptr())
        ctx.synchronize()
        label = torch.floor(60 * torch.rand(rows, device="cuda", generator=g) ** 3)
        s["t"] = torch.log2(1 + label)
        s["y"] = torch.zeros(rows, dtype=torch.float32, device="cuda")
        s["params"] = _model()[0]
        s["net"] = mauvehip.Mlp(ctx, params=s["params"])
    else:
        base = _genome(case["length"], g)
        seqs = [_ascii(_relative(base, 0.015, g)), _ascii(base)]
        s["seqs"] = seqs
        s["host"] = [q.cpu().numpy().tobytes() for q in seqs]
        s["seed"] = mauvehip.get_seed(case["weight"], CODING)
        folder = _Folder()
        s["folder"], s["xmfa"] = folder, os.path.join(folder.path, "pair.xmfa")
        s["rows"] = np.zeros((2, 2 * case["length"]), dtype=np.uint8)
    torch.cuda.synchronize()
    return s


class _Folder:
    """A temporary folder that goes with its state."""

    def __init__(self):
        self.path = tempfile.mkdtemp(prefix="pair_")
        self._gone = weakref.finalize(self, shutil.rmtree, self.path, True)


# ---- one pass ----------------------------------------------------------------

def run(s):
    ctx, kind = s["ctx"], s["kind"]
    if kind in ("match", "unique"):
        smls = [mauvehip.SortedMerList.from_device(ctx, q.data_ptr(), q.numel(), s["seed"]) for q in s["seqs"]]
        stats = (_pairwise if kind == "match" else _unique)(s, smls)
        for m in smls:
            m.free()
        out = [s["matches"].view(np.int64)] if kind == "match" else [s["starts"], s["lengths"]]
        return out + [int(stats.seed_tuples), int(stats.collisions), int(stats.matches)]
    if kind == "dp":
        mauvehip.global_align_device(ctx, s["a"].data_ptr(), s["b"].data_ptr(), s["jobs"], s["paths"].data_ptr(),
                                     s["results"].data_ptr())
        return [s["paths"], s["results"]]
    if kind == "band":
        a, b = s["a"].data_ptr(), s["b"].data_ptr()
        mauvehip.gap_features_device(ctx, a, b, s["jobs"], s["features"].data_ptr())
        bands = s["net"].predict_bands_device(s["features"].data_ptr(), len(s["jobs"]), s["delta"], s["min_band"])
        mauvehip.global_align_banded_device(ctx, a, b, s["jobs"], bands, s["paths"].data_ptr(),
                                            s["results"].data_ptr(), s["dev"].data_ptr())
        return [s["paths"], s["results"], s["dev"]]
    if kind == "net":
        rows = s["y"].numel()
        s["net"].forward_device(s["x"].data_ptr(), rows, s["y"].data_ptr())
        loss, grad = s["net"].grad_device(s["x"].data_ptr(), s["t"].data_ptr(), rows)
        return [s["y"], float(loss), grad]
    row_1, row_2, lut, _ = pipeline.align_pair(ctx, [q.data_ptr() for q in s["seqs"]], s["host"], s["seed"], s["xmfa"],
                                               ["genome1.fa", "genome2.fa"])
    s["rows"][0, :len(row_1)] = row_1
    s["rows"][1, :len(row_2)] = row_2
    return [s["rows"], lut]


def _checked(ctx, rc):
    if rc != mauvehip.MH_OK:
        raise RuntimeError(ctx.L.mh_last_error().decode())


def _pairwise(s, smls):
    """mh_find_matches_pairwise into the program's records."""
    ctx, out = s["ctx"], s["matches"]
    k, found, stats = len(smls), C.c_uint64(), mauvehip.MatchStats()
    _checked(ctx, ctx.L.mh_find_matches_pairwise(ctx.h, (C.c_void_p * k)(*[m.h.value for m in smls]), k,
                                                 out.ctypes.data, len(out), C.byref(found), C.byref(stats)))
    if found.value > len(out):
        raise RuntimeError("more matches than the program's records hold")
    return stats


def _unique(s, smls):
    """mh_find_matches_unique, its list copied into the program's arrays."""
    ctx, starts, lengths = s["ctx"], s["starts"], s["lengths"]
    k, h, stats = len(smls), C.c_void_p(), mauvehip.MatchStats()
    _checked(ctx, ctx.L.mh_find_matches_unique(ctx.h, (C.c_void_p * k)(*[m.h.value for m in smls]), k, C.byref(h),
                                               C.byref(stats)))
    try:
        n = ctx.L.mh_match_k_list_size(h)
        if n > len(starts):
            raise RuntimeError("more matches than the program's arrays hold")
        if n:
            C.memmove(starts.ctypes.data, ctx.L.mh_match_k_list_starts(h), n * k * 8)
            C.memmove(lengths.ctypes.data, ctx.L.mh_match_k_list_lengths(h), n * 8)
    finally:
        ctx.L.mh_match_k_list_free(h)
    return stats


# ---- what a pass cannot do without ------------------------------------------

# Integer operations of a DP cell: M, D and I each add once and take a maximum
# of two or three values.
CELL_OPS = 7


def _mean_cells(case):
    """Cells of the average job: A log-uniform on [shortest, longest], B of about its length."""
    lo, hi = case["shortest"], case["longest"] + 1
    return (hi * hi - lo * lo) / (2 * np.log(hi / lo))


def work(case):
    kind = case["kind"]
    if kind in ("match", "unique"):
        # the genomes read, a list entry per base (an 8-byte key, a 4-byte
        # position) written and read
        total = case["genomes"] * case["length"]
        return {"bytes": 25 * total, "flops": 0}
    if kind in ("dp", "band"):
        cells = case["jobs"] * _mean_cells(case)
        length = case["jobs"] * (case["longest"] + 1 - case["shortest"]) / np.log((case["longest"] + 1) / case["shortest"])
        if kind == "band":
            # the cells of bands of about a hundred columns each side of the diagonal
            cells = min(cells, 200 * length)
        return {"bytes": 4 * length + 40 * case["jobs"], "flops": CELL_OPS * cells}
    if kind == "net":
        layers = mauvehip.MLP_IN * mauvehip.MLP_H1 + mauvehip.MLP_H1 * mauvehip.MLP_H2 + mauvehip.MLP_H2
        return {"bytes": 4 * case["rows"] * (mauvehip.MLP_IN + 2) + 8 * mauvehip.MLP_NPARAMS,
                "flops": 2 * case["rows"] * layers * 4}
    # genomes, lists, rows, file and LUT; a 200-column window over each base in the DP of two passes
    return {"bytes": 62 * 2 * case["length"], "flops": CELL_OPS * 2 * 150 * case["length"]}


def tolerance(case):
    """Matches, paths, scores, rows and LUTs are whole numbers.  The network
    rounds activations and gradients to bf16 between its layers."""
    if case["kind"] == "net":
        return {"rel": 1e-2}
    return "exact"


def exact(case, seed):
    """The network's output, loss and gradient in 64 bits, without the
    rounding between its layers; the other kinds give whole numbers."""
    if case["kind"] != "net":
        return None
    s = prepare(case, seed)
    x, t = (s[k].cpu().numpy().astype(np.float64) for k in ("x", "t"))
    p = s["params"].astype(np.float64)
    parts, at = [], 0
    for shape in ((mauvehip.MLP_H1, mauvehip.MLP_IN), (mauvehip.MLP_H1,), (mauvehip.MLP_H2, mauvehip.MLP_H1),
                  (mauvehip.MLP_H2,), (mauvehip.MLP_H2,), (1,)):
        size = int(np.prod(shape))
        parts.append(p[at:at + size].reshape(shape))
        at += size
    w1, b1, w2, b2, w3, b3 = parts
    z1 = x @ w1.T + b1
    h1 = np.maximum(z1, 0)
    z2 = h1 @ w2.T + b2
    h2 = np.maximum(z2, 0)
    y = h2 @ w3 + b3[0]
    rows = len(t)
    d = (y - t) / rows
    g3, gb3 = h2.T @ d, d.sum()
    d2 = np.outer(d, w3) * (z2 > 0)
    g2, gb2 = d2.T @ h1, d2.sum(0)
    d1 = (d2 @ w2) * (z1 > 0)
    g1, gb1 = d1.T @ x, d1.sum(0)
    grad = np.concatenate([v.reshape(-1) for v in (g1, gb1, g2, gb2, g3, np.array([gb3]))])
    return [y, float(((y - t) ** 2).sum() / (2 * rows)), grad]
