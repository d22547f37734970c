"""Workloads for timing and checking the library through its public entry points.

listed() gives the fixed cases, draw(rng) one more of the same ranges. For a
case, prepare(case, seed) makes what a program holds before the call (tensors,
factors, handles, plans), run(state) makes one pass through the library,
work(case) the bytes and operations the pass cannot do without, and
exact(case, seed) the pass's results in 64-bit floating point with torch.

Kinds of case:
  mttkrp  one mode-0 MTTKRP of a device-resident CSF on device factors
  ttv     one TTV over the last mode of a device-resident CSF
  modes   the MTTKRPs of every non-root mode of one device-resident CSF
  batch   every mode of several uneven tensors, one captured graph replay
  cp_als  a CP-ALS sweep over several tensors, factors read back
  host    the drop-in call on host operands: validation, transfers, kernel
"""

import ctypes
import math

import numpy as np
import torch

import tentaco_amd as tt

LEAF_MEAN = 7.4  # mean nonzeros per level N-2 node of the generator's log-normal(1.5, 1)
MID_MEAN = 4.5   # mean children of the levels between
DEVICE = "cuda:0"


def listed():
    return [
        # the smallest calls: a 10k-nonzero block inside an outer loop, where
        # launches and latency are the cost
        {"name": "mttkrp_small", "kind": "mttkrp", "dims": "1003,2017,1511", "nnz": 10007, "rank": 16,
         "skew": 1.1, "variant": "auto"},
        # the headline benchmark tensor: uniform coordinates, one nonzero per fibre
        {"name": "mttkrp_uniform", "kind": "mttkrp", "dims": "4096,4096,4096", "nnz": 500000, "rank": 32,
         "skew": 0.0, "variant": "auto"},
        # the largest benchmark tensor: 100M nonzeros, giant Zipf slices
        {"name": "mttkrp_3way_large", "kind": "mttkrp", "dims": "500000,500000,500000", "nnz": 100000000,
         "rank": 32, "skew": 1.1, "variant": "auto"},
        # the 4-mode benchmark tensor at the widest benchmark rank
        {"name": "mttkrp_4way_r64", "kind": "mttkrp", "dims": "200000,200000,200000,200000",
         "nnz": 60000000, "rank": 64, "skew": 1.1, "variant": "auto"},
        # an ordinary 5-mode tensor with ragged dims at the narrow benchmark rank
        {"name": "mttkrp_5way_mid", "kind": "mttkrp", "dims": "12007,5003,20011,3001,9001", "nnz": 1500007,
         "rank": 16, "skew": 1.1, "variant": "auto"},
        # a rank that is no power of two (users pick 10, 20, 50, 100 freely)
        {"name": "mttkrp_rank50", "kind": "mttkrp", "dims": "60013,45007,30011", "nnz": 5000011, "rank": 50,
         "skew": 1.1, "variant": "auto"},
        # the TTV benchmark tensor: c wider than one LDS window
        {"name": "ttv_large", "kind": "ttv", "dims": "100000,100000,100000", "nnz": 20000000, "skew": 1.1},
        # a small 4-mode TTV inside a loop
        {"name": "ttv_small", "kind": "ttv", "dims": "1003,317,523,2011", "nnz": 200003, "skew": 1.1},
        # all non-root modes on one CSF, for programs that cannot hold a CSF per mode
        {"name": "one_csf_modes", "kind": "modes", "dims": "100000,100000,100000", "nnz": 20000000,
         "rank": 32, "skew": 1.1},
        # a batch of uneven tensors, every mode, replayed from a graph
        {"name": "batch_uneven", "kind": "batch", "tensors": 8, "nnz_lo": 10000, "nnz_hi": 2000000,
         "dim_lo": 1000, "dim_hi": 300000, "rank": 32},
        # CP-ALS of several tensors (orders 3, 4, 5): a sweep, its fit and its factors
        {"name": "cp_als_uneven", "kind": "cp_als", "tensors": 3, "nnz_lo": 200000, "nnz_hi": 1000000,
         "dim_lo": 2000, "dim_hi": 40000, "rank": 32, "sweeps": 1},
        # the reference's own call with host operands, as a relinked program makes it
        {"name": "host_dropin", "kind": "host", "op": "mttkrp_gpu_taco", "dims": "10007,20011,5003",
         "nnz": 2000003, "rank": 32, "skew": 1.1},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dims(rng, order, lo, hi):
    return ",".join(str(_log_int(rng, lo, hi)) for _ in range(order))


def draw(rng):
    kind = rng.choice(["mttkrp"] * 5 + ["ttv", "ttv", "modes", "batch", "cp_als", "host"])
    order = rng.choice([3, 3, 4, 5])
    if kind == "mttkrp":
        rank = rng.choice([16, 32, 64, 16, 32, 64, 7, 10, 20, 25, 50, 100, 128])
        if order == 3 and rng.random() < 0.25:  # uniform coordinates, short fibres
            nnz = _log_int(rng, 1e4, 4e6)
            return {"kind": kind, "dims": _dims(rng, 3, 1000, 50000), "nnz": nnz, "rank": rank, "skew": 0.0,
                    "variant": "auto"}
        default = rng.random() < 0.1
        nnz = _log_int(rng, 1e4, 2e6 if default else 3e7)
        return {"kind": kind, "dims": _dims(rng, order, 1000, 200000), "nnz": nnz, "rank": rank,
                "skew": round(rng.uniform(0.8, 1.5), 2), "variant": "default" if default else "auto"}
    if kind == "ttv":
        return {"kind": kind, "dims": _dims(rng, order, 1000, 200000), "nnz": _log_int(rng, 1e4, 2e7),
                "skew": round(rng.uniform(0.8, 1.5), 2)}
    if kind == "modes":
        return {"kind": kind, "dims": _dims(rng, order, 1000, 100000), "nnz": _log_int(rng, 1e5, 1e7),
                "rank": rng.choice([16, 32, 64, 20]), "skew": round(rng.uniform(0.8, 1.5), 2)}
    if kind == "batch":
        return {"kind": kind, "tensors": rng.randint(4, 10), "nnz_lo": 10000, "nnz_hi": _log_int(rng, 1e5, 2e6),
                "dim_lo": 1000, "dim_hi": _log_int(rng, 1e4, 3e5), "rank": rng.choice([16, 32, 32, 64])}
    if kind == "cp_als":
        return {"kind": kind, "tensors": rng.randint(1, 3), "nnz_lo": 100000, "nnz_hi": _log_int(rng, 2e5, 1e6),
                "dim_lo": 1000, "dim_hi": _log_int(rng, 1e4, 4e4), "rank": rng.choice([16, 32, 64]), "sweeps": 1}
    op = rng.choice(["mttkrp_gpu_taco", "mttkrp", "ttv"])
    order = 3 if op == "mttkrp_gpu_taco" else order
    return {"kind": kind, "op": op, "dims": _dims(rng, order, 1000, 50000), "nnz": _log_int(rng, 1e4, 2e6),
            "rank": rng.choice([16, 32, 64]), "skew": round(rng.uniform(0.8, 1.5), 2)}


# ---------------------------------------------------------------------------
# inputs
class Buffer:
    """A torch tensor handed to the handle API, which takes objects with a
    device pointer in .ptr."""

    def __init__(self, t):
        assert t.is_contiguous()
        self.t = t
        self.ptr = ctypes.c_void_p(t.data_ptr())


def _dims_of(case):
    return [int(d) for d in case["dims"].split(",")]


def _uniform(shape, gen):
    return torch.rand(shape, generator=gen, device=DEVICE, dtype=torch.float32) * 2 - 1


def _gen(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _tensor(dims, nnz, skew, seed):
    """Host CSF: skew > 0 the Zipf slice / log-normal fibre generator, else
    uniform coordinates with duplicates summed."""
    if skew > 0:
        return tt.Csf.synth(len(dims), dims, nnz, slice_s=skew, seed=seed)
    rng = np.random.default_rng(seed)
    coords = np.stack([rng.integers(0, d, nnz) for d in dims]).astype(np.int32)
    return tt.Csf.from_coo(dims, coords, rng.uniform(-1, 1, nnz).astype(np.float32))


def _ttv_tensor(case, seed):
    """The tensor of a TTV: the output has one entry per fibre, so its pattern
    depends on the case alone and its values on the seed."""
    B = _tensor(_dims_of(case), case["nnz"], case["skew"], 17)
    B.vals = np.random.default_rng(seed).uniform(-1, 1, B.nnz).astype(np.float32)
    return B


def _is_ttv(case):
    return case["kind"] == "ttv" or case.get("op") == "ttv"


def _uneven(case, seed):
    """The uneven tensor list of a batch: its shape depends on the case
    alone, its entries on the seed."""
    rng = np.random.default_rng(7)
    out = []
    for t in range(case["tensors"]):
        order = 3 + t % 3
        dims = [int(round(math.exp(rng.uniform(math.log(case["dim_lo"]), math.log(case["dim_hi"])))))
                for _ in range(order)]
        nnz = int(round(math.exp(rng.uniform(math.log(case["nnz_lo"]), math.log(case["nnz_hi"])))))
        out.append((dims, nnz, float(rng.uniform(0.8, 1.5)), seed * 1000 + t))
    return [_tensor(*a) for a in out]


def prepare(case, seed):
    kind = case["kind"]
    gen = _gen(seed)
    s = {"case": case}
    if kind == "batch" or kind == "cp_als":
        R = case["rank"]
        hosts = _uneven(case, seed)
        s["R"] = R
        handles = [[tt.DeviceCsf(Bm) for Bm in B.mode_csfs()] for B in hosts]
        s["handles"] = handles
        if kind == "batch":
            factors = [[_uniform((d, R), gen) for d in B.dims] for B in hosts]
            s["outs"] = [torch.empty((B.dims[m], R), device=DEVICE) for B in hosts for m in range(B.order)]
            s["batch"] = tt.Batch([h for hs in handles for h in hs], R)
            operands = [[Buffer(f[k]) for k in range(B.order) if k != m]
                        for B, f in zip(hosts, factors) for m in range(B.order)]
            s["batch"].set_operands(operands, [Buffer(o) for o in s["outs"]], [o.shape[0] for o in s["outs"]])
            s["batch"].set_output_mode(tt.Batch.OUTPUTS_RETAINED)
            s["batch"].capture()
            s["factors"] = factors
        else:
            s["cpd"] = tt.Cpd(handles, R, seed=seed)
            for t, B in enumerate(hosts):
                for m, f in enumerate(_als_start(B, R, seed, t)):
                    s["cpd"].set_factor(t, m, f)
            s["orders"] = [B.order for B in hosts]
        return s
    B = _ttv_tensor(case, seed) if _is_ttv(case) else _tensor(_dims_of(case), case["nnz"], case["skew"], seed)
    s["R"] = R = case.get("rank", 1)
    if kind == "host":
        s["B"] = B
        if case["op"] == "ttv":
            s["c"] = _uniform((B.dims[-1],), gen).cpu().numpy()
        else:
            s["factors"] = [_uniform((d, R), gen).cpu().numpy() for d in B.dims[1:]]
        if case["op"] == "mttkrp_gpu_taco":
            s["A"] = np.zeros((B.dims[0], R), np.float32)
            s["taco"] = [tt.dense_taco(s["A"]), B.as_taco()] + [tt.dense_taco(f) for f in s["factors"]]
        return s
    H = tt.DeviceCsf(B)
    s["H"] = H
    if kind == "ttv":
        s["c"] = _uniform((B.dims[-1],), gen)
        s["y"] = torch.empty(B.nodes(B.order - 2), device=DEVICE)
    elif kind == "mttkrp":
        s["factors"] = [_uniform((d, R), gen) for d in B.dims[1:]]
        s["A"] = torch.empty((B.dims[0], R), device=DEVICE)
        s["variant"] = tt.VARIANT_DEFAULT if case["variant"] == "default" else tt.VARIANT_AUTO
        H.reserve(R, s["variant"])
    else:
        s["factors"] = [_uniform((d, R), gen) for d in B.dims]
        s["outs"] = [torch.empty((d, R), device=DEVICE) for d in B.dims[1:]]
        for level in range(1, B.order):
            H.reserve_level(level)
    return s


def _als_start(B, R, seed, t):
    rng = np.random.default_rng([seed, t])
    return [rng.normal(size=(d, R)).astype(np.float32) for d in B.dims]


# ---------------------------------------------------------------------------
# one pass
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "mttkrp":
        s["H"].mttkrp([Buffer(f) for f in s["factors"]], Buffer(s["A"]), s["R"], s["variant"])
        return s["A"]
    if kind == "ttv":
        s["H"].ttv(Buffer(s["c"]), Buffer(s["y"]))
        return s["y"]
    if kind == "modes":
        factors = [Buffer(f) for f in s["factors"]]
        for level, out in enumerate(s["outs"], 1):
            s["H"].mttkrp_level(level, factors, Buffer(out), s["R"])
        return s["outs"]
    if kind == "batch":
        s["batch"].launch()
        return s["outs"]
    if kind == "cp_als":
        fits = s["cpd"].iterate(case["sweeps"], use_graphs=True)
        # (factors, the weights of the last mode updated, and the fit, in the
        # precision of the factors it is computed from)
        out = [[s["cpd"].factor(t, m) for m in range(n)] for t, n in enumerate(s["orders"])]
        return {"factors": [[a for a, _ in f] for f in out], "weights": [f[-1][1] for f in out],
                "fits": fits.astype(np.float32)}
    if case["op"] == "ttv":
        return tt.ttv(s["B"], s["c"])
    if case["op"] == "mttkrp":
        return tt.mttkrp(s["B"], s["factors"])
    tt.lib().mttkrp_gpu_taco(*[ctypes.byref(t) for t, _ in s["taco"]])
    return s["A"]


# ---------------------------------------------------------------------------
# what a pass cannot do without
def _nodes(dims, nnz, skew):
    """Node counts per level, root first, as the generator makes them on
    average (uniform coordinates: one nonzero per fibre)."""
    n = [nnz]
    for m in range(len(dims) - 2, 0, -1):
        n.insert(0, max(1, nnz if skew == 0 else n[0] / (LEAF_MEAN if m == len(dims) - 2 else MID_MEAN)))
    return [dims[0]] + n


def _mttkrp_work(dims, nnz, skew, R):
    n = _nodes(dims, nnz, skew)
    b = 4 * (n[0] + 1) + 4 * nnz + sum(4 * c for c in n[1:]) + sum(4 * c for c in n[1:-1])
    b += 4 * R * sum(dims)
    return {"bytes": b, "flops": 2 * R * sum(n[1:])}


def work(case):
    kind = case["kind"]
    if kind in ("batch", "cp_als"):
        rng = np.random.default_rng(7)
        total = {"bytes": 0.0, "flops": 0.0}
        R = case["rank"]
        for t in range(case["tensors"]):
            dims = [math.exp(rng.uniform(math.log(case["dim_lo"]), math.log(case["dim_hi"]))) for _ in range(3 + t % 3)]
            nnz = math.exp(rng.uniform(math.log(case["nnz_lo"]), math.log(case["nnz_hi"])))
            skew = float(rng.uniform(0.8, 1.5))
            for m in range(len(dims)):
                w = _mttkrp_work([dims[m]] + dims[:m] + dims[m + 1:], nnz, skew, R)
                if kind == "cp_als":  # the solve and the Gram of the mode's rows, its read of M and write of A
                    w = {"bytes": w["bytes"] + 4 * R * dims[m], "flops": w["flops"] + 4 * R * R * dims[m]}
                for k in total:
                    total[k] += w[k] * case.get("sweeps", 1)
        return total
    dims, nnz, skew = _dims_of(case), case["nnz"], case["skew"]
    if _is_ttv(case):
        n = _nodes(dims, nnz, skew)
        b = 4 * (n[0] + 1) + sum(8 * c for c in n[1:-2]) + 8 * n[-2] + 8 * nnz + 4 * dims[-1]
        return {"bytes": b, "flops": 2 * nnz}
    w = _mttkrp_work(dims, nnz, skew, case["rank"])
    if kind == "modes":
        return {k: v * (len(dims) - 1) for k, v in w.items()}
    return w


# ---------------------------------------------------------------------------
# 64-bit results
CHUNK = 1 << 22


class _Tree:
    """Device copies of a host CSF's levels: coordinates and, per node, its
    parent."""

    def __init__(self, B):
        self.order, self.dims = B.order, B.dims
        self.crd = [torch.from_numpy(np.array(B.crd[m])).to(DEVICE) for m in range(B.order)]
        self.parent = [None]
        for m in range(1, B.order):
            pos = torch.from_numpy(np.array(B.pos[m])).to(DEVICE).long()
            ids = torch.arange(pos.numel() - 1, device=DEVICE, dtype=torch.int32)
            self.parent.append(torch.repeat_interleave(ids, pos[1:] - pos[:-1]))
        self.vals = torch.from_numpy(np.array(B.vals)).to(DEVICE)

    def below(self, factors, level):
        """Per level-`level` node, the sum over its subtree below it (its own
        factor row not applied): nodes x R; for the leaves, their values."""
        s = self.vals.double()[:, None]
        for m in range(self.order - 1, level, -1):
            n, R = self.crd[m - 1].numel(), factors[m].shape[1]
            up = torch.zeros((n, R), dtype=torch.float64, device=DEVICE)
            for a in range(0, self.crd[m].numel(), CHUNK):
                z = slice(a, a + CHUNK)
                up.index_add_(0, self.parent[m][z], s[z] * factors[m][self.crd[m][z]].double())
            s = up
        return s

    def mttkrp(self, factors, level):
        """MTTKRP of the mode at `level`; factors by level (None at `level`)."""
        R = next(f.shape[1] for f in factors if f is not None)
        below = self.below(factors, level)
        above = torch.ones((self.crd[0].numel(), 1), dtype=torch.float64, device=DEVICE)
        for m in range(level):
            above = above * factors[m][self.crd[m]].double()
            if m + 1 < level:
                above = above[self.parent[m + 1]]
        out = torch.zeros((self.dims[level], R), dtype=torch.float64, device=DEVICE)
        for a in range(0, self.crd[level].numel(), CHUNK):
            z = slice(a, a + CHUNK)
            v = below[z] if level == 0 else below[z] * above[self.parent[level][z]]
            out.index_add_(0, self.crd[level][z], v.expand(-1, R))
        return out


def _als64(B, start, sweeps):
    """CP-ALS in 64 bits: factors normalised by their column 2-norms in the
    first sweep and by max(1, largest magnitude) after it; the fit is
    1 - ||X - model|| / ||X||."""
    tree = _Tree(B)
    A = [torch.from_numpy(f).to(DEVICE).double() for f in start]
    gram = [a.T @ a for a in A]
    norm2 = float(tree.vals.double().square().sum())
    for sweep in range(sweeps):
        for m in range(B.order):
            M = tree.mttkrp([None if k == m else A[k] for k in range(B.order)], m)
            V = torch.ones_like(gram[0])
            for k in range(B.order):
                if k != m:
                    V = V * gram[k]
            a = torch.linalg.solve(V, M.T).T
            lam = a.norm(dim=0) if sweep == 0 else a.abs().amax(dim=0).clamp(min=1.0)
            A[m] = a / lam
            gram[m] = A[m].T @ A[m]
    V = torch.ones_like(gram[0])
    for g in gram:
        V = V * g
    inner = float((M * A[-1] * lam).sum())
    left = max(0.0, norm2 + float(lam @ V @ lam) - 2 * inner)
    return [a.cpu() for a in A], lam.cpu(), 1 - math.sqrt(left / norm2)


def exact(case, seed):
    kind = case["kind"]
    gen = _gen(seed)
    if kind == "batch":
        hosts = _uneven(case, seed)
        factors = [[_uniform((d, case["rank"]), gen) for d in B.dims] for B in hosts]
        out = []
        for B, f in zip(hosts, factors):
            tree = _Tree(B)
            out += [tree.mttkrp([None if k == m else f[k] for k in range(B.order)], m) for m in range(B.order)]
        return out
    if kind == "cp_als":
        hosts = _uneven(case, seed)
        got = [_als64(B, _als_start(B, case["rank"], seed, t), case["sweeps"]) for t, B in enumerate(hosts)]
        return {"factors": [g[0] for g in got], "weights": [g[1] for g in got],
                "fits": torch.tensor([g[2] for g in got], dtype=torch.float64)}
    B = _ttv_tensor(case, seed) if _is_ttv(case) else _tensor(_dims_of(case), case["nnz"], case["skew"], seed)
    tree = _Tree(B)
    if _is_ttv(case):
        c = _uniform((B.dims[-1],), gen)
        return tree.below([None] * (B.order - 1) + [c[:, None]], B.order - 2)[:, 0]
    if kind == "modes":
        f = [_uniform((d, case["rank"]), gen) for d in B.dims]
        return [tree.mttkrp([None if k == m else f[k] for k in range(B.order)], m) for m in range(1, B.order)]
    f = [_uniform((d, case["rank"]), gen) for d in B.dims[1:]]
    return tree.mttkrp([None] + f, 0)
