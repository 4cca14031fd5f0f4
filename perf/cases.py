"""The work this framework is measured on: cases over its public entry points.

Four kinds of work, as a program that clusters or quantises vectors does them:

* "lloyd": one `batch_kmeans_Euclid` call, the trainer;
* "assign": one `euclid_assign` call, encoding points with a finished codebook;
* "step": one iteration by the separate operations (assign, update, finalize),
  as a program that owns its loop runs it;
* "evaluate": one `quality.evaluate` call, judging finished centroids.

Points are Gaussian mixtures (blob centres N(0, 4 I), noise 0.5, as many
blobs as clusters, uniform or Zipf(1.1) blob sizes) or plain N(0, I) noise;
initial centroids are distinct random points, finished centroids are the blob
centres a little off.
"""

from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "flash-kmeans-cuda_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import flash_kmeans_cuda as fk  # noqa: E402
from flash_kmeans_cuda import ops, quality  # noqa: E402

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}

SAMPLE_POINTS = 4096  # quality.evaluate's defaults
SAMPLE_SEED = 1000


def _case(name, op, dtype, B, N, K, D, iters=1, tol=0.0, data="mixture"):
    c = {"op": op, "dtype": dtype, "B": B, "N": N, "K": K, "D": D, "iters": iters,
         "tol": tol, "data": data}
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # The smallest training call of the benchmark: a few thousand fp32
        # points, where launches and latency are all there is.
        _case("lloyd_f32_4k", "lloyd", "f32", 1, 4096, 64, 128, 10, data="normal"),
        # The reference's smallest published shape: one codebook of 256.
        _case("lloyd_f16_32k", "lloyd", "f16", 1, 32768, 256, 128, 10),
        # The middle published shape: an inverted-file index of 2048 lists.
        _case("lloyd_f16_131k", "lloyd", "f16", 1, 131072, 2048, 128, 10),
        # Batched heads in bf16, stopped by the convergence test.
        _case("lloyd_bf16_batch8", "lloyd", "bf16", 8, 65536, 1024, 64, 15, tol=1e-4),
        # The largest published shape, clusters of very unequal size.  (Three
        # iterations: many centroids start in one large blob here, and what
        # one near-tie label moves grows from iteration to iteration.)
        _case("lloyd_f16_524k", "lloyd", "f16", 1, 524288, 8192, 128, 3, data="zipf"),
        # Full-precision training at an ordinary size.
        _case("lloyd_f32_131k", "lloyd", "f32", 1, 131072, 1024, 128, 10),
        # A feature width that no tile divides.
        _case("lloyd_f16_odd", "lloyd", "f16", 1, 100000, 300, 37, 10),
        # Wide rows, as embedding vectors have.
        _case("lloyd_bf16_wide", "lloyd", "bf16", 1, 262144, 2048, 256, 5),
        # The smallest encode call: a request's worth of points.
        _case("assign_f16_small", "assign", "f16", 1, 1000, 64, 64),
        # Few points against a very large codebook.
        _case("assign_f16_65k_codes", "assign", "f16", 1, 16384, 65536, 128),
        # One iteration of a caller-owned loop over four batch rows.
        _case("step_bf16_batch4", "step", "bf16", 4, 131072, 512, 128),
        # Judging the centroids of a larger fp16 run.
        _case("evaluate_f16_262k", "evaluate", "f16", 1, 262144, 4096, 128),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """The listed cases' ranges: 1e3 to 5e5 points, 16 to 8192 clusters (up to
    65536 to encode with), widths 8 to 512, every type.  16-bit widths that
    the matrix units take whole cost at most the largest 16-bit listed call,
    the others at most the largest fp32 one."""
    while True:
        op = rng.choice(["lloyd"] * 5 + ["assign"] * 3 + ["step"] * 2 + ["evaluate"])
        dtype = rng.choice(["f16", "f16", "bf16", "bf16", "f32"])
        B = rng.choice([1, 1, 1, 2, 3, 4, 8])
        N = _log_int(rng, 1000, 524288) // B
        K = _log_int(rng, 16, 65536 if op == "assign" else 8192)
        D = (rng.choice([16, 32, 64, 64, 96, 128, 128, 128, 256, 512])
             if rng.random() < 0.6 else _log_int(rng, 8, 512))
        data = rng.choice(["mixture", "mixture", "zipf", "normal"])
        iters = rng.choice([1, 2] if data == "zipf" else [1, 2, 5, 10]) if op == "lloyd" else 1
        tol = 1e-4 if op == "lloyd" and rng.random() < 0.2 else 0.0
        if op != "assign" and K * 4 > N or N < 200:
            continue
        matrix_units = dtype != "f32" and D % 8 == 0
        if 2.0 * B * N * K * D * iters > (3.2e12 if matrix_units else 3.3e11):
            continue
        if 4.0 * B * N * D > 5.4e8:
            continue
        return _case(None, op, dtype, B, N, K, D, iters, tol, data)


def _points(case, seed):
    """(x, blob centres), x (B, N, D) in the case's type, centres fp32."""
    B, N, K, D = case["B"], case["N"], case["K"], case["D"]
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    centres = 2.0 * torch.randn(B, K, D, device="cuda", generator=g)
    noise = torch.randn(B, N, D, device="cuda", generator=g)
    if case["data"] == "normal":
        return noise.to(DTYPES[case["dtype"]]), centres, g
    if case["data"] == "zipf":
        w = torch.arange(1, K + 1, device="cuda", dtype=torch.float64).pow(-1.1)
        cdf = (w / w.sum()).cumsum(0)
        u = torch.rand(B, N, device="cuda", generator=g, dtype=torch.float64)
        blob = torch.searchsorted(cdf, u).clamp_(max=K - 1)
    else:
        blob = torch.randint(0, K, (B, N), device="cuda", generator=g)
    x = noise.mul_(0.5)
    for b in range(B):
        x[b] += centres[b, blob[b]]
    return x.to(DTYPES[case["dtype"]]), centres, g


def prepare(case, seed):
    x, centres, g = _points(case, seed)
    B, N, K = case["B"], case["N"], case["K"]
    s = {"case": case, "x": x}
    if case["op"] == "lloyd":
        pick = torch.stack([torch.randperm(N, device="cuda", generator=g)[:K] for _ in range(B)])
        s["init"] = torch.gather(x, 1, pick.unsqueeze(-1).expand(-1, -1, x.shape[2])).contiguous()
        return s
    if case["data"] == "normal":
        centres *= 0.5
    else:
        centres += 0.05 * torch.randn(centres.shape, device="cuda", generator=g)
    s["centroids"] = centres.to(x.dtype)
    if case["op"] in ("assign", "step"):
        # A program that assigns the same points again keeps their norms.
        s["x_sq"] = ops.row_sqnorm(x)
    return s


def run(s):
    case, x = s["case"], s["x"]
    K = case["K"]
    if case["op"] == "lloyd":
        ids, centroids, n = fk.batch_kmeans_Euclid(
            x, K, max_iters=case["iters"], tol=case["tol"], init_centroids=s["init"])
        return {"ids": ids, "centroids": centroids, "n_iters": n}
    if case["op"] == "assign":
        return {"ids": fk.euclid_assign(x, s["centroids"], s["x_sq"])}
    if case["op"] == "step":
        ids = fk.euclid_assign(x, s["centroids"], s["x_sq"])
        sums, counts = fk.centroid_update_sorted(x, ids, K)
        new = fk.centroid_finalize(sums, counts, s["centroids"])
        return {"ids": ids, "sums": sums, "counts": counts, "centroids": new}
    return quality.evaluate(x, s["centroids"])


def _esize(case):
    return 4 if case["dtype"] == "f32" else 2


def work(case):
    """Each pass over the points scores all B N K pairs over D features and
    has to read x once (the centroids of the pass before decide the labels of
    this one); the update adds every row once.  A call that its tolerance may
    stop early is counted with the iterations it is allowed."""
    B, N, K, D, it = case["B"], case["N"], case["K"], case["D"], case["iters"]
    e = _esize(case)
    x, cent, ids = B * N * D * e, B * K * D * e, B * N * 4
    score, add = 2.0 * B * N * K * D, 1.0 * B * N * D
    if case["op"] == "lloyd":
        return {"bytes": it * (x + 2 * cent) + ids, "flops": it * (score + add)}
    if case["op"] == "assign":
        return {"bytes": x + cent + B * N * 4 + ids, "flops": score}
    if case["op"] == "step":
        return {"bytes": x + 2 * cent + B * N * 4 + ids + B * K * (4 * D + 4),
                "flops": score + add}
    sample = 2.0 * B * min(SAMPLE_POINTS, N) * K * D
    return {"bytes": x + cent + ids, "flops": score + sample + 3 * add}


def tolerance(case):
    """Four times the largest difference from `exact` seen over the listed and
    about a hundred drawn cases.  What differs are labels of points at nearly
    equal distance from two centroids (fp32 distances are rounded at the size
    of the squared norms), at most 2.5e-5 of the points in one pass, and what
    such a point moves: one centroid by up to 0.09 of the values' size where
    the cluster is small.  Over several iterations both spread to the labels
    that depend on the moved centroids (1.4e-3 of them, centroids 5e-3 as a
    whole).  Without such a point, sums in fp32 are within 1e-7 of theirs and
    16-bit centroids within the type's rounding (f16 2.1e-4, bf16 1.7e-3)."""
    ties = max(1e-4, 2.0 / (case["B"] * case["N"]))
    if case["op"] == "evaluate":
        return {"rel": 1e-5, "differ": min(0.01, ties)}
    if case["op"] == "assign":
        return {"differ": min(0.01, ties)}
    if case["op"] == "step" or case["iters"] == 1:
        return {"rel": 0.007 if case["dtype"] == "bf16" else 0.002, "max": 0.35,
                "differ": min(0.01, ties)}
    return {"rel": 0.01, "max": 0.35, "differ": max(0.005, ties)}


def _nearest64(x, c):
    """Labels and squared distances of x (N, D) to c (K, D), both float64."""
    ids = torch.empty(x.shape[0], dtype=torch.int64, device=x.device)
    best = torch.empty(x.shape[0], dtype=torch.float64, device=x.device)
    c_sq = (c * c).sum(1)
    step = max(1, (1 << 28) // c.shape[0])
    for i in range(0, x.shape[0], step):
        xs = x[i:i + step]
        d = torch.addmm(c_sq, xs, c.t(), alpha=-2.0)
        ids[i:i + step] = d.argmin(1)
        best[i:i + step] = ((xs - c[ids[i:i + step]]) ** 2).sum(1)
    return ids, best


def _sums64(x, ids, K):
    sums = torch.zeros(K, x.shape[1], dtype=torch.float64, device=x.device)
    sums.index_add_(0, ids, x)
    return sums, torch.bincount(ids, minlength=K)


def _means64(sums, counts, old):
    return torch.where((counts > 0).unsqueeze(1), sums / counts.clamp(min=1).unsqueeze(1), old)


def exact(case, seed):
    """The same work in float64.  Centroids pass from one iteration to the
    next in the case's type, as the path defines; the last ones are returned
    unrounded."""
    s = prepare(case, seed)
    x, B, K = s["x"], case["B"], case["K"]
    if case["op"] == "lloyd":
        cur = s["init"]
        n = 0
        for _ in range(case["iters"]):
            n += 1
            ids, new = [], []
            for b in range(B):
                xb = x[b].double()
                ib, _ = _nearest64(xb, cur[b].double())
                sb, nb = _sums64(xb, ib, K)
                ids.append(ib)
                new.append(_means64(sb, nb, cur[b].double()))
            new = torch.stack(new)
            stored = new.to(x.dtype)
            shift = (stored.double() - cur.double()).norm(dim=-1).max().item()
            cur = stored
            if case["tol"] > 0 and shift < case["tol"]:
                break
        return {"ids": torch.stack(ids).to(torch.int32), "centroids": new, "n_iters": n}
    cent = s["centroids"].double()
    out = [_nearest64(x[b].double(), cent[b]) for b in range(B)]
    ids = torch.stack([o[0] for o in out])
    if case["op"] == "assign":
        return {"ids": ids.to(torch.int32)}
    if case["op"] == "step":
        sums, counts = zip(*[_sums64(x[b].double(), ids[b], K) for b in range(B)])
        new = torch.stack([_means64(sums[b], counts[b], cent[b]) for b in range(B)])
        return {"ids": ids.to(torch.int32), "sums": torch.stack(sums),
                "counts": torch.stack(counts).to(torch.int32), "centroids": new}
    per_row = [float(o[1].sum()) for o in out]
    g = torch.Generator(device="cuda").manual_seed(SAMPLE_SEED)
    idx = torch.randperm(case["N"], generator=g, device="cuda")[:min(SAMPLE_POINTS, case["N"])]
    return {"ids": ids.to(torch.int32), "inertia": sum(per_row), "inertia_per_batch": per_row,
            "empty_clusters": int((torch.bincount(ids.flatten(), minlength=K) == 0).sum()),
            "sample_exact_inertia": sum(float(o[1][idx].sum()) for o in out)}
