"""The measured work of this library: what a program that uses it has it do.

Every case names a ``kind`` (one of the public calls) and its sizes:

* ``search``    exhaustive kNN on vectors resident in HBM: ``yk_norms`` and
  ``yk_knn_f32`` (the FP32 form), or with ``kp`` > 0 the precision form
  (``yk_to_bf16`` and ``yk_knn_bf16`` keeping kp candidates per query).  The
  queries of a call are new, so their norms and BF16 copies are part of the
  pass; the base's are too with ``rebuild`` (a base searched once), else
  they are kept beside the base (a base served for long).
* ``knn``       the same through ``yael_amd.knn`` on host arrays.
* ``kmeans``    ``yael_kmeans_device`` on points resident in HBM, or with
  ``host`` ``yael_amd.kmeans`` on a host array.
* ``batched``   ``yael_kmeans_batched_device``: the nodes of one level of a
  hierarchical k-means, sizes after a Zipf law.
* ``subspaces`` ``yael_kmeans_subspaces_device``: a product quantiser's
  training, one k-means per block of columns.
* ``descent``   ``yk_hkm_quantize``: points to the leaves of a learned tree.

``data``: "sift" -- a Gaussian mixture (centres uniform in [0, 255]^d, sigma
20) clipped to [0, 255] and rounded, as byte descriptors are; "float" -- the
same without the rounding; "unit" -- rows of |N(0, 1)| scaled to unit length.
"""
import ctypes
import math

import numpy as np
import torch

import yael_amd
from yael_amd import hkm
from yael_amd.workloads import zipf_sizes

QUIET, INIT_RANDOM = 0x10000, 0x80000  # kmeans() flags
KMEANS_SEED = 7


def listed():
    return [
        # one query against a served base: the latency of a search request
        dict(name="one_query", kind="search", nq=1, nb=1_000_000, d=128, k=10, kp=0, type=2,
             weighted=False, rebuild=False, data="sift"),
        # a small search from a host program: the cost of a call
        dict(name="small_knn_host", kind="knn", nq=200, nb=3000, d=128, k=10, type=2,
             weighted=False, data="sift"),
        # an ordinary batch of odd sizes, a short list per query
        dict(name="ragged_knn_k10", kind="search", nq=1003, nb=100_003, d=100, k=10, kp=0, type=2,
             weighted=False, rebuild=True, data="float"),
        # base weights, which only the FP32 form takes, a long list per query
        dict(name="weighted_knn_k100", kind="search", nq=2000, nb=200_000, d=128, k=100, kp=0,
             type=2, weighted=True, rebuild=True, data="sift"),
        # the large exact search, every derived array made by the call
        dict(name="large_knn_k100", kind="search", nq=10_000, nb=1_000_000, d=128, k=100, kp=200,
             type=2, weighted=False, rebuild=True, data="sift"),
        # long vectors against a served base
        dict(name="long_vectors_k10", kind="search", nq=10_000, nb=1_000_000, d=960, k=10, kp=64,
             type=2, weighted=False, rebuild=False, data="unit"),
        # a small clustering from a host program
        dict(name="small_kmeans_host", kind="kmeans", n=20_000, d=32, k=50, niter=20, host=True,
             data="float"),
        # a codebook of ordinary size
        dict(name="kmeans_k1024", kind="kmeans", n=100_000, d=128, k=1024, niter=10, host=False,
             data="sift"),
        # a large codebook
        dict(name="kmeans_k65536", kind="kmeans", n=1_000_000, d=128, k=65_536, niter=2,
             host=False, data="sift"),
        # one level of a hierarchical k-means
        dict(name="batched_256", kind="batched", ninst=256, total=2_000_000, d=128, k=64,
             niter=15, data="sift"),
        # a product quantiser
        dict(name="subspaces_8", kind="subspaces", n=1_000_000, d=128, nsub=8, k=256, niter=10,
             data="sift"),
        # encoding with a learned tree
        dict(name="tree_descent", kind="descent", n=1_000_000, d=128, nlevel=2, bf=32,
             data="sift"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed kinds: sizes spread over the logarithm of
    their ranges, the last one held to what the listed cases cost."""
    kind = rng.choice(["fp32", "fp32", "bf16", "bf16", "knn", "kmeans", "kmeans", "batched",
                       "subspaces", "descent"])
    if kind == "fp32":
        d, nq = _log(rng, 16, 256), _log(rng, 1, 4000)
        nb = min(_log(rng, 5000, 1_000_000), max(5000, int(2e11 / (nq * d))))
        typ = rng.choice([2, 2, 16])
        return dict(kind="search", nq=nq, nb=nb, d=d, k=rng.choice([1, _log(rng, 2, 16),
                                                                    _log(rng, 17, 200)]),
                    kp=0, type=typ, weighted=rng.random() < 0.2, rebuild=rng.random() < 0.5,
                    data="unit" if typ == 16 else rng.choice(["sift", "float"]))
    if kind == "bf16":
        d, nq = _log(rng, 32, 960), _log(rng, 256, 10_000)
        nb = min(_log(rng, 100_000, 1_000_000), max(100_000, int(4e12 / (nq * d))))
        k = rng.choice([1, _log(rng, 2, 30), _log(rng, 31, 200)])
        return dict(kind="search", nq=nq, nb=nb, d=d, k=k, kp=max(32, 2 * k), type=2,
                    weighted=False, rebuild=rng.random() < 0.5,
                    data=rng.choice(["sift", "float", "unit"]))
    if kind == "knn":
        return dict(kind="knn", nq=_log(rng, 1, 1000), nb=_log(rng, 1000, 20_000),
                    d=_log(rng, 16, 256), k=rng.choice([1, _log(rng, 2, 100)]),
                    type=rng.choice([2, 2, 16]), weighted=rng.random() < 0.2, data="float")
    if kind == "kmeans":
        host = rng.random() < 0.3
        n, d = _log(rng, 2000, 50_000 if host else 1_000_000), _log(rng, 16, 128)
        k = _log(rng, 8, 256 if host else max(64, min(65_536, n // 20)))
        k = min(k, n // 20)
        niter = max(1, min(20, int(4e12 / (float(n) * k * d))))
        return dict(kind="kmeans", n=n, d=d, k=k, niter=niter, host=host,
                    data=rng.choice(["sift", "float"]))
    if kind == "batched":
        ninst, k = _log(rng, 8, 256), _log(rng, 8, 128)
        lo = ninst * max(256, 8 * k)
        return dict(kind="batched", ninst=ninst, total=_log(rng, lo, max(lo + 1, 2_000_000)),
                    d=_log(rng, 16, 128), k=k, niter=rng.randint(5, 15),
                    data=rng.choice(["sift", "float"]))
    if kind == "subspaces":
        nsub = rng.choice([4, 8, 16])
        return dict(kind="subspaces", n=_log(rng, 10_000, 1_000_000),
                    d=nsub * rng.randint(4, 128 // nsub), nsub=nsub, k=_log(rng, 16, 256),
                    niter=rng.randint(3, 10), data=rng.choice(["sift", "float"]))
    levels = rng.choice([2, 2, 3])
    return dict(kind="descent", n=_log(rng, 10_000, 1_000_000), d=_log(rng, 16, 128),
                nlevel=levels, bf=rng.randint(4, 32 if levels == 2 else 10),
                data=rng.choice(["sift", "float"]))


# ---------------------------------------------------------------------------
# inputs


def _rng(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000 + salt)
    return g


def _rows(seed, salt, n, d, data, ncomp=1024):
    """n x d float32 rows on the GPU.  The mixture's centres depend on the
    seed alone, so base, queries and points come from the same mixture."""
    g = _rng(seed, salt)
    if data == "unit":
        x = torch.randn((n, d), generator=g, device="cuda").abs_()
        return x.div_(x.norm(dim=1, keepdim=True))
    cen = torch.rand((ncomp, d), generator=_rng(seed, 0), device="cuda") * 255
    x = cen[torch.randint(0, ncomp, (n,), generator=g, device="cuda")]
    x += 20 * torch.randn((n, d), generator=g, device="cuda")
    x.clamp_(0, 255)
    return x.round_() if data == "sift" else x


def _components(case):
    """Mixture components of a case: 1,024, and as many as centroids where a
    clustering asks for more."""
    return max(1024, case["k"]) if case["kind"] == "kmeans" else 1024


def _padded(x):
    """The library's device layout: rows of yk_ld(d) floats, zero padded."""
    n, d = x.shape
    ld = yael_amd.lib().yk_ld(d)
    if ld == d:
        return x.contiguous()
    p = torch.zeros((n, ld), device="cuda")
    p[:, :d] = x
    return p


def _inputs(case, seed):
    """The case's vectors (unpadded, on the GPU), from the seed alone."""
    d, data = case["d"], case["data"]
    if case["kind"] in ("search", "knn"):
        v = {"b": _rows(seed, 1, case["nb"], d, data), "q": _rows(seed, 2, case["nq"], d, data)}
        if case["weighted"]:
            v["w"] = torch.rand(case["nb"], generator=_rng(seed, 3), device="cuda") * 1.5 + 0.5
        return v
    n = case["total"] if case["kind"] == "batched" else case["n"]
    return {"v": _rows(seed, 1, n, d, data, _components(case))}


def _instances(case):
    """Rows and seeds of a batched call's instances."""
    lo = max(256, 4 * case["k"])
    sizes = zipf_sizes(case["ninst"], case["total"], lo, max(case["total"] // 16, 2 * lo,
                                                             2 * case["total"] // case["ninst"]))
    return sizes, np.arange(1, case["ninst"] + 1, dtype=np.int64)


def _ptr(a):
    if a is None:
        return None
    return ctypes.c_void_p(a.data_ptr() if isinstance(a, torch.Tensor) else a.ctypes.data)


def _dev(n, dtype):
    return torch.zeros(n, dtype=dtype, device="cuda")


def _pad32(n):
    return (n + 31) // 32 * 32


# ---------------------------------------------------------------------------
# what a program holds before the call


def prepare(case, seed):
    L = yael_amd.lib()
    yael_amd.init()
    s = dict(case)
    x = _inputs(case, seed)
    kind, d = case["kind"], case["d"]
    if kind == "search":
        nq, nb, k, typ = case["nq"], case["nb"], case["k"], case["type"]
        s.update(b=_padded(x["b"]), q=_padded(x["q"]), bn=_dev(_pad32(nb), torch.float32),
                 qn=_dev(nq, torch.float64), w=None, idx=_dev((nq, k), torch.int32),
                 dis=_dev((nq, k), torch.float32))
        if case["weighted"]:
            s["w"] = _dev(_pad32(nb), torch.float32)
            s["w"][:nb] = x["w"]
        if case["kp"]:
            s.update(bh=_dev(L.yk_bf16_bytes(nb, d, typ, 0) // 2, torch.int16),
                     qh=_dev(L.yk_bf16_bytes(nq, d, typ, 1) // 2, torch.int16),
                     bst=_dev(4 * nb, torch.float32), qst=_dev(4 * nq, torch.float32),
                     mx=_dev(4, torch.float32), fallback=ctypes.c_int(0))
        torch.cuda.synchronize()
        if not case["rebuild"]:
            _base_arrays(L, s)
            yael_amd.check(L.yk_sync(), "sync")
    elif kind == "knn":
        s.update({n: a.cpu().numpy() for n, a in x.items()})
    elif kind == "kmeans" and case["host"]:
        s["v"] = x["v"].cpu().numpy()
    elif kind == "descent":
        _descent_state(L, s, x["v"])
    else:
        n, k = len(x["v"]), case["k"]
        s["v"] = _padded(x["v"])
        rows = 1
        if kind == "batched":
            s["sizes"], s["seeds"] = _instances(case)
            rows = case["ninst"]
        elif kind == "subspaces":
            s["seeds"] = np.arange(1, case["nsub"] + 1, dtype=np.int64)
            rows = case["nsub"]
        dsub = d // rows if kind == "subspaces" else d
        pts = n * rows if kind == "subspaces" else n
        s.update(cent=np.empty((rows, k, dsub), np.float32), dis=np.empty(pts, np.float32),
                 assign=np.empty(pts, np.int32), nassign=np.empty((rows, k), np.int32),
                 qerr=np.empty(rows, np.float32))
        torch.cuda.synchronize()
    return s


def _base_arrays(L, s):
    """A base's derived arrays: its float norms, in the precision form
    written by the conversion to BF16."""
    l2 = s["type"] == 2
    if s["kp"]:
        yael_amd.check(L.yk_to_bf16(_ptr(s["b"]), s["nb"], s["d"], s["type"], 0, _ptr(s["bh"]),
                                    _ptr(s["bst"]), _ptr(s["mx"]),
                                    _ptr(s["bn"]) if l2 else None), "to_bf16")
    elif l2:
        yael_amd.check(L.yk_norms(_ptr(s["b"]), s["nb"], s["d"], _ptr(s["bn"]), None), "norms")


def _descent_state(L, s, v):
    """A tree learned on the first points, its levels stacked on the GPU, and
    the points with their norms."""
    leaves = s["bf"] ** s["nlevel"]
    ctypes.CDLL(None).srand48(ctypes.c_long(1))
    learn = v[:min(len(v), max(10_000, 16 * leaves))].cpu().numpy()
    # a node left with fewer points than children ends the learning: a
    # smaller tree is tried, as its user would
    while True:
        try:
            tree, _ = hkm.hkm_learn(learn, s["nlevel"], s["bf"], niter=4)
            break
        except yael_amd.YaelGPUError:
            if s["bf"] <= 4:
                raise
            s["bf"] = s["bf"] * 3 // 4
    cent = np.concatenate([tree.centroids(level) for level in range(s["nlevel"])])
    s.update(v=_padded(v), vn=_dev(len(v), torch.float64),
             cent=_padded(torch.from_numpy(cent).cuda()),
             cn=_dev(_pad32(len(cent)), torch.float32), idx=_dev(len(v), torch.int32))
    torch.cuda.synchronize()
    yael_amd.check(L.yk_norms(_ptr(s["cent"]), len(cent), s["d"], _ptr(s["cn"]), None), "norms")
    yael_amd.check(L.yk_sync(), "sync")


# ---------------------------------------------------------------------------
# one pass


def run(s):
    L = yael_amd.lib()
    kind = s["kind"]
    if kind == "search":
        return _search(L, s)
    if kind == "knn":
        idx, dis = yael_amd.knn(s["q"], s["b"], s["k"], distance_type=s["type"],
                                weights=s.get("w"))
        return {"idx": idx, "dis": dis}
    if kind == "descent":
        yael_amd.check(L.yk_norms(_ptr(s["v"]), s["n"], s["d"], None, _ptr(s["vn"])), "norms")
        yael_amd.check(L.yk_hkm_quantize(_ptr(s["v"]), _ptr(s["vn"]), s["n"], s["d"], s["nlevel"],
                                         s["bf"], _ptr(s["cent"]), _ptr(s["cn"]),
                                         _ptr(s["idx"])), "hkm_quantize")
        return {"idx": s["idx"]}
    if kind == "kmeans" and s["host"]:
        cent, qerr, dis, assign, nassign = yael_amd.kmeans(
            s["v"], s["k"], niter=s["niter"], seed=KMEANS_SEED, verbose=False, output="all")
        return {"cent": cent, "qerr": float(qerr), "dis": dis, "assign": assign,
                "nassign": nassign}
    flags = QUIET | INIT_RANDOM
    out = [_ptr(s[n]) for n in ("cent", "dis", "assign", "nassign")]
    if kind == "kmeans":
        err = ctypes.c_float(0)
        yael_amd.check(L.yael_kmeans_device(s["d"], s["n"], s["k"], s["niter"], _ptr(s["v"]),
                                            flags, KMEANS_SEED, 1, *out, ctypes.byref(err)),
                       "kmeans")
        s["qerr"][0] = err.value
    elif kind == "batched":
        yael_amd.check(L.yael_kmeans_batched_device(
            s["d"], s["ninst"], _ptr(s["sizes"]), s["k"], s["niter"], _ptr(s["v"]), flags,
            _ptr(s["seeds"]), *out, _ptr(s["qerr"]), None, 1, None), "batched")
    else:
        yael_amd.check(L.yael_kmeans_subspaces_device(
            s["d"], s["n"], s["nsub"], s["k"], s["niter"], _ptr(s["v"]), flags, _ptr(s["seeds"]),
            *out, _ptr(s["qerr"]), None, None), "subspaces")
    return {n: s[n] for n in ("cent", "dis", "assign", "nassign", "qerr")}


def _search(L, s):
    l2, qn, bn = s["type"] == 2, _ptr(s["qn"]), _ptr(s["bn"])
    if s["rebuild"]:
        _base_arrays(L, s)
    if l2:
        yael_amd.check(L.yk_norms(_ptr(s["q"]), s["nq"], s["d"], None, qn), "norms")
    if not s["kp"]:
        yael_amd.check(L.yk_knn_f32(s["type"], s["nq"], s["nb"], s["d"], s["k"], _ptr(s["q"]),
                                    qn, _ptr(s["b"]), bn, _ptr(s["w"]), _ptr(s["idx"]),
                                    _ptr(s["dis"])), "knn_f32")
        return {"idx": s["idx"], "dis": s["dis"]}
    yael_amd.check(L.yk_to_bf16(_ptr(s["q"]), s["nq"], s["d"], s["type"], 1, _ptr(s["qh"]),
                                _ptr(s["qst"]), None, None), "to_bf16")
    yael_amd.check(L.yk_knn_bf16(s["type"], s["nq"], s["nb"], s["d"], s["k"], s["kp"],
                                 _ptr(s["q"]), qn, _ptr(s["qh"]), _ptr(s["qst"]), _ptr(s["b"]),
                                 bn, _ptr(s["bh"]), _ptr(s["mx"]), _ptr(s["idx"]),
                                 _ptr(s["dis"]), ctypes.byref(s["fallback"])), "knn_bf16")
    return {"idx": s["idx"], "dis": s["dis"]}


# ---------------------------------------------------------------------------
# what a pass cannot do without


def work(case):
    """Inputs read once and outputs written once; 2 d operations per
    (query, base vector) or (point, centroid) pair.  A clustering reads its
    points once per iteration."""
    kind, d = case["kind"], case["d"]
    if kind in ("search", "knn"):
        nq, nb, k = case["nq"], case["nb"], case["k"]
        return {"bytes": 4.0 * d * (nq + nb) + 8.0 * nq * k + (4.0 * nb if case["weighted"] else 0),
                "flops": 2.0 * d * nq * nb}
    if kind == "descent":
        n, bf, levels = case["n"], case["bf"], case["nlevel"]
        rows = sum(bf ** (level + 1) for level in range(levels))
        return {"bytes": 4.0 * d * (n + rows) + 4.0 * n, "flops": 2.0 * d * n * bf * levels}
    k, it = case["k"], case["niter"]
    n = case["total"] if kind == "batched" else case["n"]
    sets = {"kmeans": 1, "batched": case.get("ninst"), "subspaces": 1}[kind]
    pts = n * case["nsub"] if kind == "subspaces" else n
    return {"bytes": 4.0 * d * n * it + 8.0 * pts + 4.0 * sets * k * (d + 1),
            "flops": 2.0 * d * n * k * it}


# ---------------------------------------------------------------------------
# the values in 64 bits


def exact(case, seed):
    kind = case["kind"]
    x = _inputs(case, seed)
    if kind in ("search", "knn"):
        return {"idx": None, "dis": _exact_search(case, x)}
    if kind == "descent":
        return None  # leaf numbers only
    v = x["v"]
    if kind == "kmeans":
        runs = [(v, KMEANS_SEED)]
    elif kind == "batched":
        sizes, seeds = _instances(case)
        at = np.concatenate([[0], np.cumsum(sizes)])
        runs = [(v[at[i]:at[i + 1]], int(seeds[i])) for i in range(len(sizes))]
    else:
        w = case["d"] // case["nsub"]
        runs = [(v[:, i * w:(i + 1) * w], i + 1) for i in range(case["nsub"])]
    got = [_exact_kmeans(p, case["k"], case["niter"], seed) for p, seed in runs]
    if any(g is None for g in got):
        return None
    out = {"dis": torch.cat([g[1] for g in got]), "assign": None, "nassign": None}
    if case.get("host"):
        out.update(cent=got[0][0], qerr=float(got[0][2]))
    else:
        out.update(cent=torch.stack([g[0] for g in got]), qerr=torch.stack([g[2] for g in got]))
    return out


def _exact_search(case, x):
    b, k = x["b"].double(), case["k"]
    bn = (b * b).sum(1)
    out = []
    step = max(1, min(256, int(3e8 // case["nb"])))
    for i in range(0, case["nq"], step):
        q = x["q"][i:i + step].double()
        dis = q @ b.T
        if case["type"] == 2:
            dis = dis.mul_(-2).add_(bn).add_((q * q).sum(1, keepdim=True))
        if case["weighted"]:
            dis *= x["w"].double()
        out.append(dis.topk(k, dim=1, largest=False, sorted=True).values)
    return torch.cat(out)


def _exact_kmeans(v, k, niter, seed):
    """(centroids, distances, objective / n) of the library's own run --
    random initialisation from its seed, Lloyd steps -- in 64 bits; None
    when a cluster becomes empty (its split depends on the rounding)."""
    n = len(v)
    libc = ctypes.CDLL(None)
    outer = ctypes.c_uint(seed)
    inner = ctypes.c_uint(libc.rand_r(ctypes.byref(outer)))
    moved, sel = {}, []
    for i in range(k):  # the first k places of a shuffle
        j = i + (libc.rand_r(ctypes.byref(inner)) % (n - i) if i < n - 1 else 0)
        sel.append(moved.get(j, j))
        moved[j] = moved.get(i, i)
    v = v.double()
    vn = (v * v).sum(1, keepdim=True)
    cent = v[torch.tensor(sel, device=v.device)]
    step = max(1, int(2e8 // k))
    last = None
    for _ in range(niter):
        cn = (cent * cent).sum(1)
        best = [torch.min((v[i:i + step] @ cent.T).mul_(-2).add_(cn).add_(vn[i:i + step]), dim=1)
                for i in range(0, n, step)]
        dis, assign = (torch.cat([b[j] for b in best]) for j in (0, 1))
        if last is not None and torch.equal(assign, last):
            break
        last = assign
        count = torch.bincount(assign, minlength=k)
        if int(count.min()) == 0:
            return None
        cent = torch.zeros_like(cent).index_add_(0, assign, v) / count[:, None]
    return cent, dis, dis.sum() / n
