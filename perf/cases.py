"""Performance cases of the PQ search framework: what a user's program has it do, through its public entry points.

Four kinds of work, on synthetic data of the shape the benchmark and the tests use (a 1000-component Gaussian mixture
with sigma 0.3, k-means codebooks, nearest-centroid codes):

  search   PQSearcher: exhaustive ADC search, fp32 tables (v8) or fp16 tables (v9), from device or host buffers
  ivf      IVFIndex: inverted-file search over the nprobe nearest lists
  rerank   Reranker: exact distances of each query's candidates, then the k best
  encode   vk_pq_encode_device: PQ codes of vectors that are in HBM

Every result is bit-identical to the CPU's by contract (ids, distance bits and codes), so the tolerance is "exact".
"""
import ctypes
import math

import numpy as np
import torch

import veckern_amd as vk

KSUB = 256
MIXTURE, SIGMA = 1000, 0.3
TRAIN_ROWS, TRAIN_ROUNDS = 16384, 4

# The most work of a drawn search, in table lookups (queries x vectors x sub-spaces), and its most code bytes.
MOST_LOOKUPS, MOST_CODE_BYTES = 16_000_000_000, 160_000_000


def listed():
    return [
        # One interactive query against a 10M-vector database: latency, one launch, codes read once.
        {"name": "one_query_10m", "kind": "search", "n": 10_000_000, "d": 128, "m": 16, "nq": 1, "k": 10, "q": 4,
         "f16": False, "host": False},
        # A small database answering a small batch from host memory, default tuning: the smallest ordinary call.
        {"name": "batch100_100k_host", "kind": "search", "n": 100_000, "d": 128, "m": 16, "nq": 100, "k": 10, "q": 2,
         "f16": False, "host": True},
        # A serving batch of odd size over an odd number of vectors: between the latency and the throughput ends.
        {"name": "batch37_1m_ragged", "kind": "search", "n": 1_000_003, "d": 128, "m": 16, "nq": 37, "k": 20, "q": 4,
         "f16": False, "host": False},
        # The headline benchmark: a throughput batch over 1M vectors.
        {"name": "batch1000_1m", "kind": "search", "n": 1_000_000, "d": 128, "m": 16, "nq": 1000, "k": 10, "q": 4,
         "f16": False, "host": False},
        # Finer codes and long result lists, as searched before an exact re-rank.
        {"name": "batch1000_1m_m32_k100", "kind": "search", "n": 1_000_000, "d": 128, "m": 32, "nq": 1000, "k": 100,
         "q": 4, "f16": False, "host": False},
        # The finest codes: two dimensions per sub-space, the largest work.
        {"name": "batch1000_1m_m64_k100", "kind": "search", "n": 1_000_000, "d": 128, "m": 64, "nq": 1000, "k": 100,
         "q": 2, "f16": False, "host": False},
        # fp16 tables, eight queries per block: the precision option, at the headline's shape.
        {"name": "batch1000_1m_f16", "kind": "search", "n": 1_000_000, "d": 128, "m": 16, "nq": 1000, "k": 10, "q": 8,
         "f16": True, "host": False},
        # Another dimension, with a sub-space count that no kernel is specialised for (d = 96, m = 48).
        {"name": "batch64_200k_m48", "kind": "search", "n": 200_003, "d": 96, "m": 48, "nq": 64, "k": 20, "q": 4,
         "f16": False, "host": False},
        # Inverted file, throughput batch: 1024 lists, the 32 nearest probed.
        {"name": "ivf_batch1000", "kind": "ivf", "n": 1_000_000, "d": 128, "m": 16, "nlist": 1024, "nprobe": 32,
         "nq": 1000, "k": 10, "host": False},
        # Inverted file, one interactive query: a chain of small launches.
        {"name": "ivf_one_query", "kind": "ivf", "n": 1_000_000, "d": 128, "m": 16, "nlist": 1024, "nprobe": 8,
         "nq": 1, "k": 10, "host": False},
        # Exact re-rank of the 100 candidates of each of 1000 queries.
        {"name": "rerank_1000x100", "kind": "rerank", "n": 1_000_000, "d": 128, "nq": 1000, "r": 100, "k": 10},
        # Encoding a database (the build side of every index).
        {"name": "encode_1m", "kind": "encode", "n": 1_000_000, "d": 128, "m": 16},
    ]


def _log_int(rng, lo, hi):
    """A whole number in [lo, hi], uniform over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(["search", "ivf", "rerank", "encode"], weights=[11, 4, 3, 2])[0]
    if kind == "search":
        m, d = rng.choice([(16, 128), (16, 128), (16, 64), (16, 96), (32, 128), (48, 96), (64, 128)])
        n = _log_int(rng, 50_000, min(10_000_000, MOST_CODE_BYTES // m))
        nq = _log_int(rng, 1, max(1, min(1000, MOST_LOOKUPS // (n * m))))
        return {"kind": kind, "n": n, "d": d, "m": m, "nq": nq, "k": rng.choice([1, 10, 10, 20, 64, 100, 128]),
                "q": rng.choice([1, 2, 4, 4, 8]), "f16": rng.random() < 0.2, "host": rng.random() < 0.25}
    if kind == "ivf":
        m, d = rng.choice([(16, 128), (16, 128), (16, 64), (32, 128), (48, 96)])
        nlist = rng.choice([200, 256, 1000, 1024, 2048])
        return {"kind": kind, "n": _log_int(rng, 50_000, 1_000_000), "d": d, "m": m, "nlist": nlist,
                "nprobe": _log_int(rng, 1, 64), "nq": _log_int(rng, 1, 1000), "k": rng.choice([1, 10, 10, 100]),
                "host": rng.random() < 0.25}
    if kind == "rerank":
        r = _log_int(rng, 10, 1000)
        return {"kind": kind, "n": _log_int(rng, 100_000, 1_000_000), "d": rng.choice([96, 128, 128, 130, 200]),
                "nq": _log_int(rng, 1, min(2000, 200_000 // r)), "r": r, "k": min(r, rng.choice([1, 10, 10, 100]))}
    m, d = rng.choice([(16, 128), (32, 128), (64, 128), (8, 64), (16, 96), (16, 256)])
    return {"kind": kind, "n": _log_int(rng, 1000, 1_000_000), "d": d, "m": m}


# ---------------------------------------------------------------------------------------------- inputs


def _generator(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1_000_003 + stream) % (1 << 62))
    return g


class _Mixture:
    """Rows of a Gaussian mixture on the GPU, made from the seed."""

    def __init__(self, d, seed):
        self.d, self.seed = d, seed
        self.centres = torch.randn(MIXTURE, d, device="cuda", generator=_generator(seed, 1))

    def rows(self, count, stream):
        g = _generator(self.seed, stream)
        which = torch.randint(0, MIXTURE, (count,), device="cuda", generator=g)
        x = torch.randn(count, self.d, device="cuda", generator=g)
        return x.mul_(SIGMA).add_(self.centres[which])

    def chunks(self, n, step=1 << 18):
        for i, start in enumerate(range(0, n, step)):
            yield start, self.rows(min(step, n - start), 1000 + i)


def _sub(x, m):
    """x as [m][rows][d / m]."""
    return x.view(x.shape[0], m, -1).transpose(0, 1).contiguous()


def _nearest(xs, cent):
    """Nearest centroid per sub-space: xs [m][rows][dsub], cent [m][256][dsub] -> [m][rows]."""
    norms = (cent * cent).sum(-1).unsqueeze(1)
    return torch.baddbmm(norms, xs, cent.transpose(1, 2).contiguous(), alpha=-2.0).argmin(-1)


def _codebook(mix, m):
    """Codebook [m][256][dsub] by a few Lloyd rounds on a sample."""
    xs = _sub(mix.rows(TRAIN_ROWS, 2), m)
    cent = xs[:, :KSUB].clone()
    for _ in range(TRAIN_ROUNDS):
        one_hot = torch.nn.functional.one_hot(_nearest(xs, cent), KSUB).to(torch.float32).transpose(1, 2).contiguous()
        counts = one_hot.sum(-1, keepdim=True)
        cent = torch.where(counts > 0, torch.bmm(one_hot, xs) / counts.clamp(min=1), cent)
    return cent.contiguous()


def _codes(mix, cent, n):
    """uint8 codes n x m, on the GPU."""
    m = cent.shape[0]
    out = torch.empty(n, m, dtype=torch.uint8, device="cuda")
    step = max(1, (1 << 21) // m)
    for start, x in mix.chunks(n):
        for i in range(0, x.shape[0], step):
            part = x[i:i + step]
            out[start + i:start + i + part.shape[0]] = _nearest(_sub(part, m), cent).t().to(torch.uint8)
    return out


def _coarse(mix, nlist, n):
    """Coarse centroids (one Lloyd round over a sample) and the list of each of the n vectors."""
    sample = mix.rows(max(TRAIN_ROWS, 16 * nlist), 3)
    co = sample[:nlist].clone()
    one_hot = torch.nn.functional.one_hot(_nearest(sample[None], co[None])[0], nlist).to(torch.float32).t().contiguous()
    counts = one_hot.sum(-1, keepdim=True)
    co = torch.where(counts > 0, one_hot @ sample / counts.clamp(min=1), co).contiguous()
    lists = torch.empty(n, dtype=torch.int32, device="cuda")
    for start, x in mix.chunks(n):
        lists[start:start + x.shape[0]] = _nearest(x[None], co[None])[0].to(torch.int32)
    return co, lists


def _inputs(case, seed):
    """The case's inputs as torch tensors on the GPU."""
    mix = _Mixture(case["d"], seed)
    kind = case["kind"]
    if kind in ("search", "ivf"):
        cent = _codebook(mix, case["m"])
        got = {"cent": cent, "codes": _codes(mix, cent, case["n"]), "queries": mix.rows(case["nq"], 4)}
        if kind == "ivf":
            got["coarse"], got["lists"] = _coarse(mix, case["nlist"], case["n"])
        return got
    if kind == "rerank":
        base = torch.empty(case["n"], case["d"], device="cuda")
        for start, x in mix.chunks(case["n"]):
            base[start:start + x.shape[0]] = x
        g = _generator(seed, 5)
        cand = torch.zeros(case["nq"], case["r"], 2, dtype=torch.int32, device="cuda")  # (dist, id) records
        cand[..., 1] = torch.randint(0, case["n"], (case["nq"], case["r"]), device="cuda", generator=g)
        return {"base": base, "cand": cand, "queries": mix.rows(case["nq"], 4)}
    x = torch.empty(case["n"], case["d"], device="cuda")
    for start, part in mix.chunks(case["n"]):
        x[start:start + part.shape[0]] = part
    return {"cent": _codebook(mix, case["m"]), "x": x}


def prepare(case, seed):
    got = _inputs(case, seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "encode":
        s["x"], s["cent"] = got["x"], got["cent"]
        s["codes"] = torch.empty(case["n"], case["m"], dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        return s
    if kind == "search":
        handle = vk.PQSearcher(got["cent"].cpu().numpy(), got["codes"].cpu().numpy(), case["d"])
        handle.set_tuning(vk.Tuning(queries_per_block=case["q"]))
    elif kind == "ivf":
        handle = vk.IVFIndex(got["coarse"].cpu().numpy(), got["cent"].cpu().numpy(), got["codes"].cpu().numpy(),
                             got["lists"].cpu().numpy())
    else:
        handle = vk.Reranker(got["base"].cpu().numpy())
        s["cand"] = got["cand"]
    s["handle"] = handle
    s["variant"] = vk.ScanVariant.FusedWarpF16 if case.get("f16") else vk.ScanVariant.FusedWarp
    if case.get("host"):
        s["queries"] = got["queries"].cpu().numpy()
    else:
        s["queries"] = got["queries"].contiguous()
        out = torch.zeros(case["nq"], case["k"], 2, dtype=torch.int32, device="cuda")  # (dist, id) records
        s["out"], s["dist"], s["ids"] = out, out.view(torch.float32)[..., 0], out[..., 1]
    torch.cuda.synchronize()
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "encode":
        rc = vk.library().vk_pq_encode_device(ctypes.c_void_p(s["cent"].data_ptr()), case["d"], case["m"],
                                              ctypes.c_void_p(s["x"].data_ptr()), case["n"],
                                              ctypes.c_void_p(s["codes"].data_ptr()))
        if rc != vk.VK_OK:
            raise RuntimeError(vk.library().vk_last_error().decode())
        return s["codes"]
    h = s["handle"]
    if kind == "search":
        if case["host"]:
            dist, ids, _ = h.search(s["queries"], case["k"], s["variant"])
            return {"dist": dist, "ids": ids}
        h.search_device(s["queries"].data_ptr(), case["nq"], case["k"], s["variant"], s["out"].data_ptr())
    elif kind == "ivf":
        if case["host"]:
            dist, ids, _ = h.search(s["queries"], case["nprobe"], case["k"])
            return {"dist": dist, "ids": ids}
        h.search_device(s["queries"].data_ptr(), case["nq"], case["nprobe"], case["k"], s["out"].data_ptr())
    else:
        h.rerank_device(s["queries"].data_ptr(), case["nq"], s["cand"].data_ptr(), case["r"], case["k"],
                        s["out"].data_ptr())
    return {"dist": s["dist"], "ids": s["ids"]}


def work(case):
    kind = case["kind"]
    d = case["d"]
    if kind == "encode":
        n, m = case["n"], case["m"]
        return {"bytes": 4.0 * n * d + n * m + 4.0 * KSUB * d, "flops": 3.0 * n * KSUB * d}
    nq, k = case["nq"], case["k"]
    ends = 4.0 * nq * d + 8.0 * nq * k  # queries in, results out
    if kind == "rerank":
        rows = nq * case["r"]
        return {"bytes": ends + 8.0 * rows + 4.0 * d * min(rows, case["n"]), "flops": 3.0 * rows * d}
    n, m = case["n"], case["m"]
    tables = 3.0 * nq * KSUB * d
    if kind == "search":
        return {"bytes": ends + 4.0 * KSUB * d + 1.0 * n * m, "flops": tables + 1.0 * nq * n * m}
    share = min(1.0, case["nprobe"] / case["nlist"])  # of the vectors, for lists of equal size
    return {"bytes": ends + 4.0 * KSUB * d + 4.0 * case["nlist"] * d + min(1.0, nq * share) * n * (m + 4.0),
            "flops": tables + 3.0 * nq * case["nlist"] * d + nq * share * n * m}


def tolerance(case):
    # Ids, distances and codes are bit-identical to the CPU's by contract: every sum has one order, and equal
    # distances are ordered by id.
    return "exact"


# ---------------------------------------------------------------------------------------------- 64-bit results


def _best(dist, ids, k):
    """The k smallest of each row by (dist, id)."""
    d, at = torch.topk(dist, k, dim=-1, largest=False)
    i = torch.gather(ids, -1, at) if ids is not None else at
    order = torch.argsort(i, dim=-1, stable=True)
    d, i = torch.gather(d, -1, order), torch.gather(i, -1, order)
    order = torch.argsort(d, dim=-1, stable=True)
    return torch.gather(d, -1, order), torch.gather(i, -1, order)


def exact(case, seed):
    got = _inputs(case, seed)
    kind = case["kind"]
    if kind == "encode":
        cent = got["cent"].double()
        out = torch.empty(case["n"], case["m"], dtype=torch.uint8, device="cuda")
        for start in range(0, case["n"], 8192):
            xs = _sub(got["x"][start:start + 8192].double(), case["m"])
            best = torch.stack([((xs[s][:, None, :] - cent[s][None]) ** 2).sum(-1).argmin(-1)
                                for s in range(case["m"])], 1)
            out[start:start + best.shape[0]] = best.to(torch.uint8)
        return out
    queries = got["queries"].double()
    dists, ids = [], []
    if kind == "rerank":
        for q0 in range(0, case["nq"], 64):
            cand = got["cand"][q0:q0 + 64, :, 1].long()
            d = ((got["base"][cand].double() - queries[q0:q0 + 64, None, :]) ** 2).sum(-1)
            bd, bi = _best(d, cand, case["k"])
            dists.append(bd)
            ids.append(bi)
    else:
        m, n, k = case["m"], case["n"], case["k"]
        cent = got["cent"].double()
        lut = ((queries.view(-1, m, 1, case["d"] // m) - cent[None]) ** 2).sum(-1)  # [nq][m][256]
        codes = got["codes"].t().long() if n * m <= 70_000_000 else None
        step = max(1, min(64, (1 << 27) // n))
        for q0 in range(0, case["nq"], step):
            acc = torch.zeros(min(step, case["nq"] - q0), n, dtype=torch.float64, device="cuda")
            for s in range(m):
                column = codes[s] if codes is not None else got["codes"][:, s].long()
                acc += lut[q0:q0 + step, s][:, column]
            if kind == "ivf":
                co = got["coarse"].double()
                cd = ((queries[q0:q0 + step, None, :] - co[None]) ** 2).sum(-1)
                _, probes = _best(cd, None, case["nprobe"])
                probed = torch.zeros(cd.shape, dtype=torch.bool, device="cuda").scatter_(1, probes, True)
                acc = acc.masked_fill_(~probed[:, got["lists"].long()], math.inf)
            bd, bi = _best(acc, None, k)
            dists.append(bd)
            ids.append(torch.where(torch.isinf(bd), torch.full_like(bi, -1), bi))
    return {"dist": torch.cat(dists), "ids": torch.cat(ids).to(torch.int32)}
