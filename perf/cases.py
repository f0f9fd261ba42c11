"""The work a user of this package has it do on one MI355X, as cases that can be timed and compared.

A case is one pass of a tensor-parallel rank's share of a row-parallel linear and the norm behind it, in the
forms the package offers:

  allreduce      signalling GEMM, the groups released to the staging buffer, reorder + RMSNorm
  reducescatter  the same with the row remap and one rank's receive buffer [M / world, N]
  serial         plain GEMM (any M and N, which is what a batch of a few tokens or a ragged one needs), one bulk
                 copy to the staging buffer, RMSNorm
  norm           RMSNorm alone

through the torch classes and ops (`api` "class") or through the nn.Module wrappers (`api` "module").
Shapes are those of bench.py's workloads, of the tests, or generic ones of the same kind; activations are
N(0, 1), weights N(0, 0.02), gamma N(1, 0.1).
"""
from __future__ import annotations

import math

import torch

import flashoverlap_amd
from flashoverlap_amd import capi, layers, tiling

# tiles of 128x128 / 128x256 / 256x128, in the order of the Algo index
ALGO_TILES = [(128, 128), (128, 128), (128, 256), (128, 256), (256, 128), (256, 128)]
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def _overlap(path, name, api, dtype, m, n, k, algo, group, world=1, rank=0):
    """`group`: layout tiles per signal group (the last group takes what is left)."""
    return {"name": name, "path": path, "api": api, "dtype": dtype, "m": m, "n": n, "k": k, "algo": algo,
            "group": group, "world": world, "rank": rank, "eps": 1e-5}


def _serial(name, dtype, m, n, k):
    return {"name": name, "path": "serial", "api": "class", "dtype": dtype, "m": m, "n": n, "k": k, "algo": 1,
            "eps": 1e-5}


def _norm(name, dtype, m, n):
    return {"name": name, "path": "norm", "api": "class", "dtype": dtype, "m": m, "n": n, "eps": 1e-5}


def listed():
    return [
        # Prefill of a large batch: bench.py's four GPU workloads and its plumbing shape.
        # down_proj of a model with hidden size 4096, half of its 14336 columns; one hardware wave per group
        _overlap("allreduce", "allreduce_8192x4096x7168", "class", "bf16", 8192, 4096, 7168, 1, 1024),
        # o_proj of a model with hidden size 8192, an eighth of its columns: small K, in the eight groups of its tuning file
        _overlap("allreduce", "allreduce_16384x8192x1024", "class", "bf16", 16384, 8192, 1024, 0, 1024),
        # the square shape: one hardware wave, in sixteen groups
        _overlap("allreduce", "allreduce_4096x4096x4096", "class", "fp16", 4096, 4096, 4096, 1, 64),
        # a small problem in sixteen groups: launches and latency
        _overlap("allreduce", "allreduce_1024x1024x1024", "class", "fp16", 1024, 1024, 1024, 1, 4),
        # a decode batch of 128 sequences through the nn.Module wrappers, the layer in one group
        _overlap("allreduce", "allreduce_128x4096x7168", "module", "bf16", 128, 4096, 7168, 1, 32),
        # ReduceScatter in a world of eight: the large prefill, and a chunk of 1024 tokens through the wrappers
        _overlap("reducescatter", "reducescatter_8192x8192x3584", "class", "bf16", 8192, 8192, 3584, 1, 1024, 8, 0),
        _overlap("reducescatter", "reducescatter_1024x8192x3584", "module", "bf16", 1024, 8192, 3584, 1, 256, 8, 3),
        # Decode: one token, and a batch of sixteen (M is no multiple of a tile: the plain GEMM)
        _serial("serial_1x8192x3584", "bf16", 1, 8192, 3584),
        _serial("serial_16x4096x7168", "bf16", 16, 4096, 7168),
        # a prompt of an odd number of tokens, and the test suite's large shape with nothing even in it but K
        _serial("serial_2041x4096x7168", "fp16", 2041, 4096, 7168),
        _serial("serial_8191x4097x7168", "bf16", 8191, 4097, 7168),
        # RMSNorm alone over the longest rows that a wavefront takes whole
        _norm("norm_4096x16384", "bf16", 4096, 16384),
    ]


def _spread(rng, low, high, step=1):
    """A multiple of `step` between low and high, spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return max(low, min(high, int(round(v / step)) * step))


def _cost(case):
    """Seconds of a pass, roughly: for keeping drawn cases within the listed ones."""
    w = work(case)
    return w["flops"] / 1.5e15 + w["bytes"] / 5e12


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        path = rng.choice(["allreduce", "allreduce", "allreduce", "reducescatter", "serial", "serial", "serial", "norm"])
        dtype = rng.choice(["fp16", "bf16"])
        if path == "norm":
            case = _norm("", dtype, _spread(rng, 128, 16384), _spread(rng, 1024, 65536, 8))
            if case["m"] * case["n"] < 1 << 23:   # a norm that small is one launch, and is timed behind the small GEMMs
                continue
        elif path == "serial":
            n = _spread(rng, 512, 8192, rng.choice([1, 8, 8, 8, 128]))
            case = _serial("", dtype, _spread(rng, 1, 8192), n, _spread(rng, 512, 8192, rng.choice([8, 64])))
        else:
            algo = rng.choice([0, 1, 1, 1, 2, 4])
            bm, bn = ALGO_TILES[algo]
            m, n = _spread(rng, bm, 16384, bm), _spread(rng, 1024, 8192, bn)
            k = _spread(rng, 512, 8192, rng.choice([8, 64, 64]))
            tiles = (m // bm) * (n // bn)
            group = max(1, tiles // rng.randrange(1, 17))   # up to some thirty groups: tuning files name one to eight
            world = rng.choice([2, 4, 8]) if path == "reducescatter" else 1
            case = _overlap(path, "", rng.choice(["class", "module"]), dtype, m, n, k, algo, group, world,
                            rng.randrange(world))
        del case["name"]
        if _cost(case) <= most:
            return case


def work(case):
    m, n = case["m"], case["n"]
    if case["path"] == "norm":
        return {"bytes": 2 * (2 * m * n + n), "flops": 4 * m * n}
    k = case["k"]
    inputs = m * k + n * k                            # A, B
    if case["path"] == "serial":
        outputs = 2 * m * n                           # C, staging
        normed = m * n if n % 8 == 0 else 0
    else:
        outputs = m * n + m * n // case["world"]      # C, and the staging or receive buffer
        normed = m * n // case["world"]
    return {"bytes": 2 * (inputs + outputs + normed + (n if normed else 0)), "flops": 2 * m * n * k + 4 * normed}


def tolerance(case):
    # Sums are taken in fp32; results are rounded to the storage type up to three times (C, the scaled value,
    # the product with gamma): unit roundoff 2^-9 for bf16 and 2^-12 for fp16, in each of two implementations.
    return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 1.5e-3}


def _object(case):
    o = torch.classes.flashoverlap_class.OverlapImpl()
    o.mccl_init(case.get("rank", 0), case.get("world", 1), torch.ops.flashoverlap_op.generate_mccl_id())
    o.mutlass_init()
    o.overlap_init()
    return o


def prepare(case, seed):
    flashoverlap_amd.load()
    dev, dtype = torch.device("cuda"), DTYPES[case["dtype"]]
    g = torch.Generator(device=dev).manual_seed(seed)

    def normal(*shape, mean=0.0, std=1.0):
        return torch.empty(shape, dtype=dtype, device=dev).normal_(mean, std, generator=g)

    m, n = case["m"], case["n"]
    s = {"case": case, "gamma": normal(n, mean=1.0, std=0.1)}
    if case["path"] == "norm":
        s["x"], s["out"] = normal(m, n), torch.empty(m, n, dtype=dtype, device=dev)
        return s
    k = case["k"]
    s["a"], s["b"] = normal(m, k), normal(n, k, std=0.02)
    if case["path"] == "serial":
        s["overlap"] = _object(case)
        s["c"] = torch.empty(m, n, dtype=dtype, device=dev)
        s["staging"] = torch.empty(m, n, dtype=dtype, device=dev)
        s["overlap"].set_staging(s["staging"])
        s["out"] = torch.empty(m, n, dtype=dtype, device=dev) if n % 8 == 0 else None
        return s

    world, rank, algo = case["world"], case["rank"], case["algo"]
    bm, bn, _ = capi.algo_tile(algo)
    tm, tn = m // bm, n // bn
    hint = tiling.raster_hint(m, n, algo)
    cseg = tiling.uniform_cseg(tm * tn, case["group"])
    if case["api"] == "module":
        config = {"BM": bm, "BN": bn, "Algo": algo, "hint": hint, "cSeg": cseg}
        comm_op = "all_reduce" if case["path"] == "allreduce" else "reduce_scatter"
        s["linear"] = layers.OverlapRowParallelLayer(rank, world, k, n, m, config, comm_op, dtype=dtype, device=dev)
        s["linear"].weight = torch.nn.Parameter(s["b"], requires_grad=False)
        s["norm"] = layers.ReorderRMSNorm(n, m // world, bm // world, bn, hint, eps=case["eps"], dtype=dtype, device=dev)
        s["norm"].weight = torch.nn.Parameter(s["gamma"], requires_grad=False)
        return s
    s["overlap"] = _object(case)
    s["ra"] = tiling.reorder_indices(tm * tn, hint, dev).reshape(tm, tn)
    s["cseg_cpu"] = torch.tensor(cseg, dtype=torch.int32)
    s["cseg_gpu"] = s["cseg_cpu"].to(dev)
    s["counters"] = torch.zeros(len(cseg), dtype=torch.int32, device=dev)
    s["c"] = torch.empty(m, n, dtype=dtype, device=dev)
    s["recv"] = torch.empty(m // world, n, dtype=dtype, device=dev)
    s["out"] = torch.empty(m // world, n, dtype=dtype, device=dev)
    s["tile"] = (bm // world, bn)
    if case["path"] == "reducescatter":
        s["re"] = tiling.generate_row_remap_array(m, n, bm, bn, cseg, world, dev)
    else:
        s["overlap"].set_staging(s["recv"])
    return s


def run(s):
    case, ops = s["case"], torch.ops.flashoverlap_op
    if case["path"] == "norm":
        ops.rmsnorm_eps(s["x"], s["out"], s["gamma"], case["eps"])
        return [s["out"]]
    if case["path"] == "serial":
        s["overlap"].gemm_allreduce(s["a"], s["b"], s["c"], case["algo"])
        if s["out"] is None:
            return [s["c"], s["staging"]]
        ops.rmsnorm_eps(s["staging"], s["out"], s["gamma"], case["eps"])
        return [s["c"], s["staging"], s["out"]]
    if case["api"] == "module":
        y = s["linear"](s["a"])
        return [y, s["norm"](y)]
    if case["path"] == "allreduce":
        s["overlap"].gemm_allreduce_overlap(s["a"], s["b"], s["c"], s["counters"], s["ra"], 1, s["cseg_cpu"],
                                            s["cseg_gpu"], case["algo"], False)
    else:
        s["overlap"].gemm_reducescatter_overlap(s["a"], s["b"], s["c"], s["recv"], s["counters"], s["ra"], s["re"], 1,
                                                s["cseg_cpu"], s["cseg_gpu"], case["algo"], False)
    ops.reorder_rmsnorm_eps(s["recv"], s["out"], s["gamma"], s["tile"][0], s["tile"][1], 1, s["ra"], case["eps"])
    return [s["c"], s["recv"], s["out"], s["counters"]]
