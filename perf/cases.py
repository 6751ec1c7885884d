"""Performance cases of the sparse side of a recommendation model.

Twelve listed cases and a generator of more cover what a caller of this
package runs per batch: jagged tensors to and from dense, the feature permute
with its offsets, training steps of the table-batched embedding (lookup,
backward and fused rowwise Adagrad), sequence lookups, quantized inference
lookups and the row codecs.  Sizes follow the benchmark configurations of
``mx_fbgemm.bench_inputs`` and the tests; each kind spans the smallest batch
(online inference, debugging runs) to the largest.

``listed()``/``draw(rng)`` give cases (dicts of plain values),
``prepare(case, seed)`` what a program holds before the call, ``run(state)``
one pass through the public entry points, ``work(case)`` the bytes and
operations a pass cannot do without, ``tolerance(case)`` how far two correct
implementations may differ and ``exact(case, seed)`` the same outputs in 64
bits from plain torch.
"""

from __future__ import annotations

import functools
import itertools
import math
import random
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "torchlib-xpu_amd"))

import mx_fbgemm  # noqa: E402,F401  (registers torch.ops.fbgemm.*)
from mx_fbgemm import (  # noqa: E402
    ComputeDevice,
    EmbeddingLocation,
    PoolingMode,
    SparseType,
)
from mx_fbgemm.split_table_batched_embeddings_ops_inference import (  # noqa: E402
    IntNBitTableBatchedEmbeddingBagsCodegen,
)
from mx_fbgemm.split_table_batched_embeddings_ops_training import (  # noqa: E402
    SplitTableBatchedEmbeddingBagsCodegen,
)

DEV = "cuda"
DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16,
          "int32": torch.int32, "int64": torch.int64}
BYTES = {"float32": 4, "float16": 2, "bfloat16": 2, "int32": 4, "int64": 8}
LR, EPS = 0.01, 1.0e-8


def listed() -> list[dict]:
    return [
        # Padding a batch of short user histories for a dense tower and
        # flattening the result back: one feature, one launch each way.
        dict(name="jagged_round_trip", kind="jagged", op="round_trip", B=512, L=64, L2=0, D=128,
             dtype="float32", index="int64"),
        # Sessions of events (two jagged dimensions) padded for an attention
        # tower in bf16, and the gradient brought back to the events.
        dict(name="jagged_nested_grad", kind="jagged", op="grad", B=256, L=20, L2=50, D=64,
             dtype="bfloat16", index="int64"),
        # Reordering a batch's features into the tables' order after the input
        # exchange, and the new offsets the lookup takes.
        dict(name="permute_features", kind="permute", T=40, T_out=40, B=4096, L=10,
             weighted=True, index="int64"),
        # One step of a small model or a small local batch: the launches count.
        dict(name="train_small", kind="train", T=5, E=5000, dims="64", B=128, L=5,
             lengths="uniform", zipf=1.05, pooling="sum", weights="float32", weighted=False,
             ranks=0, index="int64"),
        # The benchmark model's training step: 8 tables of 1M x 128 fp32 rows,
        # 4096 samples of about 20 lookups, skewed ids.
        dict(name="train_step", kind="train", T=8, E=1_000_000, dims="128", B=4096, L=20,
             lengths="uniform", zipf=1.05, pooling="sum", weights="float32", weighted=False,
             ranks=0, index="int64"),
        # A weighted lookup over many features of different widths with fp16
        # weights, whose per-sample weights are learned too (position weights).
        dict(name="train_weighted_mixed", kind="train", T=20, E=200_000,
             dims="32,64,100,128,256,36", B=2048, L=8, lengths="poisson", zipf=1.05,
             pooling="sum", weights="float16", weighted=True, ranks=0, index="int32"),
        # Sequence features (no pooling): one row and one gradient row per event.
        dict(name="train_sequence", kind="sequence", T=4, E=500_000, D=96, B=1024, L=50,
             lengths="uniform", zipf=1.05, weights="float32", index="int64"),
        # One online request batch against a small quantized model.
        dict(name="nbit_small", kind="nbit", T=6, E=20_000, types="int8,int4", dims="64", B=32,
             L=10, lengths="uniform", zipf=1.05, pooling="sum", weighted=False, out="float16",
             index="int32"),
        # The benchmark's inference batch: 16 INT8 + 16 INT4 tables, fixed
        # length 20, MEAN, uniform ids over 32M rows.
        dict(name="nbit_pooled", kind="nbit", T=32, E=1_000_000, types="int8,int4", dims="128",
             B=16384, L=20, lengths="fixed", zipf=0.0, pooling="mean", weighted=False,
             out="float16", index="int64"),
        # A ranking model's tables as they come: three row types, seven widths,
        # Poisson lengths with a tenth of the bags empty.
        dict(name="nbit_mixed", kind="nbit", T=42, E=300_000, types="float16,int4,int8",
             dims="32,64,96,128,256,200,48", B=16384, L=15, lengths="poisson", zipf=1.1,
             pooling="sum", weighted=False, out="float16", index="int64"),
        # Quantized sequence features for an inference attention tower.
        dict(name="nbit_sequence", kind="nbit_sequence", T=4, E=300_000, types="int8", D=96,
             B=1024, L=100, lengths="uniform", zipf=1.05, out="float16", index="int32"),
        # Quantizing a trained table for serving, and reading it back.
        dict(name="quantize_rows", kind="codec", rows=500_000, D=120, bits=4, fused8=False,
             dtype="float32"),
    ]


def _log(rng: random.Random, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["jagged", "permute", "train", "train", "sequence", "nbit", "nbit",
                       "nbit_sequence", "codec"])
    index = rng.choice(["int32", "int64"])
    if kind == "jagged":
        nested = rng.random() < 0.5
        B, L = _log(rng, 8, 1024), _log(rng, 4, 40 if nested else 400)
        return dict(kind=kind, op=rng.choice(["round_trip", "grad", "add"]), B=B, L=L,
                    L2=_log(rng, 4, 40) if nested else 0, D=_log(rng, 8, 200),
                    dtype=rng.choice(["float32", "float16", "bfloat16"]), index=index)
    if kind == "permute":
        T = _log(rng, 2, 100)
        return dict(kind=kind, T=T, T_out=max(1, T - rng.choice([0, 0, 1, 3])),
                    B=_log(rng, 16, 8192), L=_log(rng, 2, 24), weighted=rng.random() < 0.5,
                    index=index)
    lengths = rng.choice(["uniform", "poisson"])
    zipf = rng.choice([0.0, 1.05, 1.2])
    if kind == "train":
        dims = ",".join(str(4 * _log(rng, 1, 64)) for _ in range(rng.randint(1, 6)))
        return dict(kind=kind, T=_log(rng, 1, 40), E=_log(rng, 500, 300_000), dims=dims,
                    B=_log(rng, 16, 4096), L=_log(rng, 1, 12), lengths=lengths, zipf=zipf,
                    pooling=rng.choice(["sum", "mean"]),
                    weights=rng.choice(["float32", "float32", "float16"]),
                    weighted=rng.random() < 0.3, ranks=rng.choice([0, 0, 0, 2]), index=index)
    if kind == "sequence":
        return dict(kind=kind, T=_log(rng, 1, 12), E=_log(rng, 500, 300_000),
                    D=4 * _log(rng, 2, 64), B=_log(rng, 16, 1024), L=_log(rng, 2, 40),
                    lengths=lengths, zipf=zipf, weights=rng.choice(["float32", "float16"]),
                    index=index)
    types = ["float16", "int8", "int4", "int2", "fp8", "float32"]
    out = rng.choice(["float16", "float16", "bfloat16", "float32"])
    if kind == "nbit":
        k = rng.randint(1, 3)
        dims = ",".join(str(8 * _log(rng, 1, 48)) for _ in range(rng.randint(1, 7)))
        return dict(kind=kind, T=_log(rng, 2, 48), E=_log(rng, 500, 300_000),
                    types=",".join(rng.sample(types, k)), dims=dims, B=_log(rng, 8, 8192),
                    L=_log(rng, 1, 24), lengths=lengths, zipf=zipf,
                    pooling=rng.choice(["sum", "mean"]), weighted=rng.random() < 0.25, out=out,
                    index=index)
    if kind == "nbit_sequence":
        return dict(kind=kind, T=_log(rng, 1, 12), E=_log(rng, 500, 300_000),
                    types=",".join(rng.sample(types, rng.randint(1, 2))), D=8 * _log(rng, 1, 40),
                    B=_log(rng, 8, 1024), L=_log(rng, 2, 100), lengths=lengths, zipf=zipf,
                    out=out, index=index)
    fused8 = rng.random() < 0.3
    return dict(kind=kind, rows=_log(rng, 100, 400_000), D=_log(rng, 8, 300),
                bits=8 if fused8 else rng.choice([2, 4, 8]), fused8=fused8,
                dtype=rng.choice(["float32", "float16"]))


# ---- inputs ------------------------------------------------------------------


def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _offsets(lengths: torch.Tensor) -> torch.Tensor:
    out = torch.zeros(lengths.numel() + 1, dtype=torch.int64, device=DEV)
    out[1:] = torch.cumsum(lengths.view(-1).long(), 0)
    return out


def _shuffled(case: dict, n: int, g: torch.Generator, make) -> torch.Tensor:
    """n lengths whose values belong to the case and whose order to the seed,
    so that a case's outputs have one shape whatever the seed."""
    key = repr(sorted((k, v) for k, v in case.items() if k != "name"))
    own = _gen(random.Random(key).getrandbits(48))
    return make(own)[torch.randperm(n, generator=g, device=DEV)]


def _lengths(case: dict, n: int, g: torch.Generator) -> torch.Tensor:
    """n bag lengths of mean about L: U{1..2L}, Poisson(L) clipped to 100 with
    a tenth of the bags empty, or L each."""
    L = case["L"]
    if case["lengths"] == "uniform":
        return _shuffled(case, n, g, lambda own: torch.randint(1, 2 * L + 1, (n,), generator=own,
                                                               device=DEV))
    if case["lengths"] == "poisson":
        def poisson(own):
            x = torch.poisson(torch.full((n,), float(L), device=DEV), generator=own)
            return x.long().clamp(max=100) * (torch.rand(n, generator=own, device=DEV) >= 0.1)
        return _shuffled(case, n, g, poisson)
    return torch.full((n,), L, dtype=torch.int64, device=DEV)


def _mean_length(case: dict) -> float:
    return {"uniform": case["L"] + 0.5, "poisson": 0.9 * case["L"], "fixed": case["L"]}[
        case["lengths"]]


def _ids(case: dict, E: int, n: int, g: torch.Generator) -> torch.Tensor:
    """n row ids of a table: uniform, or Zipf ranks spread by a permutation."""
    a = case["zipf"]
    if a == 0.0:
        return torch.randint(0, E, (n,), generator=g, device=DEV)
    cdf = torch.cumsum(torch.arange(1, E + 1, dtype=torch.float64, device=DEV).pow_(-a), 0)
    u = torch.rand(n, generator=g, device=DEV, dtype=torch.float64) * cdf[-1]
    rank = torch.searchsorted(cdf, u, right=True).clamp_(max=E - 1)
    return torch.randperm(E, generator=g, device=DEV)[rank]


@functools.lru_cache(maxsize=None)
def _distinct(E: int, n: float, a: float) -> float:
    """Expected distinct rows among n draws of ``_ids``."""
    p = np.full(E, 1.0 / E) if a == 0.0 else np.arange(1, E + 1, dtype=np.float64) ** -a
    p /= p.sum()
    return float(-np.expm1(n * np.log1p(-np.minimum(p, 1.0 - 1e-12))).sum())


def _dims(case: dict) -> list[int]:
    ds = [int(d) for d in str(case["dims"]).split(",")] if "dims" in case else [case["D"]]
    return [ds[t % len(ds)] for t in range(case["T"])]


def _types(case: dict) -> list[str]:
    ts = case["types"].split(",")
    return [ts[t % len(ts)] for t in range(case["T"])]


def _batch_sizes(case: dict) -> list[list[int]]:
    """Samples per feature and rank of a variable batch (ranks > 0)."""
    B, R = case["B"], case["ranks"]
    return [[max(1, B // (1 + (t + r) % 3) // R) for r in range(R)] for t in range(case["T"])]


def _bags_per_feature(case: dict) -> list[int]:
    if case.get("ranks", 0):
        return [sum(b) for b in _batch_sizes(case)]
    return [case["B"]] * case["T"]


def _batch(case: dict, g: torch.Generator) -> dict:
    """Feature-major bag lengths, 64-bit offsets and row ids of a lookup batch."""
    bags = _bags_per_feature(case)
    lengths = _lengths(case, sum(bags), g)
    off = _offsets(lengths)
    first = [0] + list(itertools.accumulate(bags))
    at = off[torch.tensor(first, device=DEV)].tolist()
    ids = [_ids(case, case["E"], at[t + 1] - at[t], g) for t in range(case["T"])]
    return dict(bags=bags, first=first, at=at, lengths=lengths, offsets=off,
                indices=torch.cat(ids))


def _train_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    s = _batch(case, g)
    dims, T, E = _dims(case), case["T"], case["E"]
    s["dims"] = dims
    s["weights"] = (torch.rand(E * sum(dims), generator=g, device=DEV) * 0.02 - 0.01).to(
        DTYPES[case["weights"]])
    # Momentum as some way into training: every row has been updated before.
    s["momentum"] = torch.rand(E * T, generator=g, device=DEV) * 1e-4 + 1e-6
    N = s["indices"].numel()
    if case["kind"] == "sequence":
        shape = (N, case["D"])
    elif case["ranks"]:
        shape = (sum(b * d for b, d in zip(s["bags"], dims)),)
    else:
        shape = (case["B"], sum(dims))
    s["grad"] = torch.randn(shape, generator=g, device=DEV) * 0.01
    s["psw"] = (torch.rand(N, generator=g, device=DEV) + 0.5 if case.get("weighted") else None)
    return s


def _row_bytes(ty: str, D: int) -> int:
    return {"float32": 4 * D, "float16": 2 * D, "fp8": D, "int8": D + 4, "int4": D // 2 + 4,
            "int2": D // 4 + 4}[ty]


def _nbit_inputs(case: dict, seed: int) -> dict:
    """The batch and each table's rows: [E, row bytes padded to 16] uint8,
    quantized rows with fp16 scale and bias in front of the codes."""
    g = _gen(seed)
    s = _batch(case, g)
    E, tables = case["E"], []
    for ty, D in zip(_types(case), _dims(case)):
        rb = -(-_row_bytes(ty, D) // 16) * 16
        w = torch.randint(0, 256, (E, rb), generator=g, device=DEV, dtype=torch.uint8)
        if ty.startswith("int"):
            qp = torch.empty((E, 2), device=DEV, dtype=torch.float16)
            qp[:, 0] = torch.rand(E, generator=g, device=DEV) * 9e-3 + 1e-3
            qp[:, 1] = torch.rand(E, generator=g, device=DEV) * 0.2 - 0.1
            w[:, :4] = qp.view(torch.uint8)
        elif ty == "fp8":
            w &= 0xBF  # magnitudes below 2, as an encoder of small weights gives
        else:
            v = (torch.randn((E, D), generator=g, device=DEV) * 0.01).to(DTYPES[ty])
            w[:, : _row_bytes(ty, D)] = v.view(torch.uint8)
        tables.append(w)
    s["tables"] = tables
    N = s["indices"].numel()
    s["psw"] = torch.rand(N, generator=g, device=DEV) + 0.5 if case.get("weighted") else None
    return s


def _jagged_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    B, L, L2 = case["B"], case["L"], case["L2"]
    def upto(top, n):
        return _offsets(_shuffled(case, n, g, lambda own: torch.randint(
            0, top + 1, (n,), generator=own, device=DEV)))

    offs = [upto(L, B)]
    if L2:
        offs.append(upto(L2, int(offs[0][-1])))
    N, dt = int(offs[-1][-1]), DTYPES[case["dtype"]]
    dense = [B, L] + ([L2] if L2 else []) + [case["D"]]
    return dict(offs=offs, N=N, max_lengths=dense[1:-1],
                values=torch.randn((N, case["D"]), generator=g, device=DEV).to(dt),
                dense=torch.randn(dense, generator=g, device=DEV).to(dt))


def _permute_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    T, B = case["T"], case["B"]
    # Each feature keeps its lengths over the seeds (in another order), and
    # the same features are kept.
    top = 2 * case["L"] + 1
    lengths = _shuffled(case, B, g, lambda own: torch.randint(
        0, top, (B, T), generator=own, device=DEV)).t().contiguous()
    perm = torch.randperm(case["T_out"], generator=g, device=DEV)
    N = int(lengths.sum())
    return dict(lengths=lengths, perm=perm, N_out=int(lengths[perm].sum()),
                values=torch.randint(0, 1_000_000, (N,), generator=g, device=DEV),
                psw=torch.rand(N, generator=g, device=DEV) if case["weighted"] else None)


def _codec_input(case: dict, seed: int) -> torch.Tensor:
    g = _gen(seed)
    scale = torch.rand((case["rows"], 1), generator=g, device=DEV) * 0.1 + 0.01
    return (torch.randn((case["rows"], case["D"]), generator=g, device=DEV) * scale).to(
        DTYPES[case["dtype"]])


# ---- what the program holds, and one pass ------------------------------------

SPARSE = {"float32": SparseType.FP32, "float16": SparseType.FP16, "bfloat16": SparseType.BF16,
          "int8": SparseType.INT8, "int4": SparseType.INT4, "int2": SparseType.INT2,
          "fp8": SparseType.FP8}
POOL = {"sum": PoolingMode.SUM, "mean": PoolingMode.MEAN}


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    ix = DTYPES[case["index"]] if "index" in case else None
    st: dict = dict(case=case, kind=kind)
    if kind == "jagged":
        s = _jagged_inputs(case, seed)
        st.update(offs=[o.to(ix) for o in s["offs"]], N=s["N"], max_lengths=s["max_lengths"],
                  values=s["values"], dense=s["dense"])
        if case["op"] == "grad":
            st["values"].requires_grad_(True)
    elif kind == "permute":
        s = _permute_inputs(case, seed)
        st.update(perm=s["perm"].int(), lengths=s["lengths"].to(ix), values=s["values"].to(ix),
                  psw=s["psw"], N_out=s["N_out"])
    elif kind in ("train", "sequence"):
        s = _train_inputs(case, seed)
        tbe = SplitTableBatchedEmbeddingBagsCodegen(
            [(case["E"], d, EmbeddingLocation.DEVICE, ComputeDevice.CUDA) for d in s["dims"]],
            pooling_mode=PoolingMode.NONE if kind == "sequence" else POOL[case["pooling"]],
            learning_rate=LR, eps=EPS, device=torch.device(DEV, torch.cuda.current_device()),
            weights_precision=SPARSE[case["weights"]], stochastic_rounding=False)
        with torch.no_grad():
            tbe.weights_dev.copy_(s["weights"])
            tbe.momentum1_dev.copy_(s["momentum"])
        st.update(tbe=tbe, indices=s["indices"].to(ix), offsets=s["offsets"].to(ix),
                  grad=s["grad"], psw=s["psw"].requires_grad_(True) if case.get("weighted") else None,
                  bs=_batch_sizes(case) if case.get("ranks") else None)
    elif kind in ("nbit", "nbit_sequence"):
        s = _nbit_inputs(case, seed)
        tbe = IntNBitTableBatchedEmbeddingBagsCodegen(
            [("t%d" % t, case["E"], d, SPARSE[ty], EmbeddingLocation.DEVICE)
             for t, (ty, d) in enumerate(zip(_types(case), _dims(case)))],
            pooling_mode=PoolingMode.NONE if kind == "nbit_sequence" else POOL[case["pooling"]],
            output_dtype=SPARSE[case["out"]],
            device=torch.device(DEV, torch.cuda.current_device()))
        for dst, src in zip(tbe.split_embedding_weights(), s["tables"]):
            dst.copy_(src)
        st.update(tbe=tbe, indices=s["indices"].to(ix), offsets=s["offsets"].to(ix),
                  psw=s["psw"])
    else:
        st.update(x=_codec_input(case, seed))
    return st


def run(st: dict):
    kind, case = st["kind"], st["case"]
    ops = torch.ops.fbgemm
    if kind == "jagged":
        if case["op"] == "add":
            return ops.jagged_dense_elementwise_add_jagged_output(st["values"], st["offs"],
                                                                  st["dense"])[0]
        if case["op"] == "round_trip":
            dense = ops.jagged_to_padded_dense(st["values"], st["offs"], st["max_lengths"], 0.0)
            return dense, ops.dense_to_jagged(dense, st["offs"], st["N"])[0]
        st["values"].grad = None
        dense = ops.jagged_to_padded_dense(st["values"], st["offs"], st["max_lengths"], 0.0)
        dense.backward(st["dense"])
        return dense.detach(), st["values"].grad
    if kind == "permute":
        lengths, values, psw = ops.permute_2D_sparse_data(st["perm"], st["lengths"], st["values"],
                                                          st["psw"], st["N_out"])
        return lengths, values, psw, ops.asynchronous_complete_cumsum(lengths.view(-1))
    if kind == "train":
        if st["psw"] is not None:
            st["psw"].grad = None
        tbe = st["tbe"]
        out = tbe(st["indices"], st["offsets"], st["psw"],
                  batch_size_per_feature_per_rank=st["bs"])
        out.backward(st["grad"])
        return dict(out=out.detach(), weights=tbe.weights_dev.detach(),
                    momentum=tbe.momentum1_dev,
                    grad=st["psw"].grad if st["psw"] is not None else None)
    if kind == "sequence":
        tbe = st["tbe"]
        out = tbe(st["indices"], st["offsets"])
        out.backward(st["grad"])
        return dict(out=out.detach(), weights=tbe.weights_dev.detach(),
                    momentum=tbe.momentum1_dev)
    if kind == "nbit":
        return st["tbe"](st["indices"], st["offsets"], st["psw"])
    if kind == "nbit_sequence":
        return st["tbe"](st["indices"], st["offsets"])
    if case["fused8"]:
        q = (ops.FloatToFused8BitRowwiseQuantized(st["x"]) if case["dtype"] == "float32"
             else ops.HalfToFused8BitRowwiseQuantized(st["x"]))
        return q, ops.Fused8BitRowwiseQuantizedToFloat(q)
    q = ops.FloatOrHalfToFusedNBitRowwiseQuantizedSBHalf(st["x"], case["bits"])
    return q, ops.FusedNBitRowwiseQuantizedSBHalfToFloat(q, case["bits"])


# ---- the work of a pass --------------------------------------------------------


def work(case: dict) -> dict:
    kind = case["kind"]
    ib = BYTES[case["index"]] if "index" in case else 0
    if kind == "jagged":
        rows = case["B"] * case["L"] * (case["L2"] or 1)
        N = case["B"] * case["L"] / 2 * (case["L2"] / 2 if case["L2"] else 1)
        eb = case["D"] * BYTES[case["dtype"]]
        off = ib * (case["B"] + (case["B"] * case["L"] / 2 if case["L2"] else 0))
        if case["op"] == "add":  # values and the dense rows they meet read, values written
            return {"bytes": 3 * N * eb + off, "flops": N * case["D"]}
        # values read, dense written; then the covered dense rows read and
        # values (or their gradient) written
        return {"bytes": N * eb + rows * eb + 2 * N * eb + 2 * off, "flops": 0.0}
    if kind == "permute":
        bags_in, bags = case["T"] * case["B"], case["T_out"] * case["B"]
        N = bags * case["L"]
        return {"bytes": ib * (bags_in + 2 * bags) + 2 * N * ib + (8 * N if case["weighted"] else 0),
                "flops": 0.0}
    if kind == "codec":
        n, q = case["rows"] * case["D"], case["rows"] * (
            case["D"] + 8 if case["fused8"] else -(-case["D"] * case["bits"] // 8) + 4)
        return {"bytes": n * BYTES[case["dtype"]] + 2 * q + 4 * n, "flops": 4.0 * n}
    dims, bags, L = _dims(case), _bags_per_feature(case), _mean_length(case)
    lookups = [b * L for b in bags]
    N = sum(lookups)
    rows = [_distinct(case["E"], n, case["zipf"]) for n in lookups]
    idx = N * ib + (sum(bags) + 1) * ib
    if kind in ("nbit", "nbit_sequence"):
        table = sum(u * _row_bytes(ty, d) for u, ty, d in zip(rows, _types(case), dims))
        per = lookups if kind == "nbit_sequence" else bags
        out = sum(n * d for n, d in zip(per, dims)) * BYTES[case["out"]]
        return {"bytes": idx + table + out + (4 * N if case.get("weighted") else 0),
                "flops": 2.0 * sum(n * d for n, d in zip(lookups, dims))}
    # A training step: the batch, the touched rows and momentum read and
    # written, the output written, its gradient read (and the per-sample
    # weights read and their gradient written).
    wb = BYTES[case["weights"]]
    table = sum(u * (2 * d * wb + 8) for u, d in zip(rows, dims))
    per = lookups if kind == "sequence" else bags
    dense = 2 * 4 * sum(n * d for n, d in zip(per, dims))
    macs = sum(n * d for n, d in zip(lookups, dims))
    weighted = bool(case.get("weighted"))
    flops = (0 if kind == "sequence" else macs) + macs + (4 * macs if weighted else 0)
    return {"bytes": idx + table + dense + (8 * N if weighted else 0),
            "flops": flops + 5.0 * sum(u * d for u, d in zip(rows, dims))}


def tolerance(case: dict):
    """Copies, integer work and the codecs' bytes are exact.  Pooled fp32 sums,
    the rowwise Adagrad update and the per-sample gradients differ by the
    order of their fp32 sums; fp16 weights and 16-bit outputs by a rounding
    that falls the other way now and then."""
    kind = case["kind"]
    if kind in ("permute", "codec") or kind == "jagged":
        return "exact"
    if kind in ("train", "sequence"):
        if case["weights"] == "float16":
            return {"rel": 1e-5, "max": 5e-3}
        return {"rel": 2e-6, "max": 2e-4}
    out = case["out"]
    return {"float32": {"rel": 2e-6, "max": 2e-4}, "float16": {"rel": 2e-4, "max": 5e-3},
            "bfloat16": {"rel": 2e-3, "max": 4e-2}}[out]


# ---- 64-bit results from plain torch -------------------------------------------


def _exact_jagged(case: dict, s: dict):
    off0, N = s["offs"][0], s["N"]
    i = torch.arange(N, device=DEV)
    if case["L2"]:
        off1 = s["offs"][1]
        seg = torch.searchsorted(off1, i, right=True) - 1
        b = torch.searchsorted(off0, seg, right=True) - 1
        row = (b * case["L"] + (seg - off0[b])) * case["L2"] + (i - off1[seg])
    else:
        b = torch.searchsorted(off0, i, right=True) - 1
        row = b * case["L"] + (i - off0[b])
    v, d = s["values"].double(), s["dense"].double().reshape(-1, case["D"])
    if case["op"] == "add":
        return v + d[row]
    dense = torch.zeros_like(d)
    dense[row] = v
    return dense.view(s["dense"].shape), (v if case["op"] == "round_trip" else d[row])


def _exact_train(case: dict, s: dict):
    kind, E, dims = case["kind"], case["E"], s["dims"]
    w = s["weights"].double()
    h = s["momentum"].double()
    N = s["indices"].numel()
    gpsw = torch.zeros(N, dtype=torch.float64, device=DEV) if s["psw"] is not None else None
    grad = s["grad"].double()
    out = torch.empty_like(grad)
    bs = _batch_sizes(case) if case.get("ranks") else None
    w0 = d0 = 0
    for t, D in enumerate(dims):
        lo, hi, nb = s["at"][t], s["at"][t + 1], s["bags"][t]
        idx = s["indices"][lo:hi]
        W = w[w0:w0 + E * D].view(E, D)
        if kind == "sequence":
            rows = W[idx]
            out[lo:hi] = rows
            g = grad[lo:hi]
        else:
            lens = s["lengths"][s["first"][t]:s["first"][t] + nb]
            bag = torch.repeat_interleave(torch.arange(nb, device=DEV), lens)
            if bs:  # rank-major, then feature-major, flat
                spans, o = [], 0
                for r in range(case["ranks"]):
                    for f, d in enumerate(dims):
                        n = bs[f][r] * d
                        if f == t:
                            spans.append((o, o + n))
                        o += n
                gt = torch.cat([grad[a:b] for a, b in spans]).view(nb, D)
            else:
                gt = grad[:, d0:d0 + D]
            p = s["psw"].double()[lo:hi] if s["psw"] is not None else torch.ones(
                hi - lo, dtype=torch.float64, device=DEV)
            scale = (1.0 / lens.clamp(min=1).double())[bag] if case["pooling"] == "mean" else 1.0
            rows = W[idx]
            res = torch.zeros((nb, D), dtype=torch.float64, device=DEV).index_add_(
                0, bag, rows * (p * scale).unsqueeze(1))
            if bs:
                n0 = 0
                for a, b in spans:
                    k = (b - a) // D
                    out[a:b] = res[n0:n0 + k].reshape(-1)
                    n0 += k
            else:
                out[:, d0:d0 + D] = res
            g = gt[bag]
            if gpsw is not None:
                gpsw[lo:hi] = (g * rows).sum(1) * scale
            g = g * (p * scale).unsqueeze(1)
        uniq, inv = torch.unique(idx, return_inverse=True)
        G = torch.zeros((uniq.numel(), D), dtype=torch.float64, device=DEV).index_add_(0, inv, g)
        ht = h[t * E:(t + 1) * E]
        hn = ht[uniq] + G.square().mean(1)
        ht[uniq] = hn
        W[uniq] -= (LR / (hn.sqrt() + EPS)).unsqueeze(1) * G
        w0 += E * D
        d0 += D
    res = dict(out=out, weights=w, momentum=h)
    if kind == "train":
        res["grad"] = gpsw
    return res


def _decode(ty: str, rows: torch.Tensor, D: int) -> torch.Tensor:
    """Rows of uint8 in the lookup's layout as float64 values."""
    if ty in ("float32", "float16"):
        return rows[:, : _row_bytes(ty, D)].contiguous().view(DTYPES[ty]).double()
    if ty == "fp8":  # sign, 4 exponent bits of bias 7, 3 mantissa bits
        c = rows[:, :D].long()
        e, m = (c >> 3) & 15, (c & 7).double()
        mag = torch.where(e > 0, torch.ldexp(1.0 + m / 8, e - 7), torch.ldexp(m / 8, e - 6))
        return torch.where(c >= 128, -mag, mag)
    bits = int(ty[3:])
    codes = rows[:, 4:4 + D * bits // 8]
    q = torch.stack([(codes >> s) & ((1 << bits) - 1) for s in range(0, 8, bits)], 2).reshape(
        rows.shape[0], D).double()
    qp = rows[:, :4].contiguous().view(torch.float16).double()
    return q * qp[:, :1] + qp[:, 1:]


def _exact_nbit(case: dict, s: dict):
    res = []
    for t, (ty, D) in enumerate(zip(_types(case), _dims(case))):
        lo, hi, B = s["at"][t], s["at"][t + 1], s["bags"][t]
        idx = s["indices"][lo:hi]
        if case["kind"] == "nbit_sequence":
            res.append(_decode(ty, s["tables"][t][idx], D))
            continue
        lens = s["lengths"][s["first"][t]:s["first"][t] + B]
        bag = torch.repeat_interleave(torch.arange(B, device=DEV), lens)
        v = _decode(ty, s["tables"][t][idx], D)
        if s["psw"] is not None:
            v *= s["psw"].double()[lo:hi].unsqueeze(1)
        o = torch.zeros((B, D), dtype=torch.float64, device=DEV).index_add_(0, bag, v)
        if case["pooling"] == "mean":
            o /= lens.clamp(min=1).double().unsqueeze(1)
        res.append(o)
    return torch.cat(res, 0 if case["kind"] == "nbit_sequence" else 1)


def _exact_codec(case: dict, x: torch.Tensor):
    x = x.double()
    lo, hi = x.amin(1, keepdim=True), x.amax(1, keepdim=True)
    if case["fused8"]:
        scale = (hi - lo) / 255
        return None, torch.round((x - lo) * (255 / (hi - lo + 1e-8))) * scale + lo
    top = float((1 << case["bits"]) - 1)
    lo = lo.half().double()
    scale = ((hi - lo) / top).half().double()
    scale = torch.where(scale == 0, torch.ones_like(scale), scale)
    return None, torch.round((x - lo) / scale).clamp(0, top) * scale + lo


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "jagged":
        return _exact_jagged(case, _jagged_inputs(case, seed))
    if kind == "permute":
        # Whole numbers and copies only: compared bit for bit.
        return None
    if kind in ("train", "sequence"):
        return _exact_train(case, _train_inputs(case, seed))
    if kind in ("nbit", "nbit_sequence"):
        return _exact_nbit(case, _nbit_inputs(case, seed))
    return _exact_codec(case, _codec_input(case, seed))
