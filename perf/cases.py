"""The work whose speed matters here, as cases: the audit of a decode step, the attention shares, the
budget split under each objective, and the views of vLLM's block table and SGLang's token list.

Sizes are this repository's own: the Llama-3-8B decode shape, the fp8 full step, the skewed
long-context mix, the 1024 x 8192 view build, the 4-row fp32 check and the controller's batch at the
decode shape.  ``draw`` spreads over the ranges between and around them.

A case's ``op`` is the call it makes:

  audit       RecordingPlane over the layers of a decode step; ``mode`` says how: ``record`` is the
              engine's hook called eagerly, ``graph`` the same captured once and replayed, ``layers``
              the plan and one launch (the only form with a key scale, for fp8 keys).  With ``shares``
              the step goes on to the shares, the uniform ranking and the view.
  shares      tile_shares over the recorded planes of many layers
  uniform     uniform_view: the uniform ranking and the view in one call
  view        DecodeView.build on a committed keep mask
  controller  keep_rows: the controller's rule under ``sum`` or ``maxmin`` on float32 shares
  objective   sum_keep / maxmin_keep on float64 scores
  slots       SlotCompactor.compact on SGLang's list
"""

from __future__ import annotations

import math
import os
import sys
import time

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sigmod-kvscope_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from observe.allocation import (maxmin_keep, maxmin_workspace_bytes, sum_keep, sum_workspace_bytes)  # noqa: E402
from observe.controller import keep_rows, keep_rows_workspace_bytes  # noqa: E402
from observe.tile_shares import shares_workspace_bytes, tile_shares  # noqa: E402
from runtime.audit_kernel import TILE_BLOCKS, RecordingPlane  # noqa: E402
from runtime.block_view import DecodeView, uniform_view  # noqa: E402
from runtime.sglang_compact import SlotCompactor  # noqa: E402

DTYPES = {"fp32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "fp8": torch.float8_e4m3fn}
ELEMENT = {"fp32": 4, "f16": 2, "bf16": 2, "fp8": 1}
K_SCALE = 6.0 / 448.0  # N(0, 1) fills the e4m3 range up to 6 sigma
FRACTION, RECENT = 0.5, 4


def listed():
    audit = {"op": "audit", "heads_audited": "group", "long_rows": 0, "timer": False, "shares": False}
    return [
        # a small batch audited through the whole path, eager: a handful of launches and little data
        dict(audit, name="step_small_fp32", mode="record", rows=4, low=17, high=512, block=16, kv_heads=2, group=4,
             dim=64, dtype="fp32", layers=2, shares=True),
        # the ordinary audit step of a captured decode: Llama-3-8B, 32 layers, then shares, ranking and view
        dict(audit, name="step_llama_bf16", mode="graph", rows=128, low=512, high=8192, block=16, kv_heads=8, group=4,
             dim=128, dtype="bf16", layers=32, shares=True),
        # every KV head of each layer: the fuller audit, the most bytes
        dict(audit, name="audit_all_heads_bf16", mode="record", rows=128, low=512, high=8192, block=16, kv_heads=8,
             group=4, dim=128, dtype="bf16", layers=4, heads_audited="all"),
        # long contexts among many shorter ones, fp8 keys in 32-token blocks, the per-row timer on
        dict(audit, name="audit_long_fp8", mode="layers", rows=256, low=2048, high=8192, long_rows=8, long=131072,
             block=32, kv_heads=8, group=4, dim=128, dtype="fp8", layers=8, timer=True),
        # shares of a few very long requests over 32 layers
        {"name": "shares_long", "op": "shares", "rows": 16, "low": 256, "high": 8192, "layers": 32, "cells": 4,
         "aggregate": "mean"},
        # the ranking and view of many long requests
        {"name": "uniform_1024x8192", "op": "uniform", "rows": 1024, "low": 1, "high": 8192, "block": 16, "recent": 0,
         "paired": False},
        # what every decode step pays: the view of the committed mask
        {"name": "view_128x512", "op": "view", "rows": 128, "low": 32, "high": 512, "block": 16, "prefill": 0},
        # the controller's rule at the decode shape, each of its float64 objectives
        {"name": "controller_sum_128x512", "op": "controller", "objective": "sum", "rows": 128, "low": 32, "high": 512,
         "released": True, "weights": False, "paired": True},
        {"name": "controller_maxmin_128x512", "op": "controller", "objective": "maxmin", "rows": 128, "low": 32,
         "high": 512, "released": True, "weights": False, "paired": True},
        # the same objectives over many long requests
        {"name": "sum_1024x8192", "op": "objective", "objective": "sum", "rows": 1024, "low": 1, "high": 8192,
         "weights": False, "paired": False},
        {"name": "maxmin_1024x8192", "op": "objective", "objective": "maxmin", "rows": 1024, "low": 1, "high": 8192,
         "weights": False, "paired": False},
        # SGLang's list of a decode batch, and a graph's padding rows
        {"name": "slots_256x8192", "op": "slots", "rows": 256, "padding": 8, "low": 512, "high": 8192, "block": 16,
         "wide": False},
    ]


def _log(rng, low, high):
    """A whole number spread over the logarithm of low .. high."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _draw_audit(rng):
    dtype = rng.choice(["bf16", "bf16", "f16", "fp8", "fp32"])
    block = rng.choice([8, 16, 16, 32])
    dim = rng.choice([64, 128, 128, 256])
    kv_heads = rng.choice([1, 2, 4, 8])
    group = rng.choice([1, 2, 4, 4, 7, 8])
    heads = "all" if rng.random() < 0.25 and kv_heads * group <= 64 else "group"
    rows = _log(rng, 1, 256)
    high = _log(rng, 64, 32768)
    layers = _log(rng, 1, 32)
    case = {"op": "audit", "mode": "layers" if dtype == "fp8" else rng.choice(["record", "graph", "layers"]),
            "rows": rows, "low": max(1, high // 16), "high": high, "long_rows": 0, "block": block,
            "kv_heads": kv_heads, "group": group, "dim": dim, "dtype": dtype, "layers": layers,
            "heads_audited": heads, "timer": rng.random() < 0.25, "shares": heads == "group" and rng.random() < 0.5}
    # at most about 3 GB of keys in a pass, 8 GB of cache and 256 MB of records
    while case["rows"] > 1 and (work(case)["bytes"] > 3e9 or _cache_bytes(case) > 8e9 or _record_bytes(case) > 256e6):
        if case["layers"] > 4:
            case["layers"] //= 2
        else:
            case["rows"] = max(1, case["rows"] * 3 // 4)
    return case


def draw(rng):
    op = rng.choice(["audit"] * 5 + ["shares", "uniform", "uniform", "view", "controller", "controller", "objective",
                                     "objective", "slots"])
    if op == "audit":
        return _draw_audit(rng)
    rows = _log(rng, 1, 1024)
    high = _log(rng, 16, 8192)
    case = {"op": op, "rows": rows, "low": max(1, high // 64), "high": high}
    if op == "shares":
        case.update(rows=min(rows, 256), layers=_log(rng, 1, 48), cells=rng.choice([1, 4, 4, 7, 8, 32]),
                    aggregate=rng.choice(["mean", "mean", "max"]))
        while _record_bytes(case) > 256e6:
            case["rows" if case["rows"] > 1 else "layers"] //= 2
    elif op == "uniform":
        case.update(block=rng.choice([8, 16, 32]), recent=rng.choice([0, 4]), paired=rng.random() < 0.5)
    elif op == "view":
        case.update(rows=min(rows, 512), block=rng.choice([8, 16, 32]), prefill=rng.choice([0, 0, 1, 3]))
        case["prefill"] = min(case["prefill"], case["rows"] - 1)
    elif op in ("controller", "objective"):
        case.update(objective=rng.choice(["sum", "maxmin"]), paired=rng.random() < 0.5)
        case["weights"] = case["objective"] == "sum" and rng.random() < 0.5
        if op == "controller":
            case["released"] = rng.random() < 0.5
    else:
        case.update(rows=min(rows, 512), padding=rng.choice([0, 3, 8]), high=_log(rng, 16, 16384),
                    block=rng.choice([8, 16, 32]), wide=rng.random() < 0.5)
        case["low"] = max(1, case["high"] // 16)
    return case


# -- sizes ----------------------------------------------------------------------------------------

def _mean_len(case):
    """The mean of a case's uniform lengths (tokens for audit and slots, blocks for the rest)."""
    return (case["low"] + case["high"]) / 2


def _tokens(case):
    long_rows = case["long_rows"]
    return (case["rows"] - long_rows) * _mean_len(case) + long_rows * case.get("long", 0)


def _width(case):
    if case["op"] in ("audit", "slots"):
        return -(-max(case["high"], case.get("long", 0)) // case["block"])
    return case["high"]


def _cells(case):
    if case["op"] == "shares":
        return case["cells"]
    return case["group"] * (case["kv_heads"] if case["heads_audited"] == "all" else 1)


def _record_bytes(case):
    return 2 * 4 * case["layers"] * case["rows"] * _width(case) * _cells(case)


def _cache_bytes(case):
    return 2 * _tokens(case) * case["kv_heads"] * case["dim"] * ELEMENT[case["dtype"]]


def work(case):
    op, rows, width = case["op"], case["rows"], _width(case)
    if op == "audit":
        tokens, cells = _tokens(case), _cells(case)
        heads = case["kv_heads"] if case["heads_audited"] == "all" else 1
        blocks = tokens / case["block"] + rows / 2
        query = rows * cells * case["dim"] * max(2, ELEMENT[case["dtype"]])
        layer = tokens * heads * case["dim"] * ELEMENT[case["dtype"]] + query + 2 * blocks * cells * 4
        total = case["layers"] * layer + blocks * 4 + rows * 8
        if case["shares"]:  # records read, shares written and read, keep written, table rows read and written
            total += case["layers"] * 2 * blocks * cells * 4 + rows * width * (4 + 1 + 8) + blocks * 4
        return {"bytes": total, "flops": 2.0 * case["layers"] * tokens * cells * case["dim"]}
    blocks = rows * _mean_len(case)
    if op == "shares":
        return {"bytes": case["layers"] * 2 * blocks * case["cells"] * 4 + rows * width * 4, "flops": 0}
    if op == "uniform":  # scores, the table row, the view row, the keep
        return {"bytes": blocks * 4 + rows * width * (4 + 4 + 1), "flops": 0}
    if op == "view":
        return {"bytes": rows * width * (4 + 4) + blocks, "flops": 0}
    if op in ("controller", "objective"):
        score = 8 if op == "objective" else 4 + (1 if case["released"] else 0)
        return {"bytes": blocks * score + rows * width, "flops": 0}
    slot = 8 if case["wide"] else 4
    blocks /= case["block"]  # about half the blocks stay
    return {"bytes": rows * _mean_len(case) * slot * 1.0 + blocks, "flops": 0}


def tolerance(case):
    # Audit records are float32 sums of dim products of the keys' own type, and of exponentials of them; the shares
    # are means of softmaxes over those.  Measured 0.8 to 1.2e-7 (records) and 0.4 to 0.9e-7 (shares) from 64 bits,
    # so two orders of summing differ by up to about 2.5e-7.  Everything else is whole numbers, and only a ranking
    # of computed shares can turn on their last bit (one swapped block shifts the view between the two).
    if case["op"] == "audit":
        return {"rel": 1e-6, "max": 2e-5, "differ": 0.005 if case["shares"] else 0.0}
    if case["op"] == "shares":
        return {"rel": 1e-6, "max": 2e-5}
    return "exact"


# -- inputs ---------------------------------------------------------------------------------------

def _lengths(case, rng):
    lens = rng.integers(case["low"], case["high"] + 1, size=case["rows"])
    if case.get("long_rows"):
        lens[rng.permutation(case["rows"])[: case["long_rows"]]] = case["long"]
    return lens.astype(np.int32)


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _shares(case, blocks, gen, dtype):
    """Dirichlet(0.1) scores of each row, zero past its blocks; ``paired`` gives the two blocks of a tile one
    value, as shares from an audit have."""
    rows, width = case["rows"], case["high"]
    g = torch._standard_gamma(torch.full((rows, width), 0.1, device="cuda"), generator=gen)
    if case["paired"]:
        g = g[:, ::2].repeat_interleave(2, dim=1)[:, :width]
    live = torch.arange(width, device="cuda")[None, :] < blocks[:, None]
    g = torch.where(live, g, torch.zeros((), device="cuda")).double()
    return (g / g.sum(dim=1, keepdim=True)).float().to(dtype)


class _Device:
    """Raw device memory of the plane as a tensor."""

    def __init__(self, address, shape):
        self.__cuda_array_interface__ = {"data": (address, False), "shape": shape, "typestr": "<f4", "version": 2}


def _audit_inputs(case, seed):
    rng, gen = np.random.default_rng(seed), _generator(seed)
    lens, width = _lengths(case, rng), _width(case)
    blocks = (lens + case["block"] - 1) // case["block"]
    used = int(blocks.sum())
    pool = used + used // 16 + 2
    ids = torch.randperm(pool - 1, generator=gen, device="cuda", dtype=torch.int64) + 1
    live = torch.arange(width)[None, :] < torch.from_numpy(blocks)[:, None]
    table = torch.zeros(case["rows"], width, dtype=torch.int32, device="cuda")
    table[live.cuda()] = ids[:used].to(torch.int32)
    shape = (pool, 2, case["block"], case["kv_heads"], case["dim"])
    dtype = DTYPES[case["dtype"]]
    caches = []
    for _ in range(min(2, case["layers"])):  # consecutive layers read different memory
        cache = torch.empty(shape, dtype=dtype, device="cuda")  # the values' half is never read
        step = max(1, (1 << 27) // (case["block"] * case["kv_heads"] * case["dim"]))
        for start in range(0, pool, step):
            part = torch.randn((min(step, pool - start), *shape[2:]), generator=gen, device="cuda")
            if case["dtype"] == "fp8":
                part = (part / K_SCALE).clamp_(-448.0, 448.0)
            cache[start : start + step, 0] = part.to(dtype)
        caches.append(cache)
    q_type = torch.bfloat16 if case["dtype"] == "fp8" else dtype
    queries = torch.randn(case["layers"], case["rows"], case["kv_heads"] * case["group"], case["dim"], generator=gen,
                          device="cuda").to(q_type)
    return {"lens_host": lens, "table": table, "lens": torch.from_numpy(lens).cuda(),
            "blocks": torch.from_numpy(blocks.astype(np.int32)).cuda(), "caches": caches, "queries": queries}


class _Audit:
    """A plane set up as an engine sets it up, and the step it runs."""

    def __init__(self, case, seed):
        self.case = case
        for name, value in _audit_inputs(case, seed).items():
            setattr(self, name, value)
        rows, width, layers = case["rows"], _width(case), case["layers"]
        self.plane = RecordingPlane(layers, rows, width, case["group"], case["block"], timer=case["timer"],
                                    kv_heads=case["kv_heads"] if case["heads_audited"] == "all" else None)
        self.cache_of = [self.caches[layer % len(self.caches)] for layer in range(layers)]
        self.plane.attach([c.data_ptr() for c in self.cache_of])
        self.plane.select(np.ones(rows, dtype=bool), np.arange(rows))
        self.plane.set(True)
        self.scale = case["dim"] ** -0.5
        self.k_scale = K_SCALE if case["dtype"] == "fp8" else 1.0
        self.records = torch.as_tensor(_Device(self.plane.lse_address, (2, layers, rows, width, _cells(case))),
                                       device="cuda")
        if case["shares"]:
            need = shares_workspace_bytes(rows, width, layers)
            self.workspace = torch.zeros(max(need, 1), dtype=torch.uint8, device="cuda")
        self.graph = None
        if case["mode"] == "graph":
            self.record()  # the layers are numbered as they first run
            self.step()
            torch.cuda.synchronize()
            self.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(self.graph):
                self.out = self.step()

    def record(self):
        for layer in range(self.case["layers"]):
            self.plane.record(f"layer.{layer}", self.table, self.lens, self.queries[layer], self.cache_of[layer],
                              self.scale)

    def step(self):
        case, plane = self.case, self.plane
        if case["mode"] == "layers":
            plane.plan(self.table, self.lens)
            entries = [plane.direct(layer, self.queries[layer], self.cache_of[layer][:, 0], self.scale,
                                    k_scale=self.k_scale) for layer in range(case["layers"])]
            plane.launch_layers(entries, self.cache_of[0][:, 0], self.queries[0], staged=False)
        else:
            self.record()
        out = {"records": self.records}
        if case["shares"]:
            out["shares"] = tile_shares(plane.lse_address, case["layers"], case["layers"], plane.rows, plane.width,
                                        plane.cells, None, self.blocks, TILE_BLOCKS, workspace=self.workspace)
            keep, summary, view, view_lens = uniform_view(out["shares"], self.blocks, self.table, self.lens,
                                                          case["block"], fraction=FRACTION, recent_blocks=RECENT)
            out.update(keep=keep, summary=summary, view=view, view_lens=view_lens)
        return out

    def run(self):
        if self.graph is None:
            return self.step()
        self.graph.replay()
        return self.out


def _share_inputs(case, seed):
    """Recorded planes: the two blocks of a tile hold its record, the cells past a row were never written."""
    rng, gen = np.random.default_rng(seed), _generator(seed)
    blocks = torch.from_numpy(_lengths(case, rng)).cuda()
    rows, width, cells = case["rows"], case["high"], case["cells"]
    tiles = -(-width // TILE_BLOCKS)
    planes = torch.empty(2, case["layers"], rows, width, cells, device="cuda")
    dead = torch.arange(width, device="cuda")[None, :] >= blocks[:, None]
    for layer in range(case["layers"]):
        m = 2.0 + torch.randn(rows, tiles, cells, generator=gen, device="cuda")
        total = 1.0 + 15.0 * torch.rand(rows, tiles, cells, generator=gen, device="cuda")
        for plane, value in enumerate((m, total)):
            value = value.repeat_interleave(TILE_BLOCKS, dim=1)[:, :width]
            planes[plane, layer] = torch.where(dead[:, :, None], torch.full((), float("nan"), device="cuda"), value)
    return planes, blocks


class _Shares:
    def __init__(self, case, seed):
        self.case = case
        self.planes, self.blocks = _share_inputs(case, seed)
        need = shares_workspace_bytes(case["rows"], case["high"], case["layers"])
        self.workspace = torch.zeros(max(need, 1), dtype=torch.uint8, device="cuda")
        self.out = torch.empty(case["rows"], case["high"], device="cuda")

    def run(self):
        case = self.case
        return tile_shares(self.planes.data_ptr(), case["layers"], case["layers"], case["rows"], case["high"],
                           case["cells"], None, self.blocks, TILE_BLOCKS, case["aggregate"], out=self.out,
                           workspace=self.workspace)


def _table(case, gen):
    return torch.randint(1, 2_000_000, (case["rows"], case["high"]), generator=gen, device="cuda", dtype=torch.int32)


def _fill(case, blocks, rng):
    """Token lengths whose last block is partly filled."""
    bs = case["block"]
    return ((blocks.astype(np.int64) - 1) * bs + rng.integers(1, bs + 1, size=case["rows"])).astype(np.int32)


class _Uniform:
    def __init__(self, case, seed):
        rng, gen = np.random.default_rng(seed), _generator(seed)
        self.case = case
        blocks = _lengths(case, rng)
        self.blocks = torch.from_numpy(blocks).cuda()
        self.lens = torch.from_numpy(_fill(case, blocks, rng)).cuda()
        self.scores = _shares(case, self.blocks, gen, torch.float32)
        self.table = _table(case, gen)

    def run(self):
        return uniform_view(self.scores, self.blocks, self.table, self.lens, self.case["block"], fraction=FRACTION,
                            recent_blocks=self.case["recent"])


class _View:
    def __init__(self, case, seed):
        rng, gen = np.random.default_rng(seed), _generator(seed)
        self.table = _table(case, gen)
        self.lens = torch.from_numpy(_fill(case, _lengths(case, rng), rng)).cuda()
        query = np.ones(case["rows"], dtype=np.int32)
        query[rng.permutation(case["rows"])[: case["prefill"]]] = 37
        self.query_lens = torch.from_numpy(query)
        self.view = DecodeView(case["rows"], case["high"], case["block"])
        self.view.write_row_controls(rng.random((case["rows"], case["high"])) < FRACTION)
        self.view.write_lease_deadline(time.monotonic_ns() + 3600 * 10**9)

    def run(self):
        return self.view.build(self.table, self.lens, self.query_lens)


class _Controller:
    def __init__(self, case, seed):
        rng, gen = np.random.default_rng(seed), _generator(seed)
        self.case = case
        rows, width = case["rows"], case["high"]
        blocks = _lengths(case, rng)
        self.lengths = torch.from_numpy(blocks).cuda()
        self.shares = _shares(case, self.lengths, gen, torch.float32)
        self.evidence = torch.ones(rows, dtype=torch.bool, device="cuda")
        self.audited = torch.from_numpy(np.maximum(1, blocks - rng.integers(0, 4, size=rows)).astype(np.int32)).cuda()
        # one block in twenty was released: never the first, which every view reads
        released = rng.random((rows, width)) < 0.05
        released[:, 0] = False
        self.released = torch.from_numpy(released).cuda() if case["released"] else None
        self.weights = torch.from_numpy(rng.uniform(0.5, 2.0, size=rows)).cuda() if case["weights"] else None
        self.out = torch.empty(rows, width, dtype=torch.uint8, device="cuda")
        need = keep_rows_workspace_bytes(case["objective"], rows, width)
        self.workspace = torch.empty(need, dtype=torch.uint8, device="cuda")

    def run(self):
        return keep_rows(self.shares, self.lengths, self.evidence, FRACTION, objective=self.case["objective"],
                         recent_blocks=RECENT, audited_blocks=self.audited, released=self.released,
                         weights=self.weights, out=self.out, workspace=self.workspace)


class _Objective:
    def __init__(self, case, seed):
        rng, gen = np.random.default_rng(seed), _generator(seed)
        rows, width = case["rows"], case["high"]
        blocks = _lengths(case, rng)
        self.blocks = torch.from_numpy(blocks).cuda()
        self.scores = _shares(case, self.blocks, gen, torch.float64)
        total = int(blocks.sum())
        self.budget = max(math.ceil(FRACTION * total), int(np.minimum(blocks, 2).sum()))
        self.out = torch.empty(rows, width, dtype=torch.uint8, device="cuda")
        if case["objective"] == "sum":
            weights = torch.from_numpy(rng.uniform(0.5, 2.0, size=rows)).cuda() if case["weights"] else None
            self.call, need, self.more = sum_keep, sum_workspace_bytes(rows), {"weights": weights}
        else:
            self.call, need, self.more = maxmin_keep, maxmin_workspace_bytes(rows, width), {}
        self.workspace = torch.empty(need, dtype=torch.uint8, device="cuda")

    def run(self):
        return self.call(self.scores, self.blocks, budget=self.budget, out=self.out, workspace=self.workspace,
                         **self.more)


class _Slots:
    def __init__(self, case, seed):
        rng, gen = np.random.default_rng(seed), _generator(seed)
        self.case = case
        lens = np.concatenate([_lengths(case, rng), np.ones(case["padding"], np.int32)])
        self.entries, self.all_rows = int(lens.sum()), len(lens)
        self.engine_indptr = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)).cuda()
        slot = torch.int64 if case["wide"] else torch.int32
        room = self.all_rows * case["high"]  # the engine's buffer holds the longest batch
        self.engine_slots = torch.zeros(room, dtype=slot, device="cuda")
        self.engine_slots[: self.entries] = torch.randperm(self.entries, generator=gen, device="cuda").to(slot)
        self.indptr, self.slots = self.engine_indptr.clone(), self.engine_slots.clone()
        width = _width(case)
        self.keep = torch.from_numpy(rng.random((case["rows"], width)) < FRACTION).cuda()
        self.compactor = SlotCompactor(width, case["block"], torch.device("cuda"))

    def run(self):
        # the engine writes its list anew each step, and the compaction rewrites it in place
        self.indptr.copy_(self.engine_indptr)
        self.slots[: self.entries].copy_(self.engine_slots[: self.entries])
        lens = self.compactor.compact(self.indptr, self.slots, self.keep, None, True, self.case["rows"],
                                      self.all_rows, self.entries)
        return {"indptr": self.indptr, "slots": self.slots, "lens": lens}


_STATES = {"audit": _Audit, "shares": _Shares, "uniform": _Uniform, "view": _View, "controller": _Controller,
           "objective": _Objective, "slots": _Slots}


def prepare(case, seed):
    return _STATES[case["op"]](case, seed)


def run(state):
    return state.run()


# -- the same in 64 bits --------------------------------------------------------------------------

def _exact_records(case, seed):
    inputs = _audit_inputs(case, seed)
    rows, width, block, dim, group = case["rows"], _width(case), case["block"], case["dim"], case["group"]
    cells, tile = _cells(case), block * TILE_BLOCKS
    scale = dim ** -0.5 * (K_SCALE if case["dtype"] == "fp8" else 1.0)
    planes = torch.full((2, case["layers"], rows, width, cells), float("nan"), dtype=torch.float64, device="cuda")
    for layer in range(case["layers"]):
        keys = inputs["caches"][layer % len(inputs["caches"])][:, 0]
        heads = range(case["kv_heads"]) if case["heads_audited"] == "all" else [layer % case["kv_heads"]]
        for row, length in enumerate(inputs["lens_host"].tolist()):
            n = -(-length // block)
            tiles = -(-n // TILE_BLOCKS)
            ids = inputs["table"][row, :n].long()
            for i, head in enumerate(heads):
                query = inputs["queries"][layer, row, head * group : (head + 1) * group].double()
                k = keys[ids, :, head].reshape(n * block, dim)[:length].double()
                scores = torch.full((tiles * tile, group), float("-inf"), dtype=torch.float64, device="cuda")
                scores[:length] = (k @ query.t().contiguous()) * scale
                scores = scores.reshape(tiles, tile, group)
                m = scores.amax(dim=1)
                total = (scores - m[:, None]).exp().sum(dim=1)
                for plane, value in enumerate((m, total)):
                    planes[plane, layer, row, :n, i * group : (i + 1) * group] = (
                        value.repeat_interleave(TILE_BLOCKS, dim=0)[:n])
    return planes, inputs["blocks"]


def _exact_shares(planes, blocks, aggregate):
    """Each (layer, query row)'s softmax over its row's blocks, a lone last block with its tile's whole mass,
    then their mean or the renormalised maximum."""
    layers, rows, width, cells = planes.shape[1:]
    position = torch.arange(width, device="cuda")
    out = torch.zeros(rows, width, dtype=torch.float64, device="cuda")
    for row, n in enumerate(blocks.tolist()):
        u = planes[0, :, row, :n].double() + planes[1, :, row, :n].double().log()
        if n % TILE_BLOCKS:
            u = u + torch.where(position[:n] >= n - n % TILE_BLOCKS, math.log(TILE_BLOCKS / (n % TILE_BLOCKS)), 0.0)[
                None, :, None]
        share = torch.softmax(u, dim=1)
        if aggregate == "mean":
            out[row, :n] = share.mean(dim=(0, 2))
        else:
            peak = share.amax(dim=(0, 2))
            out[row, :n] = peak / peak.sum()
    return out


def exact(case, seed):
    if case["op"] == "audit":
        planes, blocks = _exact_records(case, seed)
        out = {"records": planes}
        if case["shares"]:
            out.update(shares=_exact_shares(planes, blocks, "mean"), keep=None, summary=None, view=None, view_lens=None)
        return out
    if case["op"] == "shares":
        planes, blocks = _share_inputs(case, seed)
        return _exact_shares(planes, blocks, case["aggregate"])
    return None  # whole numbers
