"""Pins the CPU model of the batched runtime (oracle/runtime.py) against the
reference runtime's own recorded trajectories (tests/golden/runtime_*.npz,
written by the reference TieredKVRuntime, tierkv_policy.py:1534-1912).

One oracle instance per layer (the reference serves one sequence per
layer); prefill, appends and policy ticks are replayed with the recorded
inputs.  After every recorded operation the oracle's per-block tier states
and lengths must equal the reference's BlockManager states and length table
exactly.  Ticks take the recorded block scores directly (the block mass of
probability sums is pinned on its own by closed forms).

Slot ids of a batch follow an allocation order of their own (the reference has
no batch); they are checked by invariants: every resident block owns a
distinct slot of its tier, and free stacks plus owned slots cover every slot
exactly once."""

from __future__ import annotations

import json
import os

import numpy as np
import pytest
import torch

from oracle.runtime import BatchedRuntimeOracle
from paged_tierkv_amd.runtime import LayerStorage, _prefill_tiers, _score_rows, prefill_states, recency_scores

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
CASES = ["runtime_compact_hot_warm", "runtime_compact_hot_warm_cold", "runtime_dense_hot_warm",
         "runtime_dense_hot_warm_cold"]
HOT_SLOTS = WARM_SLOTS = 64


def _invariants(orc: BatchedRuntimeOracle, where: str) -> None:
    n = int(orc.nb[0])
    for tier, free, cap in ((0, orc.hot_free, HOT_SLOTS), (1, orc.warm_free, WARM_SLOTS)):
        owned = [int(orc.table[0, i]) for i in range(n) if orc.states[0, i] == tier]
        assert len(set(owned)) == len(owned), f"{where}: tier {tier} slot shared"
        assert sorted(owned + list(free)) == list(range(cap)), f"{where}: tier {tier} slots lost or duplicated"
    cold = [i for i in range(n) if orc.states[0, i] == 2]
    assert all(orc.table[0, i] == -1 for i in cold), f"{where}: COLD block keeps a slot"


@pytest.mark.parametrize("name", CASES)
def test_oracle_runtime_follows_reference_trajectory(name):
    fx = np.load(os.path.join(GOLDEN, name + ".npz"))
    cfg = json.loads(str(fx["config"]))
    ops = json.loads(str(fx["ops"]))
    kv_all, scores_all = fx["kv"], fx["scores"]
    bs, hot_b, warm_b = cfg["block_size"], cfg["hot_budget"], cfg["warm_budget"]
    max_blocks = -(-cfg["max_seq_len"] // bs)
    mode = cfg["mode"]
    orcs = [BatchedRuntimeOracle(1, cfg["kv_heads"], cfg["head_dim"], bs, max_blocks, HOT_SLOTS, WARM_SLOTS,
                                 policy_mode=mode, warm_format="ref_u8") for _ in range(cfg["num_layers"])]
    len_row = 3 if cfg["layout"] == "compact" else 2
    checked = 0
    for op in ops:
        kind, where = op["op"], f"{name} op {op['i']} ({op['op']})"
        if kind == "prefill":
            off, t = op["kv"]
            k, v = kv_all[0, :, off:off + t][None], kv_all[1, :, off:off + t][None]
            so, sn = op["scores"]
            orcs[op["layer"]].prefill(k, v, scores_all[so:so + sn][None], hot_b, warm_b)
        elif kind == "append":
            off, t = op["kv"]
            for j in range(t):
                orcs[op["layer"]].append(kv_all[0, :, off + j:off + j + 1][None], kv_all[1, :, off + j:off + j + 1][None])
        elif kind == "policy":
            orc = orcs[op["layer"]]
            n = int(orc.nb[0])
            so, sn = op["scores"]
            assert sn == n, where
            orc.tick(None, hot_b, warm_b, scores=scores_all[so:so + sn].reshape(1, n))
        if "snap" in op and op.get("layer") is not None and kind in ("prefill", "append", "policy"):
            layer = op["layer"]
            orc = orcs[layer]
            n = int(orc.nb[0])
            want_states = op["snap"]["bm"][layer][1]
            assert orc.states[0, :n].tolist() == want_states, where
            want_len = op["snap"]["tables"][len_row][layer][:n]
            assert orc.lengths[0, :n].tolist() == want_len, where
            _invariants(orc, where)
            checked += 1
    assert checked > 60


@pytest.mark.parametrize("mode", ["hot_warm", "hot_warm_cold"])
@pytest.mark.parametrize("n", [0, 1, 2, 3, 4, 17])
def test_prefill_tiers_of_many_rows(n, mode):
    # Every row at once equals the rows one by one: ties, signed zeros,
    # infinities, a NaN, and budgets from below zero to above the row.
    rng = np.random.default_rng(n)
    rows = np.concatenate([rng.random((4, n)), rng.choice([0.0, -0.0, 1.0, np.inf, -np.inf], (6, n)),
                           np.zeros((1, n))])
    nan = rows.copy()
    nan[0, n // 2: n // 2 + 1] = np.nan
    for scores in (rows, nan):
        for hot in (-1, 0, 2, 3, 5, n, n + 3):
            for warm in (-1, 0, 1, 4, n + 1):
                got = _prefill_tiers(scores, hot, warm, mode)
                assert got.shape == scores.shape and got.dtype == np.int32
                assert got.tolist() == [prefill_states(n, r, hot, warm, mode) for r in scores], (hot, warm)


@pytest.mark.parametrize("make", [
    lambda x: x.tolist(), lambda x: x, lambda x: x.numpy(), lambda x: x.double(), lambda x: x.bfloat16(),
    lambda x: x.clone().requires_grad_(), lambda x: (x.clone().requires_grad_() * 2.0) / 2.0,
    lambda x: x.t().contiguous().t() if x.ndim == 2 else x[:, None].expand(-1, 2).contiguous()[:, 0],
], ids=["list", "tensor", "numpy", "double", "bf16", "leaf", "graph", "strided"])
def test_prefill_scores_of_every_kind(make):
    # Scores come as lists, arrays or tensors, of a graph or not, shared by
    # the sequences or one row each; the last block's may be missing.
    torch.manual_seed(0)
    n, batch = 7, 3
    for shape in ((n,), (n - 1,), (n + 2,), (batch, n), (batch + 1, n - 1)):
        given = make(torch.rand(shape))
        want = torch.as_tensor(given, dtype=torch.float32).tolist()
        got = _score_rows(given, batch, n)
        rows = [want] if len(shape) == 1 else want[:batch]
        assert got.shape == (len(rows), n) and got.dtype == np.float64
        for g, w in zip(got.tolist(), rows):
            assert g == (w + [0.0])[:n]
    assert _score_rows(None, batch, n).tolist() == [recency_scores(n)]
    for short in (torch.rand(n - 2), torch.rand(batch, n - 2), torch.rand(batch - 1, n)):
        with pytest.raises(IndexError):
            _score_rows(short, batch, n)


def test_layer_tensors_replaced_by_the_caller_are_loaded():
    # A prefill fills the tensors the layer holds, whether they are still the
    # views of its one buffer or the caller's own (a restored table).
    views = {"table": (0, 6, (2, 3)), "states": (64, 6, (2, 3)), "lengths": (128, 6, (2, 3)), "nblocks": (192, 2, (2,)),
             "open": (256, 2, (2,)), "hot_free": (320, 4, (4,)), "warm_free": (384, 5, (5,)), "ctl": (448, 4, (4,))}
    flat = torch.arange(512, dtype=torch.int32)
    for replaced in ((), ("table",), ("ctl", "nblocks"), tuple(views)):
        meta = torch.zeros(512, dtype=torch.int32)
        parts = {n: meta[at: at + size].view(shape) for n, (at, size, shape) in views.items()}
        st = LayerStorage(*[None] * 8, meta=meta, **parts)
        for name in replaced:
            setattr(st, name, torch.zeros_like(parts[name]))
        st.load(flat, views)
        for name, (at, size, shape) in views.items():
            assert torch.equal(getattr(st, name), flat[at: at + size].view(shape)), (replaced, name)
    bare = LayerStorage(*[None] * 8, **{n: torch.zeros(shape, dtype=torch.int32) for n, (_, _, shape) in views.items()})
    bare.load(flat, views)
    assert torch.equal(bare.warm_free, flat[384:389])
