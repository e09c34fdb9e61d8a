"""GPU parity of the prefill block-score kernel (tierkv_prefill_block_mass)
against the float64 oracle (oracle.policy.prefill_block_mass): per-sequence
mean causal attention probability per block over heads and queries, the
quantity compute_block_scores (tierkv_policy.py:1380-1389) takes from the
eager prefill attention.  fp16 / bf16 inputs are exact in the oracle; the
kernel accumulates q . k in fp32 on MFMA and uses exp2f, so the result is
compared at 1e-4 relative.  Covers ragged prompt lengths (not multiples of
16 or 64), GQA groups 1 / 4 / 8, head_dim 64 / 128, block sizes 16 / 32,
HF's transposed projection layout, bf16, and agreement with the tier
engine's compute_block_scores on materialised weights."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle.policy import prefill_block_mass as oracle_mass
from paged_tierkv_amd import _lib, kernels, tierkv_policy as tp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Hkv,T,D,bs,dtype", [
    (1, 32, 8, 130, 128, 16, torch.float16),
    (2, 8, 8, 77, 64, 16, torch.float16),
    (2, 16, 2, 200, 128, 32, torch.float16),
    (1, 32, 4, 64, 128, 16, torch.bfloat16),
    (3, 4, 1, 1, 64, 16, torch.float16),
    (1, 16, 4, 513, 128, 16, torch.float16),
    (1, 12, 2, 300, 128, 16, torch.float16),     # GQA group 6: the guarded 8-head variant
    (2, 4, 2, 97, 64, 32, torch.bfloat16),       # GQA group 2: the guarded 4-head variant
])
def test_prefill_block_mass_matches_oracle(device, B, H, Hkv, T, D, bs, dtype):
    print(f"[prefill] B={B} H={H} Hkv={Hkv} T={T} D={D} bs={bs} {dtype}", flush=True)
    g = torch.Generator().manual_seed(T * 7 + H)
    q = (torch.randn((B, H, T, D), generator=g) * 1.5).to(dtype)
    k = (torch.randn((B, Hkv, T, D), generator=g) * 1.5).to(dtype)
    scaling = D ** -0.5
    got = kernels.prefill_block_mass(q.to(device), k.to(device), bs, scaling).cpu().numpy()
    want = oracle_mass(q.float().numpy(), k.float().numpy(), scaling, bs)
    np.testing.assert_allclose(got, want, rtol=1e-4, atol=1e-9)


def test_prefill_block_mass_hf_layout(device):
    """q / k as HF produces them: [B, T, H, D] storage viewed as [B, H, T, D]."""
    B, H, Hkv, T, D = 2, 32, 8, 150, 128
    g = torch.Generator().manual_seed(3)
    q = torch.randn((B, T, H, D), generator=g).half().to(device).transpose(1, 2)
    k = torch.randn((B, T, Hkv, D), generator=g).half().to(device).transpose(1, 2)
    got = kernels.prefill_block_mass(q, k, 16, D ** -0.5).cpu().numpy()
    want = oracle_mass(q.float().cpu().numpy(), k.float().cpu().numpy(), D ** -0.5, 16)
    np.testing.assert_allclose(got, want, rtol=1e-4, atol=1e-9)


def test_prefill_block_mass_agrees_with_compute_block_scores(device):
    """One sequence: the kernel equals the tier engine's compute_block_scores
    on the materialised fp32 causal probabilities (block-mass kernel)."""
    H, Hkv, T, D = 8, 2, 96, 64
    g = torch.Generator().manual_seed(9)
    q = torch.randn((1, H, T, D), generator=g).half().to(device)
    k = torch.randn((1, Hkv, T, D), generator=g).half().to(device)
    kk = k.float().repeat_interleave(H // Hkv, dim=1)
    logits = (q.float() @ kk.transpose(2, 3).contiguous()) * D ** -0.5
    logits = logits.masked_fill(~torch.tril(torch.ones(T, T, dtype=torch.bool, device=device)), float("-inf"))
    probs = torch.softmax(logits, dim=-1)
    engine = tp.TierKVPolicyEngine(block_size=16, block_manager=None)
    ref = engine.compute_block_scores(probs)
    got = kernels.prefill_block_mass(q, k, 16, D ** -0.5)[0]
    torch.testing.assert_close(got, ref, rtol=1e-4, atol=1e-8)


@pytest.mark.parametrize("B,H,Hkv,T,D,dtype", [
    (1, 1, 1, 2048, 64, torch.float16),      # one head per workgroup; the last length with four waves
    (1, 2, 1, 2049, 64, torch.bfloat16),     # two heads; the first with eight
    (1, 3, 1, 1000, 128, torch.float16),     # an idle slot
    (1, 5, 1, 530, 128, torch.bfloat16),     # two head sets, the second with three idle slots
    (1, 2, 2, 4096, 64, torch.float16),      # the last one-pass length
    (1, 2, 1, 4100, 64, torch.float16),      # two passes, partial last tile
    (128, 5, 1, 250, 64, torch.float16),     # 2048 rows: the last launch with head sets side by side
    (129, 5, 1, 250, 64, torch.bfloat16),    # the first with one after the other
    (3, 8, 2, 1001, 64, torch.float16),      # six pairs dealt together
    (1, 18, 18, 2048, 128, torch.float16),   # 18 pairs dealt four at a time, the last two by themselves
    (9, 1, 1, 65, 128, torch.float16),       # pairs not a multiple of the XCDs, one row past a 64-query block
])
def test_prefill_block_mass_edges(device, B, H, Hkv, T, D, dtype):
    print(f"[prefill-edge] B={B} H={H} Hkv={Hkv} T={T} D={D} {dtype}", flush=True)
    g = torch.Generator().manual_seed(T + H)
    q = torch.randn((B, H, T, D), generator=g).to(dtype)
    k = torch.randn((B, Hkv, T, D), generator=g).to(dtype)
    got = kernels.prefill_block_mass(q.to(device), k.to(device), 16, D ** -0.5).cpu().numpy()
    want = oracle_mass(q.float().numpy(), k.float().numpy(), D ** -0.5, 16)
    np.testing.assert_allclose(got, want, rtol=1e-4, atol=1e-9)


@pytest.mark.parametrize("T,growth", [(700, 30.0), (700, -30.0), (4200, 30.0)])
def test_prefill_block_mass_growing_logits(device, T, growth):
    """Logits that grow along the prompt by far more than 2^64 in probability
    (the rows' references are raised and their earlier sums rescaled), or
    fall (later sums are tiny).  Logits reach about |growth| * 10 in log2
    units: a few fp32 roundings of 300 * 2^-24 in the exponent are 1e-4
    relative, so the bound is 5e-4."""
    g = torch.Generator().manual_seed(5)
    ramp = torch.linspace(0.1, 1.0, T) if growth > 0 else torch.linspace(1.0, 0.1, T)
    q = torch.randn((1, 4, T, 64), generator=g).half()
    k = (torch.randn((1, 1, T, 64), generator=g) * (ramp * abs(growth))[None, None, :, None]).half()
    got = kernels.prefill_block_mass(q.to(device), k.to(device), 16, 64 ** -0.5).cpu().numpy()
    want = oracle_mass(q.float().numpy(), k.float().numpy(), 64 ** -0.5, 16)
    np.testing.assert_allclose(got, want, rtol=5e-4, atol=1e-9)


def _mass_in(q, k, scaling, nbytes):
    """Block masses (16-token blocks) in a workspace of nbytes of a larger buffer."""
    (B, H, T, D), Hkv = q.shape, k.shape[1]
    out = torch.full((B, -(-T // 16)), -1.0, dtype=torch.float32, device=q.device)
    ws = torch.full((nbytes + 4096,), 255, dtype=torch.uint8, device=q.device)   # NaN where it is read unwritten
    rc = _lib.lib().tierkv_prefill_block_mass(
        _lib.ptr(q), *q.stride()[:3], _lib.ptr(k), *k.stride()[:3],
        _lib.DTYPE_BF16 if q.dtype == torch.bfloat16 else _lib.DTYPE_F16, _lib.ptr(out), B, H, Hkv, T, D, 16, scaling,
        _lib.ptr(ws), nbytes, _lib.stream_of(q.device))
    _lib.check(rc, "tierkv_prefill_block_mass")
    torch.cuda.synchronize()
    assert bool((ws[nbytes:] == 255).all()), "wrote past the workspace"
    return out


@pytest.mark.parametrize("G,T,D,dtype,growth", [
    (5, 2100, 64, torch.float16, 0.0),       # eight waves, the second head set with three idle slots
    (8, 2100, 128, torch.bfloat16, 0.0),
    (6, 4090, 128, torch.float16, 0.0),      # the last one-pass length in tiles, a partial last tile
    (5, 4100, 128, torch.bfloat16, 0.0),     # two passes
    (8, 4100, 64, torch.float16, 0.0),
    (7, 2500, 64, torch.float16, 30.0),      # references raised with eight waves and two head sets
    (7, 4300, 64, torch.float16, 30.0),
])
def test_prefill_head_sets_beyond_2048_tokens(device, G, T, D, dtype, growth):
    """Groups above four heads in the eight-wave and the two-pass kernels, the
    two head sets one after the other and side by side (the two workspace
    sizes), and through the wrapper, which takes the second."""
    print(f"[prefill-sets] G={G} T={T} D={D} {dtype} growth={growth}", flush=True)
    g = torch.Generator().manual_seed(T + G)
    q = torch.randn((1, G, T, D), generator=g).to(dtype)
    k = torch.randn((1, 1, T, D), generator=g)
    if growth:
        k = k * (torch.linspace(0.1, 1.0, T) * growth)[None, None, :, None]
    k = k.to(dtype)
    want = oracle_mass(q.float().numpy(), k.float().numpy(), D ** -0.5, 16)
    lib = _lib.lib()
    least = lib.tierkv_prefill_block_mass_workspace_bytes(1, 1, T)
    full = lib.tierkv_prefill_block_mass_full_workspace_bytes(1, G, 1, T)
    assert full == 2 * least
    qd, kd = q.to(device), k.to(device)
    one, two = (_mass_in(qd, kd, D ** -0.5, n) for n in (least, full))
    # Logits of several hundred carry a few roundings of 300 * 2^-24 in the exponent.
    tol = 5e-4 if growth else 1e-4
    for got in (one, two):
        np.testing.assert_allclose(got.cpu().numpy(), want, rtol=tol, atol=1e-9)
    assert torch.equal(kernels.prefill_block_mass(qd, kd, 16, D ** -0.5), two)


def test_prefill_scores_do_not_depend_on_earlier_calls(device):
    """Launches too long for head sets side by side give the same bits before
    and after a call that made the shared scratch larger."""
    g = torch.Generator().manual_seed(2)
    q = torch.randn((129, 5, 250, 64), generator=g).half().to(device)
    k = torch.randn((129, 1, 250, 64), generator=g).half().to(device)
    lib = _lib.lib()
    least = lib.tierkv_prefill_block_mass_workspace_bytes(129, 1, 250)
    assert lib.tierkv_prefill_block_mass_full_workspace_bytes(129, 5, 1, 250) == least
    want = _mass_in(q, k, 0.125, least)
    kernels.prefill_block_mass(torch.cat([q] * 3), torch.cat([k] * 3), 16, 0.125)
    assert torch.equal(kernels.prefill_block_mass(q, k, 16, 0.125), want)
    assert torch.equal(_mass_in(q, k, 0.125, 4 * least), want)
