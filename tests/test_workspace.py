"""Decode-workspace ownership rules, checked on the CPU (no kernel launches).

* A fixed workspace never replaces its buffer: a launch that needs more
  raises, so a captured graph can never replay on a released buffer.
* A growable workspace carries its error flags into the new buffer.
* A workspace first bound under stream capture becomes fixed, so a later,
  larger eager launch cannot free memory a captured graph replays on.
* A workspace that cannot be replaced serves every launch the library accepts
  it for, also where the launch's free plan would use more.
* The batched runtime sizes its fixed workspace once, for ``max_blocks``
  with score sums; every smaller launch of the same geometry (any block
  count, with or without scores) fits in it, so nothing it launches can ask
  for more.
"""

from __future__ import annotations

import pytest
import torch

from paged_tierkv_amd import _lib
from paged_tierkv_amd.tierkv_hip import DecodeWorkspace, launch_bytes


def test_fixed_workspace_never_replaces_its_buffer():
    ws = DecodeWorkspace("cpu", 4096, growable=False)
    before = ws.data_ptr()
    ws.reserve(4096)
    ws.reserve(100)
    assert ws.data_ptr() == before
    with pytest.raises(RuntimeError, match="fixed workspace"):
        ws.reserve(4097)
    assert ws.data_ptr() == before and ws.nbytes == 4096


def test_growable_workspace_keeps_error_flags():
    ws = DecodeWorkspace("cpu", 256)
    ws.buf[:4].view(torch.int32).fill_(2)
    ws.reserve(1 << 16)
    assert ws.nbytes == 1 << 16
    assert int(ws.buf[:4].view(torch.int32).item()) == 2
    assert int(ws.buf[4:].abs().sum()) == 0
    assert ws.error_word() == 2
    assert ws.error_word() == 0


def test_capture_pins_a_growable_workspace(monkeypatch):
    ws = DecodeWorkspace("cpu", 4096)
    assert ws.growable
    monkeypatch.setattr(DecodeWorkspace, "_capturing", lambda self: True)
    ws.reserve(1024)                    # bound under capture: fits, and is fixed from now on
    assert not ws.growable
    with pytest.raises(RuntimeError, match="during HIP graph capture"):
        ws.reserve(8192)
    monkeypatch.setattr(DecodeWorkspace, "_capturing", lambda self: False)
    before = ws.data_ptr()
    with pytest.raises(RuntimeError, match="fixed workspace"):
        ws.reserve(8192)                # eager growth after the capture is refused
    assert ws.data_ptr() == before and ws.nbytes == 4096


@pytest.mark.parametrize("batch,heads,kv,dim,max_blocks", [
    (16, 32, 8, 128, 144),     # C5: Llama-3-8B, 2048 + 256 tokens
    (1, 32, 4, 64, 33),        # TinyLlama shape, batch 1
    (4, 32, 8, 128, 2048),     # C4 rows
    (3, 48, 3, 128, 700),      # GQA 16, four waves per workgroup
])
def test_runtime_workspace_covers_every_launch(batch, heads, kv, dim, max_blocks):
    full = DecodeWorkspace.bytes_for(batch, heads, kv, max_blocks, dim, return_scores=True)
    for nb in range(1, max_blocks + 1):
        for scores in (False, True):
            assert DecodeWorkspace.bytes_for(batch, heads, kv, nb, dim, return_scores=scores) <= full, (nb, scores)


def test_graph_runner_reserves_before_capture(monkeypatch):
    """DecodeGraphRunner reserves the runtime's decode workspace in its
    constructor, before any step could be captured."""
    from paged_tierkv_amd import hf_llama

    calls = []

    class Rt:
        is_batched = True
        batch = 2
        device = torch.device("cpu")
        fixed_launch_bound = False

        def reserve_decode_workspace(self, heads):
            calls.append(heads)

    class Cfg:
        num_attention_heads = 32

    class Model:
        config = Cfg()

    runner = hf_llama.DecodeGraphRunner(Model(), Rt())
    assert calls == [32]
    assert runner.rt.fixed_launch_bound


@pytest.mark.parametrize("batch,heads,kv,dim", [(1, 32, 4, 64), (12, 32, 8, 128), (31, 32, 8, 128), (3, 16, 16, 64),
                                                (2, 64, 4, 128), (200, 8, 8, 128)])
@pytest.mark.parametrize("scores", [False, True])
def test_reported_bytes_cover_every_shorter_row(batch, heads, kv, dim, scores):
    """The split count a launch takes is not monotonic in its row length; the
    reported workspace is, so one sized for the longest row fits every launch."""
    last = 0
    for nb in list(range(1, 140)) + [143, 144, 255, 256, 257, 400, 511, 512, 768, 1024, 1025, 2048, 2600, 5000]:
        need = DecodeWorkspace.bytes_for(batch, heads, kv, nb, dim, return_scores=scores)
        assert need >= last, (nb, need, last)
        last = need


def _plain_rule_bytes(batch, heads, kv, nb, dim, scores, splits=0):
    """Workspace of the plain split rule: about 2048 waves on the chip, at
    least four tiles per wave, rows under 12 tiles per wave whole."""
    units, nw = batch * kv, 8 if heads // kv <= 8 else 4
    if not splits:
        splits = min(max(1, -(-2048 // (units * nw))), max(1, nb // (4 * nw)))
        if nb < 12 * nw:
            splits = 1
    splits = max(1, min(max(splits, -(-nb // 511)), nb))
    up = lambda x: -(-x // 256) * 256
    partials = up(batch * heads * splits * dim * 4) + up(batch * heads * splits * 2 * 4) if splits > 1 else 0
    return 256 + (1 << 16) * 4 + partials + (up(batch * heads * nb * 2 * 4) if scores else 0)


@pytest.mark.parametrize("heads,kv,dim", [(32, 8, 128), (32, 4, 64), (16, 16, 64), (64, 4, 128)])
def test_least_bytes_are_the_plain_split_rules(heads, kv, dim):
    lib = _lib.lib()
    for batch in (1, 2, 7, 31, 32, 33, 40, 64, 65, 128):
        for nb in (1, 9, 33, 95, 96, 144, 256, 511, 512, 1100, 2048):
            for scores in (0, 1):
                for splits in (0, 1, 3, 8):
                    full, least = launch_bytes(lib, batch, heads, kv, nb, 16, dim, scores, splits)
                    assert least == _plain_rule_bytes(batch, heads, kv, nb, dim, scores, splits), (batch, nb, splits)
                    assert least <= full
    assert lib.tierkv_decode_workspace_least_bytes(0, 32, 8, 256, 16, 128, 0, 0) < 0


@pytest.mark.parametrize("batch", [32, 33, 40, 48, 63, 64])
def test_fixed_workspace_serves_smaller_batches(batch, monkeypatch):
    """A workspace sized for a large batch holds no split partials, where a
    smaller batch's free plan would split: it is served unsplit, eagerly in a
    fixed workspace and under capture in a growable one."""
    shape = (batch, 32, 8, 256, 16, 128, 0, 0)
    full, least = launch_bytes(_lib.lib(), *shape)
    ws = DecodeWorkspace.for_shape("cpu", 128, 32, 8, 256, 128, return_scores=False)
    assert least <= ws.nbytes < full
    before = ws.data_ptr()
    ws.reserve(full, least)
    assert ws.data_ptr() == before and ws.nbytes < full
    warmed = DecodeWorkspace("cpu")
    warmed.reserve(*launch_bytes(_lib.lib(), 128, *shape[1:]))
    before = warmed.data_ptr()
    monkeypatch.setattr(DecodeWorkspace, "_capturing", lambda self: True)
    warmed.reserve(full, least)
    assert warmed.data_ptr() == before and not warmed.growable
    monkeypatch.setattr(DecodeWorkspace, "_capturing", lambda self: False)
    warmed.reserve(full, least)         # fixed by the capture
    assert warmed.data_ptr() == before
    grown = DecodeWorkspace("cpu", least)
    grown.reserve(full, least)          # growable: room for the free plan
    assert grown.nbytes == full


def test_workspace_below_the_least_bytes_is_refused():
    full, least = launch_bytes(_lib.lib(), 16, 32, 8, 256, 16, 128, 1, 0)
    assert least < full
    DecodeWorkspace("cpu", least, growable=False).reserve(full, least)
    with pytest.raises(RuntimeError, match=f"needs {least}:"):
        DecodeWorkspace("cpu", least - 1, growable=False).reserve(full, least)
