"""Scratch memory when several host threads run modules on one stream: no call may find its scratch handed to another call
between its own launches.  The library is a stand-in here (two "launches" with a pause between them on host memory), so what
is tested is who gets which memory, and when."""
import threading
import time

import pytest
import torch

from sensenova_u1_amd import GGUFLinear, GGUFParameter, modality, ops


@pytest.fixture
def host_scratch(monkeypatch):
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(ops, "_stream", lambda dev: 7)
    monkeypatch.setattr(ops, "_workspaces", {})


def _in_threads(n, fn):
    errors = []

    def body(i):
        try:
            fn(i)
        except BaseException as e:   # (reported in the test's own thread)
            errors.append(e)
    threads = [threading.Thread(target=body, args=(i,)) for i in range(n)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


def test_a_short_prompt_s_gate_outputs_are_the_call_s_own(host_scratch, monkeypatch):
    """17 .. 64 rows: the gate projection is written by one launch and read by the next."""
    m, n, k = 40, 64, 256
    monkeypatch.setattr(modality, "_gated_tile_route", lambda *a: True)
    monkeypatch.setattr(GGUFLinear, "_checked_rows", lambda self, x, *o: x)
    both = threading.Barrier(4)

    def two_launches(x2d, gate, up, qt, h2d, ws, numerics, nbytes=None):
        scratch = ws.view(-1)[:2 * m * n].view(torch.bfloat16).view(m, n)
        scratch.copy_(x2d[:, :n])           # "gate"
        both.wait(20)                       # every thread is between its two launches now
        h2d.copy_(scratch)                  # "up, with the product"

    monkeypatch.setattr(ops, "gate_up_silu_ws_into", two_launches)
    bs, ts = ops.GGML_QUANT_SIZES[ops.Q8_0]
    mods = []
    for _ in range(2):
        lin = GGUFLinear(k, n, bias=False, compute_dtype=torch.bfloat16, device="meta")
        lin.weight = GGUFParameter(torch.zeros((n, k // bs * ts), dtype=torch.uint8), quant_type=ops.Q8_0)
        mods.append(lin)

    def one(i):
        x = torch.full((m, k), float(i + 1), dtype=torch.bfloat16)
        assert torch.equal(modality._gated_activations(x, m, *mods, None, 1e-6), x[:, :n])
    _in_threads(4, one)
