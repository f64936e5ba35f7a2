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


@pytest.mark.parametrize("entry", ["linear_ws", "linear_static", "gate_up_silu_ws", "grouped_linear_ws"])
def test_calls_that_share_a_pooled_workspace_do_not_interleave(host_scratch, monkeypatch, entry):
    """The pool hands the threads of one stream the same memory; one call's launches are then enqueued as one run."""
    import contextlib
    import types
    scratch, seen = [None], []

    def launches(*args):
        me = threading.get_ident()
        scratch[0] = me                     # the first launch fills the workspace
        time.sleep(0.01)                    # (a foreign call: the interpreter lock is free)
        seen.append(scratch[0] == me)       # the second launch reads it
        return 0

    monkeypatch.setattr(ops, "_on", lambda dev: contextlib.nullcontext())
    monkeypatch.setattr(ops, "load_library", lambda: types.SimpleNamespace(**{f"sngguf_{entry}": launches}))
    x, y, w = torch.zeros((80, 64), dtype=torch.bfloat16), torch.zeros((80, 32), dtype=torch.bfloat16), torch.zeros((32, 68), dtype=torch.uint8)

    def one(i):
        for _ in range(5):
            ws = ops.pooled_workspace(x.device, 4096 * (i + 1))
            if entry == "linear_ws":
                ops.linear_ws_into(x, w, ops.Q8_0, None, y, ws, 1)
            elif entry == "linear_static":
                ops.linear_static_into(x, w, ops.Q8_0, None, y, 1)
            elif entry == "gate_up_silu_ws":
                ops.gate_up_silu_ws_into(x, w, w, ops.Q8_0, y, ws, 1)
            else:
                ops.grouped_linear_ws_into(x, None, 40, w, ops.Q8_0, w, ops.Q8_0, None, None, y, None, ws, 1)
    _in_threads(4, one)
    assert len(seen) == 20 and all(seen)
