"""GPU: silu of a gated pair at every finite bf16 gate, on every route that ends in one: the decode kernel, the mid-size kernel
(narrow and wide form, with K split and without), the tile kernels' split launch and the dense launch.

A gate row holds one weight of 1 and an up row one that meets an activation of 1, so gates are the activations themselves and the
pair's output is bf16(silu(gate)).  Bound: fp32 arithmetic is good to a few units in its last place, so each output is the bf16
rounding of g / (1 + exp(-g)) in fp64, the same bits on every route - but for four gates whose value lies within 2^-21 (relative) of the
middle between two bf16 values, where either is right.  exp(-g) beyond fp32's range is infinite, as in fp32, which gives -0 from g = -89
on."""
import pytest
import torch

from oracle import gguf_oracle as go
from sensenova_u1_amd import ops

pytestmark = pytest.mark.gpu


def _rows(n, k, columns, scale, dev):
    """Q8_0 rows with a single weight: 1 x scale[n] at column columns[n]."""
    w = torch.zeros((n, k // 32, 34), dtype=torch.uint8)
    at, row = columns // 32, torch.arange(n)
    w[row, at, 0:2] = scale.to(torch.float16).view(torch.uint8).reshape(n, 2)
    w[row, at, 2 + columns % 32] = 1
    return w.reshape(n, -1).to(dev)


# rows, columns, K, copies of the sums that the workspace holds (None: what the least form takes), and the mid-size kernel's (columns
# of a workgroup, K slices) where it runs
ROUTES = {"decode": (16, 4104, 4352, 0, None), "narrow": (64, 1032, 1280, 1, (64, 1)), "narrow, K split": (64, 1032, 2560, 4, (64, 3)),
          "wide": (128, 12296, 768, 1, (128, 1)), "wide, K split": (100, 4104, 4352, 2, (128, 2)), "long": (1500, 4104, 512, 0, (256, 1)),
          "tiles, K split": (128, 520, 640, 1, None), "dense": (256, 392, 384, 0, None)}


@pytest.mark.parametrize("route", ROUTES)
def test_every_finite_gate(dev, route):
    m, n, k, copies, mid = ROUTES[route]
    print(f"case gated silu {route} {m}x{n}x{k}", flush=True)
    distinct = min(n - 8, -(-65536 // m))
    bits = torch.arange(m * distinct, dtype=torch.int32) % 65536
    values = bits.to(torch.int16).view(torch.bfloat16)
    values = torch.where(torch.isfinite(values.float()), values, torch.ones((), dtype=torch.bfloat16))
    x = torch.zeros((m, k), dtype=torch.bfloat16)
    x[:, :distinct], x[:, k - 1] = values.reshape(m, distinct), 1.0
    # (the last eight columns: gates 2^-9 times as large, among them negative ones that round to -0)
    scale = torch.ones(n)
    scale[-8:] = 2.0 ** -9
    gate = _rows(n, k, torch.arange(n) % distinct, scale, dev)
    up = _rows(n, k, torch.full((n,), k - 1), torch.ones(n), dev)
    xd, h = x.to(dev), torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=dev)
    if route == "decode":
        ops.gate_up_silu_into(xd, gate, up, go.Q8_0, h, 1)
    else:
        nbytes = max(copies * 8 * m * n, ops.gate_up_silu_workspace_bytes(n, k) if not copies else 2 * m * n)
        plan = ops.mid_plan(go.Q8_0, m, n, k, True, nbytes)
        assert (plan and (plan[0], plan[3])) == mid, plan
        ops.gate_up_silu_ws_into(xd, gate, up, go.Q8_0, h, torch.empty(nbytes, dtype=torch.uint8, device=dev), 1)
    # (an activation of -0 is added to a sum of +0)
    g = ((x[:, torch.arange(n) % distinct].float() + 0.0) * scale).to(torch.bfloat16)
    e = torch.exp(-g.double())
    want = g.double() / (1.0 + torch.where(e > torch.finfo(torch.float32).max, float("inf"), e))
    exact, lo, hi, got = (t.view(torch.int16) for t in (*((want * (1.0 + e * 2.0 ** -21)).float().to(torch.bfloat16) for e in (0, -1, 1)), h.cpu()))
    bad = (got != exact) & ((want.abs() < 2.0 ** -126) | ((got != lo) & (got != hi)))
    assert not bool(bad.any()), (int(bad.sum()), sorted(set(zip(g[bad].tolist(), h.cpu()[bad].tolist(), want[bad].tolist())))[:8])
