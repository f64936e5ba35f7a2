"""GPU: the SiLU-gated pair over a few hundred rows - both matrices in one launch with K split over workgroups, the
reduction ending in the gated product - against the oracle (rel-L2 <= 1e-3: bf16 outputs, decoded weights the same bits)
and against the two projections and the product as bf16 tensors.  K in whole super-blocks of 256 runs on the mid-size kernel
below 2048 rows, everything else on the tile kernels.  Sizes around the 256 x 256 tile, one and several K
slices, and a workspace with room for exactly one copy of the sums and for none; the form of
17 .. 64 rows, scratch sizes, and what hangs on the projections' calls."""
import threading

import pytest
import torch

from oracle import gguf_oracle as go
from sensenova_u1_amd import GGUFLinear, GGUFParameter, ops, synthetic
from sensenova_u1_amd.modality import gated_mlp

pytestmark = pytest.mark.gpu


def _run(dev, qt, m, n, k, num=1, x=None, gate=None, ws_bytes=None):
    gate = synthetic.make_packed(qt, n, k, seed=n + k) if gate is None else gate
    up = synthetic.make_packed(qt, n, k, seed=n + k + 1)
    x = synthetic.make_activations(m, k, seed=m) if x is None else x
    ws = torch.empty(ws_bytes or ops.gate_up_silu_workspace_bytes(n, k), dtype=torch.uint8, device=dev)
    h = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=dev)
    ops.gate_up_silu_ws_into(x.to(dev), gate.to(dev), up.to(dev), qt, h, ws, num)
    return h.cpu(), go.gguf_linear_forward(x, gate, qt, numerics=num), go.gguf_linear_forward(x, up, qt, numerics=num)


@pytest.mark.parametrize("qt", [go.Q8_0, go.Q4_K])
@pytest.mark.parametrize("num", [0, 1])
@pytest.mark.parametrize("m,n,k", [(65, 8, 1024), (256, 264, 512), (257, 248, 1280), (511, 520, 1024), (100, 2056, 2048)])
def test_pair_with_split_k(dev, c_oracle, qt, num, m, n, k):
    print(f"case gated split qt={qt} num={num} {m}x{n}x{k}", flush=True)
    h, g, u = _run(dev, qt, m, n, k, num, ws_bytes=16 * 8 * m * n + ops.gate_up_silu_workspace_bytes(n, k))
    assert go.rel_l2(h, c_oracle.silu_mul(g, u)) <= 1e-3


@pytest.mark.parametrize("qt", [go.Q8_0, go.Q4_K])
@pytest.mark.parametrize("num", [0, 1])
@pytest.mark.parametrize("room", [0, 1])
@pytest.mark.parametrize("m,n,k", [(300, 1032, 256), (511, 520, 512), (65, 2056, 128)])
def test_room_for_one_copy_and_for_none(dev, c_oracle, qt, num, room, m, n, k):
    """Ragged rows and several column tiles per matrix.  One copy: K in one slice, fp32 sums and the gated reduction.  None: 16
    bytes less, or what the dense launch needs if that is more, which must hold less than one copy then."""
    if qt == go.Q4_K and k % 256:
        k = 256
    print(f"case pair room={room} qt={qt} num={num} {m}x{n}x{k}", flush=True)
    copy, dense = 8 * m * n, ops.gate_up_silu_workspace_bytes(n, k)
    if room == 0:
        m += -(-max(dense - copy + 16, 0) // (8 * n))     # rows enough for a copy that the dense launch's workspace cannot hold
        copy = 8 * m * n
        assert dense <= copy - 16 and 65 <= m < 1024
    h, g, u = _run(dev, qt, m, n, k, num, ws_bytes=copy if room else copy - 16)
    assert go.rel_l2(h, c_oracle.silu_mul(g, u)) <= 1e-3


def test_infinite_and_huge_gates(dev, c_oracle):
    """silu(+inf) = +inf, silu(-inf) = NaN, silu(-1e30) = -0, as on bf16 tensors."""
    qt, m, n, k = go.Q8_0, 130, 256, 256
    gate = synthetic.make_packed(qt, n, k, seed=71)
    gate[:64, 0:2] = torch.tensor([100.0], dtype=torch.float16).view(torch.uint8)
    x = synthetic.make_activations(m, k, seed=5)
    x[:3] = 0
    x[0, 0], x[1, 0], x[2, 0] = 1e38, -1e38, 1e30
    h, g, u = _run(dev, qt, m, n, k, x=x, gate=gate, ws_bytes=64 << 20)
    want = c_oracle.silu_mul(g, u)
    assert bool(torch.isnan(want.float()).any()) and bool(torch.isinf(want.float()).any())
    assert torch.equal(torch.isnan(h.float()), torch.isnan(want.float()))
    inf = torch.isinf(want.float())
    assert torch.equal(torch.isinf(h.float()), inf) and torch.equal(h[inf], want[inf])
    fin = torch.isfinite(want.float())
    assert torch.equal(torch.signbit(h[:3][fin[:3]].float()), torch.signbit(want[:3][fin[:3]].float()))
    assert go.rel_l2(torch.where(fin, h.float(), 0.0), torch.where(fin, want.float(), 0.0)) <= 1e-3


@pytest.mark.parametrize("num", [0, 1])
@pytest.mark.parametrize("qt,m,n,k,copies", [(go.Q8_0, 65, 8, 1152, 9), (go.Q8_0, 256, 264, 640, 1), (go.Q8_0, 257, 248, 1408, 2),
                                             (go.Q8_0, 100, 2056, 2176, 4), (go.Q8_0, 511, 520, 1152, 2), (go.Q4_K, 2100, 264, 512, 2), (go.Q8_0, 3000, 72, 768, 3)])
def test_pair_on_the_split_tile_launch(dev, c_oracle, qt, num, m, n, k, copies):
    """Where the mid-size kernel does not take a pair - K in half super-blocks, 2048 rows and more - the tile kernel's own split
    launch, one slice and several."""
    print(f"case gated split tiles qt={qt} num={num} {m}x{n}x{k}", flush=True)
    nbytes = copies * 8 * m * n
    assert ops.mid_plan(qt, m, n, k, True, nbytes) is None
    h, g, u = _run(dev, qt, m, n, k, num, ws_bytes=nbytes)
    assert go.rel_l2(h, c_oracle.silu_mul(g, u)) <= 1e-3


@pytest.mark.parametrize("k", [384, 640])
def test_infinite_and_huge_gates_on_the_split_tile_launch(dev, c_oracle, k):
    qt, m, n = go.Q8_0, 130, 256
    assert ops.mid_plan(qt, m, n, k, True, 64 << 20) is None
    gate = synthetic.make_packed(qt, n, k, seed=71)
    gate[:64, 0:2] = torch.tensor([100.0], dtype=torch.float16).view(torch.uint8)
    x = synthetic.make_activations(m, k, seed=5)
    x[:3] = 0
    x[0, 0], x[1, 0], x[2, 0] = 1e38, -1e38, 1e30
    h, g, u = _run(dev, qt, m, n, k, x=x, gate=gate, ws_bytes=8 * m * n)
    want = c_oracle.silu_mul(g, u)
    assert bool(torch.isnan(want.float()).any()) and bool(torch.isinf(want.float()).any())
    assert torch.equal(torch.isnan(h.float()), torch.isnan(want.float()))
    inf = torch.isinf(want.float())
    assert torch.equal(torch.isinf(h.float()), inf) and torch.equal(h[inf], want[inf])
    fin = torch.isfinite(want.float())
    assert torch.equal(torch.signbit(h[:3][fin[:3]].float()), torch.signbit(want[:3][fin[:3]].float()))


@pytest.mark.parametrize("qt,m", [(go.Q4_K, 65), (go.Q8_0, 203), (go.Q8_0, 511)])
def test_gated_mlp_takes_it(dev, monkeypatch, qt, m):
    n, k = 1024, 2048
    mods = []
    for j, (o, i) in enumerate(((n, k), (n, k), (k, n))):
        lin = GGUFLinear(i, o, bias=False, compute_dtype=torch.bfloat16, device="meta")
        lin.weight = GGUFParameter(synthetic.make_packed(qt, o, i, seed=40 + j, device=dev), quant_type=qt)
        mods.append(lin)
    gate, up, down = mods
    x = synthetic.make_activations(m, k, seed=m, device=dev)
    calls = []
    real = ops.gate_up_silu_ws_into
    monkeypatch.setattr(ops, "gate_up_silu_ws_into", lambda *a, **kw: (calls.append(a[0].shape[0]), real(*a, **kw))[1])
    got = gated_mlp(x, gate, up, down)
    assert calls == [m]
    # (another order of the fp32 sums: one bf16 step of a gated value now and then)
    assert go.rel_l2(got.cpu(), down(torch.nn.functional.silu(gate(x)) * up(x)).cpu()) <= 5e-4


@pytest.mark.parametrize("qt", [go.Q8_0, go.Q4_1, go.Q3_K, go.Q4_K, go.Q6_K])
@pytest.mark.parametrize("m,n,k", [(17, 8, 256), (33, 136, 512), (40, 4104, 1024), (64, 264, 768)])
def test_pair_of_17_to_64_rows(dev, c_oracle, qt, m, n, k):
    """silu and the product in the up projection's epilogue: the outputs of the two projections and of silu are rounded as
    the tensors of the separate calls are, so only the last place of exp() can differ from those."""
    print(f"case gated 17..64 rows qt={qt} {m}x{n}x{k}", flush=True)
    h, g, u = _run(dev, qt, m, n, k)
    assert go.rel_l2(h, c_oracle.silu_mul(g, u)) <= 1e-3
    x = synthetic.make_activations(m, k, seed=m).to(dev)
    gt, ut = (ops.linear(x, synthetic.make_packed(qt, n, k, seed=n + k + j).to(dev), qt) for j in (0, 1))
    assert go.rel_l2(h, (torch.nn.functional.silu(gt) * ut).cpu()) <= 1e-4


def test_infinite_gates_at_40_rows(dev, c_oracle):
    qt, m, n, k = go.Q8_0, 40, 256, 256
    gate = synthetic.make_packed(qt, n, k, seed=71)
    gate[:64, 0:2] = torch.tensor([100.0], dtype=torch.float16).view(torch.uint8)
    x = synthetic.make_activations(m, k, seed=5)
    x[:3] = 0
    x[0, 0], x[1, 0], x[2, 0] = 1e38, -1e38, 1e30
    h, g, u = _run(dev, qt, m, n, k, x=x, gate=gate)
    want = c_oracle.silu_mul(g, u)
    assert torch.equal(torch.isnan(h.float()), torch.isnan(want.float()))
    inf = torch.isinf(want.float())
    assert torch.equal(torch.isinf(h.float()), inf) and torch.equal(h[inf], want[inf])


def test_hooked_projections_are_called(dev):
    """A forward hook on a projection keeps the module calls."""
    n, k, m = 512, 1024, 40
    mods = []
    for j, (o, i) in enumerate(((n, k), (n, k), (k, n))):
        lin = GGUFLinear(i, o, bias=False, compute_dtype=torch.bfloat16, device="meta")
        lin.weight = GGUFParameter(synthetic.make_packed(go.Q8_0, o, i, seed=60 + j, device=dev), quant_type=go.Q8_0)
        mods.append(lin)
    x = synthetic.make_activations(m, k, seed=m, device=dev)
    want = gated_mlp(x, *mods)
    seen = []
    handle = mods[1].register_forward_hook(lambda mod, args, out: seen.append(out.shape))
    got = gated_mlp(x, *mods)
    handle.remove()
    assert seen == [(m, n)] and go.rel_l2(got.cpu(), want.cpu()) <= 1e-4


class _Adapted(GGUFLinear):
    def forward(self, inputs):
        return super().forward(inputs) * 2


@pytest.mark.parametrize("m,n,k", [(40, 512, 1024), (203, 1024, 2048), (512, 6144, 2048)])
def test_projections_with_their_own_forward_are_called(dev, m, n, k):
    """An overriding subclass and a hook that replaces the output, at sizes of each form that was module calls."""
    print(f"case own forward {m}x{n}x{k}", flush=True)
    mods = []
    for j, (o, i, cls) in enumerate(((n, k, GGUFLinear), (n, k, _Adapted), (k, n, GGUFLinear))):
        lin = cls(i, o, bias=False, compute_dtype=torch.bfloat16, device="meta")
        lin.weight = GGUFParameter(synthetic.make_packed(go.Q8_0, o, i, seed=80 + j, device=dev), quant_type=go.Q8_0)
        mods.append(lin)
    gate, up, down = mods
    x = synthetic.make_activations(m, k, seed=m, device=dev)
    assert torch.equal(gated_mlp(x, gate, up, down), down(torch.nn.functional.silu(gate(x)) * up(x)))
    plain = GGUFLinear(k, n, bias=False, compute_dtype=torch.bfloat16, device="meta")
    plain.weight = up.weight
    handle = plain.register_forward_hook(lambda mod, args, out: out * 2)
    assert torch.equal(gated_mlp(x, gate, plain, down), gated_mlp(x, gate, up, down))
    handle.remove()


@pytest.mark.parametrize("m,n,k", [(40, 512, 1024), (203, 1024, 2048), (512, 6144, 2048)])
def test_bf16_input_to_an_fp16_projection_is_refused(dev, m, n, k):
    mods = []
    for j, (o, i, dtype) in enumerate(((n, k, torch.bfloat16), (n, k, torch.float16), (k, n, torch.bfloat16))):
        lin = GGUFLinear(i, o, bias=False, compute_dtype=dtype, device="meta")
        lin.weight = GGUFParameter(synthetic.make_packed(go.Q8_0, o, i, seed=20 + j, device=dev), quant_type=go.Q8_0)
        mods.append(lin)
    with pytest.raises(RuntimeError, match="compute dtype"):
        gated_mlp(synthetic.make_activations(m, k, seed=m, device=dev), *mods)


@pytest.mark.parametrize("qt,m,n,k", [(go.Q8_0, 40, 264, 512), (go.Q6_K, 17, 8, 256), (go.Q4_K, 64, 4104, 256), (go.Q8_0, 257, 264, 2048),
                                      (go.Q4_K, 203, 1024, 2048), (go.Q6_K, 130, 264, 512)])
def test_workspace_of_exactly_the_form_s_size(dev, c_oracle, qt, m, n, k):
    """As many bytes as the form asks for, the 64 behind them untouched; 16 bytes less are refused where no smaller form exists."""
    print(f"case exact workspace qt={qt} {m}x{n}x{k}", flush=True)
    nbytes = ops.gate_up_silu_ws_bytes(qt, m, n, k)
    gate, up = (synthetic.make_packed(qt, n, k, seed=n + j, device=dev) for j in (0, 1))
    x = synthetic.make_activations(m, k, seed=m, device=dev)
    ws = torch.full((nbytes + 64,), 0xA5, dtype=torch.uint8, device=dev)
    h = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=dev)
    ops.gate_up_silu_ws_into(x, gate, up, qt, h, ws, 1, nbytes)
    g, u = (go.gguf_linear_forward(x.cpu(), w.cpu(), qt, numerics=1) for w in (gate, up))
    assert go.rel_l2(h.cpu(), c_oracle.silu_mul(g, u)) <= 1e-3
    assert bool((ws[nbytes:] == 0xA5).all())
    if m <= 64 or qt == go.Q6_K:
        with pytest.raises(ops.SnGgufError):
            ops.gate_up_silu_ws_into(x, gate, up, qt, h, ws, 1, nbytes - 16)


def test_forty_rows_leave_no_weight_sized_workspace(dev):
    n, k, m = 2048, 1024, 40
    mods = []
    for j, (o, i) in enumerate(((n, k), (n, k), (k, n))):
        lin = GGUFLinear(i, o, bias=False, compute_dtype=torch.bfloat16, device="meta")
        lin.weight = GGUFParameter(synthetic.make_packed(go.Q8_0, o, i, seed=30 + j, device=dev), quant_type=go.Q8_0)
        mods.append(lin)
    ops.release_workspaces()
    gated_mlp(synthetic.make_activations(m, k, seed=m, device=dev), *mods)
    assert sum(ws.numel() for ws in ops._workspaces.values()) <= 2 * m * n


@pytest.mark.parametrize("qt_down", [go.Q8_0, go.Q6_K])
@pytest.mark.parametrize("m", [40, 203, 600])
def test_captured_passes_replay_the_eager_ones(dev, qt_down, m):
    """Scratch of the call's own and workspaces handed out during a capture: replays on new rows, eager passes between them."""
    print(f"case captured gated pair m={m} down={qt_down}", flush=True)
    n, k = 1024, 2560
    mods = []
    for j, (o, i, qt) in enumerate(((n, k, go.Q8_0), (n, k, go.Q8_0), (k, n, qt_down))):
        lin = GGUFLinear(i, o, bias=False, compute_dtype=torch.bfloat16, device="meta")
        lin.weight = GGUFParameter(synthetic.make_packed(qt, o, i, seed=60 + j, device=dev), quant_type=qt)
        mods.append(lin)
    x = synthetic.make_activations(m, k, seed=m, device=dev)
    gated_mlp(x, *mods)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = gated_mlp(x, *mods)
    for seed in (1, 2, 3):
        rows = synthetic.make_activations(m, k, seed=seed, device=dev)
        want = gated_mlp(rows, *mods)
        torch.cuda.synchronize()
        x.copy_(rows)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)


@pytest.mark.parametrize("m", [17, 40, 64, 203])
def test_threads_on_one_stream(dev, m):
    """Four host threads, each with rows of its own, through one MLP on the default stream: scratch of the call (up to 64
    rows) and of the pool (beyond)."""
    print(f"case threads on one stream m={m}", flush=True)
    n, k = 1024, 2048
    mods = []
    for j, (o, i) in enumerate(((n, k), (n, k), (k, n))):
        lin = GGUFLinear(i, o, bias=False, compute_dtype=torch.bfloat16, device="meta")
        lin.weight = GGUFParameter(synthetic.make_packed(go.Q8_0, o, i, seed=50 + j, device=dev), quant_type=go.Q8_0)
        mods.append(lin)
    xs = [synthetic.make_activations(m, k, seed=100 + t, device=dev) for t in range(4)]
    want = [gated_mlp(x, *mods) for x in xs]
    got = [[] for _ in xs]

    def body(t):
        for _ in range(16):
            got[t].append(gated_mlp(xs[t], *mods))
    threads = [threading.Thread(target=body, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for w, outs in zip(want, got):
        assert len(outs) == 16 and all(torch.equal(o, w) for o in outs)
