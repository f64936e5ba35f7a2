"""GPU parity of the kernel for 17 rows to a few thousand (csrc/gemm_mid.hip): every block format on every instance (16-row tiles a
workgroup holds x columns it covers), with and without K split over workgroups, each in both numerics modes, as a projection with
bias and as a gated pair; K shares that end early, ragged rows and columns, the residual.

Bound: the decoded weights are the oracle's bits and the sums are fp32 in another order, so an output differs from the oracle's
by at most one bf16 step now and then; rel-L2 1e-3 is every output half a step off (2^-9 / sqrt(3))."""
import pytest
import torch

from oracle import gguf_oracle as go
from sensenova_u1_amd import ops, synthetic

pytestmark = pytest.mark.gpu
TOL = 1e-3
TYPES = [go.Q4_0, go.Q4_1, go.Q5_0, go.Q5_1, go.Q8_0, go.Q2_K, go.Q3_K, go.Q4_K, go.Q5_K, go.Q6_K]


def _columns(n, seed, count=40):
    cols = torch.randint(0, n, (count,), generator=torch.Generator().manual_seed(seed))
    cols[0], cols[1] = 0, n - 1
    return cols


def _check(got, want):
    assert bool(torch.isfinite(got.float()).all())
    assert go.rel_l2(got, want) <= TOL


@pytest.mark.parametrize("qt", TYPES)
@pytest.mark.parametrize("num", [0, 1])
@pytest.mark.parametrize("m,n,k", [(17, 264, 256), (33, 515, 768), (48, 1032, 2304), (64, 136, 4096), (50, 2050, 512)])
def test_projection_of_17_to_64_rows(dev, qt, num, m, n, k):
    """One super-block, shares of unequal length, a K split with scratch; columns that end inside a wavefront's rows."""
    print(f"case mid rows qt={qt} num={num} {m}x{n}x{k}", flush=True)
    packed, x = synthetic.make_packed(qt, n, k, seed=n + k), synthetic.make_activations(m, k, seed=m)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(k)) * 0.5).to(torch.bfloat16)
    res = synthetic.make_activations(m, n, seed=m + 1)
    want = go.gguf_linear_forward(x, packed, qt, bias, numerics=num)
    xd, pd, bd = x.to(dev), packed.to(dev), bias.to(dev)
    _check(ops.linear(xd, pd, qt, bd, num).cpu(), want)
    _check(ops.linear_residual(xd, pd, qt, res.to(dev), bd, num).cpu(), (res.float() + want.float()).to(torch.bfloat16))
    y = torch.empty((m, n), dtype=torch.bfloat16, device=dev)   # without scratch: no K split
    rc = ops.load_library().sngguf_linear(xd.data_ptr(), m, pd.data_ptr(), qt, n, k, bd.data_ptr(), y.data_ptr(), num, ops._stream(dev))
    assert rc == 0
    _check(y.cpu(), want)


# (rows, columns, K) that the plan gives each instance: narrow 32 / 48 / 64 rows, wide 32 .. 208, long 160 .. 256
INSTANCES = [(17, 264, 256), (1024, 264, 256), (1500, 264, 256), (17, 8200, 2048), (100, 4104, 1280), (150, 4104, 1280), (65, 12296, 512),
             (100, 12296, 512), (400, 4104, 512), (509, 4104, 512), (257, 12296, 512), (400, 12296, 512), (1500, 4104, 512)]


@pytest.mark.parametrize("qt", [go.Q8_0, go.Q6_K, go.Q5_0])
@pytest.mark.parametrize("m,n,k", INSTANCES)
def test_pair_of_every_instance(dev, c_oracle, qt, m, n, k):
    num = (m + k // 256) & 1
    print(f"case mid pair qt={qt} num={num} {m}x{n}x{k}", flush=True)
    gate, up = (synthetic.make_packed(qt, n, k, seed=n + j, device=dev) for j in (0, 1))
    x = synthetic.make_activations(m, k, seed=m, device=dev)
    ws = torch.empty(ops.gate_up_silu_workspace_bytes(n, k) + 2 * m * n, dtype=torch.uint8, device=dev)
    h = torch.full((m + 1, n), 7.0, dtype=torch.bfloat16, device=dev)
    ops.gate_up_silu_ws_into(x, gate, up, qt, h[:m], ws, num)
    cols = _columns(n, m)
    g, u = (go.gguf_linear_forward(x.cpu(), w[cols.to(dev)].cpu(), qt, numerics=num) for w in (gate, up))
    _check(h[:m, cols.to(dev)].cpu(), c_oracle.silu_mul(g, u))
    assert bool((h[m] == 7.0).all())   # nothing behind the last row


@pytest.mark.parametrize("qt", TYPES)
@pytest.mark.parametrize("m,n,k", [(17, 520, 12288), (48, 1032, 4096), (64, 2048, 2304)])
def test_pair_of_few_columns_in_any_workspace(dev, c_oracle, qt, m, n, k):
    """The K split that the shape asks for, one slice fewer, and the least workspace: the gate outputs alone, which the decode kernel's
    two launches or the launch without a K split take.  Nothing behind the bytes handed over."""
    num = (m + n // 8) & 1
    gate, up = (synthetic.make_packed(qt, n, k, seed=n + j, device=dev) for j in (0, 1))
    x = synthetic.make_activations(m, k, seed=m, device=dev)
    cols = _columns(n, m)
    g, u = (go.gguf_linear_forward(x.cpu(), w[cols.to(dev)].cpu(), qt, numerics=num) for w in (gate, up))
    want, asked = c_oracle.silu_mul(g, u), ops.gate_up_silu_ws_bytes(qt, m, n, k)
    assert asked >= 2 * 8 * m * n
    for nbytes in (asked, asked - 16, 2 * m * n):
        print(f"case mid few columns qt={qt} num={num} {m}x{n}x{k} workspace {nbytes}", flush=True)
        ws = torch.full((nbytes + 64,), 0xA5, dtype=torch.uint8, device=dev)
        h = torch.full((m + 1, n), 7.0, dtype=torch.bfloat16, device=dev)
        ops.gate_up_silu_ws_into(x, gate, up, qt, h[:m], ws, num, nbytes)
        _check(h[:m, cols.to(dev)].cpu(), want)
        assert bool((ws[nbytes:] == 0xA5).all()) and bool((h[m] == 7.0).all())


# (rows, columns, K) -> (columns of a workgroup, 16-row tiles of its instance, row tiles, K slices), the same for all formats
PROJECTIONS = {
    (65, 136, 256): (64, 2, 3, 1), (64, 136, 2048): (64, 2, 2, 4), (1000, 520, 256): (64, 3, 21, 1), (700, 136, 2048): (64, 3, 15, 4),
    (150, 4104, 256): (64, 4, 3, 1), (1500, 136, 2304): (64, 4, 24, 3), (203, 4104, 1280): (128, 2, 7, 1), (1000, 1032, 1280): (128, 3, 21, 1),
    (1500, 1032, 1280): (128, 4, 24, 1), (65, 16392, 256): (128, 6, 1, 1), (65, 8200, 2304): (128, 6, 1, 3), (100, 16392, 256): (128, 8, 1, 1),
    (1000, 1032, 2304): (128, 8, 8, 3), (130, 16392, 512): (128, 10, 1, 1), (1000, 1032, 2048): (128, 10, 7, 4), (203, 16392, 512): (128, 13, 1, 1),
    (130, 16392, 256): (256, 10, 1, 1), (100, 16392, 2304): (256, 10, 1, 3), (509, 16392, 1280): (256, 13, 3, 1), (203, 16392, 2304): (256, 13, 1, 3),
    (209, 16392, 2048): (256, 16, 1, 3)}
PAIRS = {
    (17, 136, 256): (64, 2, 1, 1), (17, 136, 2048): (64, 2, 1, 4), (1000, 264, 256): (64, 3, 21, 1), (400, 136, 2048): (64, 3, 9, 4),
    (1500, 264, 256): (64, 4, 24, 1), (509, 264, 2304): (64, 4, 8, 3), (203, 2056, 1280): (128, 2, 7, 1), (1000, 520, 1280): (128, 3, 21, 1),
    (1500, 520, 1280): (128, 4, 24, 1), (65, 8200, 256): (128, 6, 1, 1), (65, 4104, 2304): (128, 6, 1, 3), (100, 8200, 256): (128, 8, 1, 1),
    (100, 4104, 2304): (128, 8, 1, 3), (130, 8200, 512): (128, 10, 1, 1), (150, 4104, 2304): (128, 10, 1, 3), (509, 4104, 512): (128, 13, 3, 1),
    (130, 8200, 256): (256, 10, 1, 1), (100, 8200, 2304): (256, 10, 1, 3), (203, 16392, 256): (256, 13, 1, 1), (203, 8200, 2304): (256, 13, 1, 3),
    (209, 16392, 256): (256, 16, 1, 1), (209, 8200, 2048): (256, 16, 1, 3),
    # more workgroups than run at once: narrow form of 32 rows with 512 (packed rows two units ahead) and 513 (one), wide form with 385
    (32, 16384, 512): (64, 2, 1, 1), (31, 16392, 512): (64, 2, 1, 1), (29, 24584, 1280): (128, 2, 1, 1), (44, 24584, 1280): (128, 3, 1, 1)}


def workspace_bytes(qt, m, n, k, pair):
    if pair:
        return ops.gate_up_silu_ws_bytes(qt, m, n, k)
    return ops.load_library().sngguf_linear_scratch_bytes(qt, m, n, k) if m <= 64 else ops.linear_ws_bytes(qt, m, n, k)


@pytest.mark.parametrize("qt", TYPES)
@pytest.mark.parametrize("m,n,k", PROJECTIONS)
def test_projection_on_each_instance(dev, qt, m, n, k):
    num = (TYPES.index(qt) + list(PROJECTIONS).index((m, n, k))) & 1
    print(f"case mid projection qt={qt} num={num} {m}x{n}x{k}", flush=True)
    nbytes = workspace_bytes(qt, m, n, k, False)
    assert ops.mid_plan(qt, m, n, k, False, nbytes) == PROJECTIONS[m, n, k]
    packed, x = synthetic.make_packed(qt, n, k, seed=n, device=dev), synthetic.make_activations(m, k, seed=m, device=dev)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(k)) * 0.5).to(torch.bfloat16).to(dev)
    ws = torch.full((nbytes + 64,), 0xA5, dtype=torch.uint8, device=dev)
    y = torch.full((m + 1, n), 7.0, dtype=torch.bfloat16, device=dev)
    call = ops.load_library().sngguf_linear_scratch if m <= 64 else ops.load_library().sngguf_linear_ws
    args = (x.data_ptr(), m, packed.data_ptr(), qt, n, k, bias.data_ptr())
    assert call(*args, *((None,) if m <= 64 else ()), y.data_ptr(), ws.data_ptr(), nbytes, num, ops._stream(dev)) == 0
    cols = _columns(n, m)
    _check(y[:m, cols.to(dev)].cpu(), go.gguf_linear_forward(x.cpu(), packed[cols.to(dev)].cpu(), qt, bias.cpu()[cols], numerics=num))
    assert bool((ws[nbytes:] == 0xA5).all()) and bool((y[m] == 7.0).all())


@pytest.mark.parametrize("qt", TYPES)
@pytest.mark.parametrize("m,n,k", PAIRS)
def test_pair_on_each_instance(dev, c_oracle, qt, m, n, k):
    num = (TYPES.index(qt) + list(PAIRS).index((m, n, k))) & 1
    print(f"case mid pair instance qt={qt} num={num} {m}x{n}x{k}", flush=True)
    nbytes = workspace_bytes(qt, m, n, k, True)
    assert ops.mid_plan(qt, m, n, k, True, nbytes) == PAIRS[m, n, k]
    gate, up = (synthetic.make_packed(qt, n, k, seed=n + j, device=dev) for j in (0, 1))
    x = synthetic.make_activations(m, k, seed=m, device=dev)
    ws = torch.full((nbytes + 64,), 0xA5, dtype=torch.uint8, device=dev)
    h = torch.full((m + 1, n), 7.0, dtype=torch.bfloat16, device=dev)
    ops.gate_up_silu_ws_into(x, gate, up, qt, h[:m], ws, num, nbytes)
    cols = _columns(n, m)
    g, u = (go.gguf_linear_forward(x.cpu(), w[cols.to(dev)].cpu(), qt, numerics=num) for w in (gate, up))
    _check(h[:m, cols.to(dev)].cpu(), c_oracle.silu_mul(g, u))
    assert bool((ws[nbytes:] == 0xA5).all()) and bool((h[m] == 7.0).all())


@pytest.mark.parametrize("qt", [go.Q8_0, go.Q4_K, go.Q3_K, go.Q6_K])
@pytest.mark.parametrize("m,n,k", [(65, 1024, 2304), (203, 515, 4096), (300, 2050, 1280), (509, 4096, 2048), (1000, 1032, 768), (130, 264, 12288)])
def test_projection_beyond_64_rows(dev, qt, m, n, k):
    """The workspace that the shape asks for and not a byte more; with K split where the columns are few."""
    print(f"case mid ws qt={qt} {m}x{n}x{k}", flush=True)
    packed, x = synthetic.make_packed(qt, n, k, seed=n, device=dev), synthetic.make_activations(m, k, seed=m, device=dev)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(k)) * 0.5).to(torch.bfloat16).to(dev)
    nbytes = ops.linear_ws_bytes(qt, m, n, k)
    ws = torch.full((nbytes + 64,), 0xA5, dtype=torch.uint8, device=dev)
    y = torch.full((m + 1, n), 7.0, dtype=torch.bfloat16, device=dev)[:m] if n % 8 == 0 else torch.empty((m, n), dtype=torch.bfloat16, device=dev)
    rc = ops.load_library().sngguf_linear_ws(x.data_ptr(), m, packed.data_ptr(), qt, n, k, bias.data_ptr(), y.data_ptr(), ws.data_ptr(), nbytes,
                                             1, ops._stream(dev))
    assert rc == 0
    cols = _columns(n, m)
    _check(y[:, cols.to(dev)].cpu(), go.gguf_linear_forward(x.cpu(), packed[cols.to(dev)].cpu(), qt, bias.cpu()[cols]))
    assert bool((ws[nbytes:] == 0xA5).all())


@pytest.mark.parametrize("qt", [go.Q8_0, go.Q6_K])
@pytest.mark.parametrize("m", [40, 203])
def test_captured_projection_replays_the_eager_one(dev, qt, m):
    """Partial sums in scratch of the call's own (up to 64 rows) or a workspace handed out during the capture."""
    from sensenova_u1_amd import GGUFLinear, GGUFParameter
    print(f"case mid captured qt={qt} m={m}", flush=True)
    n, k = 1024, 4096
    lin = GGUFLinear(k, n, bias=False, compute_dtype=torch.bfloat16, device="meta")
    lin.weight = GGUFParameter(synthetic.make_packed(qt, n, k, seed=3, device=dev), quant_type=qt)
    x = synthetic.make_activations(m, k, seed=m, device=dev)
    lin(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = lin(x)
    for seed in (1, 2, 3):
        rows = synthetic.make_activations(m, k, seed=seed, device=dev)
        want = lin(rows)
        torch.cuda.synchronize()
        x.copy_(rows)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
