"""A projection's sums are cut into the K slices of its shape, whatever a pooled workspace has grown to through other modules'
calls: every call asks the library how much workspace the shape can use."""
import pytest
import torch

from sensenova_u1_amd import GGUFLinear, GGUFParameter, grouped_linear, modality, ops, synthetic

TYPES = [ops.Q4_0, ops.Q8_0, ops.Q3_K, ops.Q4_K, ops.Q5_K, ops.Q6_K, ops.BF16]


def test_what_a_shape_can_use():
    """Whole fp32 copies of the output for a K split (behind the decoded weight where the tile kernel does not decode the
    type), the decoded weight without one, nothing up to 64 rows and where K is not whole K steps."""
    for qt in TYPES:
        for m, n, k in ((65, 4096, 12288), (203, 4096, 12288), (509, 1024, 4096), (300, 2050, 1024), (1024, 12288, 4096)):
            nbytes = ops.linear_ws_bytes(qt, m, n, k)
            rest = nbytes - (0 if qt in (ops.Q8_0, ops.Q4_K, ops.BF16) else 2 * n * k)
            if -(-m // 256) * -(-n // 256) <= 128:
                # one workgroup per compute unit at most: 256 tiles of partial sums
                assert rest % (4 * m * n) == 0 and 2 <= rest // (4 * m * n) <= 64 and rest <= 256 * 256 * 256 * 4
            else:
                assert nbytes == (0 if qt == ops.BF16 else 2 * n * k)
        assert ops.linear_ws_bytes(qt, 64, 4096, 4096) == 0 and ops.linear_ws_bytes(qt, 0, 4096, 4096) == 0
    # four K steps of 64 a slice, two where K has fewer than eight; fewer copies where they lie a power of two apart
    for qt in (ops.Q8_0, ops.BF16):
        assert ops.linear_ws_bytes(qt, 100, 512, 1024) == 4 * 4 * 100 * 512 and ops.linear_ws_bytes(qt, 100, 512, 256) == 2 * 4 * 100 * 512
    assert ops.linear_ws_bytes(ops.Q8_0, 512, 2048, 6144) < 48 << 20 and ops.linear_ws_bytes(ops.Q8_0, 512, 2048, 128) == 2 * 2048 * 128
    assert ops.linear_ws_bytes(ops.Q8_0, 300, 512, 96) == 0 and ops.linear_ws_bytes(16, 300, 512, 256) == 0
    assert ops.linear_ws_bytes(ops.Q8_0, 4096, 1024, 4096) == 2 * 1024 * 4096 + 4 * 4 * 4096 * 1024   # weight pass from 4096 rows on


def _linear(qt, n, k, seed, dev):
    lin = GGUFLinear(k, n, bias=False, compute_dtype=torch.bfloat16, device="meta")
    lin.weight = GGUFParameter(synthetic.make_packed(qt, n, k, seed=seed, device=dev), quant_type=qt)
    return lin


@pytest.mark.gpu
@pytest.mark.parametrize("qt", TYPES)
@pytest.mark.parametrize("m,n,k", [(65, 512, 4096), (203, 1024, 12288), (300, 264, 1024), (513, 4096, 2048)])
def test_a_grown_pool_changes_nothing(dev, qt, m, n, k):
    print(f"case grown pool qt={qt} {m}x{n}x{k}", flush=True)
    lin, x = _linear(qt, n, k, 3, dev), synthetic.make_activations(m, k, seed=4, device=dev)
    for policy in ("auto", "resident"):
        lin.gemm_policy = policy
        ops.release_workspaces()
        fresh = lin(x)
        ops.pooled_workspace(dev, 2 * n * k + 64 * 4 * m * n)
        assert torch.equal(lin(x), fresh)
    ops.release_workspaces()


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_text", [(512, 100), (515, 101), (515, 96)])
def test_a_grown_pool_changes_no_mixed_rows(dev, n, n_text):
    """(515 columns: the image rows start at an address that only the launch over both groups takes)"""
    m, k = 400, 2048
    und, gen = _linear(ops.Q8_0, n, k, 5, dev), _linear(ops.Q8_0, n, k, 6, dev)
    x = synthetic.make_activations(m, k, seed=7, device=dev)
    ops.release_workspaces()
    fresh = grouped_linear(x, None, und, gen, n_text=n_text)
    ops.pooled_workspace(dev, 1 << 28)
    assert torch.equal(grouped_linear(x, None, und, gen, n_text=n_text), fresh)
    ops.release_workspaces()


@pytest.mark.gpu
def test_a_grown_pool_changes_no_stacked_projections(dev):
    qt, m, k = ops.Q6_K, 203, 4096
    mods = [_linear(qt, n, k, 8 + n, dev) for n in (1024, 256, 256)]
    want = [mod(synthetic.make_activations(m, k, seed=9, device=dev)) for mod in mods]
    holder = torch.nn.Module()
    holder.q_proj, holder.k_proj, holder.v_proj = mods
    assert modality.stack_shared_input_projections(holder) == 1
    x = synthetic.make_activations(m, k, seed=9, device=dev)
    ops.release_workspaces()
    fresh = [mod(x).clone() for mod in mods]
    ops.pooled_workspace(dev, 1 << 28)
    again = [mod(x) for mod in mods]
    assert all(torch.equal(a, b) for a, b in zip(again, fresh))
    for a, b in zip(fresh, want):
        assert float((a.float() - b.float()).norm() / b.float().norm()) <= 4e-4
    ops.release_workspaces()
