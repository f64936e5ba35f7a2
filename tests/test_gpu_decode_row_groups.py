"""GPU: 17 .. 64 activation rows around the width from which a workgroup takes two 16-row groups of the weight (4096), and
the arg-max over a vocabulary-sized Q6_K matrix.  The K pieces do not depend on the number of row groups, so the first 4096
columns are the narrow matrix's, bit for bit."""
import pytest
import torch

from oracle import gguf_oracle as go
from sensenova_u1_amd import ops, synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qt", [go.Q8_0, go.Q4_0, go.Q5_1, go.Q3_K, go.Q4_K, go.Q6_K])
@pytest.mark.parametrize("n,k,m", [(4097, 256, 17), (4127, 512, 33), (4128, 768, 64), (6144, 2048, 40)])
def test_two_row_groups_per_workgroup(dev, qt, n, k, m):
    print(f"case row groups qt={qt} {m}x{n}x{k}", flush=True)
    packed = synthetic.make_packed(qt, n, k, seed=n + m)
    x = synthetic.make_activations(m, k, seed=m)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(n)) * 0.5).to(torch.bfloat16)
    got = ops.linear(x.to(dev), packed.to(dev), qt, bias.to(dev), 1)
    narrow = ops.linear(x.to(dev), packed[:4096].contiguous().to(dev), qt, bias[:4096].to(dev), 1)
    assert torch.equal(got[:, :4096], narrow)
    assert go.rel_l2(got.cpu(), go.gguf_linear_forward(x, packed, qt, bias, numerics=1)) <= 1e-3


@pytest.mark.parametrize("k,m", [(256, 1), (512, 2), (4096, 1), (1024, 5)])
def test_vocabulary_sized_q6_k(dev, k, m):
    """One super-block (one wavefront per workgroup) and more (two)."""
    n = 32771
    print(f"case vocabulary q6_k {m}x{n}x{k}", flush=True)
    packed = synthetic.make_packed(go.Q6_K, n, k, seed=k)
    x = synthetic.make_activations(m, k, seed=m)
    y = ops.linear(x.to(dev), packed.to(dev), go.Q6_K, None, 1)
    assert go.rel_l2(y.cpu(), go.gguf_linear_forward(x, packed, go.Q6_K, numerics=1)) <= 1e-3
    assert torch.equal(ops.lm_head_argmax(x.to(dev), packed.to(dev), go.Q6_K), y.float().argmax(dim=-1))
