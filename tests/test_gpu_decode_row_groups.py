"""GPU: 17 .. 64 activation rows around the widths and lengths at which the number of 16-row groups of the weight and of
wavefronts per workgroup changes, and the arg-max over a vocabulary-sized Q6_K matrix."""
import pytest
import torch

from oracle import gguf_oracle as go
from sensenova_u1_amd import ops, synthetic

pytestmark = pytest.mark.gpu


def _both(dev, qt, n, k, m, numerics=1):
    packed = synthetic.make_packed(qt, n, k, seed=n + m)
    x = synthetic.make_activations(m, k, seed=m)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(n)) * 0.5).to(torch.bfloat16)
    got = ops.linear(x.to(dev), packed.to(dev), qt, bias.to(dev), numerics)
    return got, go.gguf_linear_forward(x, packed, qt, bias, numerics=numerics), packed, x, bias


@pytest.mark.parametrize("qt", [go.Q8_0, go.Q4_0, go.Q5_1, go.Q3_K, go.Q4_K, go.Q6_K])
@pytest.mark.parametrize("n,k,m", [(4097, 256, 17), (4127, 512, 33), (4128, 768, 64), (6144, 2048, 40)])
def test_two_row_groups_per_workgroup(dev, qt, n, k, m):
    """Up to 8176 columns and K < 8192 a row's K is cut into the same pieces with one and two row groups per workgroup, so the
    first 4096 columns are the narrow matrix's, bit for bit."""
    print(f"case row groups qt={qt} {m}x{n}x{k}", flush=True)
    got, want, packed, x, bias = _both(dev, qt, n, k, m)
    narrow = ops.linear(x.to(dev), packed[:4096].contiguous().to(dev), qt, bias[:4096].to(dev), 1)
    assert torch.equal(got[:, :4096], narrow)
    assert go.rel_l2(got.cpu(), want) <= 1e-3


@pytest.mark.parametrize("qt", [go.Q8_0, go.Q5_0, go.Q2_K, go.Q4_K, go.Q5_K, go.Q6_K])
@pytest.mark.parametrize("n,k,m", [(8192, 1536, 17), (8193, 1536, 33), (12272, 1280, 50), (12304, 512, 64), (4096, 8192, 21), (4096, 8192, 26),
                                   (4080, 8192, 40), (4112, 8192, 33), (8200, 8192, 49)])
def test_wavefronts_per_workgroup(dev, qt, n, k, m):
    """Both sides of 256 workgroups, of K = 8192 and of the row counts from which four wavefronts take such rows."""
    print(f"case wavefronts qt={qt} {m}x{n}x{k}", flush=True)
    got, want, *_ = _both(dev, qt, n, k, m)
    assert go.rel_l2(got.cpu(), want) <= 1e-3


@pytest.mark.parametrize("numerics", [0, 1])
@pytest.mark.parametrize("n,k,m", [(8192, 256, 49), (8193, 768, 49), (12288, 256, 64), (12289, 512, 64), (16385, 256, 49), (24575, 256, 63),
                                   (24576, 256, 49), (12280, 1280, 48)])
def test_q5_k_row_groups(dev, numerics, n, k, m):
    """The widths between which Q5_K beyond 48 rows keeps one row group per workgroup."""
    print(f"case q5_k {m}x{n}x{k}", flush=True)
    got, want, *_ = _both(dev, go.Q5_K, n, k, m, numerics)
    assert go.rel_l2(got.cpu(), want) <= 1e-3


@pytest.mark.parametrize("n", [32771, 98339])
@pytest.mark.parametrize("k,m", [(256, 1), (512, 2), (1024, 1), (512, 5), (512, 16)])
def test_vocabulary_sized_q6_k(dev, n, k, m):
    """98339 columns: one super-block (one wavefront per workgroup) and more (two, by the rule for such widths); 32771: up to
    three by the count that fills the chip.  One and two rows are staged, more are not."""
    print(f"case vocabulary q6_k {m}x{n}x{k}", flush=True)
    packed = synthetic.make_packed(go.Q6_K, n, k, seed=k)
    x = synthetic.make_activations(m, k, seed=m)
    y = ops.linear(x.to(dev), packed.to(dev), go.Q6_K, None, 1)
    assert go.rel_l2(y.cpu(), go.gguf_linear_forward(x, packed, go.Q6_K, numerics=1)) <= 1e-3
    assert torch.equal(ops.lm_head_argmax(x.to(dev), packed.to(dev), go.Q6_K), y.float().argmax(dim=-1))
