"""GPU: the packed-half decode of Q4_K / Q6_K (fp16 and bf16 outputs of the fp16 rounding chain) against the one that
widens to fp32, bit for bit: one super-block, odd row counts, and more super-blocks than one pass of the grid covers."""
import pytest
import torch

from oracle import gguf_oracle as go
from sensenova_u1_amd import ops, synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qt", [go.Q4_K, go.Q6_K])
@pytest.mark.parametrize("n,k", [(1, 256), (7, 768), (129, 1280), (40003, 4096)])
def test_half_chain_decode_is_the_fp32_form_rounded(dev, qt, n, k):
    print(f"case half chain qt={qt} {n}x{k}", flush=True)
    packed = synthetic.make_packed(qt, n, k, seed=n + qt, device=dev)
    wide = ops.dequantize(packed, qt, torch.float32, ops.NUM_UPSTREAM_FP16)   # fp16 values, widened exactly
    half = ops.dequantize(packed, qt, torch.float16, ops.NUM_UPSTREAM_FP16)
    assert torch.equal(half.view(torch.int16), wide.half().view(torch.int16))
    bf16 = ops.dequantize(packed, qt, torch.bfloat16, ops.NUM_UPSTREAM_FP16)
    assert torch.equal(bf16.view(torch.int16), half.to(torch.bfloat16).view(torch.int16))
