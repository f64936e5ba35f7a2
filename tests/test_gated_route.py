"""Which gate / up pairs beyond 16 rows ``gated_mlp`` hands to one library call: the rule needs no device, only sizes, types
and what is registered on the two projections."""
import types

import pytest
import torch

from sensenova_u1_amd import GGUFLinear, GGUFParameter, modality, ops

SPLIT_PAIRS = [(ops.Q8_0, 6144, 2048, 203), (ops.Q4_K, 9728, 2560, 511), (ops.Q8_0, 6144, 2048, 512), (ops.Q4_K, 9728, 2560, 512),
               (ops.Q8_0, 4096, 4096, 768), (ops.Q8_0, 8960, 3584, 512)]
FILLED = (ops.Q8_0, 12288, 4096, 4096)   # the dense gated launch, whose tiles fill the chip


class Adapted(GGUFLinear):
    def forward(self, inputs):
        return super().forward(inputs) + 1


def _linear(qt, n, k, cls=GGUFLinear, compute_dtype=torch.bfloat16):
    bs, ts = ops.GGML_QUANT_SIZES[qt]
    lin = cls(k, n, bias=False, compute_dtype=compute_dtype, device="meta")
    lin.weight = GGUFParameter(torch.empty((n, k // bs * ts), dtype=torch.uint8, device="meta"), quant_type=qt)
    return lin


def _route(rows, gate, up):
    x = types.SimpleNamespace(is_cuda=True, dtype=torch.bfloat16)   # (what the rule reads of its input beyond 64 rows)
    return modality._gated_tile_route(x, rows, True, gate, up)


@pytest.mark.parametrize("qt,n,k,rows", SPLIT_PAIRS)
def test_a_forward_of_its_own_is_called(qt, n, k, rows):
    plain = _linear(qt, n, k)
    assert _route(rows, plain, _linear(qt, n, k))
    assert not _route(rows, plain, _linear(qt, n, k, cls=Adapted)) and not _route(rows, _linear(qt, n, k, cls=Adapted), plain)
    patched = _linear(qt, n, k)
    patched.forward = lambda inputs: inputs
    assert not _route(rows, patched, plain)


@pytest.mark.parametrize("qt,n,k,rows", SPLIT_PAIRS)
def test_hooks_keep_the_module_calls(qt, n, k, rows):
    gate, up = _linear(qt, n, k), _linear(qt, n, k)
    every = torch.nn.modules.module
    hook = lambda *args: None
    for register in (up.register_forward_hook, gate.register_forward_pre_hook, up.register_full_backward_hook,
                     gate.register_full_backward_pre_hook, every.register_module_forward_hook, every.register_module_forward_pre_hook,
                     every.register_module_full_backward_hook, every.register_module_full_backward_pre_hook):
        handle = register(hook)
        try:
            assert not _route(rows, gate, up), register
        finally:
            handle.remove()
    assert _route(rows, gate, up)


@pytest.mark.parametrize("qt,n,k,rows", SPLIT_PAIRS)
def test_another_compute_dtype_is_left_to_the_modules(qt, n, k, rows):
    """(a bf16 input to an fp16 or fp32 module: its forward raises)"""
    for other in (torch.float16, torch.float32):
        assert not _route(rows, _linear(qt, n, k), _linear(qt, n, k, compute_dtype=other))
        assert not _route(rows, _linear(qt, n, k, compute_dtype=other), _linear(qt, n, k))
    assert _route(rows, _linear(qt, n, k, compute_dtype=None), _linear(qt, n, k))


def test_the_filled_dense_launch_stays_what_it_was():
    qt, n, k, rows = FILLED
    assert _route(rows, _linear(qt, n, k), _linear(qt, n, k, cls=Adapted))


def test_the_route_follows_the_form():
    """Everything the library has a faster form for, and nothing else; the dense launch where its tiles fill the chip."""
    for qt in (ops.Q8_0, ops.Q4_K, ops.Q6_K, ops.BF16):
        for n, k in ((12288, 4096), (9728, 2560), (6144, 2048), (4096, 4096), (512, 16384), (1536, 1024), (14336, 8192), (516, 1024)):
            gate, up = _linear(qt, n, k), _linear(qt, n, k)
            for rows in (1, 16, 65, 203, 511, 512, 768, 1000, 1024, 2048, 4095, 4096, 5000):
                form = ops.gate_up_silu_ws_form(qt, rows, n, k)
                assert _route(rows, gate, up) == (form != ops.PAIR_SEPARATE)
                fits = ops.gate_up_silu_ws_fits(qt, rows, n, k)
                filled = rows >= modality.GATED_TILE_MIN_ROWS and modality.gated_tile_fill(rows, n) >= modality.GATED_TILE_MIN_FILL
                assert (form == ops.PAIR_DENSE) == (fits and filled)
                few = -(-rows // 256) * -(-n // 256) <= 128 and 65 <= rows < 4096 and 4 * rows <= k
                assert (form == ops.PAIR_SPLIT) == (fits and not filled and few and qt in (ops.Q8_0, ops.Q4_K))
    # thousands of rows on a narrow pair with very long rows: no form but the dense launch, and that one badly filled
    assert ops.gate_up_silu_ws_form(ops.Q8_0, 4096, 512, 16384) == ops.PAIR_SEPARATE
    assert ops.gate_up_silu_ws_form(ops.Q6_K, 40, 512, 1024) == ops.PAIR_DECODE
    assert ops.gate_up_silu_ws_form(ops.Q8_0, 40, 512, 1152) == ops.PAIR_SEPARATE   # K in whole 128, not 256, elements


def test_workspace_is_what_the_form_needs():
    """2 M N bytes for the gate outputs up to 64 rows; whole fp32 copies of both outputs for a K split, within what the dense
    form would take; the interleaved weights for the dense form; never more than the size that is enough at any M."""
    for qt, m, n, k in ((ops.Q8_0, 17, 12288, 4096), (ops.Q6_K, 64, 9728, 2560), (ops.Q2_K, 33, 8, 256)):
        assert ops.gate_up_silu_ws_bytes(qt, m, n, k) == 2 * m * n
    for qt, m, n, k in ((ops.Q8_0, 65, 12288, 4096), (ops.Q4_K, 203, 12288, 4096), (ops.Q8_0, 509, 12288, 4096), (ops.Q4_K, 512, 9728, 2560)):
        nbytes = ops.gate_up_silu_ws_bytes(qt, m, n, k)
        assert 0 < nbytes <= ops.gate_up_silu_workspace_bytes(n, k) and nbytes % (8 * m * n) == 0
    for qt, m, n, k in ((ops.Q8_0, 40, 512, 384), (ops.Q6_K, 203, 12288, 4096), FILLED[:1] + FILLED[3:] + FILLED[1:3], (ops.Q8_0, 300, 512, 256)):
        assert ops.gate_up_silu_ws_bytes(qt, m, n, k) == ops.gate_up_silu_workspace_bytes(n, k)
    for qt, m, n, k in ((ops.Q8_0, 16, 512, 256), (ops.Q8_0, 300, 516, 256), (ops.Q8_0, 300, 512, 192), (ops.BF16, 300, 512, 256)):
        assert ops.gate_up_silu_ws_bytes(qt, m, n, k) == 0
