"""What 17 rows to two thousand ask for and how they run, without a device: whole fp32 copies of the outputs where a K split pays,
nothing elsewhere."""
import pytest

from sensenova_u1_amd import ops
from tests.test_gpu_mid_rows import INSTANCES, PAIRS, PROJECTIONS, workspace_bytes

TYPES = [ops.Q4_0, ops.Q4_1, ops.Q5_0, ops.Q5_1, ops.Q8_0, ops.Q2_K, ops.Q3_K, ops.Q4_K, ops.Q5_K, ops.Q6_K]


@pytest.mark.parametrize("qt", TYPES)
def test_scratch_of_17_to_64_rows(qt):
    size = ops.load_library().sngguf_linear_scratch_bytes
    for m in (17, 32, 40, 64):
        for n, k in ((512, 12288), (1024, 4096), (4096, 4096), (6144, 4096), (4096, 12288), (515, 2048), (12288, 4096)):
            nbytes = size(qt, m, n, k)
            copies = nbytes // (4 * m * n)
            # two halves of K per workgroup: at least two super-blocks of 256 in a slice
            assert nbytes % (4 * m * n) == 0 and copies != 1 and copies <= min(16, k // 512) and nbytes <= 64 << 20
        assert size(qt, m, 4096, 12288) > 0          # 64 workgroups of 64 columns would leave three quarters of the device idle
        assert size(qt, m, 4096, 256) == 0 and size(qt, m, 12288, 512) == 0
    assert size(qt, 16, 4096, 12288) == 0 and size(qt, 0, 4096, 12288) == 0 and size(qt, 513, 4096, 4096) == 0
    assert size(qt, 40, 0, 4096) == 0 and size(qt, 40, 4096, 4096 + 128) == 0 and size(qt, 40, 4096, -256) == 0


def test_no_scratch_for_other_types():
    size = ops.load_library().sngguf_linear_scratch_bytes
    assert size(ops.BF16, 40, 4096, 12288) == 0 and size(16, 40, 4096, 12288) == 0


@pytest.mark.parametrize("qt", TYPES)
def test_pairs_of_few_columns_split_k_at_17_to_64_rows(qt):
    """A pair of few columns leaves most of the device idle unless K is split; the least workspace (the gate outputs) still runs, and
    more than the shape asks for changes nothing."""
    for m in (17, 33, 64):
        for n, k in ((512, 12288), (1024, 4096), (2048, 12288), (4096, 4096), (4096, 12288)):
            nbytes, copy = ops.gate_up_silu_ws_bytes(qt, m, n, k), 8 * m * n
            plan = ops.mid_plan(qt, m, n, k, True, nbytes)
            assert plan[3] >= 2 and nbytes == plan[3] * copy <= min(64 << 20, ops.gate_up_silu_workspace_bytes(n, k))
            assert ops.mid_plan(qt, m, n, k, True, 1 << 40) == plan
            least = ops.mid_plan(qt, m, n, k, True, 2 * m * n)
            assert least is None or least[3] == 1
        # (17 rows: two launches of the decode kernel, 37 - 42 us, instead of 48 super-blocks one after the other, 42 - 58)
        assert m > 17 or ops.mid_plan(qt, m, 512, 12288, True, 2 * m * 512) is None
        assert ops.gate_up_silu_ws_bytes(qt, m, 12288, 4096) == 2 * m * 12288 and ops.gate_up_silu_ws_bytes(qt, m, 512, 256) == 2 * m * 512


@pytest.mark.parametrize("qt,m,n,k,workspace", [
    (ops.Q6_K, 17, 24576, 2048, 1 << 30),      # decode kernel 22 us, mid-size kernel 25
    (ops.Q4_K, 17, 1024, 4096, 1 << 30),       # 8.6, 9.4
    (ops.Q5_K, 17, 1024, 4096, 1 << 30),       # 8.8, 9.8
    (ops.Q6_K, 64, 4096, 12288, 0),            # no scratch, no K split: 51, 67
    (ops.Q6_K, 1024, 12288, 4096, 1 << 40),    # weight pass and dense launch 110, mid-size kernel 123
    (ops.Q6_K, 1024, 24576, 2048, 1 << 40)])   # 125, 134
def test_projections_stay_on_the_faster_kernel(qt, m, n, k, workspace):
    """Formats whose decode takes longer than the one that a shared estimate was fitted to, and 17 rows, where the decode kernel's
    second operand is nearly empty."""
    assert ops.mid_plan(qt, m, n, k, False, workspace) is None


def test_projections_on_the_mid_size_kernel():
    """(us as above, all ten formats within a few per cent): 48 rows of 4096 x 12288 37 / 21, 64 rows of 12288 x 4096 44 / 24, 203 rows of
    6144 x 4096 37 / 31; 1024 rows of 12288 x 4096 in Q8_0 108 / 105."""
    for qt in TYPES:
        for m, n, k in ((48, 4096, 12288), (64, 12288, 4096), (203, 6144, 4096), (509, 4096, 12288)):
            assert ops.mid_plan(qt, m, n, k, False, 1 << 40) is not None
    assert ops.mid_plan(ops.Q8_0, 1024, 12288, 4096, False, 1 << 40) is not None
    assert ops.mid_plan(ops.Q8_0, 2048, 12288, 4096, False, 1 << 40) is None and ops.mid_plan(ops.BF16, 40, 4096, 4096, False, 1 << 30) is None


@pytest.mark.parametrize("qt", TYPES)
@pytest.mark.parametrize("pair", [False, True])
def test_more_than_what_is_asked_for_changes_nothing(qt, pair):
    """Which kernel runs and how K is cut is the shape's own, whatever a caller's scratch or a pool has grown to."""
    for m in (17, 33, 48, 64, 65, 130, 300, 509, 1024, 1500):
        for n in (8, 512, 515, 1024, 2056, 4096, 6144, 9728, 24576):
            for k in (256, 1024, 2048, 4096, 12288):
                nbytes = workspace_bytes(qt, m, n, k, pair)
                if (nbytes == 0 and m > 64) or (pair and n % 8):
                    continue
                plan = ops.mid_plan(qt, m, n, k, pair, nbytes)
                for more in (nbytes + 16, 2 * nbytes + (32 << 20), 1 << 40):
                    assert ops.mid_plan(qt, m, n, k, pair, more) == plan, (m, n, k, more)


FORMS = {64: (2, 3, 4), 128: (2, 3, 4, 6, 8, 10, 13), 256: (10, 13, 16)}   # columns of a workgroup: 16-row tiles of its instances


@pytest.mark.parametrize("qt", TYPES)
@pytest.mark.parametrize("pair,shapes", [(False, PROJECTIONS), (True, PAIRS)])
def test_the_parity_tests_run_every_instance(qt, pair, shapes):
    """What the shapes of the parity tests are listed for: all thirteen forms and sizes, with and without a K split in each form."""
    assert {s: ops.mid_plan(qt, *s, pair, workspace_bytes(qt, *s, pair)) for s in shapes} == shapes
    assert {p[:2] for p in shapes.values()} == {(cols, mt) for cols in FORMS for mt in FORMS[cols]}
    assert {(p[0], p[3] > 1) for p in shapes.values()} == {(cols, split) for cols in FORMS for split in (False, True)}
    enough = lambda m, n, k: ops.gate_up_silu_workspace_bytes(n, k) + 2 * m * n
    assert len({ops.mid_plan(qt, *s, True, enough(*s))[:2] for s in INSTANCES}) == 13
