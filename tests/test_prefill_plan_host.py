"""Which kernel a prefill GEMM call runs and what workspace it takes (hxq_prefill_gemm_plan), and
the bound over all types and formats.  No GPU: the plans count on 256 compute units then."""
import pytest

from helix_substrate import _hxq
from helix_substrate._hxq import FMT_SCALAR, FMT_SCALAR_U16, FMT_VQ2_P12

BF16, F32 = 1, 0


def plan(m, out, k, dt=BF16, fmt=FMT_SCALAR, group=128):
    return _hxq.lib().hxq_prefill_gemm_plan(m, out, k, dt, fmt, group)


def test_dtype_codes():
    import torch
    assert (_hxq.dtype_code(torch.float32), _hxq.dtype_code(torch.bfloat16)) == (F32, BF16)


@pytest.mark.parametrize("m,out,k", [(16, 3584, 18944), (64, 3584, 18944), (80, 8512, 2048),
                                     (512, 512, 3584), (5, 256, 256)])
def test_few_row_calls_take_no_workspace(m, out, k):
    assert plan(m, out, k) == -1
    if m <= 64:
        assert plan(m, out, k, F32) == -1


@pytest.mark.parametrize("m,out,k", [(m, out, k) for m in (1, 16, 64, 65, 128, 129, 300, 1001, 8192)
                                     for out in (16, 512, 1000, 3584, 18944)
                                     for k in (64, 512, 2048, 18944, 32768)])
def test_bound_covers_every_type_and_format(m, out, k):
    most = _hxq.lib().hxq_prefill_gemm_workspace_bytes(m, out, k)
    plans = [plan(m, out, k, dt, fmt, g) for dt in (BF16, 2, F32)
             for fmt in (FMT_SCALAR, FMT_SCALAR_U16, FMT_VQ2_P12) for g in (0, 16, 128, 16384)
             if not (fmt == FMT_VQ2_P12 and g)]
    assert most == max(0, max(plans))


def test_tiled_plan_splits_k():
    assert plan(1001, 1000, 512) > 0        # 32 tiles of 128 x 256, K in two ranges
    assert plan(8192, 8192, 3584) == 0      # 1024 tiles of 256 x 256: whole rounds, no split


@pytest.mark.parametrize("fmt,dt,few,tiled", [
    # two row blocks of X: W's subtiles times the row blocks, per CU, decide
    (FMT_SCALAR, BF16, [(65, 11008, 2048), (128, 10240, 8192), (128, 6144, 16384), (65, 3584, 18944)],
     [(65, 14336, 4096), (128, 14336, 4096), (96, 18944, 18944)]),
    (FMT_VQ2_P12, 2, [(65, 11008, 2048), (128, 6144, 16384)], [(65, 14336, 4096)]),
    (FMT_SCALAR_U16, BF16, [(65, 9216, 3584), (128, 8512, 2048), (65, 3584, 18944)],
     [(65, 10240, 2048), (65, 10240, 8192), (128, 18944, 3584), (65, 6144, 16384)]),
    (FMT_SCALAR_U16, F32, [(33, 18944, 3584), (64, 6144, 16384)], []),
    (FMT_SCALAR, F32, [(33, 18944, 3584), (64, 3584, 18944)], []),
])
def test_line_between_the_kernels(fmt, dt, few, tiled):
    group = 0 if fmt == FMT_VQ2_P12 else 128
    for s in few:
        assert plan(*s, dt, fmt, group) == -1, s
    for s in tiled:
        assert plan(*s, dt, fmt, group) >= 0, s


@pytest.mark.parametrize("experts,top_k,few,tiled", [
    (8, 2, (1, 16, 48), (49,)), (16, 2, (4, 96), (97, 112)), (32, 4, (8, 64), (80, 96)),
    (64, 8, (1, 4, 16, 48), (56, 64, 96)), (128, 8, (4, 64), (80,)), (256, 8, (8, 64), (97,)),
])
def test_grouped_line_holds_for_uneven_routing(experts, top_k, few, tiled):
    """Tokens up to which 16-row tiles are no slower than 64-row ones, however few experts they go to."""
    tile = _hxq.lib().hxq_moe_grouped_tile
    for t in few:
        assert tile(t * top_k, experts, BF16, 2048, 128) == 16, t
        assert tile(t * top_k, experts, F32, 2048, 128) == 128
        assert tile(t * top_k, experts, BF16, 2046, 128) == 64   # no whole 16-byte rows of Y
        assert tile(t * top_k, experts, BF16, 2048, 16384) == 64
    for t in tiled:
        assert tile(t * top_k, experts, BF16, 2048, 128) == 64, t
    assert tile(97 * experts, experts, BF16, 2048, 128) == 128
    assert tile(193 * experts, experts, BF16, 2048, 128) == 256
