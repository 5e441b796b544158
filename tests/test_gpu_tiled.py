"""hxq_prefill_gemm past the line where the tiled kernel takes over from the few-row one: ragged
tiles of X and W, one and several launches, K in one and several ranges, every index format and
affine group layout, dense and repeated sidecars, operands bit for bit.  Each case asserts which
kernel its call runs."""
import numpy as np
import pytest
import torch

import oracle
from helix_substrate import _hxq
from helix_substrate.hxq_format import padded_in_features
from test_gpu_anyk import _check_module, _scalar
from test_gpu_formats import FMTS, _case, _dev, _grp, _wide_layer
from test_gpu_rows import _check

pytestmark = pytest.mark.gpu

U8, U16 = _hxq.FMT_SCALAR, _hxq.FMT_SCALAR_U16


def _plan(m, out, inp, xdt, fmt=U8, G=128):
    has_affine = G and fmt in (U8, U16, _hxq.FMT_AF6)
    p = _hxq.lib().hxq_prefill_gemm_plan(m, out, inp, _hxq.dtype_code(xdt), fmt, G if has_affine else 0)
    assert p >= 0, "the few-row kernel would run"
    return p


@pytest.mark.parametrize("fmt", [U8, U16] + FMTS)
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float16, torch.float32])
def test_tiled_formats(dev, fmt, xdt):
    assert _plan(1001, 1000, 1024, xdt, fmt) > 0   # K in ranges
    _check(dev, fmt, 1001, 1000, 1024, 128, xdt)


@pytest.mark.parametrize("m,out,inp,G", [
    (1001, 1000, 576, 48), (515, 3000, 512, 16), (1001, 1000, 1088, 32), (777, 1100, 1344, 96),
    (1030, 8200, 448, 64),   # 256-row tiles
    (2300, 8200, 512, 128),  # more tiles than compute units: the last ones in a launch of their own
])
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float32])
def test_tiled_groups_and_tiles(dev, m, out, inp, G, xdt):
    _plan(m, out, inp, xdt, U8, G)
    _check(dev, U8, m, out, inp, G, xdt)


@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float32])
def test_tiled_dense_sidecar(dev, xdt):
    """5 % of the weights: some 200 entries per row group and step."""
    _plan(1001, 1000, 512, xdt)
    _check(dev, U8, 1001, 1000, 512, 128, xdt, density=0.05)


@pytest.mark.parametrize("fmt,G", [(U8, 16), (U8, 48), (U8, 64), (U8, 192), (U16, 64), (U16, 48)]
                         + [(f, 64) for f in FMTS])
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float16, torch.float32])
def test_tiled_operands_bit_exact(dev, fmt, G, xdt):
    """Rows of the identity, six times over: each output element is one operand times 1."""
    out, inp, reps = 1000, 192, 6
    if fmt == U16:
        mod, W, Wf = _wide_layer(out, inp, 3000, seed=G, group_size=G, density=0.01, fma=True)
        raw, cb, aff, gp, gk, gv = _dev(dev, mod.indices, mod.codebook, mod._affine_t,
                                        mod._sc_grp_ptr, mod._sc_grp_key, mod._sc_grp_val)
    elif fmt == U8:
        mod, W, Wf = _scalar(out, inp, G, seed=G, fma=True)
        raw, cb, aff, gp, gk, gv = _dev(dev, mod.indices, mod._kcb, mod._affine_t,
                                        mod._sc_grp_ptr, mod._sc_grp_key, mod._sc_grp_val)
    else:
        raw, cb, s, o, pos, val, W, _ = _case(fmt, out, inp, G=G, nsc=0.01, seed=3)
        Wf = W if s is None else _case(fmt, out, inp, G=G, nsc=0.01, seed=3, fma=True)[6]
        aff = None if s is None else np.ascontiguousarray(np.stack([s.T, o.T], axis=-1))
        raw, cb, aff = _dev(dev, raw, cb, aff)
        gp, gk, gv = _grp(dev, pos, val, out, inp)
    _plan(reps * inp, out, inp, xdt, fmt, G)
    x = torch.eye(inp, dtype=xdt, device=dev).repeat(reps, 1)
    print(f"tiled one-hot fmt={fmt} G={G} x={xdt}", flush=True)
    y = _hxq.prefill_gemm(x, raw, cb, aff, G, gp, gk, gv, out_dtype=torch.float32, fmt=fmt,
                          out_features=out)
    want = torch.from_numpy(np.ascontiguousarray(W if xdt == torch.float32 else Wf)).to(xdt).float()
    want = want.t().to(dev)
    for r in range(reps):
        assert torch.equal(y[r * inp:(r + 1) * inp], want), r


@pytest.mark.parametrize("out_f,in_f,G", [
    (1000, 1000, 0),    # no affine, K padded to 1024
    (1040, 1040, 16),   # 16-column groups, padded groups of zeros
    (1000, 4000, 32),
])
def test_tiled_any_k(dev, out_f, in_f, G):
    print(f"tiled any-K out={out_f} in={in_f} G={G}", flush=True)
    for xdt in (torch.float32, torch.bfloat16):
        _plan(1001, out_f, padded_in_features(in_f), xdt, U8, G)
    m, W = _scalar(out_f, in_f, G, seed=in_f + G)
    _check_module(m.to(dev), W, dev, rows=(1001,))


def test_tiled_without_sidecar(dev):
    L = _scalar(1000, 512, 128, seed=1)[0].to(dev)
    _plan(1001, 1000, 512, torch.bfloat16)
    x = torch.randn(1001, 512, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16)
    y = _hxq.prefill_gemm(x.to(dev), L.indices, L._kcb, L._affine_t, 128, None, None, None, None,
                          out_dtype=torch.float32)
    t = [a.cpu().numpy() for a in (L.indices, L.codebook, L.group_scale, L.group_offset)]
    W = oracle.reconstruct(*t, 128, None, None, fma=True)
    W16 = torch.from_numpy(W).to(torch.bfloat16).float().numpy()
    ref = oracle.linear_np(x.float().numpy(), W16)
    assert np.abs(y.cpu().numpy() - ref).max() <= 2e-5 * np.abs(ref).max()
