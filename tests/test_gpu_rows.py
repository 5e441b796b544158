"""hxq_prefill_gemm on few rows of X (hxq_rows.h) at the edges of its tiles: 16-row tiles of X
and W, 64-row blocks, one 64-column step up to several per wave, runs of 1, 2, 3 and 5 subtiles,
every affine group layout and index format, sidecars denser than the 32 entries a row group
holds per iteration."""
import numpy as np
import pytest
import torch

import oracle
from helix_substrate import _hxq
from test_gpu_formats import FMTS, _case, _dev, _grp, _maxrel, _wide_layer

pytestmark = pytest.mark.gpu


def _check(dev, fmt, m, out, inp, G, xdt, density=0.001):
    if fmt == _hxq.FMT_SCALAR_U16:
        mod, W, Wf = _wide_layer(out, inp, 3000, seed=m + out, group_size=G, density=density, fma=True)
        raw, cb, aff, gp, gk, gv = _dev(dev, mod.indices, mod.codebook, mod._affine_t,
                                        mod._sc_grp_ptr, mod._sc_grp_key, mod._sc_grp_val)
    elif fmt == _hxq.FMT_SCALAR:
        from helix_substrate import synth
        L = synth.make_layer_np(out, inp, seed=m + inp, group_size=G, density=density)
        args = (L["indices"], L["codebook"], L["group_scale"], L["group_offset"], G,
                L["sidecar_positions"], L["sidecar_values"])
        W, Wf = oracle.reconstruct(*args), oracle.reconstruct(*args, fma=True)
        aff = np.ascontiguousarray(np.stack([L["group_scale"].T, L["group_offset"].T], axis=-1))
        raw, cb, aff = _dev(dev, L["indices"], L["codebook"], aff)
        gp, gk, gv = _grp(dev, L["sidecar_positions"], L["sidecar_values"], out, inp)
    else:
        raw, cb, s, o, pos, val, W, _ = _case(fmt, out, inp, G=G, seed=m + inp)
        Wf = W if s is None else _case(fmt, out, inp, G=G, seed=m + inp, fma=True)[6]
        aff = None if s is None else np.ascontiguousarray(np.stack([s.T, o.T], axis=-1))
        raw, cb, aff = _dev(dev, raw, cb, aff)
        gp, gk, gv = _grp(dev, pos, val, out, inp)
    g = torch.Generator().manual_seed(m)
    x = torch.randn(m, inp, generator=g).to(xdt)
    bias = torch.randn(out, generator=g) * 0.1
    print(f"rows fmt={fmt} m={m} out={out} in={inp} G={G} x={xdt}", flush=True)
    args = (x.to(dev), raw, cb, aff, G, gp, gk, gv, bias.to(dev))
    y = _hxq.prefill_gemm(*args, out_dtype=torch.float32, fmt=fmt, out_features=out)
    xf = x.float().numpy()
    # fp32 X: order of fp32 sums only; 16-bit X: likewise, once W is rounded as the operands are
    Wr, bar = (W, 1e-5) if xdt == torch.float32 else (torch.from_numpy(Wf).to(xdt).float().numpy(), 2e-5)
    rel = _maxrel(y.cpu().numpy(), oracle.linear_np(xf, Wr, bias.numpy()))
    assert rel <= bar, rel
    assert torch.equal(_hxq.prefill_gemm(*args, out_dtype=torch.float32, fmt=fmt, out_features=out), y)
    y16 = _hxq.prefill_gemm(*args, fmt=fmt, out_features=out)
    assert torch.equal(y16, y.to(xdt))   # the same sums, rounded once


@pytest.mark.parametrize("m,out,inp,G", [
    (1, 16, 64, 64), (5, 15, 64, 16), (16, 17, 1088, 32), (17, 81, 1024, 128), (33, 300, 2048, 128),
    (64, 4100, 448, 64), (65, 530, 576, 48), (130, 100, 4160, 64), (16, 12300, 320, 64),
    (40, 20500, 192, 64), (48, 256, 8256, 64),
])
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float32])
def test_rows_edges(dev, m, out, inp, G, xdt):
    _check(dev, _hxq.FMT_SCALAR, m, out, inp, G, xdt)


@pytest.mark.parametrize("fmt", FMTS + [_hxq.FMT_SCALAR_U16])
@pytest.mark.parametrize("m,out,inp", [(7, 48, 128), (31, 5000, 640), (63, 258, 1152)])
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float16, torch.float32])
def test_rows_formats(dev, fmt, m, out, inp, xdt):
    _check(dev, fmt, m, out, inp, 128 if inp % 128 == 0 else 64, xdt)


@pytest.mark.parametrize("fmt", [_hxq.FMT_SCALAR, _hxq.FMT_SCALAR_U16] + FMTS)
@pytest.mark.parametrize("out", [6400, 11200, 18944])   # runs of 2, 3 and 5 (uint16: 3) subtiles
@pytest.mark.parametrize("m", [5, 20, 40, 64])          # 1 to 4 row tiles (fp32: 1 or 2)
def test_rows_every_run_and_row_tile(dev, fmt, out, m):
    for xdt in [torch.bfloat16, torch.float32] if m != 64 else [torch.float16]:
        assert _hxq.lib().hxq_prefill_gemm_plan(m, out, 192, _hxq.dtype_code(xdt), fmt,
                                                0 if fmt in FMTS[:2] else 64) == -1
        _check(dev, fmt, m, out, 192, 64, xdt)


@pytest.mark.parametrize("m,out,inp", [(9, 130, 512), (20, 8200, 256)])
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float32])
def test_rows_dense_sidecar(dev, m, out, inp, xdt):
    """5 % of the weights: some 200 entries per row group and step."""
    _check(dev, _hxq.FMT_SCALAR, m, out, inp, 128, xdt, density=0.05)


@pytest.mark.parametrize("m,out,inp", [(16, 48, 192), (16, 48, 64 * 67), (40, 48, 192)])
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float32])
def test_rows_infinite_unused_entry(dev, m, out, inp, xdt):
    """Step counts that are no multiple of a wave's steps per iteration, with an infinite
    codebook entry 0 that no index uses: the result is the one with that entry finite."""
    g = torch.Generator().manual_seed(inp)
    idx = torch.randint(1, 256, (out, inp), generator=g, dtype=torch.uint8).to(dev)
    cb = torch.randn(256, generator=g)
    x = torch.randn(m, inp, generator=g).to(xdt).to(dev)
    print(f"rows inf entry m={m} out={out} in={inp} x={xdt}", flush=True)
    ys = []
    for v in (0.0, float("inf")):
        cb[0] = v
        ys.append(_hxq.prefill_gemm(x, idx, cb.to(dev), None, 128, None, None, None, None,
                                    out_dtype=torch.float32))
    assert torch.isfinite(ys[0]).all() and torch.equal(ys[0], ys[1])


_MANY = tuple((0, 1, 0, 0, 2, 0, 18)[e % 7] if e % 5 == 0 else e % 2 for e in range(150))


@pytest.mark.parametrize("counts,out,inp", [
    (c, out, inp) for out, inp in ((64, 64), (336, 576), (1024, 2048))
    for c in ((1,), (0, 1, 0, 16), (17, 0, 3, 33), (0, 0, 5), (2, 2, 2, 2, 2, 2, 2),
              (0, 17, 0, 0, 33, 0, 0, 1))] + [(_MANY, 64, 64)])
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float16])
def test_rows_grouped(dev, counts, out, inp, xdt):
    """Experts of few, no and just over 16 or 32 rows, more experts than lanes of a wave; runs of
    five subtiles that end inside a block.  (17, 0, 3, 33) is past the line: 64-row tiles."""
    from helix_substrate import synth
    from helix_substrate.moe import bank_to, stack_bank
    E, n = len(counts), sum(counts)
    tile = _hxq.lib().hxq_moe_grouped_tile(n, E, _hxq.dtype_code(xdt), out, 64)
    assert tile == (64 if counts == (17, 0, 3, 33) else 16)
    Ls = [synth.make_layer_np(out, inp, seed=e, group_size=64, density=0.01) for e in range(E)]
    bank = bank_to(stack_bank([synth.to_torch(L) for L in Ls]), dev)
    bank["group_size"] = 64
    g = torch.Generator().manual_seed(n)
    rows = torch.randint(0, 9, (n,), generator=g).to(torch.int32)
    x = torch.randn(9, inp, generator=g).to(xdt)
    off = torch.tensor(np.concatenate([[0], np.cumsum(counts)]), dtype=torch.int32)
    print(f"rows grouped counts={counts} out={out} in={inp} x={xdt}", flush=True)
    y = _hxq.moe_grouped_gemm(x.to(dev), rows.to(dev), off.to(dev), bank, n).cpu().numpy()
    for e, L in enumerate(Ls):
        lo, hi = int(off[e]), int(off[e + 1])
        if lo == hi:
            continue
        W = oracle.reconstruct(L["indices"], L["codebook"], L["group_scale"], L["group_offset"], 64,
                               L["sidecar_positions"], L["sidecar_values"], fma=True)
        W16 = torch.from_numpy(W).to(xdt).float().numpy()
        ref = oracle.linear_np(x[rows[lo:hi].long()].float().numpy(), W16)
        assert _maxrel(y[lo:hi], ref) <= 2e-5, e   # operands equal: order of fp32 sums


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_rows_paired_banks(dev, dt):
    """Gate and up of one launch against the two run by themselves: the same sums, so what is
    left is how the product gate / (1 + exp(-gate)) * up rounds to 16 bits (at most one step
    of 2^-8 on a few of 256 terms)."""
    from helix_substrate import moe
    from test_gpu_moe import _bank, _skewed_logits
    T, E, k, H, I = 25, 12, 3, 320, 256
    bg, bu, bd = (_bank(E, o, i, seed=s, dev=dev, group_size=64)[1]
                  for o, i, s in ((I, H, 10), (I, H, 30), (H, I, 50)))
    for n_out in (I, H):
        assert _hxq.lib().hxq_moe_grouped_tile(T * k, E, _hxq.dtype_code(dt), n_out, 64) == 16
    x = torch.randn(T, H, generator=torch.Generator().manual_seed(3)).to(dt).to(dev)
    r = _hxq.moe_route(_skewed_logits(T, E, 2, dev), k, False)
    print(f"paired banks {dt}", flush=True)
    y = _hxq.moe_ffn(x, r, bg, bu, bd, out_dtype=torch.float32)
    gate, up = (_hxq.moe_grouped_gemm(x, r.sorted_rows, r.expert_offsets, b, T * k, out_dtype=dt).float()
                for b in (bg, bu))
    act = (torch.nn.functional.silu(gate) * up).to(dt)
    o = _hxq.moe_grouped_gemm(act, None, r.expert_offsets, bd, T * k, out_dtype=dt).float()
    ref = (o[r.assign_pos.long().view(T, k)] * r.topk_weights.view(T, k, 1)).sum(1)
    assert float((y - ref).abs().max()) <= 2.0 ** -8 * float(ref.abs().max())


def test_rows_allocate_nothing(dev):
    """A few-row call into a given output allocates no workspace, whatever K is."""
    m, out, inp = 16, 512, 18944
    idx = torch.randint(0, 256, (out, inp), dtype=torch.uint8, device=dev)
    cb = torch.randn(256, device=dev)
    x = torch.randn(m, inp, device=dev).to(torch.bfloat16)
    y = torch.empty(m, out, dtype=torch.bfloat16, device=dev)
    args = (x, idx, cb, None, 128, None, None, None)
    _hxq.prefill_gemm(*args, out=y)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    _hxq.prefill_gemm(*args, out=y)
    assert torch.cuda.max_memory_allocated() == before
