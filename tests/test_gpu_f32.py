"""fp32 attention up to head dim 128 on the wave-split kernels (born_f32.h):
32 stationary rows per workgroup, every fourth 32-row tile per wave.  Cases
sit where that split can go wrong: fewer tiles than waves, a partial last
tile or block, one and four waves per block, padded head dims of each column count, and every mask.

The bounds are those of the Born and purified backward tests: 1e-5 (Born,
forward) and 1e-4 (purified gradients) of the largest value, or 1e-6 (17 ulps)
of the largest sum of terms for gradients that cancel.  dscale (sum of delta / Z) is checked where every row
sees many keys: a single overlap near zero carries its own relative error into
1 / Z, whatever sums it.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import born_oracle as orc
from test_gpu_backward import _check_bwd
from test_gpu_purified import FLOOR, GTOL
from util import TOL, f64, max_abs, rel_err, seeded_inputs

pytestmark = pytest.mark.gpu

MASKS = {
    "causal": (True, 0, False),
    "dense": (False, 0, False),
    "window": (True, 37, False),
    "window_nc": (False, 37, False),
    "docs": (True, 0, True),
    "docs_window": (True, 50, True),
    "docs_dense": (False, 0, True),
}


def check_pur_fixed(B, H, T, D, dtype, mask, scale, tau, std, device, doc):
    """Purified attention with a fixed scale and tau (one that is trained keeps
    the other kernels in fp32 and fp16): output, dq, dk, dv."""
    from quantumdlblocks_amd import flash_purified_born_attention

    causal, window, _ = mask
    q, k, v, do = (x.to(device) for x in seeded_inputs((B, H, T, D), seed=T + D, std=std, n=4, dtype=dtype))
    print(f"purified, fixed scale: B{B} H{H} T{T} D{D} {dtype} {mask}", flush=True)
    q, k, v = (x.requires_grad_(True) for x in (q, k, v))
    st, tt = (torch.tensor(x, dtype=torch.float32, device=device) for x in (scale, tau))
    doc_t = None if doc is None else torch.as_tensor(doc, dtype=torch.int32, device=device)
    out = flash_purified_born_attention(q, k, v, st, tt, 0.05, is_causal=causal, window_size=window, doc_ids=doc_t)
    out.backward(do)
    n = [f64(x) for x in (q, k, v)]
    args = (*n, np.asarray(scale), np.asarray(tau))
    okw = dict(eps_base=0.05, is_causal=causal, eps=1e-8, window_size=window, doc_ids=doc)
    ref, _ = orc.purified_forward(*args, **okw)
    assert rel_err(f64(out), ref) <= TOL[dtype], rel_err(f64(out), ref)
    want = orc.purified_backward(*args, f64(do), **okw)
    mags = orc.purified_backward_magnitudes(*args, f64(do), **okw)
    for name, got, w, m in zip(("dq", "dk", "dv"), (q.grad, k.grad, v.grad), want, mags):
        er, ef = rel_err(f64(got), w), max_abs(f64(got), w) / m.max()
        assert er <= GTOL[dtype] or ef <= FLOOR[dtype], f"{name}: rel {er:.3e}, vs term scale {ef:.3e}"


def _case(H, T, D, mask, purified, device, sorted_docs=True):
    causal, window, docs = MASKS[mask]
    doc = None
    if docs:
        doc = orc.geometric_doc_ids(2, T, 23.0, seed=T + D)
        if not sorted_docs:
            doc = np.random.default_rng(T).permuted(doc, axis=1)
    scale = [1.5 - 0.2 * (h % 5) for h in range(H)]
    if purified:
        # Documents have rows that see one key, whose weight p = (gamma (x -
        # tau))^4 carries 4 err(x) / |x - tau|: with the overlaps' err(x) up to
        # 4e-7 (|x| within 3 at std 0.3) that is 1e-5 once |x - tau| < 0.16, so
        # their tau lies below every overlap.
        tau = [(-6.0 if docs else 0.05) - 0.03 * (h % 4) for h in range(H)]
        check_pur_fixed(2, H, T, D, torch.float32, MASKS[mask], scale, tau, 0.3, device, doc)
    else:
        if H > 1:
            scale[1] = -0.8
        _check_bwd(2, H, T, D, torch.float32, device, scale=scale, is_causal=causal, window_size=window, doc=doc,
                   std=0.5, seed=H + T + D, check_dscale=mask == "dense" and T > 32)


@pytest.mark.parametrize("purified", [False, True], ids=["born", "purified"])
@pytest.mark.parametrize("mask", list(MASKS))
@pytest.mark.parametrize("D", [8, 32, 40, 64, 72, 96, 104, 128])
def test_f32_masks_and_head_dims(cuda_device, D, mask, purified):
    _case(3, 141, D, mask, purified, cuda_device)


@pytest.mark.parametrize("purified", [False, True], ids=["born", "purified"])
@pytest.mark.parametrize("T", [1, 31, 32, 33, 97, 128, 160, 300])
@pytest.mark.parametrize("H", [1, 4])
def test_f32_lengths(cuda_device, T, H, purified):
    for mask in ("causal", "dense"):
        _case(H, T, 64, mask, purified, cuda_device)


@pytest.mark.parametrize("purified", [False, True], ids=["born", "purified"])
def test_f32_unsorted_documents(cuda_device, purified):
    _case(4, 150, 64, "docs", purified, cuda_device, sorted_docs=False)


@pytest.mark.parametrize("D", [40, 64, 96, 128])
def test_f32_forward(cuda_device, D):
    q, k, v = (x.to(cuda_device) for x in seeded_inputs((2, 4, 200, D), seed=D, n=3))
    from quantumdlblocks_amd import flash_born_attention

    for causal, window, _ in (MASKS["causal"], MASKS["dense"], MASKS["window"]):
        out = flash_born_attention(q, k, v, 0.7, is_causal=causal, window_size=window)
        ref, _ = orc.forward(f64(q), f64(k), f64(v), 0.7, causal, 1e-12, window, None)
        assert rel_err(f64(out), ref) <= 1e-5


@pytest.mark.parametrize("purified", [False, True], ids=["born", "purified"])
@pytest.mark.parametrize("mask", list(MASKS))
def test_f32_many_short_heads(cuda_device, mask, purified):
    """512 blocks of up to four tiles: one wave per block, and the launch
    whose second half goes out in the opposite order."""
    _case(64, 97, 40, mask, purified, cuda_device)


@pytest.mark.parametrize("purified", [False, True], ids=["born", "purified"])
@pytest.mark.parametrize("mask", ["dense", "window_nc", "docs_dense"])
@pytest.mark.parametrize("D", [72, 96, 104, 128])
def test_f32_full_chip_without_causality(cuda_device, D, mask, purified):
    """512 blocks of 128 rows (f32_staged, test_f32_rule.py): the staged
    kernels at these head dims, forward and backward or one of them."""
    _case(256, 129, D, mask, purified, cuda_device)
