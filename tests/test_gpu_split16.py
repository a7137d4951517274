"""16-bit attention of few blocks on the wave-split kernels (born_split16.h):
32 or 64 stationary rows per workgroup, every fourth 32-row tile per wave.  The
shapes are lists of test_split16_rule.py, which asserts on the host that each
takes those kernels: at the edges of their blocks and tiles, for every padded
head dim, mask and both 16-bit types.  Bounds: those of the forward, backward
and purified tests (2e-2 of the largest value for 16-bit outputs, their floors
for gradients that cancel).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import born_oracle as orc
from test_gpu_backward import _check_bwd
from test_gpu_f32 import check_pur_fixed
from test_gpu_purified import _check_pur
from test_split16_rule import (FULL_CHIP, FULL_CHIP_PURIFIED, HEAD_DIMS, LENGTHS, MASKS, RAGGED_DOCS, UNSORTED_DOCS,
                               WINDOW_NC_D128)
from util import TOL, f64, seeded_inputs

pytestmark = pytest.mark.gpu

def _case(B, H, T, D, dtype, mask, purified, device, sorted_docs=True):
    causal, window, docs = MASKS[mask]
    doc = None
    if docs:
        doc = orc.geometric_doc_ids(B, T, 90.0, seed=T + D)
        if not sorted_docs:
            doc = np.random.default_rng(T).permuted(doc, axis=1)
    kw = dict(is_causal=causal, window_size=window)
    if purified:
        scale, tau = [8.0 - 2.0 * (h % 3) for h in range(H)], [0.05 - 0.05 * (h % 3) for h in range(H)]
        if dtype == torch.bfloat16:
            _check_pur((B, H, T, D, dtype, kw, scale, tau, 0.25), device, doc)
        else:
            check_pur_fixed(B, H, T, D, dtype, MASKS[mask], scale, tau, 0.25, device, doc)
        return
    scale = [0.3 if h % 2 == 0 else -0.2 for h in range(H)]
    q, k, v = (x.to(device) for x in seeded_inputs((B, H, T, D), seed=T + D, std=0.5, n=3, dtype=dtype))
    from quantumdlblocks_amd import flash_born_attention

    doc_t = None if doc is None else torch.as_tensor(doc, dtype=torch.int32, device=device)
    out = flash_born_attention(q, k, v, torch.tensor(scale, device=device), doc_ids=doc_t, **kw)
    ref, z = orc.forward(f64(q), f64(k), f64(v), np.asarray(scale), causal, 1e-12, window, doc)
    bound = TOL[dtype] * np.abs(ref).max()
    if dtype == torch.float16:
        # The weights of P.V are rounded to fp16, as the reference's are
        # (flash_born.py:183): by at most 2^-25 each below its normal range,
        # which a document's first rows, of one or two keys, can show.
        seen = orc.visible_mask(T, causal, window, doc).astype(np.float64)
        bound = bound + 2.0 ** -25 * (seen @ np.abs(f64(v))) / z[..., None]
    assert (np.abs(f64(out) - ref) <= bound).all()
    _check_bwd(B, H, T, D, dtype, device, scale=scale, doc=doc, std=0.5, seed=T + D, check_dscale=mask == "dense", **kw)


@pytest.mark.parametrize("purified", [False, True], ids=["born", "purified"])
@pytest.mark.parametrize("case", HEAD_DIMS, ids=str)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
def test_masks_and_head_dims(cuda_device, case, purified, dtype):
    B, H, T, D, mask = case
    _case(B, H, T, D, dtype, mask, purified, cuda_device)


@pytest.mark.parametrize("purified", [False, True], ids=["born", "purified"])
@pytest.mark.parametrize("case", LENGTHS + WINDOW_NC_D128 + RAGGED_DOCS, ids=str)
def test_lengths(cuda_device, case, purified):
    """Block and tile edges; with documents also ids partly out of range, and a
    second batch whose ids start 4 bytes past a 16-byte boundary."""
    B, H, T, D, mask = case
    _case(B, H, T, D, torch.bfloat16, mask, purified, cuda_device)


@pytest.mark.parametrize("purified", [False, True], ids=["born", "purified"])
def test_unsorted_documents(cuda_device, purified):
    for B, H, T, D, mask in UNSORTED_DOCS:
        _case(B, H, T, D, torch.bfloat16, mask, purified, cuda_device, sorted_docs=False)


@pytest.mark.parametrize("purified,case", [(False, c) for c in FULL_CHIP] +
                         [(True, c) for c in FULL_CHIP + FULL_CHIP_PURIFIED], ids=str)
def test_full_chip(cuda_device, purified, case):
    """257 to 512 workgroups: where two fit a CU the second half goes out in the
    opposite order."""
    B, H, T, D, mask = case
    _case(B, H, T, D, torch.bfloat16, mask, purified, cuda_device)
