"""16-bit attention of few blocks on the wave-split kernels (born_split16.h):
32 or 64 stationary rows per workgroup, every fourth 32-row tile per wave.
Shapes few enough for those kernels (split16_rule.h; test_split16_rule.py), at the edges of their blocks and tiles, for every padded head dim, mask
and both 16-bit types.  Bounds: those of the forward, backward and purified
tests (2e-2 of the largest value for 16-bit outputs, their floors for
gradients that cancel).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import born_oracle as orc
from test_gpu_backward import _check_bwd
from test_gpu_f32 import check_pur_fixed
from test_gpu_purified import _check_pur
from util import TOL, f64, rel_err, seeded_inputs

pytestmark = pytest.mark.gpu

MASKS = {
    "causal": (True, 0, False),
    "dense": (False, 0, False),
    "window": (True, 300, False),
    "window_nc": (False, 300, False),
    "docs": (True, 0, True),
    "docs_window": (True, 300, True),
    "docs_dense": (False, 0, True),
}


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
    ref, _ = orc.forward(f64(q), f64(k), f64(v), np.asarray(scale), causal, 1e-12, window, doc)
    assert rel_err(f64(out), ref) <= TOL[dtype]
    _check_bwd(B, H, T, D, dtype, device, scale=scale, doc=doc, std=0.5, seed=T + D, check_dscale=mask == "dense", **kw)


@pytest.mark.parametrize("purified", [False, True], ids=["born", "purified"])
@pytest.mark.parametrize("mask", list(MASKS))
@pytest.mark.parametrize("D", [24, 64, 72, 96, 120, 128, 160, 256])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
def test_masks_and_head_dims(cuda_device, D, mask, purified, dtype):
    _case(1, 2, 700, D, dtype, mask, purified, cuda_device)


@pytest.mark.parametrize("purified", [False, True], ids=["born", "purified"])
@pytest.mark.parametrize("T", [384, 415, 416, 417, 447, 448, 449, 513, 1000])
@pytest.mark.parametrize("D", [64, 128])
def test_lengths(cuda_device, T, D, purified):
    for mask in ("causal", "dense"):
        _case(1, 3, T, D, torch.bfloat16, mask, purified, cuda_device)


@pytest.mark.parametrize("purified", [False, True], ids=["born", "purified"])
def test_unsorted_documents(cuda_device, purified):
    _case(2, 2, 600, 64, torch.bfloat16, "docs", purified, cuda_device, sorted_docs=False)


@pytest.mark.parametrize("purified", [False, True], ids=["born", "purified"])
@pytest.mark.parametrize("mask", ["docs", "docs_dense"])
@pytest.mark.parametrize("B,T", [(1, 1301), (2, 705), (2, 1027)])
def test_documents_of_ragged_length(cuda_device, B, T, mask, purified):
    """A last block of few rows, ids partly out of range, and a second batch
    whose ids start at 4 bytes past a 16-byte boundary."""
    _case(B, 2, T, 64, torch.bfloat16, mask, purified, cuda_device)


@pytest.mark.parametrize("H", [8, 16])
def test_two_workgroups_per_cu(cuda_device, H):
    """257 to 512 workgroups: the second half goes out in the opposite order."""
    _case(2, H, 1100, 64, torch.bfloat16, "causal", False, cuda_device)
