"""The struct-form entry points (qdl_flash_born_forward_call / _backward_call):
the packed block matches the C struct, is validated before any launch, and a
scale or tau passed by value gives what the same value in device memory does."""

from __future__ import annotations

import ctypes
import os
import re

import pytest
import torch

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "qdl_flash_born.h")


def _block(**kw):
    from quantumdlblocks_amd import _native

    args = dict(dtype=_native.DTYPE_BF16, B=1, H=2, T=8, D=64, q=0, k=0, v=0, out=0, z=0, scale=0, n_scale=1,
                scale_value=8.0, doc=0, causal=1, window=0, eps=1e-12)
    args.update(kw)
    return _native.pack_call(**args)


def test_block_has_the_structs_size():
    body = re.search(r"typedef struct qdl_born_call \{(.*?)\} qdl_born_call;", open(HEADER).read(), re.S).group(1)
    body = re.sub(r"/\*.*?\*/", "", body, flags=re.S)
    fields = 0
    for decl in body.split(";"):
        for name in decl.split(",") if decl.strip() else []:
            n = re.search(r"\[(\d+)\]", name)
            fields += int(n.group(1)) if n else 1
    assert len(_block()) == 8 * fields


def test_validation():
    from quantumdlblocks_amd import _native

    lib = _native.load()
    for fn in (lib.qdl_flash_born_forward_call, lib.qdl_flash_born_backward_call):
        assert fn(None, None) == -5
        assert fn(ctypes.c_char_p(b"\0" * 392), None) == -2  # struct_bytes
        assert fn(_block(dtype=7), None) == -1
        assert fn(_block(D=12), None) == -3
        assert fn(_block(scale=64, n_scale=3), None) == -6
        assert fn(_block(window=-1), None) == -7
        assert fn(_block(purified=1, tau=64, n_tau=3), None) == -9
        assert fn(_block(eps=-1.0), None) == -2
        assert fn(_block(), None) == -5
        assert fn(_block(T=0), None) == 0
    ptrs = dict(q=16, k=16, v=16, out=16, z=16)
    assert lib.qdl_flash_born_forward_call(_block(**{**ptrs, "q": 24}), None) == -4
    assert lib.qdl_flash_born_backward_call(_block(**ptrs, dout=16, dq=16, dk=16, dv=16), None) == -8


@pytest.mark.gpu
@pytest.mark.parametrize("purified", [False, True], ids=["born", "purified"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=str)
@pytest.mark.parametrize("D", [40, 64, 100, 128, 200])
@pytest.mark.parametrize("mask", [dict(), dict(is_causal=False), dict(window_size=30), dict(doc=True),
                                  dict(is_causal=False, window_size=20, doc=True)], ids=str)
def test_parameters_by_value(cuda_device, purified, dtype, D, mask):
    """Every kernel reads scale and tau from the block or from memory: bitwise
    the same output and gradients (no gradient of a plain number)."""
    from quantumdlblocks_amd import flash_born_attention, flash_purified_born_attention

    g = torch.Generator("cpu").manual_seed(D)
    q, k, v, do = (torch.randn(1, 2, 70, D, generator=g).mul(0.3).to(cuda_device, dtype) for _ in range(4))
    kw = dict(mask)
    if kw.pop("doc", False):
        kw["doc_ids"] = (torch.arange(70, device=cuda_device) // 25).view(1, 70)
    got = []
    for scale, tau in ((-1.5, 0.02), (torch.tensor([-1.5, -1.5], device=cuda_device,
                                                                requires_grad=not purified),
                                      torch.tensor(0.02, device=cuda_device))):
        x = [t.clone().requires_grad_(True) for t in (q, k, v)]
        if purified:
            out = flash_purified_born_attention(*x, -scale, tau, **kw)
        else:
            out = flash_born_attention(*x, scale, **kw)
        out.backward(do)
        got.append([out, *(t.grad for t in x)])
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.gpu
def test_prologue_scale_by_value(cuda_device):
    from quantumdlblocks_amd import flash_born_attention_qk_prologue

    q, k, v = (torch.randn(2, 70, 4, 64, device=cuda_device, dtype=torch.bfloat16).transpose(1, 2) for _ in range(3))
    a = flash_born_attention_qk_prologue(q, k, v, 3.0)
    b = flash_born_attention_qk_prologue(q, k, v, torch.tensor(3.0, device=cuda_device))
    assert torch.equal(a, b)


@pytest.mark.gpu
def test_a_call_captures_with_a_plain_scale(cuda_device):
    """A float scale needs no copy from the host, so the call can be captured;
    replays follow the inputs."""
    from quantumdlblocks_amd import flash_born_attention

    q, k, v = (torch.randn(1, 4, 96, 64, device=cuda_device, dtype=torch.bfloat16) for _ in range(3))
    flash_born_attention(q, k, v, 2.0)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph), torch.no_grad():
        out = flash_born_attention(q, k, v, 2.0)
    for seed in range(3):
        torch.manual_seed(seed)
        q.copy_(torch.randn_like(q))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, flash_born_attention(q, k, v, 2.0))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=str)
@pytest.mark.parametrize("D", [24, 40, 64, 96, 128, 200])
@pytest.mark.parametrize("T", [60, 600])
@pytest.mark.parametrize("mask", [dict(), dict(is_causal=False), dict(window_size=30), dict(doc=True),
                                  dict(is_causal=False, window_size=20, doc=True)], ids=str)
def test_purified_output_in_the_compute_dtype(cuda_device, dtype, D, T, mask):
    """The kernels round the output to the compute dtype themselves: it is the
    fp32 output (what a backward keeps) rounded to nearest, and a call without
    a backward, which writes no fp32 output, returns the same."""
    from quantumdlblocks_amd import flash_purified_born_attention

    g = torch.Generator("cpu").manual_seed(D)
    q, k, v = (torch.randn(1, 2, T, D, generator=g).mul(0.3).to(cuda_device, dtype) for _ in range(3))
    kw = dict(mask)
    if kw.pop("doc", False):
        kw["doc_ids"] = (torch.arange(T, device=cuda_device) // 25).view(1, T)
    with torch.no_grad():
        plain = flash_purified_born_attention(q, k, v, **kw)
    out = flash_purified_born_attention(q.requires_grad_(True), k, v, **kw)
    kept = out.grad_fn.saved_tensors[3]  # the fp32 output
    assert kept.dtype == torch.float32
    assert plain.dtype == out.dtype == dtype and out.is_contiguous()
    assert torch.equal(plain, out)
    assert torch.equal(out, kept.to(dtype)[..., :D])


def _field(block, name):
    """One field of a packed block, by its name in the C struct."""
    body = re.search(r"typedef struct qdl_born_call \{(.*?)\} qdl_born_call;", open(HEADER).read(), re.S).group(1)
    at = 0
    for decl in re.sub(r"/\*.*?\*/", "", body, flags=re.S).split(";"):
        for field in decl.split(",") if decl.strip() else []:
            word, n = re.search(r"(\w+)\s*(?:\[(\d+)\])?\s*$", field).groups()
            if word == name:
                return int.from_bytes(block[8 * at:8 * at + 8], "little")
            at += int(n or 1)
    raise KeyError(name)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("mode", ["grad", "no_grad", "inference_mode"])
def test_trained_parameters_without_a_backward(monkeypatch, mode, dtype):
    """What a purified call keeps for its backward is asked for where one can
    follow, not wherever a parameter requires a gradient."""
    from quantumdlblocks_amd.kernels import flash_born as fb

    blocks = []
    monkeypatch.setattr(fb, "_run_call", lambda fn, what, device, block: blocks.append(block))
    q = torch.zeros(1, 2, 8, 16, dtype=dtype)
    scale, tau = (torch.full((2,), x, requires_grad=True) for x in (8.0, 0.0625))
    grad_mode = {"grad": torch.enable_grad, "no_grad": torch.no_grad, "inference_mode": torch.inference_mode}[mode]
    with grad_mode():
        out = fb._run_triton_flash_purified_born(q, q, q, scale, tau, 0.05, True, 1e-8)
    assert out.requires_grad == (mode == "grad")
    assert (_field(blocks[0], "out") != 0, _field(blocks[0], "param_grads")) == (mode == "grad", mode == "grad")
    assert _field(blocks[0], "out16") != 0


@pytest.mark.parametrize("grad_enabled", [True, False])
def test_trained_scale_of_the_prologue_without_a_backward(monkeypatch, grad_enabled):
    from quantumdlblocks_amd.kernels import flash_born as fb
    from quantumdlblocks_amd.kernels.qk_prologue import _BornQKPrologueFn

    blocks = []
    monkeypatch.setattr(fb, "_run_call", lambda fn, what, device, block: blocks.append(block))
    q = torch.zeros(1, 2, 8, 16, dtype=torch.bfloat16)
    _BornQKPrologueFn.apply(q, q, q, torch.ones(2, requires_grad=True), None, None, True, 1e-12, 0, None, 1e-12,
                            grad_enabled)
    assert (_field(blocks[0], "q_rinv") != 0) == (_field(blocks[0], "k_rinv") != 0) == grad_enabled


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=str)
def test_trained_parameters_under_no_grad_on_the_gpu(cuda_device, dtype):
    """The same call as one with plain numbers, bitwise, and gradients as
    before where they are recorded."""
    from quantumdlblocks_amd import flash_purified_born_attention

    g = torch.Generator("cpu").manual_seed(0)
    q, k, v = (torch.randn(1, 2, 1000, 64, generator=g).mul(0.3).to(cuda_device, dtype) for _ in range(3))
    scale, tau = (torch.tensor(x, device=cuda_device, requires_grad=True) for x in (2.0, 0.02))
    with torch.no_grad():
        assert torch.equal(flash_purified_born_attention(q, k, v, scale, tau),
                           flash_purified_born_attention(q, k, v, 2.0, 0.02))
    flash_purified_born_attention(q, k, v, scale, tau).float().square().mean().backward()
    assert torch.isfinite(scale.grad).all() and torch.isfinite(tau.grad).all()
