"""The quantizers' row pass against the element kernels and the oracle (run with -m gpu).

Rows of whole 16-byte loads take the row pass, others (odd lengths, more than 8192 elements,
views at an odd element offset, few FP8 rows) the element kernels. The same rows are given to both, the
second time as a view one element into its storage, and must give the same bytes and scales:
row lengths either side of a wave's 512-element loads and of the register limit, few and many
rows, and rows of zeros, signed zeros, subnormals, infinities, NaN and the largest values.
"""
from __future__ import annotations

import pytest
import torch

from oracle import formats as ofmt
from oracle import quant as oquant

pytestmark = pytest.mark.gpu


def _quant(mq, fmt):
    return {"int8": mq.quantize_per_channel, "fp8": mq.quantize_fp8, "int4": mq.quantize_int4}[fmt]


def _shifted(w):
    """The same rows one element into their storage (2-byte aligned)."""
    flat = torch.empty(w.numel() + 1, dtype=w.dtype, device=w.device)
    v = flat[1:].view_as(w)
    v.copy_(w)
    return v


def _rows(M, K, dev, seed):
    g = torch.Generator().manual_seed(seed)
    w = torch.randn((M, K), generator=g) * 0.02 * torch.exp2(torch.randint(-20, 20, (M, 1), generator=g).float())
    return w.to(torch.bfloat16).to(dev)


def _same(a, b, what):
    assert torch.equal(a[0], b[0]), f"{what}: {int((a[0] != b[0]).sum())} codes differ"
    assert torch.equal(a[1].view(torch.int32), b[1].view(torch.int32)), f"{what}: scales differ"


@pytest.mark.parametrize("fmt,K", [(f, k) for f in ("int8", "fp8") for k in (8, 504, 512, 520, 1024, 1032, 2040, 4104, 8192, 8200, 1023)]
                         + [("int4", k) for k in (128, 384, 512, 640, 1024, 4224, 8192, 8320)])
@pytest.mark.parametrize("M", [1, 5, 9001])
def test_row_pass_matches_element_kernel(mq, dev, fmt, K, M):
    if M > 1000 and K > 1100:
        M = 70
    print(f"quantize {fmt} [{M}, {K}]", flush=True)
    w = _rows(M, K, dev, K + M)
    got = _quant(mq, fmt)(w)
    _same(got, _quant(mq, fmt)(_shifted(w)), f"{fmt} [{M}, {K}] against the element kernel")
    n = min(M, 5)
    c = w[:n].cpu()
    want = {"int8": oquant.quantize_per_channel, "fp8": ofmt.quantize_fp8_rows, "int4": ofmt.quantize_int4_groups}[fmt](c)
    _same((got[0][:n].cpu(), got[1][:n].cpu()), want, f"{fmt} [{M}, {K}] against the oracle")


@pytest.mark.parametrize("M", [1023, 1024, 1025])
@pytest.mark.parametrize("K", [504, 1032, 2040, 4104, 8192])
def test_fp8_row_pass_and_element_kernel_meet(mq, dev, M, K):
    """FP8 matrices of fewer rows than four per CU take the element kernel: the same bytes and scales
    on either side of the line."""
    print(f"quantize fp8 [{M}, {K}]", flush=True)
    w = _rows(M, K, dev, K + M)
    got = _quant(mq, "fp8")(w)
    _same(got, _quant(mq, "fp8")(_shifted(w)), f"fp8 [{M}, {K}] against the element kernel")
    many = _quant(mq, "fp8")(torch.cat([w, w, w, w, w]))          # by the row pass on any number of CUs up to 1278
    _same(got, (many[0][:M], many[1][:M]), f"fp8 [{M}, {K}] against the row pass")


def _special_rows(K):
    w = _rows(8, K, torch.device("cpu"), 3).float()
    w[0] = 0.0
    w[1] = -0.0
    w[2] = torch.linspace(-1e-38, 1e-38, K)               # subnormals
    w[3, 5], w[3, 900] = float("inf"), float("-inf")
    w[4, 7], w[4, 513] = float("nan"), -float("nan")
    w[5] = 3.3e38 * torch.sign(w[5])
    w[6, ::2] = -0.0
    w[7] = float("nan")
    return w.to(torch.bfloat16)


@pytest.mark.parametrize("copies", [1, 256])
@pytest.mark.parametrize("fmt", ["int8", "fp8", "int4"])
def test_row_pass_special_values(mq, dev, fmt, copies):
    w = _special_rows(1024).to(dev).repeat(copies, 1)
    print(f"quantize {fmt}: special values, {len(w)} rows", flush=True)
    _same(_quant(mq, fmt)(w), _quant(mq, fmt)(_shifted(w)), fmt)
