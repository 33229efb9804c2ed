"""GPU parity of the standalone kernels against the CPU oracle (run with -m gpu).

* quantize_per_channel (csrc/quant.hip) must equal the oracle bit for bit;
* int8_gemv (csrc/gemv.hip) must be within 1e-3 relative L2 of the fp64
  dequantized product (oracle/c/oracle.c) at the BASELINE config-2 shapes and
  at ragged shapes; so must every copy's output of its steady-state form
  (int8_gemv_repeat, several distinct weight copies in one launch).
"""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle import quant as oquant

from .conftest import GOLDEN, ROOT

pytestmark = pytest.mark.gpu

CONFIG2_SHAPES = [(4096, 1024), (1024, 2048), (6144, 1024), (1024, 3072), (151936, 1024)]
RAGGED_SHAPES = [(1, 16), (37, 48), (5, 1040), (300, 2064), (129, 4096), (3, 16384), (1000, 8192)]


def _coracle():
    return ctypes.CDLL(str(ROOT / "oracle" / "lib" / "liboracle.so"))


def _matvec_f64(q: torch.Tensor, s: torch.Tensor, x: torch.Tensor) -> np.ndarray:
    lib = _coracle()
    M, K = q.shape
    qn, sn, xn = q.numpy(), s.numpy(), x.numpy()
    y = np.empty(M, np.float64)
    lib.oracle_int8_matvec_f64(qn.ctypes.data_as(ctypes.c_void_p), sn.ctypes.data_as(ctypes.c_void_p),
                               xn.ctypes.data_as(ctypes.c_void_p), ctypes.c_int64(M), ctypes.c_int64(K),
                               y.ctypes.data_as(ctypes.c_void_p))
    return y


def test_quantize_golden_cases(mq, dev):
    d = np.load(GOLDEN / "quant_cases.npz")
    w = torch.from_numpy(d["w_bits"].view(np.int16)).view(torch.bfloat16)
    q, s = mq.quantize_per_channel(w.to(dev))
    assert np.array_equal(q.cpu().numpy(), d["q"])
    assert np.array_equal(s.cpu().numpy(), d["scale"])


@pytest.mark.parametrize("shape", [(4096, 1024), (1024, 3072), (257, 100), (3, 5), (1, 70000)])
def test_quantize_bit_exact(mq, dev, shape):
    print(f"quantize {shape}", flush=True)
    g = torch.Generator().manual_seed(shape[0] * 31 + shape[1])
    w = (torch.randn(shape, generator=g) * 0.02).to(torch.bfloat16)
    if shape[0] > 2:
        w[1] = 0
        w[2, 0] = -3.0
    q, s = mq.quantize_per_channel(w.to(dev))
    qr, sr = oquant.quantize_per_channel(w)
    assert torch.equal(s.cpu(), sr)
    assert torch.equal(q.cpu(), qr)


@pytest.mark.parametrize("shape", CONFIG2_SHAPES + RAGGED_SHAPES, ids=lambda s: f"{s[0]}x{s[1]}")
def test_int8_gemv_parity(mq, dev, shape):
    M, K = shape
    print(f"gemv {M}x{K}", flush=True)
    g = torch.Generator().manual_seed(M + 7 * K)
    w = (torch.randn(M, K, generator=g) * 0.02).to(torch.bfloat16)
    q, s = oquant.quantize_per_channel(w)
    x = torch.randn(K, generator=g, dtype=torch.float32)
    y = mq.int8_gemv(x.to(dev), q.to(dev), s.to(dev))
    torch.cuda.synchronize()
    ref = _matvec_f64(q, s, x)
    got = y.cpu().double().numpy()
    rel = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert rel <= 1e-3, rel
    assert rel <= 1e-5, f"fp32 accumulation should be far inside the 1e-3 bound, got {rel}"


@pytest.mark.parametrize("K", [16, 1008, 1024, 1040, 2048, 2064, 3072, 3088, 4096, 4112, 6144, 6160, 8192, 8208, 16384])
@pytest.mark.parametrize("M", [1, 2051])
def test_one_byte_gemv_row_lengths(mq, dev, M, K):
    """INT8 and FP8 rows either side of each number of 1 KB chunks a wave holds."""
    print(f"gemv {M}x{K}", flush=True)
    _one_byte_gemv_within_rounding(mq, dev, M, K)


def _one_byte_gemv_within_rounding(mq, dev, M, K):
    """INT8 and FP8 against float64. A lane adds 16 products per 1 KB chunk to one fp32 sum, then six
    levels add the 64 lanes' and the scale is multiplied on: within (16 chunks + 7) 2^-24 of sum |w x|,
    which one lane's columns left out or taken from elsewhere exceed many times over."""
    g = torch.Generator(device=dev).manual_seed(M + K)
    x = torch.randn(K, generator=g, device=dev)
    s = torch.rand(M, generator=g, device=dev) + 0.5
    q = torch.randint(-128, 128, (M, K), generator=g, device=dev, dtype=torch.int8)
    f = (torch.randn((M, K), generator=g, device=dev) * 40).clamp(-448, 448).to(torch.float8_e4m3fn)
    for y, w in ((mq.int8_gemv(x, q, s), q.double()), (mq.fp8_gemv(x, f.view(torch.uint8), s), f.double())):
        ref = (w @ x.double()) * s.double()
        bound = (w.abs() @ x.abs().double()) * s.double() * ((16 * ((K + 1023) // 1024) + 7) * 2.0 ** -24)
        assert bool(((y.double() - ref).abs() <= bound + 1e-30).all())


@pytest.mark.parametrize("M,K", [(70001, 16), (70001, 256), (50000, 1008), (2051, 512), (2049, 8192), (4099, 8208), (1500, 9216),
                                 (5, 10240), (3001, 10256), (2100, 12288), (2100, 12304), (9, 16384), (2300, 16384),
                                 (8192, 1024), (8193, 1024), (32768, 1024), (32769, 1024)])
def test_one_byte_gemv_forms(mq, dev, M, K):
    """Either side of the lines between the kernel's forms, with several items per wave: rows shorter
    than a chunk, activations in registers and in LDS, matrices that stay in the caches or not."""
    print(f"gemv {M}x{K}", flush=True)
    _one_byte_gemv_within_rounding(mq, dev, M, K)


def test_int8_gemv_repeatable(mq, dev):
    g = torch.Generator().manual_seed(5)
    q = torch.randint(-127, 128, (4096, 1024), generator=g, dtype=torch.int8).to(dev)
    s = torch.rand(4096, generator=g).to(dev)
    x = torch.randn(1024, generator=g).to(dev)
    a = mq.int8_gemv(x, q, s).cpu()
    b = mq.int8_gemv(x, q, s).cpu()
    assert torch.equal(a, b)


@pytest.mark.parametrize("shape,n,reps", [((1024, 2048), 3, 7), ((4096, 1024), 2, 5), ((37, 48), 2, 9),
                                          ((1000, 8192), 3, 3)], ids=lambda v: str(v))
def test_int8_gemv_repeat_parity(mq, dev, shape, n, reps):
    M, K = shape
    print(f"gemv repeat {M}x{K} copies={n} reps={reps}", flush=True)
    g = torch.Generator().manual_seed(M + 3 * K + n)
    qs, ss = [], []
    for _ in range(n):
        w = (torch.randn(M, K, generator=g) * 0.02).to(torch.bfloat16)
        q, s = oquant.quantize_per_channel(w)
        qs.append(q)
        ss.append(s)
    s = ss[0]                                         # one scale vector for every copy
    x = torch.randn(K, generator=g, dtype=torch.float32)
    y = mq.int8_gemv_repeat(x.to(dev), torch.stack(qs).to(dev), s.to(dev), reps)
    torch.cuda.synchronize()
    got = y.cpu().double().numpy()
    for c in range(n):
        ref = _matvec_f64(qs[c], s, x)
        rel = np.linalg.norm(got[c] - ref) / np.linalg.norm(ref)
        assert rel <= 1e-5, (c, rel)
