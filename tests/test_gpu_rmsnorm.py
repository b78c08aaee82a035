"""GPU parity tests of RMSNorm (``fi_rmsnorm``) and RMSNorm fused with the INT4 projection
(``fi_rmsnorm_int4_matmul``), marked ``gpu``.

* rms_norm within one fp16 ulp of the float64 form (oracle/rmsnorm.py) — the reference
  computes in fp32 with its own sum order and rsqrt, so the last bit is not pinned — and
  the fraction of elements off the correctly rounded value reported and bounded;
* the fused call against the float64 product of the normalized rows and the dequantized
  weights, for the in-GEMM norm (few rows) and the separate-pass form (more rows).
"""

import numpy as np
import pytest
import torch

from conftest import banner
from oracle import int4 as OI
from oracle import rmsnorm as ON

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _inputs(seed, M, H, scale=1.0):
    rng = np.random.default_rng(seed)
    x = (rng.standard_normal((M, H)) * scale).astype(np.float16)
    w = (rng.standard_normal(H) * 0.3 + 1.0).astype(np.float16)
    return x, w


@pytest.mark.parametrize("M,H,scale", [(1, 3072, 1.0), (64, 3072, 4.0), (1000, 3072, 0.01),
                                       (7, 256, 1.0), (3, 8192, 30.0)])
def test_rms_norm_vs_oracle(hip, M, H, scale):
    banner(f"rms_norm M={M} H={H}")
    from fast_infer_amd import rms_norm

    x, w = _inputs(M + H, M, H, scale)
    y = rms_norm(torch.from_numpy(x).to(DEV), torch.from_numpy(w).to(DEV))
    torch.cuda.synchronize()
    got = y.float().cpu().numpy().astype(np.float64)
    exact = ON.rms_norm_exact(x, w)
    assert np.all(np.abs(got - exact) <= ON.norm_bound(exact))
    off = np.mean(y.cpu().numpy() != exact.astype(np.float16))
    print(f"[rms_norm] fraction not correctly rounded: {off:.2e}")
    assert off < 0.01


def test_rms_norm_strided_rows_and_batch_dims(hip):
    banner("rms_norm strided")
    from fast_infer_amd import rms_norm

    rng = np.random.default_rng(5)
    big = rng.standard_normal((2, 5, 3072 + 64)).astype(np.float16)
    w = (rng.standard_normal(3072) * 0.3 + 1.0).astype(np.float16)
    xt = torch.from_numpy(big).to(DEV)[..., 32:32 + 3072]
    y = rms_norm(xt, torch.from_numpy(w).to(DEV))
    assert y.shape == (2, 5, 3072)
    exact = ON.rms_norm_exact(big[..., 32:32 + 3072].reshape(10, 3072), w)
    got = y.reshape(10, 3072).float().cpu().numpy()
    assert np.all(np.abs(got - exact) <= ON.norm_bound(exact))


@pytest.mark.parametrize("M", [1, 3, 4, 5, 16, 17, 64, 300])
@pytest.mark.parametrize("packed_weights", [True, False])
def test_rms_norm_int4_matmul_vs_oracle(hip, M, packed_weights):
    banner(f"rms_norm_int4_matmul M={M} packed={packed_weights}")
    from fast_infer_amd import (dequantize_int4, int4_matmul, quantize_int4_groupwise, rms_norm,
                                rms_norm_int4_matmul)

    N, K = 5120, 3072
    x, nw = _inputs(M, M, K, 2.0)
    rng = np.random.default_rng(99)
    w = (rng.standard_normal((N, K)) * 0.02).astype(np.float16)
    packed, scales = quantize_int4_groupwise(torch.from_numpy(w).to(DEV))
    w16 = dequantize_int4(packed, scales)
    weight = (packed, scales) if packed_weights else w16
    xd, nwd = torch.from_numpy(x).to(DEV), torch.from_numpy(nw).to(DEV)
    out = rms_norm_int4_matmul(xd, nwd, weight)
    two_step = int4_matmul(rms_norm(xd, nwd), weight)
    torch.cuda.synchronize()
    xn = ON.rms_norm(x, nw)
    w16n = w16.cpu().numpy()
    exact = OI.matmul_exact(xn, w16n)
    mag = np.abs(xn.astype(np.float64)) @ np.abs(w16n.astype(np.float64)).T
    # the normalized rows may differ from the oracle's by one fp16 ulp here and there
    bound = OI.matmul_bound(xn, w16n) + mag * 2.0 ** -10
    for got in (out, two_step):
        g = got.float().cpu().numpy().astype(np.float64)
        assert np.all(np.abs(g - exact) <= bound), float(np.max(np.abs(g - exact) - bound))


# The norm shared out over the workgroup (1 and 2 rows, packed weights): rows of one load and of
# several per thread, a length that leaves threads idle, the longest shared-out row, one past it,
# strided rows, and a last column tile with one column.
@pytest.mark.parametrize("M", [1, 2])
@pytest.mark.parametrize("K,pad", [(128, 0), (1024, 0), (1152, 8), (3072, 8), (4096, 0), (4224, 64),
                                   (8192, 0), (8320, 0)])
def test_rms_norm_int4_matmul_few_rows(hip, M, K, pad):
    banner(f"rms_norm_int4_matmul M={M} K={K} row pad {pad}")
    from fast_infer_amd import dequantize_int4, quantize_int4_groupwise, rms_norm_int4_matmul

    N = 145
    x, nw = _inputs(M + K, M, K, 2.0)
    w = (np.random.default_rng(K).standard_normal((N, K)) * 0.02).astype(np.float16)
    weight = quantize_int4_groupwise(torch.from_numpy(w).to(DEV))
    big = torch.full((M + 1, K + pad), float("nan"), dtype=torch.float16, device=DEV)
    big[:M, :K] = torch.from_numpy(x).to(DEV)
    out = rms_norm_int4_matmul(big[:M, :K], torch.from_numpy(nw).to(DEV), weight)
    xn, w16 = ON.rms_norm(x, nw), dequantize_int4(*weight).cpu().numpy()
    mag = np.abs(xn.astype(np.float64)) @ np.abs(w16.astype(np.float64)).T
    bound = OI.matmul_bound(xn, w16) + mag * 2.0 ** -10  # an fp16 ulp in a normalized element
    got = out.float().cpu().numpy().astype(np.float64)
    assert np.all(np.abs(got - OI.matmul_exact(xn, w16)) <= bound)


# Both norm kernels at the edges of their choice: rows of one chunk, of exactly and just over 2048
# elements (few rows and many), the longest row of a workgroup and one past it; strided rows.
@pytest.mark.parametrize("M,H,pad", [(5, 8, 0), (1023, 2048, 8), (1024, 2048, 0), (1025, 2056, 16),
                                     (33, 6152, 0), (2, 8192, 8), (2, 8200, 0), (1500, 3072, 0)])
def test_rms_norm_kernel_choice(hip, M, H, pad):
    banner(f"rms_norm M={M} H={H} row pad {pad}")
    from fast_infer_amd import rms_norm

    x, w = _inputs(M + H, M, H, 1.0)
    big = torch.full((M, H + pad), float("nan"), dtype=torch.float16, device=DEV)
    big[:, :H] = torch.from_numpy(x).to(DEV)
    got = rms_norm(big[:, :H], torch.from_numpy(w).to(DEV)).float().cpu().numpy().astype(np.float64)
    exact = ON.rms_norm_exact(x, w)
    assert np.all(np.abs(got - exact) <= ON.norm_bound(exact))


@pytest.mark.parametrize("M,H", [(12999, 2056), (13000, 2056), (13000, 2808), (13000, 2816)])
def test_rms_norm_many_rows_kernel_choice(hip, M, H):
    banner(f"rms_norm M={M} H={H}")
    from fast_infer_amd import rms_norm

    x, w = (torch.from_numpy(a).to(DEV) for a in _inputs(M + H, M, H, 1.0))
    exact = x.double() * torch.rsqrt(x.double().square().mean(-1, keepdim=True) + 1e-5) * w.double()
    got = rms_norm(x, w).double()
    # ON.norm_bound on the device
    assert bool(((got - exact).abs() <= torch.from_numpy(ON.norm_bound(exact.cpu().numpy())).to(DEV)).all())


def test_rms_norm_more_rows_than_a_workgroup_each(hip):
    """2^24 rows of 2056 elements, in place: a launch of 256 threads per row would pass the 2^32
    threads that one dimension takes."""
    banner("rms_norm of 2^24 rows x 2056")
    from fast_infer_amd import _lib

    M, H = 1 << 24, 2056
    if torch.cuda.mem_get_info()[0] < M * H * 2 + (8 << 30):
        pytest.skip("needs 77 GB of free device memory")
    row, w = _inputs(H, 3, H, 1.0)
    rows, wt = torch.from_numpy(row).to(DEV), torch.from_numpy(w).to(DEV)
    x = torch.empty(M, H, dtype=torch.float16, device=DEV)
    x[:] = rows[0]
    x[M // 2 + 1], x[M - 1] = rows[1], rows[2]
    rc = _lib.load().fi_rmsnorm(x.data_ptr(), H, M, H, wt.data_ptr(), 1e-5, x.data_ptr(), H,
                                _lib.stream_handle(torch.device(DEV)))
    _lib.check(rc, "fi_rmsnorm")
    got = x[[0, M // 2 + 1, M - 1]].double().cpu().numpy()
    exact = ON.rms_norm_exact(row, w)
    assert np.all(np.abs(got - exact) <= ON.norm_bound(exact))
    x[M // 2 + 1], x[M - 1] = x[0], x[0]
    for part in x.split(1 << 21):
        assert bool((part == x[0]).all())
    del x
    torch.cuda.empty_cache()
