"""GPU parity of the plain linear layers (kernels/h3sycl.cpp:656-739) through the C ABI against the oracle's float64
products: h3s_linear, h3s_linear_acc (row chunks included) and h3s_scale_rows. The reference's products are oneDNN's,
whose accumulation order is not restated: the parity tolerance (relative L2 < 1e-3, one ulp of the output type).
bfloat16 and half operands with K a multiple of 32 run on the matrix-core kernel (256 x 256 tiles: partial tiles at
every edge, K steps of 64 elements with a last half step where K is an odd multiple of 32, the long-K tile order
from K = 6144); h3s_linear with at most 512 rows of x or 128 of w mostly on the few-row kernel; K = 200 and
float32 operands run on rocBLAS with the separate epilogue."""
import os

import numpy as np
import pytest

from oracle import oracle as o
from helpers import assert_bits_equal, assert_close_16, launches, new, up
from sycl_minimax_h3_amd import Device, DType, ops

pytestmark = pytest.mark.gpu
o.set_threads(8)
DTS = {o.F32: DType.F32, o.F16: DType.F16, o.BF16: DType.BF16}


def mats(seed, M, K, N, dt):
    g = np.random.default_rng(seed)
    x = o.to_dt(g.standard_normal((M, K)).astype(np.float32), dt).ravel()
    w = o.to_dt((g.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32), dt).ravel()
    b = g.standard_normal(N).astype(np.float32)
    return x, w, b


def close(got, want, dt, what):
    if dt == o.F32:
        rel, _ = o.compare(np.asarray(got, np.float32).ravel(), np.asarray(want, np.float32).ravel())
        assert rel < 1e-5, f"{what}: relative L2 {rel:.2e}"
    else:
        # float32 accumulation: results that cancel to near zero carry the error of the terms (~1e-6 here)
        assert_close_16(got, want, dt, what, max_frac=2e-2, abs_floor=2e-5)


@pytest.mark.parametrize("dt,out_dt", [(o.BF16, o.BF16), (o.BF16, o.F32), (o.F16, o.F16), (o.F32, o.F32), (o.F32, o.BF16)])
@pytest.mark.parametrize("M,K,N", [(37, 256, 130), (300, 1024, 520), (8200, 64, 48), (1000, 2048, 700), (513, 6144, 300),
                                   (600, 200, 90), (257, 96, 256), (2000, 1024, 64), (2000, 1024, 100)])
@pytest.mark.parametrize("bias", [False, True])
def test_linear(dev, dt, out_dt, M, K, N, bias):
    x, w, b = mats(100 + K, M, K, N, dt)
    want = o.linear(x, dt, M, K, w, N, b if bias else None, out_dt=out_dt)
    out = new(dev, DTS[out_dt], [M, N])
    layer = ops.Linear(up(dev, w, DTS[dt], [N, K]), up(dev, b, "F32", [N]) if bias else None)
    layer.forward(up(dev, x, DTS[dt], [M, K]), out)
    close(out.to_numpy(), want, out_dt, "linear")


# at most 512 rows of x, or at most 128 of w: one row on either side, the edges of the few-row kernel's 64-row tiles along
# S and L, S past 256 rows (two tiles), a single K step, last half steps in one part and in several
@pytest.mark.parametrize("M,K,N", [(1, 32, 8), (1, 4096, 1), (64, 64, 64), (65, 992, 129), (128, 1056, 333), (192, 2048, 66), (193, 544, 1000),
                                   (256, 4128, 128), (257, 2080, 130), (512, 480, 4100), (511, 8192, 72), (513, 480, 128), (1030, 7168, 30),
                                   (20000, 96, 65), (700, 4128, 127)])
@pytest.mark.parametrize("dt,out_dt,bias", [(o.BF16, o.BF16, True), (o.F16, o.F16, False), (o.BF16, o.F32, True)])
def test_linear_few_rows(dev, dt, out_dt, bias, M, K, N):
    test_linear(dev, dt, out_dt, M, K, N, bias)


def open_with(env):
    old = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    try:
        return Device.open()
    finally:
        for k, v in old.items():
            if v is None:
                del os.environ[k]
            else:
                os.environ[k] = v


@pytest.fixture(scope="module")
def dev_by_cus(dev):
    """Contexts that size their grids for 4 and 16 compute units (H3S_CUS), and the default one (256)."""
    ds = {4: open_with({"H3S_CUS": "4"}), 16: open_with({"H3S_CUS": "16"}), 256: dev}
    yield ds
    ds[4].close()
    ds[16].close()


# every tile of the few-row kernel that a call can reach: mt x nt pieces of 64 rows of the short and of the long operand, the
# short one x or (swap) w, whole and in parts; cut tiles along both, last half steps, two tiles along S (300, 500, 512 rows)
@pytest.mark.parametrize("cus,M,K,N,mt,nt,swap,parts", [
    (16, 60, 96, 300, 1, 1, False, 1), (16, 60, 2080, 96, 1, 1, False, 7), (4, 137, 96, 33, 1, 1, True, 1), (16, 190, 2080, 33, 1, 1, True, 5),
    (4, 60, 480, 333, 1, 2, False, 1), (4, 60, 1056, 1100, 1, 2, False, 3), (16, 1500, 480, 33, 1, 2, True, 1), (4, 100, 1056, 33, 1, 2, True, 4),
    (16, 100, 96, 300, 2, 1, False, 1), (16, 128, 1056, 300, 2, 1, False, 3), (4, 190, 96, 96, 2, 1, True, 1), (16, 190, 1056, 96, 2, 1, True, 4),
    (4, 128, 480, 333, 2, 2, False, 1), (4, 100, 4128, 130, 2, 2, False, 2), (4, 500, 96, 96, 2, 2, True, 1), (16, 250, 2080, 128, 2, 2, True, 7),
    (16, 137, 96, 333, 3, 1, False, 1), (16, 190, 544, 300, 3, 1, False, 2), (4, 300, 96, 130, 3, 2, False, 1), (4, 137, 480, 600, 3, 2, False, 2),
    (256, 250, 96, 1100, 4, 1, False, 1), (16, 200, 480, 130, 4, 1, False, 2), (16, 500, 96, 600, 4, 2, False, 1), (4, 250, 480, 130, 4, 2, False, 2),
    (4, 512, 1056, 130, 4, 2, False, 1), (16, 300, 2080, 96, 3, 2, False, 7)])
@pytest.mark.parametrize("dt,out_dt,bias", [(o.BF16, o.BF16, True), (o.F16, o.F32, False)])
def test_linear_few_rows_tiles(dev_by_cus, dt, out_dt, bias, cus, M, K, N, mt, nt, swap, parts):
    dev = dev_by_cus[cus]
    x, w, b = mats(140 + K, M, K, N, dt)
    want = o.linear(x, dt, M, K, w, N, b if bias else None, out_dt=out_dt)
    out, layer = new(dev, DTS[out_dt], [M, N]), ops.Linear(up(dev, w, DTS[dt], [N, K]), up(dev, b, "F32", [N]) if bias else None)
    xt = up(dev, x, DTS[dt], [M, K])
    got = launches(dev, lambda: layer.forward(xt, out))
    close(out.to_numpy(), want, out_dt, "linear")
    S, L = (N, M) if swap else (M, N)
    tail = f"{mt}, {nt}, {str(swap).lower()}>"
    assert got[0][0].startswith("gemm_skinny_kernel<") and got[0][0].endswith(tail), got
    assert got[0][1] == -(-S // (64 * mt)) * -(-L // (64 * nt)) * parts, got
    assert [n for n, _, _ in got[1:]] == ([f"skinny_merge_kernel<{tail}"] if parts > 1 else []), got


def test_linear_few_rows_without_room(dev):
    """a context whose memory is taken: the parts' sums have no room, and the tiles run whole"""
    d = open_with({"H3S_MEM_FRACTION": "0.05"})
    M, K, N = 100, 1056, 300
    x, w, b = mats(150, M, K, N, o.BF16)
    want = o.linear(x, o.BF16, M, K, w, N, b, out_dt=o.BF16)
    xt, out = up(d, x, "BF16", [M, K]), new(d, "BF16", [M, N])
    layer = ops.Linear(up(d, w, "BF16", [N, K]), up(d, b, "F32", [N]))
    rest = new(d, "U8", [d.mem_cap() - d.mem_used() - (1 << 20)])
    got = launches(d, lambda: layer.forward(xt, out))
    close(out.to_numpy(), want, o.BF16, "linear without room")
    assert len(got) == 1 and got[0][0].startswith("gemm_skinny_kernel<"), got
    del rest
    got = launches(d, lambda: layer.forward(xt, out))
    close(out.to_numpy(), want, o.BF16, "linear with room again")
    assert len(got) == 2 and got[1][0].startswith("skinny_merge_kernel<"), got
    d.close()


@pytest.mark.parametrize("few,M,K,N", [(True, 137, 64, 512), (False, 256, 64, 512), (False, 512, 128, 2048), (True, 400, 64, 256),
                                       (False, 400, 96, 21504), (True, 64, 128, 16384), (True, 512, 2048, 2048), (False, 47104, 64, 96),
                                       (True, 47104, 64, 32), (True, 513, 64, 128), (False, 513, 64, 129),
                                       (True, 256, 512, 5376), (False, 512, 512, 10752), (True, 480, 2048, 10752)])
def test_linear_few_rows_or_tiles(dev, few, M, K, N):
    """which of the two matrix-core kernels takes a product with few rows on one side (skinny_loses): few steps with whole
    256 x 256 tiles, or more than a round of blocks, go to the tiles, the others to the few-row kernel"""
    x, w, b = mats(130, M, K, N, o.BF16)
    want = o.linear(x, o.BF16, M, K, w, N, b, out_dt=o.BF16)
    out, layer = new(dev, "BF16", [M, N]), ops.Linear(up(dev, w, "BF16", [N, K]), up(dev, b, "F32", [N]))
    xt = up(dev, x, "BF16", [M, K])
    names = [n.split("<")[0] for n, _, _ in launches(dev, lambda: layer.forward(xt, out))]
    close(out.to_numpy(), want, o.BF16, "linear")
    assert names[0] == ("gemm_skinny_kernel" if few else "gemm_f16_kernel"), names


@pytest.mark.parametrize("M,K,N", [(8300, 128, 64), (700, 1024, 600), (300, 96, 260), (130, 200, 70)])
@pytest.mark.parametrize("dt", [o.BF16, o.F16, o.F32])
def test_linear_acc(dev, dt, M, K, N):
    x, w, b = mats(110, M, K, N, dt)
    prev = o.to_dt(np.random.default_rng(111).standard_normal(M * N).astype(np.float32), dt)
    want = o.linear(x, dt, M, K, w, N, b, out_dt=dt, acc_into=prev)
    out = up(dev, prev, DTS[dt], [M, N])
    ops.Linear(up(dev, w, DTS[dt], [N, K]), up(dev, b, "F32", [N])).forward_acc(up(dev, x, DTS[dt], [M, K]), out)
    close(out.to_numpy(), want, dt, "linear_acc")


@pytest.mark.parametrize("dt", [o.BF16, o.F16, o.F32])
def test_scale_rows(dev, dt):
    N, K = 77, 200
    x, w, b = mats(120, 1, K, N, dt)
    s = np.random.default_rng(121).standard_normal(N).astype(np.float32)
    want = o.scale_rows(w, dt, N, K, s)
    layer = ops.Linear(up(dev, w, DTS[dt], [N, K]), up(dev, b, "F32", [N]))
    layer.scale_outputs(up(dev, s, "F32", [N]))
    assert_bits_equal(layer.weight.to_numpy(), want, "scale_rows")
    assert np.array_equal(layer.bias.to_numpy(), (b * s).astype(np.float32))
