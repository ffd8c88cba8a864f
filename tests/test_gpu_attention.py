"""GPU parity of h3s_attention / h3s_attention_batch (kernels/h3sycl.cpp:1433-1917) against the oracle's restatement:
the int8 (SageAttention) form and the 16-bit form, through the C ABI. The reference's kernels are third-party (Intel's
ARK, oneDNN) and their rounding inside the softmax is not restated, so the bar is the parity tolerance on the result:
relative L2 below 1e-3 against the oracle's float64 softmax of the same quantized operands."""
import os

import numpy as np
import pytest

from oracle import oracle as o
from helpers import launches, new, up

pytestmark = pytest.mark.gpu

from sycl_minimax_h3_amd import DType, Device, Error, Tensor, ops  # noqa: E402

DTS = {o.F32: DType.F32, o.F16: DType.F16, o.BF16: DType.BF16}
o.set_threads(8)


def _open_with(env):
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
def dev_sage():
    """A context that takes the int8 form at every length (H3S_SAGE_MIN_S=0)."""
    d = _open_with({"H3S_SAGE_MIN_S": "0"})
    yield d
    d.close()


@pytest.fixture(scope="module")
def dev_sage4():
    """The int8 form at every length with grids sized for 4 compute units (H3S_CUS=4): k's mean then takes 32
    features a block wherever 16 would make more than 4 blocks."""
    d = _open_with({"H3S_SAGE_MIN_S": "0", "H3S_CUS": "4"})
    yield d
    d.close()


@pytest.fixture(scope="module")
def dev_16():
    """A context that keeps every call on the 16-bit form (H3S_ATTN=onednn)."""
    d = _open_with({"H3S_ATTN": "onednn"})
    yield d
    d.close()


def qkv(seed, S, H, D, dt, stride, spread=1.0):
    g = np.random.default_rng(seed)
    mk = lambda: o.to_dt((g.standard_normal((S, stride)) * spread).astype(np.float32), dt).ravel()  # noqa: E731
    return mk(), mk(), mk()


def run(d, q, k, v, dt, S, H, D, stride, out_dt):
    qt, kt, vt = (up(d, a, DTS[dt], [S, stride]) for a in (q, k, v))
    out = new(d, DTS[out_dt], [S, H * D])
    ops.attention(ops.Rows(qt, 0, stride, S, H, D), ops.Rows(kt, 0, stride, S, H, D), ops.Rows(vt, 0, stride, S, H, D), out)
    return out.to_numpy().ravel()


def check(got, want, out_dt, what):
    g, w = o.from_dt(got, out_dt).astype(np.float32), o.from_dt(want, out_dt).astype(np.float32)
    assert np.isfinite(g).all(), f"{what}: non-finite outputs"
    rel, cos = o.compare(g, w)
    assert rel < 1e-3 and cos > 0.99999, f"{what}: relative L2 {rel:.2e}, cos {cos:.7f}"


@pytest.mark.parametrize("sage", [True, False])
@pytest.mark.parametrize("dt,out_dt", [(o.BF16, o.BF16), (o.F16, o.F32), (o.F32, o.BF16)])
@pytest.mark.parametrize("S,H,D,pad", [(64, 1, 128, 0), (130, 3, 128, 16), (257, 2, 64, 0), (1000, 2, 128, 8), (77, 4, 64, 24)])
def test_attention(dev_sage, dev_16, sage, dt, out_dt, S, H, D, pad):
    stride = H * D + pad
    q, k, v = qkv(60 + S, S, H, D, dt, stride)
    want = o.attention(q, k, v, dt, S, H, D, stride, out_dt=out_dt, sage=sage)
    want = want[0] if sage else want
    got = run(dev_sage if sage else dev_16, q, k, v, dt, S, H, D, stride, out_dt)
    check(got, want, out_dt, f"{'int8' if sage else '16-bit'} S={S} H={H} D={D}")


@pytest.mark.parametrize("dt", [o.BF16, o.F16, o.F32])
@pytest.mark.parametrize("L,Hq,Hkv,D,pad", [(512, 4, 2, 128, 0), (513, 8, 8, 128, 8), (577, 3, 1, 64, 0), (640, 2, 1, 96, 0), (705, 5, 1, 128, 3),
                                            (1090, 16, 4, 64, 0), (511, 4, 1, 128, 0), (700, 33, 3, 64, 0)])
def test_attention_causal_groups(dev, dt, L, Hq, Hkv, D, pad):
    """From 512 rows and at most 32 heads (256 CUs) a block's wavefronts share its key tiles in two groups: odd and even
    numbers of tiles, a group without a last tile, heads padded to the kernel's size, rows off 16-byte boundaries (q
    prepared), and one case on either side of the line."""
    qs, kvs = Hq * D + pad, 2 * Hkv * D + pad
    g = np.random.default_rng(L)
    q = o.to_dt(g.standard_normal((L, qs)).astype(np.float32), dt).ravel()
    kv = o.to_dt(g.standard_normal((L, kvs)).astype(np.float32), dt).ravel()
    want = o.attention_causal(q, kv, kv[Hkv * D:], dt, L, Hq, Hkv, D, qs, kvs)
    qt, kvt = up(dev, q, DTS[dt], [L, qs]), up(dev, kv, DTS[dt], [L, kvs])
    out = new(dev, DTS[dt], [L, Hq * D])
    ops.attention_causal(ops.Rows(qt, 0, qs, L, Hq, D), ops.Rows(kvt, 0, kvs, L, Hkv, D), ops.Rows(kvt, Hkv * D, kvs, L, Hkv, D), out)
    check(out.to_numpy().ravel(), want, dt, f"causal L={L} Hq={Hq} Hkv={Hkv} D={D}")


@pytest.mark.parametrize("sage", [True, False])
@pytest.mark.parametrize("S,pad", [(1, 0), (63, 2), (65, 0), (200, 6), (129, 1)])
def test_attention_edges(dev_sage, dev_16, sage, S, pad):
    """One token, tiles cut short by one key either side of 64, and row strides that are not whole 16-byte vectors
    (the element-wise preparation)."""
    H, D = 2, 64
    stride = H * D + pad
    q, k, v = qkv(75 + S, S, H, D, o.BF16, stride)
    want = o.attention(q, k, v, o.BF16, S, H, D, stride, out_dt=o.F32, sage=sage)
    want = want[0] if sage else want
    got = run(dev_sage if sage else dev_16, q, k, v, o.BF16, S, H, D, stride, o.F32)
    check(got, want, o.F32, f"edge S={S} pad={pad}")


@pytest.mark.parametrize("sage", [True, False])
def test_attention_peaked_and_shifted(dev_sage, dev_16, sage):
    """Large score spreads (the online max moves a lot, most weights underflow) and a large common offset in k (the
    int8 form takes k's mean out)."""
    S, H, D = 300, 2, 128
    q, k, v = qkv(70, S, H, D, o.BF16, H * D, spread=4.0)
    k = o.to_dt(o.from_dt(k, o.BF16) + 3.0, o.BF16)
    want = o.attention(q, k, v, o.BF16, S, H, D, out_dt=o.F32, sage=sage)
    want = want[0] if sage else want
    got = run(dev_sage if sage else dev_16, q, k, v, o.BF16, S, H, D, H * D, o.F32)
    check(got, want, o.F32, "peaked")


@pytest.mark.parametrize("blocks", ["16", "32"])
@pytest.mark.parametrize("dt", [o.BF16, o.F16, o.F32])
@pytest.mark.parametrize("S,H,D", [(1, 2, 128), (191, 1, 64), (192, 2, 64), (384, 1, 128), (385, 2, 128),
                                   (2017, 3, 64), (5000, 1, 64)])
def test_attention_kmean(request, blocks, dt, S, H, D):
    """k's mean (h3sycl.cpp:1732-1737), seen through the output. A per-feature constant taken from k moves all of a
    query's scores alike and the softmax cancels it, so in ordinary inputs a wrong mean only shows through the
    quantization. Here each feature of k is a large power of two C_f plus or minus C_f 2^-7 in pairs of rows of
    opposite sign: the float32 sum in token order is exact and the mean is C_f, so k - mean is +-C_f 2^-7. A mean
    that misses one row then moves the output by a relative L2 of about 8e-2 (a CPU model of the scores from the
    oracle's quantizer), a missed chunk or mixed-up features by 0.15 to 1. Lengths around the 384- and 192-row
    chunks of the 16-bit and float32 inputs, and past the eight-chunk ring. blocks "32": a context sized for 4 CUs,
    where the mean takes 32 features a block (its chunks of 192 and 96 rows) for every case of 128 features or more."""
    dev_sage = request.getfixturevalue("dev_sage" if blocks == "16" else "dev_sage4")
    if blocks == "32" and (H * D) // 16 <= 4:
        pytest.skip("16 features a block already fit the 4 CUs")
    stride = H * D
    g = np.random.default_rng(S + 7 * H)
    q = o.to_dt(g.standard_normal((S, stride)).astype(np.float32), dt).ravel()
    C = 2.0 ** ((10 if dt == o.F16 else 14) + g.integers(0, 4, stride))          # C (1 +- 2^-7) exact in every type
    sgn = g.choice([-1.0, 1.0], (S // 2, stride))
    e = np.zeros((S, stride))
    e[0:2 * (S // 2):2], e[1:2 * (S // 2):2] = sgn, -sgn
    k = o.to_dt((C * (1.0 + e * 2.0 ** -7)).astype(np.float32), dt).ravel()
    v = o.to_dt(g.standard_normal((S, stride)).astype(np.float32), dt).ravel()
    want, _, _, _, _, km = o.attention(q, k, v, dt, S, H, D, stride, out_dt=o.F32, sage=True)
    assert np.array_equal(km, C.astype(np.float32)), "the oracle's mean is the constant"
    got = run(dev_sage, q, k, v, dt, S, H, D, stride, o.F32)
    check(got, want, o.F32, f"k mean S={S} H={H} D={D}")


@pytest.fixture(scope="module")
def dev_split():
    """Contexts for the wide kernel's split along the keys, per form: no split (H3S_ATTN_SPLIT=1), the default, and the
    default with grids sized for 16 or 6 compute units (H3S_CUS), so that a few hundred tokens make whole rounds and
    a split last one (at 6, whole blocks that the XCD renumbering leaves in order)."""
    modes = {"none": {"H3S_ATTN_SPLIT": "1"}, "default": {}, "cus16": {"H3S_CUS": "16"}, "cus6": {"H3S_CUS": "6"}}
    ds = {}
    for sage in (True, False):
        form = {"H3S_SAGE_MIN_S": "0"} if sage else {"H3S_ATTN": "onednn"}
        for name, env in modes.items():
            ds[(sage, name)] = _open_with({**form, **env})
    yield ds
    for d in ds.values():
        d.close()


@pytest.mark.parametrize("sage", [True, False])
@pytest.mark.parametrize("mode", ["none", "default", "cus16", "cus6"])
@pytest.mark.parametrize("S,H", [(64, 1), (777, 3), (2000, 5)])
def test_attention_split_last_round(dev_split, sage, mode, S, H):
    """Heads of 128 features (the wide kernel). The grids (attn_split_plan): 64 tokens, one block of two key tiles (never
    split); 777 tokens x 3 heads, 12 blocks of 25 tiles (on 256 CUs in 5 parts each, else whole); 2000 x 5, 40 blocks of
    63 tiles (on 256 CUs in 6 parts each; on 16, 32 whole blocks and 8 in 4; on 6, 36 whole blocks and 4 in 3). The
    parts' sums are merged by attn_merge_kernel."""
    D = 128
    stride = H * D
    q, k, v = qkv(90 + S, S, H, D, o.BF16, stride)
    want = o.attention(q, k, v, o.BF16, S, H, D, stride, out_dt=o.BF16, sage=sage)
    want = want[0] if sage else want
    d = dev_split[(sage, mode)]
    got = run(d, q, k, v, o.BF16, S, H, D, stride, o.BF16)
    check(got, want, o.BF16, f"{'int8' if sage else '16-bit'} {mode} S={S} H={H}")
    t, out = new(d, "BF16", [S, stride]), new(d, "BF16", [S, stride])
    R = ops.Rows(t, 0, stride, S, H, D)
    grids = {n.split("<")[0]: b for n, b, _ in launches(d, lambda: ops.attention(R, R, R, out))}
    whole = H * -(-S // 256)
    parts = {("default", 777): (0, 5), ("default", 2000): (0, 6), ("cus16", 2000): (32, 4), ("cus6", 2000): (36, 3)}.get((mode, S))
    assert grids["attn_pl_kernel"] == (parts[0] + (whole - parts[0]) * parts[1] if parts else whole), grids
    assert ("attn_merge_kernel" in grids) == bool(parts), grids


@pytest.mark.parametrize("sage", [True, False])
@pytest.mark.parametrize("per_tile", [12.0, 30.0])
def test_attention_rising_scores(dev_sage, dev_16, sage, per_tile):
    """Scores that rise along the keys by about per_tile (base 2) every 64 keys: at 12 the weights stay inside half's
    range while the running reference lags behind the max; at 30 every tile passes the reference by more than half's
    range (the int8 kernel's overflow path: the max, the rescale, the weights again)."""
    S, H, D = 640, 2, 128
    g = np.random.default_rng(71)
    ramp = (np.arange(S, dtype=np.float32) / 64.0 * per_tile / (np.sqrt(D) * np.log2(np.e)))[:, None]
    q = o.to_dt((1.0 + 0.05 * g.standard_normal((S, H * D))).astype(np.float32), o.BF16).ravel()
    k = o.to_dt((ramp + 0.05 * g.standard_normal((S, H * D))).astype(np.float32), o.BF16).ravel()
    v = o.to_dt(g.standard_normal((S, H * D)).astype(np.float32), o.BF16).ravel()
    want = o.attention(q, k, v, o.BF16, S, H, D, out_dt=o.F32, sage=sage)
    want = want[0] if sage else want
    got = run(dev_sage if sage else dev_16, q, k, v, o.BF16, S, H, D, H * D, o.F32)
    check(got, want, o.F32, f"rising scores, {per_tile} a tile")


def test_attention_default_form_by_length(dev):
    """The default context: below 8192 tokens the 16-bit form, from 8192 on the int8 form (kernels/h3sycl.cpp:138, 1773)."""
    H, D = 1, 64
    for S, sage in ((500, False), (8200, True)):
        q, k, v = qkv(71, S, H, D, o.BF16, H * D)
        want = o.attention(q, k, v, o.BF16, S, H, D, out_dt=o.BF16, sage=sage)
        want = want[0] if sage else want
        other = o.attention(q, k, v, o.BF16, S, H, D, out_dt=o.BF16, sage=not sage)
        other = other[0] if not sage else other
        got = run(dev, q, k, v, o.BF16, S, H, D, H * D, o.BF16)
        check(got, want, o.BF16, f"default S={S}")
        # and it is measurably the form named, not the other one
        rg, _ = o.compare(o.from_dt(got, o.BF16), o.from_dt(want, o.BF16))
        ro, _ = o.compare(o.from_dt(got, o.BF16), o.from_dt(other, o.BF16))
        assert rg < ro, f"S={S}: closer to the other form ({rg:.2e} vs {ro:.2e})"


def test_attention_batch(dev_16):
    B, S, H, D = 3, 96, 2, 64
    stride = H * D
    q, k, v = qkv(72, B * S, H, D, o.BF16, stride)
    qt, kt, vt = (up(dev_16, a, "BF16", [B * S, stride]) for a in (q, k, v))
    out = new(dev_16, "BF16", [B * S, H * D])
    ops.attention_batch(ops.Rows(qt, 0, stride, B * S, H, D), ops.Rows(kt, 0, stride, B * S, H, D),
                        ops.Rows(vt, 0, stride, B * S, H, D), B, out)
    got = out.to_numpy().reshape(B, S * H * D)
    for b in range(B):
        sl = slice(b * S * stride, (b + 1) * S * stride)
        want = o.attention(q[sl], k[sl], v[sl], o.BF16, S, H, D, out_dt=o.BF16, sage=False)
        check(got[b], want, o.BF16, f"sequence {b}")


@pytest.mark.parametrize("dt", [o.F16, o.BF16, o.F32])
@pytest.mark.parametrize("L,Hq,Hkv,D", [(1, 2, 1, 128), (37, 8, 2, 128), (130, 4, 4, 64), (300, 6, 2, 128), (257, 8, 1, 64)])
def test_attention_causal(dev, dt, L, Hq, Hkv, D):
    """The text encoder's causal attention with grouped kv heads (kernels/h3sycl.cpp:873-898), q and kv in buffers of
    wider rows."""
    qs, kvs = Hq * D + 8, 2 * Hkv * D
    g = np.random.default_rng(97 + L)
    q = o.to_dt(g.standard_normal(L * qs).astype(np.float32), dt)
    kv = o.to_dt(g.standard_normal(L * kvs).astype(np.float32), dt)
    k, v = kv, kv[Hkv * D:]                                           # k and v interleaved in one buffer
    want = o.attention_causal(q, k, v, dt, L, Hq, Hkv, D, qs, kvs)
    qt, kvt = up(dev, q, DTS[dt], [L, qs]), up(dev, kv, DTS[dt], [L, kvs])
    out = new(dev, DTS[dt], [L, Hq * D])
    ops.attention_causal(ops.Rows(qt, 0, qs, L, Hq, D), ops.Rows(kvt, 0, kvs, L, Hkv, D), ops.Rows(kvt, Hkv * D, kvs, L, Hkv, D), out)
    check(out.to_numpy().ravel(), want, dt, f"causal L={L} Hq={Hq} Hkv={Hkv}")


def test_attention_refuses(dev):
    p = new(dev, "BF16", [64, 600])
    with pytest.raises(Error, match="at most 256"):
        ops.attention(ops.Rows(p, 0, 600, 64, 2, 300), ops.Rows(p, 0, 600, 64, 2, 300), ops.Rows(p, 0, 600, 64, 2, 300), p)


@pytest.mark.parametrize("sage", [True, False])
@pytest.mark.parametrize("S,H,D,pad,out_dt", [(200, 2, 256, 0, o.BF16), (130, 3, 96, 0, o.F32), (77, 2, 80, 8, o.BF16),
                                               (65, 2, 32, 0, o.F16), (150, 1, 200, 2, o.F32), (64, 2, 7, 1, o.BF16),
                                               (300, 1, 130, 0, o.BF16)])
def test_attention_head_sizes(dev_sage, dev_16, sage, S, H, D, pad, out_dt):
    """Heads of any size up to 256: 256 in its own kernel, the others zero-padded to 64, 128 or 256 features in the
    preparation and stored at their own size (odd sizes one feature at a time). The int8 form is the reference's only
    at 64 and 128 features (kernels/h3sycl.cpp:1706): on a context that asks for it at every length (dev_sage), these
    head sizes still take the 16-bit form and match the 16-bit oracle."""
    stride = H * D + pad
    q, k, v = qkv(110 + D, S, H, D, o.BF16, stride)
    assert D not in (64, 128)
    want = o.attention(q, k, v, o.BF16, S, H, D, stride, out_dt=out_dt, sage=False)
    got = run(dev_sage if sage else dev_16, q, k, v, o.BF16, S, H, D, stride, out_dt)
    check(got, want, out_dt, f"16-bit ({'a context asking for int8' if sage else 'default'}) S={S} H={H} D={D}")
    if sage:
        # and not the int8 form's result: its quantization moves the output far past the parity bar
        int8 = o.attention(q, k, v, o.BF16, S, H, D, stride, out_dt=out_dt, sage=True)[0]
        rel, _ = o.compare(o.from_dt(got, out_dt).astype(np.float32), o.from_dt(int8, out_dt).astype(np.float32))
        assert rel > 1e-3, f"S={S} D={D}: the result is the int8 form's (relative L2 {rel:.2e} from it)"


@pytest.mark.parametrize("dt", [o.BF16, o.F32])
@pytest.mark.parametrize("L,Hq,Hkv,D", [(50, 4, 2, 256), (129, 2, 1, 80), (33, 6, 3, 200), (70, 2, 2, 36)])
def test_attention_causal_head_sizes(dev, dt, L, Hq, Hkv, D):
    """The causal form at the head sizes the reference takes (D <= 256, kernels/h3sycl.cpp:877)."""
    qs, kvs = Hq * D, 2 * Hkv * D
    g = np.random.default_rng(131 + D)
    q = o.to_dt(g.standard_normal(L * qs).astype(np.float32), dt)
    kv = o.to_dt(g.standard_normal(L * kvs).astype(np.float32), dt)
    want = o.attention_causal(q, kv, kv[Hkv * D:], dt, L, Hq, Hkv, D, qs, kvs)
    qt, kvt = up(dev, q, DTS[dt], [L, qs]), up(dev, kv, DTS[dt], [L, kvs])
    out = new(dev, DTS[dt], [L, Hq * D])
    ops.attention_causal(ops.Rows(qt, 0, qs, L, Hq, D), ops.Rows(kvt, 0, kvs, L, Hkv, D), ops.Rows(kvt, Hkv * D, kvs, L, Hkv, D), out)
    check(out.to_numpy().ravel(), want, dt, f"causal L={L} Hq={Hq} Hkv={Hkv} D={D}")


@pytest.mark.parametrize("sage", [True, False])
@pytest.mark.parametrize("S", [1, 31, 32, 33, 63, 64, 65, 96, 97, 127, 160, 192, 193, 224, 255, 256, 257, 300, 511, 513])
def test_attention_wide_tiles(dev_sage, dev_16, sage, S):
    """The wide kernel (heads of 128) around its 32-key tiles, the 64-row scale blocks, the rings of six and four stages
    (sequences shorter and longer than they hold) and the 256-query blocks; the rows of q, k and v inside wider rows."""
    H, D = 3, 128
    stride = 3 * H * D
    q, k, v = qkv(110 + S, S, H, D, o.BF16, stride)
    want = o.attention(q, k, v, o.BF16, S, H, D, stride, out_dt=o.F32, sage=sage)
    want = want[0] if sage else want
    got = run(dev_sage if sage else dev_16, q, k, v, o.BF16, S, H, D, stride, o.F32)
    check(got, want, o.F32, f"wide tiles S={S}")


@pytest.mark.parametrize("sage", [True, False])
@pytest.mark.parametrize("dt", [o.BF16, o.F16, o.F32])
def test_attention_wide_split_ranges(dev_split, sage, dt):
    """Split blocks whose key ranges end inside a scale block (47 tiles of 32 keys in ranges of 6): each part's scales,
    masks and partial sums, for every type of q."""
    S, H, D = 1500, 2, 128
    q, k, v = qkv(131, S, H, D, dt, H * D)
    want = o.attention(q, k, v, dt, S, H, D, H * D, out_dt=o.F32, sage=sage)
    want = want[0] if sage else want
    got = run(dev_split[(sage, "default")], q, k, v, dt, S, H, D, H * D, o.F32)
    check(got, want, o.F32, f"wide split {sage}")


@pytest.mark.parametrize("where", ["row on row", "in the q rows", "across q", "over k", "over v"])
@pytest.mark.parametrize("form,dt,S,H,D", [("int8", o.BF16, 1100, 3, 128), ("16-bit", o.BF16, 1100, 3, 128), ("16-bit", o.F32, 900, 2, 128),
                                           ("16-bit", o.F16, 600, 2, 64), ("int8", o.BF16, 600, 2, 64), ("causal", o.BF16, 1100, 3, 128),
                                           ("causal", o.BF16, 300, 3, 64)])
def test_attention_out_over_inputs(dev, dev_sage, dev_16, form, dt, S, H, D, where):
    """out in memory that q, k or v also lie in: row on row with a contiguous q (each block has read its rows before it
    writes them), and otherwise (q prepared first: the launches say so). q, k and v are the columns of one buffer, whose
    rows out then runs along at a third of the stride, or contiguous tensors."""
    d = {"int8": dev_sage, "16-bit": dev_16, "causal": dev}[form]
    W = H * D
    q, k, v = qkv(140 + S + D, S, H, D, dt, W)
    if form == "causal":
        want = o.attention_causal(q, k, v, dt, S, H, H, D, W, W)
    else:
        want = o.attention(q, k, v, dt, S, H, D, W, out_dt=dt, sage=form == "int8")
        want = want[0] if form == "int8" else want
    two = lambda a: a.reshape(S, W)  # noqa: E731
    esz = DTS[dt].size()
    if where == "in the q rows":                                 # q | k | v in rows of 3 W, out contiguous from the start
        buf = up(d, np.concatenate([two(q), two(k), two(v)], 1).ravel(), DTS[dt], [S, 3 * W])
        qr, kr, vr = (ops.Rows(buf, i * W, 3 * W, S, H, D) for i in range(3))
        out = Tensor(DTS[dt], [S, W], buf.ptr(), buf._owner, d)
    elif where == "across q":                                    # out starts 64 rows after q in one allocation
        buf = up(d, np.concatenate([q, q[:64 * W]]), DTS[dt], [S + 64, W])
        kt, vt = (up(d, a, DTS[dt], [S, W]) for a in (k, v))
        qr, kr, vr = ops.Rows(buf, 0, W, S, H, D), ops.Rows(kt, 0, W, S, H, D), ops.Rows(vt, 0, W, S, H, D)
        out = Tensor(DTS[dt], [S, W], buf.ptr() + 64 * W * esz, buf._owner, d)
    else:
        qt, kt, vt = (up(d, a, DTS[dt], [S, W]) for a in (q, k, v))
        qr, kr, vr = (ops.Rows(t, 0, W, S, H, D) for t in (qt, kt, vt))
        out = {"row on row": qt, "over k": kt, "over v": vt}[where]
    call = lambda: (ops.attention_causal if form == "causal" else ops.attention)(qr, kr, vr, out)  # noqa: E731
    call()
    check(out.to_numpy().ravel(), want, dt, f"{form} out {where}")
    names = [n for n, _, _ in launches(d, call)]                 # (on what the first call left: only the launches are read)
    q_prepared = any("qk_prep" in n for n in names)
    assert q_prepared == (where in ("in the q rows", "across q") or (form == "int8" and D == 64)), names


@pytest.mark.parametrize("value", [-np.inf, -1e30])
@pytest.mark.parametrize("form,dt,L,Hq,D,dead", [
    ("causal", o.BF16, 600, 4, 128, [(64, 128)]),               # two key groups: the second group's first tile
    ("causal", o.BF16, 700, 3, 64, [(64, 128), (192, 256)]),    # and a later one
    ("causal", o.F32, 640, 2, 128, [(0, 63), (64, 128)]),       # nearly all of the first group's too
    ("causal", o.BF16, 200, 2, 128, [(64, 128)]),               # one group
    ("whole", o.BF16, 300, 2, 128, [(0, 32)]),                  # the wide form's first tile of 32 keys
    ("whole", o.BF16, 1500, 2, 128, [(0, 40), (192, 256), (1470, 1500)]),   # the first tiles of split ranges
    ("whole", o.F32, 300, 2, 64, [(0, 64), (250, 300)]),        # heads of 64: the first tile of 64 keys
    ("whole", o.BF16, 150, 1, 256, [(0, 100)]),
])
def test_attention_dead_keys(dev, dev_16, form, dt, L, Hq, D, dead, value):
    """Keys that every query scores at minus infinity (an infinite feature, or one past half's range: the operands are
    half) weigh nothing, wherever the tiles of a walk over the keys begin: whole tiles of them, the first of a key group,
    of a split range or of the walk itself among them."""
    g = np.random.default_rng(L + D)
    q, k, v = (g.standard_normal((L, Hq * D)).astype(np.float32) for _ in range(3))
    q = q.reshape(L, Hq, D)
    q[:, :, 3] = np.abs(q[:, :, 3]) + 0.5                        # times the infinite feature: minus infinity
    q = q.reshape(L, Hq * D)
    alive = np.ones(L, bool)
    for a, b in dead:
        alive[a:b] = False
        k[a:b, 3::D] = value
    # the same softmax in 64 bits over the other keys, of the operands as they are rounded to half
    h = lambda a: o.from_dt(o.to_dt(a, dt).ravel(), dt).reshape(a.shape).astype(np.float16).astype(np.float64)  # noqa: E731
    kf = np.where(alive[:, None], k, 0.0).astype(np.float32)
    want = np.empty((L, Hq * D))
    for hh in range(Hq):
        sl = slice(hh * D, hh * D + D)
        sc = h(q[:, sl]) @ h(kf[:, sl]).T / np.sqrt(D)
        see = np.broadcast_to(alive, (L, L)) & (np.tri(L, dtype=bool) if form == "causal" else True)
        sc = np.where(see, sc, -np.inf)
        with np.errstate(invalid="ignore"):
            p = np.exp(sc - sc.max(1, keepdims=True))
        want[:, sl] = p @ h(v[:, sl]) / p.sum(1, keepdims=True)
    rows = see.any(1)                                            # (a causal row that sees dead keys only has no value)
    q, k, v = (o.to_dt(a, dt).ravel() for a in (q, k, v))
    if form == "causal":
        qt, kt, vt = (up(dev, a, DTS[dt], [L, Hq * D]) for a in (q, k, v))
        out = new(dev, DTS[dt], [L, Hq * D])
        R = lambda t: ops.Rows(t, 0, Hq * D, L, Hq, D)  # noqa: E731
        ops.attention_causal(R(qt), R(kt), R(vt), out)
        got = out.to_numpy().ravel()
    else:
        got = run(dev_16, q, k, v, dt, L, Hq, D, Hq * D, dt)
    got = o.from_dt(got, dt).astype(np.float32).reshape(L, Hq * D)[rows]
    assert np.isfinite(got).all(), f"{int((~np.isfinite(got)).any(1).sum())} of {rows.sum()} rows are not finite"
    rel, _ = o.compare(got.ravel(), want[rows].astype(np.float32).ravel())
    # P in half, the result in dt: 2^-9 of bfloat16 (relative 2-norm 1.7e-3), under 1e-3 of half's weights
    assert rel < (3e-3 if dt == o.BF16 else 1e-3), f"relative L2 {rel:.2e}"


@pytest.mark.parametrize("sage", [True, False])
def test_attention_without_room_for_parts(sage):
    """a context whose memory is taken: the split blocks' partial sums have no room, and every block runs whole"""
    d = _open_with({"H3S_MEM_FRACTION": "0.05", **({"H3S_SAGE_MIN_S": "0"} if sage else {"H3S_ATTN": "onednn"})})
    S, H, D = 777, 3, 128
    W = H * D
    q, k, v = qkv(160, S, H, D, o.BF16, W)
    want = o.attention(q, k, v, o.BF16, S, H, D, W, out_dt=o.BF16, sage=sage)
    want = want[0] if sage else want
    qr, kr, vr = (ops.Rows(up(d, a, "BF16", [S, W]), 0, W, S, H, D) for a in (q, k, v))
    out = new(d, "BF16", [S, W])
    t = new(d, "BF16", [64, 4 * W])                              # a call of whole blocks that grows the other scratch as far
    r = ops.Rows(t, 0, 4 * W, 64, 4 * H, D)
    ops.attention(r, r, r, t)
    rest = new(d, "U8", [d.mem_cap() - d.mem_used() - (1 << 20)])
    names = [n.split("<")[0] for n, _, _ in launches(d, lambda: ops.attention(qr, kr, vr, out))]
    check(out.to_numpy().ravel(), want, o.BF16, "whole blocks")
    assert "attn_merge_kernel" not in names, names
    del rest
    names = [n.split("<")[0] for n, _, _ in launches(d, lambda: ops.attention(qr, kr, vr, out))]
    check(out.to_numpy().ravel(), want, o.BF16, "split blocks")
    assert "attn_merge_kernel" in names, names
    d.close()
