"""Parts of the native code that no call of the C ABI reaches by itself,
through tests/native (built with the library)."""
import ctypes
import os

import numpy as np
import pytest

MB = 1 << 20


@pytest.fixture(scope="module")
def unit():
    import torch  # noqa: F401  (its HIP runtime, before the library asks for one)
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "_build", "libtrc_unit.so")
    if not os.path.exists(path):
        from tensorray_amd import build
        build.build_tests()
    return ctypes.CDLL(path)


def _fit(unit, first, total, per_item, per_window, kept, may_alloc, free):
    out = (ctypes.c_uint64 * 3)()
    c = ctypes.c_uint64
    unit.unit_fit_window(c(first), c(total), c(per_item), c(per_window), c(kept), ctypes.c_int(may_alloc), c(free), out)
    return tuple(out)


KEPT, ALLOCATED = 1, 2
WINDOW = 2 << 20  # paths
DEEP = 124        # bytes per path at 8 bounces


def test_window_choice(unit):
    # small requests take the stream's memory, large ones the whole window
    assert _fit(unit, 1000, 1000, DEEP, 0, 32 * MB, 1, 1 << 40) == (1000, KEPT, 0)
    assert _fit(unit, WINDOW, 9 * WINDOW, DEEP, 0, 32 * MB, 1, 1 << 40) == (WINDOW, ALLOCATED, WINDOW * DEEP)
    # half of it where the whole cannot be had
    assert _fit(unit, WINDOW, 9 * WINDOW, DEEP, 0, 32 * MB, 1, 200 * MB)[:2] == (WINDOW // 2, ALLOCATED)
    # nothing to be had, or a captured call: the largest the stream's memory holds
    assert _fit(unit, WINDOW, 9 * WINDOW, DEEP, 0, 32 * MB, 1, 0)[:2] == (WINDOW // 8, KEPT)
    assert _fit(unit, WINDOW, 9 * WINDOW, DEEP, 0, 32 * MB, 0, 1 << 40) == (WINDOW // 8, KEPT, 0)
    # not even that: small windows, down to half a megabyte
    assert _fit(unit, WINDOW, 9 * WINDOW, DEEP, 0, 0, 1, MB)[:2] == (8192, ALLOCATED)
    assert _fit(unit, WINDOW, 9 * WINDOW, DEEP, 0, 0, 1, 0)[:2] == (4096, 0)
    # odd sizes stay multiples of 64, and a request below the smallest window is asked for once
    w, how, asked = _fit(unit, 1_000_001, 1_000_001, DEEP, 0, 0, 1, 70 * MB)
    assert how == ALLOCATED and w % 64 == 0 and w * DEEP == asked <= 70 * MB < 1_000_001 * DEEP
    assert _fit(unit, 100, 100, DEEP, 0, 0, 1, 0) == (100, 0, 100 * DEEP)


def test_window_choice_ends_when_counters_outgrow_it(unit):
    """Queues keep a kilobyte of counters per chunk: with billions of samples
    no chunk fits the stream's memory, and the search ends."""
    w, how, _ = _fit(unit, 1 << 22, 1 << 33, 90, 1024, 32 * MB, 0, 1 << 40)
    assert how == 0 and w == 4096


# ---------------------------------------------------------------------------
# Quantized nodes
# ---------------------------------------------------------------------------
def _aligned(shape, dtype):
    buf = np.zeros(int(np.prod(shape)) * np.dtype(dtype).itemsize + 128, np.uint8)
    off = -buf.ctypes.data % 128
    return buf[off:off + int(np.prod(shape)) * np.dtype(dtype).itemsize].view(dtype).reshape(shape)


def _nodes(boxes):
    """[N][4][2][3] boxes as Bvh4Node words [N][32]: all slots inner children."""
    n = len(boxes)
    w = _aligned((n, 32), np.float32)
    for k in range(3):
        w[:, 4 * k:4 * k + 4] = boxes[:, :, 0, k]
        w[:, 12 + 4 * k:16 + 4 * k] = boxes[:, :, 1, k]
    w.view(np.uint32)[:, 24:28] = np.arange(4 * n, dtype=np.uint32).reshape(n, 4)
    return w


def _decode(q, inv_scale):
    """Child planes [N][4][2][3] of QNode words in float64."""
    org = np.stack([q[:, 0] & 0xFFFFF800, (q[:, 0] << 21 | q[:, 1] >> 11) & 0xFFFFF800, (q[:, 1] << 10) & 0xFFFFF800],
                   1).astype(np.uint32).view(np.float32).astype(np.float64)
    out = np.empty((len(q), 4, 2, 3))
    for k in range(3):
        h = np.ascontiguousarray(q[:, 4 + 4 * k:8 + 4 * k]).view(np.float16).astype(np.float64)  # lower 4, upper 4
        out[:, :, 0, k] = (org[:, None, k] + h[:, :4]) / inv_scale
        out[:, :, 1, k] = (org[:, None, k] + h[:, 4:]) / inv_scale
    return out


def _quantize(unit, boxes, inv_scale):
    nodes, q = _nodes(boxes), _aligned((len(boxes), 16), np.uint32)
    unit.unit_quantize(nodes.ctypes.data_as(ctypes.c_void_p), len(boxes), ctypes.c_float(inv_scale),
                       q.ctypes.data_as(ctypes.c_void_p))
    return q


def _random_boxes(n, centre, extent, smallest, seed):
    rng = np.random.default_rng(seed)
    c = rng.uniform(-0.5, 0.5, (n, 1, 1, 3)) * extent
    size = extent * 10.0 ** rng.uniform(np.log10(smallest), 0, (n, 1, 1, 1))
    a = centre + c + size * rng.uniform(-0.5, 0.5, (n, 4, 1, 3))
    d = size * rng.uniform(0, 0.5, (n, 4, 1, 3))
    return np.concatenate([a - d, a + d], 2).astype(np.float32)


def _inv_scale(unit, boxes):
    unit.unit_quant_inv_scale.restype = ctypes.c_float
    b = np.concatenate([boxes[:, :, 0].min((0, 1)), boxes[:, :, 1].max((0, 1))]).astype(np.float32)
    return float(unit.unit_quant_inv_scale(b.ctypes.data_as(ctypes.c_void_p)))


@pytest.mark.parametrize("extent", [1e-6, 2.0, 3e5])
@pytest.mark.parametrize("distance", [0.0, 3.0, 5e3, 2e4, 1e6])
def test_quantized_planes(unit, extent, distance):
    """Planes lie outside their boxes, by no more than the formats' roundings:
    2^-11 of an offset from the node's origin (a half), the widening of 2^-20,
    and as offsets reach the node's size plus the origin's rounding of 2^-12,
    2^-10 of the node's size and 2^-22 of the coordinate in all."""
    centre = np.array([1.0, -0.7, 0.3]) * distance * extent
    boxes = _random_boxes(2000, centre, extent, 1e-4, 5)
    inv = _inv_scale(unit, boxes)
    planes = _decode(_quantize(unit, boxes, inv), inv)
    b = boxes.astype(np.float64)
    assert np.isfinite(planes).all()
    assert (planes[:, :, 0] <= b[:, :, 0]).all() and (planes[:, :, 1] >= b[:, :, 1]).all()
    size = (b[:, :, 1].max(1) - b[:, :, 0].min(1))[:, None, None]
    slack = size * 2.0**-10 + np.abs(b).max((1, 2))[:, None, None] * 2.0**-22 + extent * 2.0**-37
    assert (np.abs(planes - b) <= slack).all()


@pytest.mark.gpu
def test_device_quantizes_as_the_host(unit):
    """Half-precision subnormals, zero, the largest and infinite planes too:
    the scales run from one at which all offsets underflow to one at which
    they overflow."""
    import torch
    for distance in (0.0, 3.0, 3e4):
        boxes = _random_boxes(3001, np.array([1.0, -0.7, 0.3]) * distance, 1.0, 1e-6, 6)
        boxes[::7, 1] = boxes[::7, 0]  # flat nodes: offsets of zero
        nodes = _nodes(boxes)
        for e in (-40, -24, -20, 0, 11, 14, 16, 17, 20):
            want = _quantize(unit, boxes, 2.0**e)
            dn = torch.from_numpy(nodes.copy()).cuda()
            out = torch.zeros(len(boxes), 16, dtype=torch.int32, device="cuda")
            p = ctypes.c_void_p
            assert unit.unit_quantize_device(p(dn.data_ptr()), len(boxes), ctypes.c_float(2.0**e), p(out.data_ptr())) == 0
            torch.cuda.synchronize()
            got = out.cpu().numpy().view(np.uint32)
            # the words behind the planes of a node are not set by either
            assert np.array_equal(got, want), (distance, e)


# ---------------------------------------------------------------------------
# Correctly rounded arithmetic of the device
# ---------------------------------------------------------------------------
def _math(unit, what, a, b=None, width=1):
    import torch
    n = len(a)
    da = torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda()
    db = torch.from_numpy(np.ascontiguousarray(b if b is not None else a, np.float32)).cuda()
    out = torch.zeros(n, width, device="cuda")
    p = ctypes.c_void_p
    assert unit.unit_math(what, p(da.data_ptr()), p(db.data_ptr()), p(out.data_ptr()), n) == 0
    torch.cuda.synchronize()
    return out.cpu().numpy()


def _same(got, want):
    """The same bits; any NaN for a NaN."""
    nan = np.isnan(want)
    return np.array_equal(np.isnan(got), nan) and np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))


def _floats(rng, n, lo, hi):
    """Random signs and mantissas (some of them all ones or zeros), exponents in [lo, hi]."""
    m = rng.integers(0, 1 << 23, n, dtype=np.uint32)
    m[::17] = (1 << 23) - 1
    m[1::17] = 0
    e = rng.integers(lo + 127, hi + 128, n, dtype=np.uint32)
    return (rng.integers(0, 2, n, dtype=np.uint32) << 31 | e << 23 | m).view(np.float32)


SPECIAL = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1e-45, -1e-45, 1.1754944e-38, 3.4028235e38, -3.4028235e38, 1.0,
                    2.0**-96, 2.0**-97, 2.0**126, 2.0**127], np.float32)


@pytest.mark.gpu
def test_device_divisions(unit):
    """Quotients by a shared reciprocal are those of IEEE division (float32
    division of numpy), overflowing ones and special operands included.
    Excepted are last bits of quotients of numerators below 2^-100 and of
    subnormal quotients."""
    rng = np.random.default_rng(1)
    n = 4_000_000
    a, b = _floats(rng, n, -98, 126), _floats(rng, n, -126, 125)
    sa, sb = (x.reshape(-1) for x in np.meshgrid(SPECIAL, np.concatenate([SPECIAL, _floats(rng, 50, -126, 126)])))
    for a, b in ((a, b), (sa, sb)):
        got = _math(unit, 0, a, b, 3)
        with np.errstate(all="ignore"):
            want = np.stack([a / b, -a / b, (np.float32(0.5) * a) / b], 1)
        tiny = (np.abs(want) < 2.0**-125) | (np.abs(np.stack([a, a, 0.5 * a], 1)) < 2.0**-100)
        ulp = np.float32(2.0**-23) * np.abs(want) + np.float32(1e-45)
        with np.errstate(all="ignore"):
            near = ~tiny | ~np.isfinite(want) | (np.abs(got - want) <= ulp)
        assert near.all()
        assert _same(got[~tiny], want[~tiny])
        assert np.isinf(want).any()


@pytest.mark.gpu
def test_device_roots(unit):
    rng = np.random.default_rng(2)
    # every mantissa over two exponents, then random positive floats and special ones
    every = np.arange(0x3F800000, 0x40800000, dtype=np.uint32).view(np.float32)
    x = np.concatenate([every, np.abs(_floats(rng, 1_000_000, -126, 127)), SPECIAL])
    with np.errstate(all="ignore"):
        assert _same(_math(unit, 1, x)[:, 0], np.sqrt(x))
        inside = x[(x >= 2.0**-96) & (x < 2.0**126)]
        assert _same(_math(unit, 2, inside)[:, 0], np.float32(1.0) / np.sqrt(inside))
        want = x / x
    assert _same(_math(unit, 4, x)[:, 0], want)


@pytest.mark.gpu
def test_device_normalize(unit):
    rng = np.random.default_rng(3)
    n = 1_000_000
    v = rng.normal(size=(n, 3)).astype(np.float32) * (2.0 ** rng.integers(-45, 60, (n, 1))).astype(np.float32)
    v[: n // 2] /= np.sqrt((v[: n // 2] ** 2).sum(1, dtype=np.float32))[:, None]  # nearly normalized
    v[::1001] = 0.0
    v[1::1001, 0] = np.inf
    v[2::1001] = 1e-30
    got = _math(unit, 3, v, width=4)
    with np.errstate(all="ignore"):
        l = np.sqrt(v[:, 0] * v[:, 0] + v[:, 1] * v[:, 1] + v[:, 2] * v[:, 2])
        want = np.concatenate([v / l[:, None], l[:, None]], 1)
    tiny = (np.abs(v) < 2.0**-100) & (v != 0)
    ok = ~np.concatenate([tiny, np.zeros((n, 1), bool)], 1)
    assert _same(got[ok], want[ok])
