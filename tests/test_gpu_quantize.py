"""The GPU quantize/place and append kernels byte for byte against a float32 restatement
of the reference's quantizer (runtime/kvf_host.h:72-121): the correctly
rounded quotient (x - zero) / scale rounded half away from zero, over rows
that sit on and beside rounding ties, scales that leave binary16, infinities
and NaN, with row counts around a wave's share, layouts whose inner dimension
is smaller than it, page sizes that are no power of two, and buffers aligned
to one element only. Codes and (scale, zero) words are bytes: equal or wrong."""
import numpy as np
import pytest
import torch

import _oracle as O
from kvforge_amd import runtime as R

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    R.hip_lib()


def hard_rows(rows, d, group, levels, seed):
    """fp32 rows of every kind in turn; group boundaries cut across them."""
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((rows, d)).astype(np.float32)
    f = np.float32
    for r in range(rows):
        kind = r % 10
        if kind == 1:  # quotients on and next to ties
            sc = f(np.float16(rng.uniform(1e-3, 1.0)))
            k = rng.integers(0, levels, d).astype(np.float32) + f(0.5)
            x[r] = k * sc
            x[r] = np.nextafter(x[r], f(rng.choice([-1e9, 1e9])), dtype=np.float32) if rng.random() < 0.7 else x[r]
            x[r, ::group] = 0
            x[r, 1::group] = f(levels) * sc
        elif kind == 2:  # a large offset: the zero point's rounding exceeds the range
            x[r] = f(1000.3) + f(1e-3) * x[r]
        elif kind == 3:
            x[r] = f(rng.standard_normal())  # all equal: scale 1
        elif kind == 4:
            x[r] *= f(1e-9)  # scale rounds to binary16 zero
        elif kind == 5:
            x[r] *= f(3e-5)  # subnormal binary16 scale
        elif kind == 6:
            x[r] *= f(1e5)  # zero point overflows
        elif kind == 7:
            x[r] = np.abs(x[r]) * f(1e8)  # scale overflows
        elif kind == 8:
            x[r, rng.integers(0, d, 3)] = [np.nan, np.inf, -np.inf]
        elif kind == 9:
            x[r] *= f(1e30)
    return x


def quantized(x, fmt, group):
    """float32 restatement; returns (row bytes, uint32 words or None)."""
    rows, d = x.shape
    with np.errstate(all="ignore"):
        if fmt == R.FMT_F16:
            return x.astype(np.float16).view(np.uint8).reshape(rows, -1), None
        levels = np.float32(255 if fmt == R.FMT_INT8 else 15)
        y = x.reshape(rows, d // group, group)
        lo, hi = np.fmin.reduce(y, -1), np.fmax.reduce(y, -1)
        zero_h = lo.astype(np.float16)
        scale = (hi - lo) / levels
        scale = np.where(scale <= 0, np.float32(1), scale)
        scale_h = scale.astype(np.float16)
        q = (y - zero_h.astype(np.float32)[..., None]) / scale_h.astype(np.float32)[..., None]
        assert q.dtype == np.float32
        q = np.fmin(np.fmax(q, np.float32(0)), levels)  # NaN to 0; clamping first leaves the rounding alone
        t = np.trunc(q)
        code = (t + (q - t >= np.float32(0.5))).astype(np.uint8).reshape(rows, d)
    words = scale_h.view(np.uint16).astype(np.uint32) | zero_h.view(np.uint16).astype(np.uint32) << 16
    if fmt == R.FMT_INT4:
        code = code[:, 0::2] | code[:, 1::2] << 4
    return code, words


def _at(buf, off, dtype, n):
    """n elements of dtype that start `off` bytes into a fresh device buffer."""
    raw = torch.full((off + n * dtype.itemsize + 64,), 0xA5, dtype=torch.uint8, device="cuda:0")
    buf.append(raw)
    return raw[off:off + n * dtype.itemsize]


SHAPES = [  # B, Hkv, n, bt
    (1, 1, 1, 0), (1, 3, 5, 0), (2, 8, 33, 0), (1, 2, 257, 16), (3, 5, 47, 16), (2, 1, 100, 12), (1, 8, 4099, 16),
    (2, 40, 515, 0),
]


FORMATS = [(R.FMT_F16, 0, 64), (R.FMT_F16, 0, 128), (R.FMT_INT8, 32, 64), (R.FMT_INT8, 64, 64), (R.FMT_INT8, 32, 128),
           (R.FMT_INT8, 64, 128), (R.FMT_INT8, 128, 128), (R.FMT_INT4, 32, 64), (R.FMT_INT4, 64, 64),
           (R.FMT_INT4, 32, 128), (R.FMT_INT4, 64, 128), (R.FMT_INT4, 128, 128)]


@pytest.mark.parametrize("order", [R.ORD_HEAD, R.ORD_TOKEN], ids=["hm", "tm"])
@pytest.mark.parametrize("fmt,group,d", FORMATS)
def test_quantized_bytes(fmt, group, d, order):
    for B, Hkv, n, bt in SHAPES:
        for off in (0, 1):  # buffers at a 256-byte boundary, and one element past it
            print(f"fmt {fmt}:{group} d{d} B{B} Hkv{Hkv} n{n} bt{bt} offset {off}", flush=True)
            X = hard_rows(B * Hkv * n, d, group or d, 255 if fmt != R.FMT_INT4 else 15, seed=n + d)
            data, words = quantized(X, fmt, group)
            meta = None if words is None else words.view(np.uint16).reshape(len(X), d // group, 2)
            want, wmeta, table, mb = O.place(B, Hkv, n, fmt, group, d, order, bt, data, meta)
            used, umeta, _, _ = O.place(B, Hkv, n, fmt, group, d, order, bt, np.full_like(data, 0xFF),
                                        None if meta is None else np.full_like(meta, 0xFFFF), table=table)
            want = np.where(used == 0xFF, want, 0xA5)
            keep = []
            x = _at(keep, 4 * off, torch.float32, X.size)
            x.copy_(torch.from_numpy(X.reshape(-1).view(np.uint8)))
            dd = _at(keep, off * (2 if fmt == R.FMT_F16 else 1), torch.uint8, want.size)
            md = _at(keep, 4 * off, torch.int32, wmeta.size) if wmeta is not None else None
            tb = torch.from_numpy(table.astype(np.int32)).cuda() if bt else None
            R.quantize_place(fmt, group, d, x, B, Hkv, n, order, bt, tb, mb, dd, md)
            torch.cuda.synchronize()
            assert np.array_equal(dd.cpu().numpy(), want.reshape(-1))
            if md is not None:
                wmeta = np.where(umeta == 0xFFFFFFFF, wmeta, 0xA5A5A5A5).astype(np.uint32)
                assert np.array_equal(md.cpu().numpy().view(np.uint32), wmeta.reshape(-1))
            for raw in keep[1:]:  # nothing beyond the buffers
                assert bool((raw[-64:] == 0xA5).all())


def appended(fmt, group, d, B, Hkv, n, order, bt, off, positions, seed):
    """One append call of a row per (sequence, head) into buffers filled with
    0xA5: the rows at the positions inside the layout hold their codes and
    words, and nothing else changed."""
    print(f"append fmt {fmt}:{group} d{d} B{B} Hkv{Hkv} n{n} bt{bt} {order} offset {off}", flush=True)
    X = hard_rows(B * Hkv, d, group or d, 255 if fmt != R.FMT_INT4 else 15, seed)
    data, words = quantized(X, fmt, group)
    # the same as a whole cache: token positions[b] of every head of b (tokens
    # n..mb * bt - 1 of a paged sequence are in its last page too)
    mb = -(-n // bt) if bt else 0
    cap = mb * bt if bt else n
    at = [(b, h, int(positions[b])) for b in range(B) for h in range(Hkv)]
    hit = [(i, (b * Hkv + h) * cap + t) for i, (b, h, t) in enumerate(at) if 0 <= t < cap]
    src, dst = (np.array(v, dtype=np.int64) for v in zip(*hit))

    def whole(rows, fill):
        out = np.zeros((B * Hkv * cap,) + rows.shape[1:], rows.dtype)
        out[dst] = rows[src] if fill is None else fill
        return out

    meta = None if words is None else words.view(np.uint16).reshape(len(X), d // group, 2)
    want, wmeta, table, _ = O.place(B, Hkv, cap, fmt, group, d, order, bt, whole(data, None),
                                    None if meta is None else whole(meta, None))
    used, umeta, _, _ = O.place(B, Hkv, cap, fmt, group, d, order, bt, whole(data, 0xFF),
                                None if meta is None else whole(meta, 0xFFFF), table=table)
    keep = []
    x = _at(keep, 4 * off, torch.float32, X.size)
    x.copy_(torch.from_numpy(X.reshape(-1).view(np.uint8)))
    dd = _at(keep, off * (2 if fmt == R.FMT_F16 else 1), torch.uint8, want.size)
    md = _at(keep, 4 * off, torch.int32, wmeta.size) if wmeta is not None else None
    tb = torch.from_numpy(table.astype(np.int32)).cuda() if bt else None
    pos = torch.tensor(positions, dtype=torch.int32, device="cuda:0")
    R.append_tokens(fmt, group, d, x, B, Hkv, n, pos, order, bt, tb, mb, dd, md)
    torch.cuda.synchronize()
    assert np.array_equal(dd.cpu().numpy(), np.where(used == 0xFF, want, 0xA5).reshape(-1).astype(np.uint8))
    if md is not None:
        wmeta = np.where(umeta == 0xFFFFFFFF, wmeta, 0xA5A5A5A5).astype(np.uint32)
        assert np.array_equal(md.cpu().numpy().view(np.uint32), wmeta.reshape(-1))
    for raw in keep[1:]:
        assert bool((raw[-64:] == 0xA5).all())


@pytest.mark.parametrize("order", [R.ORD_HEAD, R.ORD_TOKEN], ids=["hm", "tm"])
@pytest.mark.parametrize("fmt,group,d", FORMATS)
def test_appended_bytes(fmt, group, d, order):
    # a wave takes 4 (d 128) or 8 (d 64) heads: less than one wave's, one and a
    # part, several; page sizes that divide by shifting and by division
    for Hkv in (1, 5, 8, 40):
        for bt in (0, 12, 16):
            n = 45
            past = -(-n // bt) * bt if bt else n
            positions = [0, n - 1, -1, past - 1, past, 17, 2 ** 31 - 1, -2 ** 31, 31]
            for off in (0, 1):
                appended(fmt, group, d, len(positions), Hkv, n, order, bt, off, positions, seed=Hkv + bt)


@pytest.mark.parametrize("order,bt", [(R.ORD_HEAD, 0), (R.ORD_TOKEN, 2)])
def test_appended_bytes_past_a_grid_of_sequences(order, bt):
    # 65535 sequences are a grid's height; the rest come round again
    B = 65535 + 70
    rng = np.random.default_rng(5)
    appended(R.FMT_INT8, 32, 64, B, 1, 3, order, bt, 0, rng.integers(-1, 5, B), seed=5)


@pytest.mark.parametrize("fmt,group,d", [f for f in FORMATS if f[1]])
def test_signalling_nans_are_skipped(fmt, group, d):
    # one signalling NaN of either sign at every place of a group, beside the
    # group's minimum and maximum at every other place: both stay
    rng = np.random.default_rng(group)
    n = 4 * group
    X = rng.standard_normal((n, d)).astype(np.float32)
    for r in range(n):
        g = X[r].reshape(-1, group)
        for i in range(len(g)):
            lo, hi, nan = rng.permutation(group)[:3]
            nan = r % group
            lo, hi = ((v + 1) % group if v == nan else v for v in (lo, hi))
            g[i, lo], g[i, hi] = -9.0 - i, 11.0 + i
            g[i].view(np.uint32)[nan] = 0x7F9CC28F if (r // group) % 2 else 0xFFA6D5A5
    # (numpy's own minimum loses its neighbour to a signalling NaN in one
    # dimension: the restatement gets them quiet, which it skips everywhere)
    quiet = np.where(np.isnan(X), np.float32(np.nan), X)
    data, words = quantized(quiet, fmt, group)
    for entry in ("place", "append"):
        B, Hkv = (1, 1) if entry == "place" else (n // 4, 4)
        x = torch.from_numpy(X.view(np.int32)).cuda()
        dd = torch.zeros(data.size, dtype=torch.uint8, device="cuda:0")
        md = torch.zeros(words.size, dtype=torch.int32, device="cuda:0")
        if entry == "place":
            R.quantize_place(fmt, group, d, x, B, Hkv, n, R.ORD_HEAD, 0, None, 0, dd, md)
        else:
            R.append_tokens(fmt, group, d, x, B, Hkv, 1, torch.zeros(B, dtype=torch.int32, device="cuda:0"), R.ORD_HEAD, 0,
                            None, 0, dd, md)
        torch.cuda.synchronize()
        assert np.array_equal(md.cpu().numpy().view(np.uint32), words.reshape(-1)), entry
        assert np.array_equal(dd.cpu().numpy(), data.reshape(-1)), entry
