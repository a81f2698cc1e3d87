"""Decode steps at the sizes where the split kernel's paths part: waves with
no, one, an odd and an even number of tiles; chunks and sequence ends inside a
tile; the XCD-affine grid over several sequences; query heads that share a KV
head without packing; a page table whose row is longer than the launch word
holds. Each against the oracle's double-precision attention over the same
dequantised cache.

Tolerances. Every product enters as a binary16 hi/lo pair (22 bits) and sums
are fp32: per head the steps measure up to 5e-6 (int8 with outlier channels),
2e-6 (f16) and 3e-5 (int4:32, whose scales are 17 times larger). A pair whose
halves do not belong together is off by a binary16 ulp of one element, 2^-11
of its share of a score: 7e-5 to 6e-4 of a head. So heads are held to 2^-15
(int8, f16), and int4 to 2^-14, twice what it measures and below 7e-5."""
import numpy as np
import pytest
import torch

import _oracle as O
from _cases import Case, args, build, reference, run, vid
from kvforge_amd import runtime as R

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    R.hip_lib()


def worst_head(got, ref):
    d = np.linalg.norm(got.astype(np.float64) - ref, axis=-1)
    return float(np.max(d / np.maximum(np.linalg.norm(ref, axis=-1), 1e-30)))


def limit(fmt):
    return 2.0 ** -14 if fmt == R.FMT_INT4 else 2.0 ** -15


@pytest.mark.parametrize("fmt,group", [(R.FMT_F16, 0), (R.FMT_INT8, 64), (R.FMT_INT8, 32), (R.FMT_INT4, 32),
                                       (R.FMT_INT4, 64)])
@pytest.mark.parametrize("H,Hkv,D", [(32, 8, 128), (16, 16, 64), (32, 4, 64)])
def test_every_head_keeps_its_precision(fmt, group, H, Hkv, D):
    b = build(Case(16, H, Hkv, D, 64, fmt, group, R.ORD_HEAD, 0, seed=3, outliers=True))
    err = worst_head(run(b, 1), reference(b))
    print(f"  {b.case.tag()}: worst head {err:.3g}", flush=True)
    assert err < limit(fmt)


@pytest.mark.parametrize("fmt", [R.FMT_INT8, R.FMT_INT4])
@pytest.mark.parametrize("order,bt", [(R.ORD_HEAD, 0), (R.ORD_TOKEN, 0), (R.ORD_TOKEN, 16)])
def test_two_column_passes(fmt, order, bt):
    # 8 heads by 4 groups: 32 (group, head) columns in two passes. Of int8 rows a
    # QK step meets one pass's groups and the other leaves it out; of int4 rows
    # every step meets both. Groups of very different size and sign show a
    # step that went to the wrong pass.
    q, K, V = O.make_data(2, 16, 2, 128, 517, 31)
    K *= np.repeat(np.float32([1, -4, 0.25, 2]), 32)
    V += np.repeat(np.float32([3, 0, -1, 5]), 32)
    b = build(Case(2, 16, 2, 128, 517, fmt, 32, order, bt), data=(q, K, V))
    for splits, warps, unroll in ((1, 4, 2), (1, 8, 4), (3, 8, 2), (5, 4, 4)):
        err = worst_head(run(b, splits, unroll=unroll, warps=warps), reference(b))
        print(f"  {b.case.tag()} S{splits} w{warps} u{unroll}: {err:.3g}", flush=True)
        assert err < limit(fmt)


@pytest.mark.parametrize("fmt,group,order,bt", [(R.FMT_F16, 0, R.ORD_HEAD, 0), (R.FMT_INT8, 64, R.ORD_HEAD, 16),
                                                (R.FMT_INT8, 64, R.ORD_TOKEN, 0), (R.FMT_INT4, 32, R.ORD_TOKEN, 16)])
def test_tiles_of_a_wave(fmt, group, order, bt):
    for n in (1, 31, 33, 127, 128, 160, 257, 385, 641, 1003):
        b = build(Case(1, 8, 2, 128, n, fmt, group, order, bt, seed=n))
        for splits, warps, unroll in ((1, 4, 2), (1, 8, 4), (3, 4, 2), (8, 4, 4), (16, 8, 2)):
            err = worst_head(run(b, splits, unroll=unroll, warps=warps), reference(b))
            print(f"  {b.case.tag()} S{splits} w{warps} u{unroll}: worst head {err:.3g}", flush=True)
            assert err < limit(fmt)


@pytest.mark.parametrize("B,H,Hkv", [(1, 32, 8), (4, 8, 2), (3, 64, 16), (2, 16, 16)])
def test_one_launch_over_the_affine_grid(B, H, Hkv):
    b = build(Case(B, H, Hkv, 128, 500, R.FMT_INT8, 64, R.ORD_HEAD, 0, seed=B))
    counters = R.fused_counters(B, Hkv)
    for splits in (2, 5):
        b.out.fill_(float("nan"))
        R.launch_fused(vid(b, True, 2), args(b, splits), counters)
        torch.cuda.synchronize()
        assert worst_head(b.out.cpu().numpy(), reference(b)) < limit(R.FMT_INT8)
        assert not bool(counters.any())


@pytest.mark.parametrize("bt", [0, 16])
def test_unpacked_query_heads(bt):
    b = build(Case(2, 12, 3, 64, 300, R.FMT_INT8, 32, R.ORD_TOKEN, bt, seed=7))
    assert worst_head(run(b, 4, pack=False), reference(b)) < limit(R.FMT_INT8)


@pytest.mark.parametrize("max_blocks", [(1 << 19) - 2, (1 << 19) - 1, (1 << 19) + 3])
def test_long_page_table_rows(max_blocks):
    b = build(Case(2, 8, 2, 128, 200, R.FMT_INT8, 64, R.ORD_HEAD, 16, seed=9))
    table = torch.zeros((2, max_blocks), dtype=torch.int32, device="cuda:0")
    table[:, :b.max_blocks] = b.table.view(2, b.max_blocks)
    b.table, b.max_blocks = table, max_blocks
    assert worst_head(run(b, 2), reference(b)) < limit(R.FMT_INT8)


@pytest.mark.parametrize("fmt,group,order", [(R.FMT_F16, 0, R.ORD_TOKEN), (R.FMT_INT8, 64, R.ORD_HEAD),
                                             (R.FMT_INT4, 32, R.ORD_TOKEN)])
@pytest.mark.parametrize("bt", [0, 16])
def test_unequal_lengths(fmt, group, order, bt):
    b = build(Case(5, 8, 2, 128, 300, fmt, group, order, bt, seed=11))
    lens = np.array([300, 0, 1, 33, 160], np.int32)
    ref = np.zeros((5, 8, 128))
    for i, n in enumerate(lens):
        if n:
            ref[i] = O.reference_attention(b.q_host[i:i + 1], np.ascontiguousarray(b.kdeq[i:i + 1, :, :n]),
                                           np.ascontiguousarray(b.vdeq[i:i + 1, :, :n]))[0]
    lens_d = torch.from_numpy(lens).cuda()
    for splits, flags in ((1, 0), (4, 0), (4, R.VARLEN_LONGEST_FIRST)):
        b.out.fill_(float("nan"))
        R.launch_varlen(vid(b, True, 2), args(b, splits), lens_d, flags=flags)
        torch.cuda.synchronize()
        got = b.out.cpu().numpy()
        assert not got[1].any()
        err = worst_head(got, ref)
        print(f"  {b.case.tag()} lengths S{splits}: worst head {err:.3g}", flush=True)
        assert err < limit(fmt)


@pytest.mark.parametrize("B,Hkv,n", [(1, 8, 24575), (1, 8, 24576), (2, 4, 24601), (1, 3, 65536)])
def test_large_two_launch_steps_on_either_grid(B, Hkv, n):
    # 48 MiB of rows from n = 24576 on (8 head groups; 3 do not divide over the
    # XCDs): the step against the partial kernel and the merge by themselves,
    # which run on the plain grid and the reference's chunks. Only fp32 sums
    # differ: 1e-5.
    b = build(Case(B, 4 * Hkv, Hkv, 128, n, R.FMT_INT8, 64, R.ORD_HEAD, 0, seed=n), check_cache=False)
    a = args(b, 12)
    R.launch(vid(b, True, 2), a)
    torch.cuda.synchronize()
    got = b.out.cpu().numpy().copy()
    b.out.fill_(float("nan"))
    R.launch_partial(vid(b, True, 2), a)
    R.launch_merge(128, a)
    torch.cuda.synchronize()
    assert worst_head(got, b.out.cpu().numpy().astype(np.float64)) < 1e-5


@pytest.mark.parametrize("bt,n,splits", [(0, 9215, 32), (0, 9216, 32), (0, 9216, 8), (16, 9220, 32)])
def test_large_steps_of_several_rounds(bt, n, splits):
    # 144 MiB of contiguous rows from n = 9216 on, in more (32 splits) and fewer
    # than two workgroups a CU; paged rows have no such line. As above.
    b = build(Case(4, 32, 8, 128, n, R.FMT_F16, 0, R.ORD_HEAD, bt, seed=n), check_cache=False)
    a = args(b, splits)
    R.launch(vid(b, True, 2), a)
    torch.cuda.synchronize()
    got = b.out.cpu().numpy().copy()
    b.out.fill_(float("nan"))
    R.launch_partial(vid(b, True, 2), a)
    R.launch_merge(128, a)
    torch.cuda.synchronize()
    assert worst_head(got, b.out.cpu().numpy().astype(np.float64)) < 1e-5


@pytest.mark.parametrize("fmt,group,D,bt,B,Hkv,n,splits", [
    (R.FMT_F16, 0, 128, 0, 1, 8, 12289, 24), (R.FMT_F16, 0, 128, 16, 4, 8, 3077, 8),
    (R.FMT_F16, 0, 64, 64, 2, 16, 6200, 5), (R.FMT_INT8, 64, 128, 16, 1, 8, 24577, 32),
    (R.FMT_INT8, 64, 128, 0, 8, 8, 3103, 16),  # 1024 workgroups: more than are resident at once
    (R.FMT_INT4, 32, 128, 0, 1, 8, 49155, 32), (R.FMT_INT4, 64, 64, 16, 4, 16, 12301, 8)])
def test_large_two_launch_steps_against_the_oracle(fmt, group, D, bt, B, Hkv, n, splits):
    # just past 48 MiB of rows in every format, contiguous and paged
    b = build(Case(B, 4 * Hkv, Hkv, D, n, fmt, group, R.ORD_HEAD, bt, seed=n), check_cache=False)
    print(f"  {b.case.tag()} S{splits}", flush=True)
    ref = O.reference_attention_mt(b.q_host, b.kdeq, b.vdeq, 16)
    for warps in (4, 8):
        err = worst_head(run(b, splits, warps=warps), ref)
        print(f"  {b.case.tag()} w{warps}: worst head {err:.3g}", flush=True)
        assert err < limit(fmt)


@pytest.mark.parametrize("fmt,group,bt", [(R.FMT_INT8, 64, 0), (R.FMT_F16, 0, 16)])
@pytest.mark.parametrize("n,splits", [(1000, 64), (1003, 8), (40, 3)])
def test_partials_of_a_whole_step(n, splits, fmt, group, bt):
    # a whole step's splits are whole tiles, ceil(n / splits) rounded up to 32
    # tokens: split s holds the attention over its own tokens alone, and the
    # splits past the end hold (-inf, 0, 0)
    b = build(Case(2, 8, 2, 128, n, fmt, group, R.ORD_HEAD, bt, seed=n))
    chunk = -(-(-(-n // splits)) // 32) * 32
    counters = R.fused_counters(2, 2)
    for entry in ("two launches", "one launch"):
        a = args(b, splits)
        if entry == "one launch":
            R.launch_fused(vid(b, True, 2), a, counters)
        else:
            R.launch(vid(b, True, 2), a)
        torch.cuda.synchronize()
        po, pm = (t.cpu().numpy().astype(np.float64) for t in a._keep)
        for s in range(splits):
            t0, t1 = min(n, s * chunk), min(n, (s + 1) * chunk)
            if t0 == t1:
                assert np.all(np.isneginf(pm[:, :, s, 0])) and not pm[:, :, s, 1].any() and not po[:, :, s].any()
                continue
            o, lse, m = O.reference_partials(b.q_host, np.ascontiguousarray(b.kdeq[:, :, t0:t1]),
                                             np.ascontiguousarray(b.vdeq[:, :, t0:t1]), 1)
            assert np.max(np.abs(pm[:, :, s, 0] - m[:, :, 0])) < 1e-4
            assert np.max(np.abs(pm[:, :, s, 0] + np.log2(pm[:, :, s, 1]) - lse[:, :, 0])) < 1e-4
            assert worst_head(po[:, :, s] / pm[:, :, s, 1:], o[:, :, 0]) < limit(fmt)


@pytest.mark.parametrize("D,H,Hkv,splits", [(128, 8, 2, 5), (64, 8, 1, 3), (128, 4, 4, 40)])
def test_partials_aligned_to_one_float(D, H, Hkv, splits):
    # part_o and part_ml are floats: buffers that start 4 bytes past a 256-byte
    # boundary give the same bits, and nothing beside them changes
    b = build(Case(2, H, Hkv, D, 1500, R.FMT_INT8, 32, R.ORD_HEAD, 0, seed=D + splits))
    counters = R.fused_counters(2, Hkv)
    pack = H > Hkv

    def step(entry, off):
        a = args(b, splits)
        bufs = []
        for field, t in zip(("part_o", "part_ml"), a._keep):
            raw = torch.full((t.numel() + 64,), 7.0, device="cuda:0")
            bufs.append((raw, t.numel()))
            setattr(a, field, raw.data_ptr() + 4 * off)
        b.out.fill_(float("nan"))
        if entry == "one launch":
            R.launch_fused(vid(b, pack, 2), a, counters)
        elif entry == "two launches":
            R.launch(vid(b, pack, 2), a)
        else:
            R.launch_partial(vid(b, pack, 2), a)
            R.launch_merge(D, a)
        torch.cuda.synchronize()
        for raw, size in bufs:
            assert bool((raw[:off] == 7).all()) and bool((raw[off + size:] == 7).all())
        return [b.out.cpu().numpy()] + [raw[off:off + size].cpu().numpy() for raw, size in bufs]

    for entry in ("two launches", "one launch", "partial and merge"):
        want = step(entry, 0)
        for off in (1, 2, 3):
            print(f"  D{D} S{splits} {entry} offset {off}", flush=True)
            for x, y in zip(step(entry, off), want):
                assert np.array_equal(x, y)


@pytest.mark.parametrize("fmt,group,D,bt,n", [(R.FMT_F16, 0, 128, 16, 12300), (R.FMT_INT8, 64, 128, 0, 24600)])
def test_large_steps_of_unpacked_query_heads(fmt, group, D, bt, n):
    # past 48 MiB of rows, four query heads a KV head without packing: the plain
    # grid, against the oracle
    b = build(Case(1, 32, 8, D, n, fmt, group, R.ORD_HEAD, bt, seed=n), check_cache=False)
    ref = O.reference_attention_mt(b.q_host, b.kdeq, b.vdeq, 16)
    for splits in (4, 8):
        assert worst_head(run(b, splits, pack=False), ref) < limit(fmt)
