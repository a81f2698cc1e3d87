"""Lengths up to the largest an int holds, where the end of the last split and
of the last tile lies past 2^31. The table names a handful of pages over and
over, so that the cache is small: page 0 holds tokens that score 0, page 1,
the last one of the sequence, tokens that score 20 (in log2), which makes its
4096 weigh as much as the 2^31 before it, so a token too many or too few at the
end moves the result by 1e-4 of it; a lost split of page 0 by more.

The one number compared is that mean; the kernel adds 2^31 / (splits * waves *
4) weights of 1 per lane, which fp32 holds exactly up to 2^24, in eights: 1e-5."""
import math

import numpy as np
import pytest
import torch

from kvforge_amd import runtime as R

pytestmark = pytest.mark.gpu

BT = 4096
D = 64


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    R.hip_lib()


def pages(fmt, n):
    """K, V and their words: page 0, page 1 up to the last token, then NaN."""
    dev = torch.device("cuda:0")
    k = torch.zeros((2, BT, D), device=dev)
    v = torch.zeros((2, BT, D), device=dev)
    k[1] = 20.0 / (D * math.log2(math.e) / math.sqrt(D))  # the query is all ones
    v[0], v[1] = 1.0, 3.0
    end = (n - 1) % BT + 1
    if fmt == R.FMT_F16:
        k[1, end:] = float("nan")
        v[1, end:] = float("nan")
        return k.half().view(torch.uint8).flatten(), v.half().view(torch.uint8).flatten(), None, None, k.half().double()
    km = torch.stack((torch.ones_like(k[..., 0]), k[..., 0]), -1).half()  # codes 0: the zero point is the value
    vm = torch.stack((torch.ones_like(v[..., 0]), v[..., 0]), -1).half()
    vm[1, end:] = float("nan")
    km[1, end:] = float("nan")
    codes = torch.zeros(2 * BT * D // 2, dtype=torch.uint8, device=dev)
    return codes, codes.clone(), km.view(torch.int32).flatten(), vm.view(torch.int32).flatten(), km[..., 1:].double()


@pytest.mark.parametrize("fmt,group", [(R.FMT_F16, 0), (R.FMT_INT4, 64)])
@pytest.mark.parametrize("lens", [False, True], ids=["uniform", "lengths"])
@pytest.mark.parametrize("n,splits", [(2 ** 31 - 1, 256), (2 ** 31 - 27, 256), (2 ** 31 - 251, 200), (2 ** 31 - 4097, 256)])
def test_last_split_and_tile(n, splits, lens, fmt, group):
    dev = torch.device("cuda:0")
    k, v, km, vm, keys = pages(fmt, n)
    mb = -(-n // BT)
    table = torch.zeros(mb, dtype=torch.int32, device=dev)
    table[-1] = 1
    q = torch.ones((1, 1, D), device=dev)
    out = torch.full((1, 1, D), float("nan"), device=dev)
    po = torch.full((1, 1, splits, D), float("nan"), device=dev)
    pm = torch.full((1, 1, splits, 2), float("nan"), device=dev)
    a = R.make_args(q, k, v, km, vm, table, out, po, pm, 1, 1, 1, n, splits, 8, group=group, block_tokens=BT,
                    max_blocks=mb, D=D)
    vid = R.variant_id(fmt, R.ORD_HEAD, True, 1, 2, D)
    print(f"n {n} splits {splits} fmt {fmt} lens {lens}", flush=True)
    if lens:
        R.launch_varlen(vid, a, torch.tensor([n], dtype=torch.int32, device=dev))
    else:
        R.launch(vid, a)
    torch.cuda.synchronize()
    end = (n - 1) % BT + 1
    s1 = float(keys[1, 0, 0]) * (D / math.sqrt(D))  # natural log units
    w = math.exp(s1)
    want = ((n - end) * 1.0 + end * w * 3.0) / ((n - end) + end * w)
    got = out.double().cpu().numpy()
    assert np.all(np.isfinite(got))
    assert np.max(np.abs(got - want)) < 1e-5 * want, (got.min(), got.max(), want)
