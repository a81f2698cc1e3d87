"""The decode-attention work that is timed and checked, case by case.

A case is one pass of a serving program through kvforge_amd.runtime:

  decode   one token's attention over a stack of `layers` layers, each with a
           KV cache of its own, every sequence at the same length n
           (runtime.launch, or runtime.launch_fused with entry "fused");
  varlen   the same over a batch of sequences of unequal lengths, with a
           binary16 query and output (runtime.launch_varlen,
           runtime.launch_fused or runtime.launch_persistent);
  step     a whole decode step: the new token's K and V rows are appended to
           every sequence (runtime.append_tokens), then attention runs over
           the cache with them in it; captured once in a HIP graph and
           replayed, as a program does whose steps are short;
  prefill  a prompt's K and V rows quantized and placed into the cache
           (runtime.quantize_place).

A case names the head counts, the head dimension d, n (the tokens of a sequence,
at most n where the lengths are unequal), the cache format and its layout (order "hm" head-major or
"tm" token-major; bt tokens per page, 0 for contiguous), and for the attention
calls the plan: splits, wavefronts per workgroup, and the unroll. Unequal
lengths are drawn from the case itself, so that its work is known; the values
come from the seed.

The caches are made here, by plain torch, and not by the library: what they
hold is then the same whichever build runs.
"""
import math
import random

import torch

from kvforge_amd import runtime as R

MIB = 1 << 20
#: Cache bytes of the largest listed case; drawn cases stay below them.
LARGEST = 512 * MIB


# ---------------------------------------------------------------- the cases
def _case(name, kind, B, H, Hkv, d, n, fmt, group, order, bt, splits=1, warps=4, unroll=2, layers=1,
          entry="launch", shortest=0, spread="uniform", longest_first=False, lens_seed=0):
    return {"name": name, "kind": kind, "B": B, "H": H, "Hkv": Hkv, "d": d, "n": n, "fmt": fmt, "group": group,
            "order": order, "bt": bt, "splits": splits, "warps": warps, "unroll": unroll, "layers": layers,
            "entry": entry, "shortest": shortest, "spread": spread, "longest_first": longest_first,
            "lens_seed": lens_seed}


def listed():
    return [
        # the first tokens of a chat: one short sequence, one layer, called
        # from Python; latency and the number of launches are all there is
        _case("short_int8", "decode", 1, 32, 8, 128, 1003, "int8", 64, "hm", 0, splits=8),
        # a small server's whole step, append and attention, over eight layers
        # of a paged pool
        _case("step_b4_paged_int8", "step", 4, 32, 8, 128, 2048, "int8", 64, "tm", 16, splits=4, layers=8,
              shortest=300, lens_seed=3),
        # the reference's plumbing shape (32 heads without grouping, 4096
        # tokens, binary16) at the split count that fills the chip
        _case("mha_4k_f16", "decode", 1, 32, 32, 128, 4096, "f16", 0, "hm", 0, splits=8, layers=4),
        # the headline decode shape, two launches per layer
        _case("gqa_32k_int8", "decode", 1, 32, 8, 128, 32768, "int8", 64, "hm", 0, splits=32, layers=4),
        # the same unquantized, one launch per layer
        _case("gqa_32k_f16_fused", "decode", 1, 32, 8, 128, 32768, "f16", 0, "hm", 0, splits=32, layers=2,
              entry="fused"),
        # a batch of eight in one shuffled pool of 16-token pages
        _case("b8_varlen_paged_int8", "varlen", 8, 32, 8, 128, 8192, "int8", 64, "tm", 16, splits=8, layers=4,
              shortest=2048, lens_seed=2),
        # long context in four bits
        _case("gqa_64k_int4", "decode", 1, 32, 8, 128, 65536, "int4", 32, "hm", 0, splits=32, warps=8, layers=4),
        # a large mixed batch, from short chats to whole books
        _case("b16_mixed_int8", "varlen", 16, 64, 8, 128, 131072, "int8", 64, "hm", 16, splits=16, layers=1,
              shortest=1024, spread="log", longest_first=True, lens_seed=9),
        # a small model's batch: head dimension 64, an odd length, token-major
        _case("b4_d64_16k_int4_tm", "decode", 4, 32, 8, 64, 16383, "int4", 32, "tm", 0, splits=8, layers=4),
        # many short sequences: the batch fills the chip, no split, no workspace
        _case("b32_2k_int8", "decode", 32, 32, 8, 128, 1999, "int8", 64, "hm", 0, splits=1, layers=2),
        # a long prompt's rows into a contiguous cache
        _case("prefill_32k_int8", "prefill", 1, 32, 8, 128, 32768, "int8", 64, "hm", 0),
        # a batch of prompts of odd length into a paged pool, four bits
        _case("prefill_b4_paged_int4", "prefill", 4, 32, 8, 128, 4093, "int4", 32, "tm", 16),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "varlen", "varlen", "step", "prefill"])
    d = rng.choice([128, 128, 64])
    H, Hkv = rng.choice([(32, 8), (32, 8), (64, 8), (32, 32), (32, 16), (16, 4)])
    fmt = rng.choice(["f16", "int8", "int8", "int4"])
    group = 0 if fmt == "f16" else rng.choice([32, 64]) if d == 64 else rng.choice([32, 64, 128])
    order = rng.choice(["hm", "tm"])
    bt = rng.choice([0, 16, 16, 64])
    layers = rng.choice([1, 2, 4, 8]) if kind == "step" else rng.choice([1, 2, 4])
    if kind == "prefill":
        layers = 1
    token = 2 * Hkv * _row_bytes(fmt, group, d)  # cache bytes of a token of one layer
    if kind == "prefill":
        token += 2 * Hkv * d * 4
    most = min(131072, LARGEST // (token * layers))
    if kind == "decode":
        n = _log_int(rng, 200, most)
        B = min(rng.choice([1, 1, 2, 4, 8, 32]), max(1, most // n))
    elif kind == "prefill":
        n = _log_int(rng, 100, min(32768, most))
        B = min(rng.choice([1, 1, 2, 4]), max(1, most // n))
    else:
        B = rng.choice([2, 4, 8, 16])
        n = _log_int(rng, 300, min(65536 if kind == "varlen" else 8192, most // B))
    # the split count that gives each of 256 compute units a workgroup (two
    # for unequal lengths), with at least 128 tokens in a split
    fill = (256 if kind == "decode" else 512) / (B * Hkv)
    splits = max(1, min(64, int(round(fill)), n // 128))
    entry = "launch"
    if kind == "decode" and splits > 1:
        entry = rng.choice(["launch", "launch", "fused"])
    elif kind == "varlen" and splits > 1:
        entry = rng.choice(["launch", "launch", "fused", "persistent"])
    spread = rng.choice(["uniform", "log"])
    c = _case("", kind, B, H, Hkv, d, n, fmt, group, order, bt, splits=splits, warps=rng.choice([4, 4, 8]),
              unroll=2 if entry == "persistent" else rng.choice([2, 2, 2, 4]), layers=layers, entry=entry,
              shortest=max(1, n // rng.choice([4, 32])), spread=spread,
              longest_first=kind == "varlen" and spread == "log", lens_seed=rng.randrange(1 << 30))
    del c["name"]
    return c


# ------------------------------------------------------- shapes, from a case
def _row_bytes(fmt, group, d):
    return d * {"f16": 16, "int8": 8, "int4": 4}[fmt] // 8 + (d // group * 4 if group else 0)


def _lens(c):
    """Tokens of each sequence."""
    if c["kind"] not in ("varlen", "step"):
        return [c["n"]] * c["B"]
    rng = random.Random(c["lens_seed"])
    lo, hi = max(1, c["shortest"]), c["n"]
    if c["spread"] == "log":
        return [min(hi, _log_int(rng, lo, hi)) for _ in range(c["B"])]
    return [rng.randint(lo, hi) for _ in range(c["B"])]


def _sized(case):
    """The case with its sequences' lengths, n the longest of them."""
    lens = _lens(case)
    return {**case, "n": max(lens)}, lens


def work(case):
    c = case
    row = _row_bytes(c["fmt"], c["group"], c["d"])
    tokens = sum(_lens(c)) * c["Hkv"] * c["layers"]
    if c["kind"] == "prefill":
        return {"bytes": 2 * tokens * (4 * c["d"] + row), "flops": 0}
    q = 2 * c["B"] * c["H"] * c["d"] * c["layers"] * (4 if c["kind"] == "decode" else 2)
    new = 2 * c["B"] * c["Hkv"] * c["layers"] * (4 * c["d"] + row) if c["kind"] == "step" else 0
    return {"bytes": 2 * tokens * row + q + new, "flops": 4 * tokens * c["H"] // c["Hkv"] * c["d"]}


def tolerance(case):
    c = case
    if c["kind"] == "prefill":
        return "exact"
    if c["kind"] != "decode":
        return {"rel": 1e-3, "max": 5e-3}  # 2.4e-4 from exact(): the output's own rounding to binary16
    # four times the measured distance from exact(): 1.3e-5 for int4 (few
    # codes, large scales), 1.3e-6 for int8, 6e-7 for unquantized rows
    return {"rel": {"int4": 5e-5, "int8": 5e-6, "f16": 2.5e-6}[c["fmt"]]}


# ------------------------------------------------------------------- inputs
def _rng(seed, *more):
    g = torch.Generator(device="cuda")
    s = int(seed)
    for m in more:
        s = (s * 1000003 + m + 12345) % (1 << 62)
    g.manual_seed(s)
    return g


def _rows(g, B, Hkv, n, d):
    """K or V rows as they come out of a projection: about N(0, 1), with one
    channel in a hundred eight times larger."""
    x = torch.randn((B, Hkv, n, d), generator=g, device="cuda")
    big = torch.rand((B, Hkv, 1, d), generator=g, device="cuda") < 0.01
    return x.mul_(torch.where(big, 8.0, 1.0))


def _quantize(x, fmt, group):
    """(payload rows as bytes [..., row], scale and zero [..., d/group, 2])."""
    if fmt == "f16":
        return x.half().view(torch.uint8), None
    levels = 255.0 if fmt == "int8" else 15.0
    y = x.view(*x.shape[:-1], x.shape[-1] // group, group)
    lo, hi = y.amin(-1), y.amax(-1)
    zero = lo.half()
    scale = ((hi - lo) / levels).half()
    scale = torch.where(scale > 0, scale, torch.ones_like(scale))
    code = ((y - zero.float().unsqueeze(-1)) / scale.float().unsqueeze(-1)).round_().clamp_(0, levels)
    code = code.to(torch.uint8).view(x.shape)
    if fmt == "int4":
        code = code[..., 0::2] | (code[..., 1::2] << 4)
    return code.contiguous(), torch.stack((scale, zero), -1)


def _dequantize(data, meta, fmt, group, d):
    if fmt == "f16":
        return data.view(torch.float16).double()
    if fmt == "int4":
        data = torch.stack((data & 15, data >> 4), -1).flatten(-2)
    y = data.view(*data.shape[:-1], d // group, group).double()
    m = meta.double()
    return (y * m[..., 0:1] + m[..., 1:2]).flatten(-2)


def _page_table(c, g):
    """[B][pages of the longest sequence] page ids, a shuffled pool's."""
    mb = -(-c["n"] // c["bt"])
    return torch.randperm(c["B"] * mb, generator=g, device="cuda").to(torch.int32).view(c["B"], mb)


def _place(c, rows, table):
    """Logical rows [B][Hkv][n][...] in the layout's order, as one flat buffer."""
    if not c["bt"]:
        return (rows if c["order"] == "hm" else rows.transpose(1, 2)).contiguous().flatten()
    B, Hkv, n = rows.shape[:3]
    mb = table.shape[1]
    tail = rows.shape[3:]
    full = rows.new_zeros((B, Hkv, mb * c["bt"], *tail))
    full[:, :, :n] = rows
    pages = full.view(B, Hkv, mb, c["bt"], *tail).transpose(1, 2)  # [B][mb][Hkv][bt]
    if c["order"] == "tm":
        pages = pages.transpose(2, 3)
    pool = torch.empty((B * mb, *pages.shape[2:]), dtype=rows.dtype, device=rows.device)
    pool[table.flatten().long()] = pages.reshape(B * mb, *pages.shape[2:])
    return pool.flatten()


def _words(meta):
    """(scale, zero) pairs as the 32-bit words the library reads."""
    return None if meta is None else meta.flatten().view(torch.int32)


def _layer(c, seed, i):
    """The values of layer i: query, K and V rows, and a step's new rows."""
    g = _rng(seed, i)
    q = torch.randn((c["B"], c["H"], c["d"]), generator=g, device="cuda")
    K = _rows(g, c["B"], c["Hkv"], c["n"], c["d"])
    V = _rows(g, c["B"], c["Hkv"], c["n"], c["d"])
    return q, K, V


def _last(x, lens):
    """Row lens[b] - 1 of each sequence: [B][Hkv][d]."""
    return torch.stack([x[b, :, n - 1] for b, n in enumerate(lens)]).contiguous()


def prepare(case, seed):
    c, lens = _sized(case)
    dev = torch.device("cuda:0")
    fmt = R.FMT_BY_NAME[c["fmt"]]
    order = R.ORD_HEAD if c["order"] == "hm" else R.ORD_TOKEN
    B, H, Hkv, d, n, S = c["B"], c["H"], c["Hkv"], c["d"], c["n"], c["splits"]
    table = _page_table(c, _rng(seed, 999)) if c["bt"] else None
    mb = table.shape[1] if c["bt"] else 0
    st = {"case": c, "fmt": fmt, "order": order, "table": table, "mb": mb, "layers": []}
    if c["kind"] == "prefill":
        rows = B * mb * Hkv * c["bt"] if c["bt"] else B * Hkv * n
        _, K, V = _layer(c, seed, 0)
        st["x"] = (K, V)
        st["to"] = [(torch.zeros(rows * R.row_bytes(fmt, d), dtype=torch.uint8, device=dev),
                     torch.zeros(rows * (d // c["group"]), dtype=torch.int32, device=dev) if c["group"] else None)
                    for _ in range(2)]
        return st
    half = c["kind"] != "decode"
    part_o = torch.empty((B, H, S, d), device=dev) if S > 1 else None
    part_ml = torch.empty((B, H, S, 2), device=dev) if S > 1 else None
    st["vid"] = R.variant_id(fmt, order, c["bt"] > 0, H // Hkv, c["unroll"], d)
    st["lens"] = torch.tensor(lens, dtype=torch.int32, device=dev) if half else None
    st["flags"] = R.VARLEN_LONGEST_FIRST if c["longest_first"] else 0
    st["counters"] = R.fused_counters(B, Hkv if H > Hkv else H, dev) if c["entry"] != "launch" else None
    st["queue"] = R.persistent_queue(dev) if c["entry"] == "persistent" else None
    st["positions"] = st["lens"] - 1 if half else None
    for i in range(c["layers"]):
        q, K, V = _layer(c, seed, i)
        L = {"q": q.half() if half else q, "part": (part_o, part_ml)}
        L["out"] = torch.zeros((B, H, d), dtype=torch.float16 if half else torch.float32, device=dev)
        if c["kind"] == "step":
            L["new"] = (_last(K, lens), _last(V, lens))
            for b, m in enumerate(lens):  # not yet in the cache
                K[b, :, m - 1:] = 0
                V[b, :, m - 1:] = 0
        L["cache"] = []
        for x in (K, V):
            data, meta = _quantize(x, c["fmt"], c["group"])
            L["cache"].append((_place(c, data, table), _words(_place(c, meta, table)) if meta is not None else None))
        (k, km), (v, vm) = L["cache"]
        if half:  # Args still names an fp32 query and output
            L["q32"], L["out32"] = q, torch.zeros((B, H, d), device=dev)
        L["args"] = R.make_args(q, k, v, km, vm, table, L["out32"] if half else L["out"], part_o, part_ml, B, H, Hkv,
                                n, S, c["warps"], group=c["group"], block_tokens=c["bt"], max_blocks=mb, D=d)
        st["layers"].append(L)
        del K, V, q
    if c["kind"] == "step":
        _step(st)  # sets the library up, as a program's first eager step does
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"]):
            _step(st)
    return st


# -------------------------------------------------------------------- a pass
def _attend(st, L):
    entry = st["case"]["entry"]
    if st["lens"] is None:
        if entry == "fused":
            R.launch_fused(st["vid"], L["args"], st["counters"])
        else:
            R.launch(st["vid"], L["args"])
        return
    more = (st["lens"], L["q"], L["out"])
    if entry == "fused":
        R.launch_fused(st["vid"], L["args"], st["counters"], varlen=more, flags=st["flags"])
    elif entry == "persistent":
        R.launch_persistent(st["vid"], L["args"], st["queue"], counters=st["counters"], varlen=more,
                            flags=st["flags"])
    else:
        R.launch_varlen(st["vid"], L["args"], *more, flags=st["flags"])


def _step(st):
    c = st["case"]
    for L in st["layers"]:
        for x, (data, meta) in zip(L["new"], L["cache"]):
            R.append_tokens(st["fmt"], c["group"], c["d"], x, c["B"], c["Hkv"], c["n"], st["positions"], st["order"],
                            c["bt"], st["table"], st["mb"], data, meta)
        _attend(st, L)


def run(state):
    st = state
    c = st["case"]
    if c["kind"] == "prefill":
        for x, (data, meta) in zip(st["x"], st["to"]):
            R.quantize_place(st["fmt"], c["group"], c["d"], x, c["B"], c["Hkv"], c["n"], st["order"], c["bt"],
                             st["table"], st["mb"], data, meta)
        return st["to"]
    if c["kind"] == "step":
        st["graph"].replay()
        return [{"out": L["out"], "cache": L["cache"]} for L in st["layers"]]
    for L in st["layers"]:
        _attend(st, L)
    return [L["out"] for L in st["layers"]]


# ---------------------------------------------------------- in 64 bits, plain
def exact(case, seed):
    c = case
    if c["kind"] == "prefill":
        return None  # bytes, compared as they are
    c, lens = _sized(c)
    H, Hkv, d = c["H"], c["Hkv"], c["d"]
    outs = []
    for i in range(c["layers"]):
        q, K, V = _layer(c, seed, i)
        if c["kind"] != "decode":
            q = q.half()
        q = q.double().view(c["B"], Hkv, H // Hkv, d)
        out = torch.zeros((c["B"], Hkv, H // Hkv, d), dtype=torch.float64, device="cuda")
        for b, m in enumerate(lens):
            k = _dequantize(*_quantize(K[b, :, :m].contiguous(), c["fmt"], c["group"]), c["fmt"], c["group"], d)
            v = _dequantize(*_quantize(V[b, :, :m].contiguous(), c["fmt"], c["group"]), c["fmt"], c["group"], d)
            for h in range(H // Hkv):
                s = (k * q[b, :, h, None, :]).sum(-1) / math.sqrt(d)
                out[b, :, h] = (torch.softmax(s, -1).unsqueeze(-1) * v).sum(-2)
            del k, v
        out = out.view(c["B"], H, d)
        outs.append({"out": out, "cache": [(None, None), (None, None)]} if c["kind"] == "step" else out)
        del K, V
    return outs
