"""Register, scratch and LDS use of every gfx950 split kernel, for the CDNA
cost model's occupancy terms (the reference reads the same facts out of its
CUDA binary with tools/dump_resources.py; here hipcc's resource-usage remarks
report them for the code objects this repository builds).

    python kvforge_amd/tools/dump_resources.py [--jobs 8] [--out machines/resources_gfx950.csv]

Compiles every explicit-instantiation source under kvforge_amd/csrc/gen with
-Rpass-analysis=kernel-resource-usage (objects go to a temporary directory)
and writes one CSV row per decode_partial instantiation:

    fmt,d,group,g,u,ord,paged,waves,vgpr,agpr,sgpr,scratch,occupancy,valu,mfma,lds,salu

fmt/ord use the kernels' numbering (f16 0, int8 1, int4 2; head-major 0,
token-major 1); `group` is the quantisation group the kernel is built for (the
head dimension for f16), `g` the GQA pack, `u` the unroll knob, `waves` the
wavefronts per workgroup; `occupancy` is the compiler's waves per SIMD.

valu, mfma, lds, salu: instructions that every 32-token tile of the kernel's
main loop runs, counted in the gfx950 assembly of the same compile (-S): the
loop is the one holding the most MFMAs in its own blocks. Of its blocks only
those count that every iteration passes through: the masking of a tile that
reaches outside the split's range, the rescaling when a score passes the
running max, and the next page ids of paged rows are behind wave-uniform
branches that a tile rarely takes. The blocks hold the tile's compute once per
unrolled step, so the counts are divided by (MFMAs in the loop / MFMAs per
tile). MFMAs per
tile follow from the kernel's column geometry: COLS = g x (d / group) query
columns (g for f16), two passes when COLS > 16, hi and lo in one MFMA when
COLS <= 8, and per pass and binary16 half 2 x d/32 QK steps (of int8:32 at d
128 and 8 heads only the half that meets the pass's groups) plus d/16 PV
steps. `lds` counts ds_* instructions (the cross-row shuffles), `salu` s_*.
"""
import argparse
import concurrent.futures as cf
import glob
import os
import re
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.dirname(HERE)
ROOT = os.path.dirname(PKG)
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = ["-std=c++17", "-O3", "--offload-arch=gfx950", "-fPIC", "-Xclang", "-target-feature",
         "-Xclang", "-packed-fp32-ops", "-mllvm", "-amdgpu-mfma-vgpr-form",
         "-mllvm", "-amdgpu-atomic-optimizer-strategy=None", "-mllvm", "-amdgpu-kernarg-preload-count=14",
         "-I" + os.path.join(ROOT, "include"),
         "-I" + os.path.join(PKG, "csrc"), "-Rpass-analysis=kernel-resource-usage"]
NAME = re.compile(r"decode_partialILi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)ELb(\d)ELi(\d+)E")
REMARK = re.compile(r"remark: (.*?) \[-Rpass-analysis")


LABEL = re.compile(r"^(_Z\w+):")
BLOCK = re.compile(r"^(\.LBB\d+_\d+):(.*)")
BB = re.compile(r"^; (%bb\.\d+):(.*)")
IN_LOOP = re.compile(r"Header=BB(\d+_\d+) Depth=\d+")
BRANCH = re.compile(r"(s_cbranch_\w+|s_branch)\s+(\.LBB\d+_\d+)")


def mfma_per_tile(fmt, d, group, g):
    cols = g * (d // group if fmt != 0 else 1)
    passes = 2 if cols > 16 else 1
    nq = 1 if cols <= 8 else 2
    # int8:32, d 128, 8 heads: a QK step holds dims of one pass's groups only
    qk_passes = 1 if (fmt, d, group, g) == (1, 128, 32, 8) else passes
    return (2 * (d // 32) * qk_passes + d // 16 * passes) * nq


def every_iteration(header, body, order, targets, falls):
    """The blocks of `body` that lie on every path from `header` back to it (all
    of them, if no branch leads back). `order` is the function's blocks as laid
    out, targets[b] where b's branches go, falls[b] whether b runs on into the
    next block."""
    body = set(body)
    after = dict(zip(order, order[1:]))

    def comes_round(without):
        seen, todo = set(), [header]
        while todo:
            b = todo.pop()
            if b in seen or b == without:
                continue
            seen.add(b)
            for t in targets[b] + ([after[b]] if falls[b] and b in after else []):
                if t == header:
                    return True
                if t in body:
                    todo.append(t)
        return False

    if not comes_round(None):
        return body
    return {b for b in body if b == header or not comes_round(b)}


def loop_mix(lines):
    """Instruction mix of the loop with the most MFMAs in its own blocks (the
    fewest vector instructions breaking a tie), over the blocks that every
    iteration runs. A
    block (a `.LBB` label or an unlabelled `; %bb.N:` fall-through) counts for
    the innermost loop holding it, as the assembler's comments on the block's
    first lines name it ("Loop Header: Depth=d" for a header, "in Loop:
    Header=BBx_y" for the others)."""
    blocks, notes, order, targets = {}, {}, [], {}
    cur, head = None, False
    for line in lines:
        m = BLOCK.match(line) or BB.match(line)
        if m:
            cur = m.group(1)
            blocks[cur], notes[cur], targets[cur], head = [], m.group(2), [], True
            order.append(cur)
            continue
        t = line.strip()
        if cur is None or not t:
            continue
        if t[0] == ";":
            if head:
                notes[cur] += " " + t
            continue
        head = False
        if t[0] != ".":
            blocks[cur].append(t.split()[0])
            if (m := BRANCH.match(t)):
                targets[cur].append(m.group(2))
    falls = {b: not (ops and ops[-1] in ("s_branch", "s_endpgm", "s_setpc_b64")) for b, ops in blocks.items()}
    loops = {}
    for b in order:
        if "Loop Header: Depth=" in notes[b]:
            owner = "BB" + b[len(".LBB"):] if b.startswith(".LBB") else b
        else:
            h = IN_LOOP.search(notes[b])
            owner = "BB" + h.group(1) if h else None
        if owner:
            loops.setdefault(owner, []).append(b)
    if not loops:
        return None

    def ops_of(body):
        return [x for b in body for x in blocks[b]]

    body = max(loops.values(), key=lambda bs: (sum(x.startswith("v_mfma") for x in ops_of(bs)),
                                               -sum(x.startswith("v_") for x in ops_of(bs))))
    ops = ops_of(every_iteration(body[0], body, order, targets, falls))
    mix = {"mfma": 0, "valu": 0, "lds": 0, "salu": 0}
    for op in ops:
        if op.startswith("v_mfma"):
            mix["mfma"] += 1
        elif op.startswith("v_"):
            mix["valu"] += 1
        elif op.startswith("ds_"):
            mix["lds"] += 1
        elif op.startswith("s_"):
            mix["salu"] += 1
    return mix


def kernel_mixes(asm):
    """{mangled decode_partial name: loop mix} of one assembly file."""
    out, name, lines = {}, None, []
    for line in asm.splitlines():
        if name is None:
            m = LABEL.match(line)
            if m and NAME.search(m.group(1)):
                name, lines = m.group(1), []
        elif line.startswith(".Lfunc_end"):
            out[name] = loop_mix(lines)
            name = None
        else:
            lines.append(line)
    return out


def remarks(src, tmp):
    asm = os.path.join(tmp, os.path.basename(src) + ".s")
    p = subprocess.run([HIPCC, *FLAGS, "--cuda-device-only", "-S", src, "-o", asm], capture_output=True,
                       text=True)
    if p.returncode != 0:
        raise RuntimeError(f"{src}: {p.stderr[-2000:]}")
    with open(asm) as fh:
        mixes = kernel_mixes(fh.read())
    rows, cur = [], None
    for line in p.stderr.splitlines():
        m = REMARK.search(line)
        if not m:
            continue
        text = m.group(1)
        if text.startswith("Function Name:"):
            cur = {"name": text.split(":", 1)[1].strip()}
            rows.append(cur)
        elif cur is not None and ":" in text:
            k, v = text.split(":", 1)
            cur[k.strip()] = v.strip()
    for r in rows:
        r["mix"] = mixes.get(r["name"])
    return rows


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=8)
    ap.add_argument("--out", default=os.path.join(ROOT, "machines", "resources_gfx950.csv"))
    args = ap.parse_args()
    srcs = sorted(glob.glob(os.path.join(PKG, "csrc", "gen", "kvf_inst_*.hip")))
    if not srcs:
        sys.exit("no instantiation sources under kvforge_amd/csrc/gen")
    table = {}
    with tempfile.TemporaryDirectory() as tmp, cf.ThreadPoolExecutor(args.jobs) as pool:
        for rows in pool.map(lambda s: remarks(s, tmp), srcs):
            for r in rows:
                m = NAME.search(r["name"])
                if not m:
                    continue
                fmt, d, group, g, u, ord_, paged, waves = (int(x) for x in m.groups())
                mix = r["mix"]
                if not mix or mix["mfma"] == 0:
                    sys.exit(f"no MFMA loop found in {r['name']}")
                copies = mix["mfma"] / mfma_per_tile(fmt, d, group, g)
                if copies != int(copies):
                    sys.exit(f"{r['name']}: {mix['mfma']} loop MFMAs is no whole number of tiles")
                per_tile = tuple(round(mix[k] / copies, 1) for k in ("valu", "mfma", "lds", "salu"))
                table[(fmt, d, group, g, u, ord_, paged, waves)] = (
                    int(r["VGPRs"]), int(r["AGPRs"]), int(r["TotalSGPRs"]),
                    int(r["ScratchSize [bytes/lane]"]), int(r["Occupancy [waves/SIMD]"]), *per_tile)
    with open(args.out, "w") as f:
        f.write("fmt,d,group,g,u,ord,paged,waves,vgpr,agpr,sgpr,scratch,occupancy,valu,mfma,lds,salu\n")
        for k in sorted(table):
            f.write(",".join(str(x) for x in (*k, *table[k])) + "\n")
    print(f"wrote {len(table)} kernels to {args.out}")


if __name__ == "__main__":
    main()
