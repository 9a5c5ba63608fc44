"""LDS reads that the bf16 attention writes in assembly, in the compiled code: the compiler does not know that their results are still on their way, so
none may be in flight where it is free to move registers about, which is where control flow joins or branches."""
import os
import re
import subprocess

from conftest import load_package

load_package()
from sd3_c_amd import build  # noqa: E402


def _functions(text):
    name, body = None, []
    for line in text.splitlines():
        start = re.match(r"(_Z\S*):", line)
        if start:
            name, body = start.group(1), []
        elif name and line.startswith(".Lfunc_end"):
            yield name, body
            name = None
        elif name:
            body.append(line)


def _in_flight(body):
    """Most reads of this kind in flight on each edge of the control flow: {(block, next block): reads}, blocks in the order of the code."""
    blocks, index, in_asm = [[]], {}, False
    for line in body:
        label, s = re.match(r"(\.LBB\S+):", line), line.strip()
        if label:
            blocks.append([])
            index[label.group(1)] = len(blocks) - 1
        elif s.startswith(";;#ASM"):
            in_asm = s == ";;#ASMSTART"
        elif s and s[0] not in ";.":
            blocks[-1].append((s.split(";")[0].split(), in_asm))
            if re.match(r"s_(c?branch|endpgm)", s):
                blocks.append([])
    entry, edges, work = {0: 0}, {}, [0]
    while work:
        i = work.pop()
        n, to = entry[i], [i + 1]
        for words, written in blocks[i]:
            op = words[0]
            if op.startswith("ds_read") and written:
                n = min(n + 1, 64)
            elif op.startswith(("ds_", "s_load")) and n:  # (counted by the same counter)
                n = min(n + 1, 64)
            elif op == "s_waitcnt":
                left = re.search(r"lgkmcnt\((\d+)\)", " ".join(words))
                n = min(n, int(left.group(1))) if left else n
            elif op.startswith("s_cbranch"):
                to = [i + 1, index[words[1]]]
            elif op == "s_branch":
                to = [index[words[1]]]
            elif op == "s_endpgm":
                to = []
        for j in to:
            if j < len(blocks):
                edges[i, j] = n
                if entry.get(j, -1) < n:
                    entry[j] = n
                    work.append(j)
    return edges


def test_no_read_is_in_flight_from_one_key_tile_to_the_next(tmp_path):
    out = tmp_path / "attention.s"
    src = "attention_bf16.hip"
    subprocess.run(["hipcc"] + build.FLAGS + build.EXTRA_FLAGS[src] + ["--offload-device-only", "-S", os.path.join(build.CSRC, src), "-o", str(out)],
                   check=True, capture_output=True)
    seen = {}
    for name, body in _functions(out.read_text()):
        kind = re.search(r"flash_attn_bf16_kernelILb(\d)ELi(\d)ELi(\d)", name)
        if kind:
            seen[kind.groups()] = _in_flight(body)
    assert sorted(seen) == [("0", "1", "4"), ("0", "1", "8"), ("0", "2", "4"), ("1", "2", "4")]
    for kind, edges in seen.items():
        assert not [e for e, n in edges.items() if n and e[1] <= e[0]], kind  # loops
        if kind[1] == "1":  # wavefronts of 32 queries: not a single branch
            assert not [e for e, n in edges.items() if n], kind
