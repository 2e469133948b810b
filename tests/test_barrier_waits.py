"""The barriers of the dense attention kernels in the assembly that the package's
own sources give: gfx950 makes no barrier wait for LDS stores by itself, and the
compiler adds no wait to the raw barrier builtin, so an LDS store that other
waves read needs its own wait before the barrier."""
import os
import re
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "selective-attention_amd"))


def device_assembly(name, out):
    import build
    subprocess.run([build.HIPCC, *build.COMMON_FLAGS, "-w", "--cuda-device-only", "-S",
                    os.path.join(build.CSRC, name), "-o", str(out)], check=True)
    return out.read_text().splitlines()


def unordered_stores(lines):
    """(kernel, line) of LDS stores from which some path reaches a barrier without
    an lgkmcnt(0) wait: a walk over the labels and branches of each kernel."""
    kernels, cur = {}, None
    for no, line in enumerate(lines):
        m = re.match(r"(_Z\w*kernel\w*):", line)
        if m:
            cur = kernels.setdefault(m.group(1), [])
        if cur is not None:
            cur.append((no, line.split(";")[0].strip()))
        if line.startswith("\t.section") or ".end_amdhsa_kernel" in line:
            cur = None
    bad = []
    for name, body in kernels.items():
        labels = {t[:-1]: i for i, (_, t) in enumerate(body) if re.match(r"\.\w+:$", t)}
        for i, (no, text) in enumerate(body):
            if not text.startswith("ds_write"):
                continue
            todo, seen = [i + 1], set()
            while todo:
                j = todo.pop()
                if j in seen or j >= len(body):
                    continue
                seen.add(j)
                t = body[j][1]
                if t.startswith("s_waitcnt") and "lgkmcnt(0)" in t or t.startswith("s_endpgm"):
                    continue
                if t.startswith("s_barrier"):
                    bad.append((name, no + 1))
                    break
                b = re.match(r"s_c?branch\w*\s+(\.\w+)", t)
                if b:
                    todo.append(labels[b.group(1)])
                if not t.startswith("s_branch"):
                    todo.append(j + 1)
    return sorted(set(bad)), len(kernels)


def test_dense_attention_orders_its_lds_stores(tmp_path):
    bad, kernels = unordered_stores(device_assembly("attention_dense.hip", tmp_path / "dense.s"))
    assert kernels >= 10
    assert not bad


def test_walk_finds_a_missing_wait():
    body = ["_Zkernel:", "\tds_write_b32 v0, v1", "\ts_waitcnt vmcnt(0)", "\ts_cbranch_scc1 .LBB0_2",
            "\ts_waitcnt lgkmcnt(0)", "\ts_barrier", ".LBB0_2:", "\ts_endpgm"]
    assert not unordered_stores(body)[0]
    del body[4]
    assert unordered_stores(body)[0] == [("_Zkernel", 2)]
