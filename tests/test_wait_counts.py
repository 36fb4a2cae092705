"""The counted waits of the expert streams (nn_amd/csrc/nnq_moe.hip) against the memory instructions that
the compiler leaves between them.  moe_stream_kernel copies its activation chunks to LDS some steps ahead
and waits for one with `vmcnt(N)`, N the instructions issued after it; a load that the compiler deletes
or moves makes N too large, and a wave then reads a chunk that has not landed.  Nothing on the GPU shows that
reliably, so the assembly of every instantiation is read here.  No GPU needed."""
import os
import re
import subprocess

import pytest

from nn_amd import build

SRC = os.path.join(build.CSRC, "nnq_moe.hip")


def problems(asm):
    """(instantiation, what) of every wait that counts more than can be in flight after its chunk's copies."""
    found, kernels = [], 0
    for m in re.finditer(r"^(\S*moe_stream_kernelILi(\d)ELb(\d)ELi(\d)ELb(\d)E\S*):(.*?)^\.Lfunc_end", asm, re.S | re.M):
        kernels += 1
        name, chunk = "moe_stream_kernel<%s, %s, %s, %s>" % m.group(2, 3, 4, 5), int(m.group(4))
        ahead = 1 if chunk == 3 else 2  # batches that may be in flight at a chunk's wait: ring depth - 2
        ops = []
        for line in m.group(6).splitlines():
            t = line.strip()
            if re.match(r"buffer_load_\w+ .*\blds\b", t):
                ops.append("copy")
            elif re.match(r"buffer_load_", t):
                ops.append("load")
            elif t.startswith("s_barrier"):
                ops.append("barrier")
            elif w := re.match(r"s_waitcnt.*vmcnt\((\d+)\)", t):
                ops.append(int(w.group(1)))
        # a step: its counted wait, the barrier, then the batch that it issues
        steps = [i for i in range(len(ops) - 1) if isinstance(ops[i], int) and ops[i] > 0 and ops[i + 1] == "barrier"]
        batches = []
        for i in steps:
            j = i + 2
            while j < len(ops) and ops[j] in ("copy", "load"):
                j += 1
            batches.append((ops[i], ops[i + 2:j].count("copy"), j - i - 2))
            if ops[i] > ahead * (j - i - 2):
                found.append((name, "waits for all but %d, its step issues %d" % (ops[i], j - i - 2)))
        if not batches:
            found.append((name, "no counted waits found"))
            continue
        # the prologue: ring depth - 1 batches of loads and copies between two barriers
        wait, copies, _ = max(batches)
        runs = re.findall(r"(?:[cl]){4,}", "".join("c" if o == "copy" else "l" if o == "load" else "." for o in ops))
        pro = [r for r in runs if r.count("c") == (ahead + 1) * copies and r.count("l")]
        if not pro:
            found.append((name, "no prologue found"))
        for r in pro:
            if "c" * copies and r.rfind("c", 0, len(r) - wait) < 0 or r[:len(r) - wait].count("c") < copies:
                found.append((name, "the prologue's order %s leaves the first chunk in flight" % r))
    return found, kernels


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="needs hipcc")
def test_expert_stream_waits_cover_their_copies(tmp_path):
    out = str(tmp_path / "moe.s")
    subprocess.run([build.HIPCC, f"--offload-arch={build.ARCH}", *build.COMMON, *build.DEVICE_FLAGS,
                    *build.EXTRA_FLAGS.get("nnq_moe.hip", []), "--cuda-device-only", "-S", SRC, "-o", out], check=True,
                   stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    found, kernels = problems(open(out).read())
    assert kernels == 8, kernels
    assert not found, found
