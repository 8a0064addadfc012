"""The barriers of the prompt kernels, in the code that the compiler makes: a wave's LDS accesses have returned when it meets
one, since behind it other waves copy over the stages that this wave has read.  Compiles for gfx950; no GPU."""
import os
import re
import shutil
import subprocess

import pytest


def _kernels(path):
    """(name, instructions and labels) of every kernel of an assembly file."""
    found = []
    for line in open(path):
        t = line.split(";")[0].strip()
        if re.match(r"_Z\w+:$", t):
            found.append((t[:-1], []))
        elif found and t and (not t.startswith(".") or t.endswith(":")):
            found[-1][1].append(t)
    return [(name, code) for name, code in found if "s_barrier" in code]


def _under_way_at_barriers(code):
    """For every barrier the largest number of LDS accesses that can be under way there, over all ways to it."""
    label = {t[:-1]: i for i, t in enumerate(code) if t.endswith(":")}
    most, work, at_barrier = {0: 0}, [0], {}
    while work:
        i = work.pop()
        n, t, after = most[i], code[i], [i + 1]
        wait = re.match(r"s_waitcnt\b.*\blgkmcnt\((\d+)\)", t)
        branch = re.match(r"s_(c?)branch\w*\s+(\S+)", t)
        if t.startswith("ds_"):
            n = min(n + 1, 64)
        elif wait:
            n = min(n, int(wait.group(1)))
        elif t == "s_barrier":
            at_barrier[i] = max(at_barrier.get(i, 0), n)
        elif branch:
            after = [label[branch.group(2)]] + (after if branch.group(1) else [])
        elif t.startswith("s_endpgm"):
            after = []
        for j in after:
            if j < len(code) and most.get(j, -1) < n:
                most[j] = n
                work.append(j)
    return at_barrier


# "late": the first step's products, which keep the compiler's own wait in front of the barrier today, are left out of the copy
# that is compiled, and what was read is used behind the barrier
@pytest.mark.parametrize("products", ["as they are", "late"])
def test_lds_accesses_have_returned_at_every_barrier(tmp_path, products):
    from moa_amd import build
    csrc = tmp_path / "moa_amd" / "csrc"
    shutil.copytree(build.CSRC, csrc, ignore=shutil.ignore_patterns("build"))
    shutil.copytree(os.path.join(build.HERE, "..", "include"), tmp_path / "include")
    source = csrc / "moa_prefill.hip"
    if products == "late":
        text = source.read_text()
        first, use = "tile_qk(", "st[nt] = T::mfma(kf[s], qf[s], st[nt]);"
        at = text.index(use, text.index(first))
        later = "for (int e = 0; e < 4; ++e) st[nt][4 * (s & 3) + e] = __builtin_bit_cast(f32x4, kf[s])[e];"
        source.write_text(text[:at] + later + text[at + len(use):])
    out = str(tmp_path / "prefill.s")
    r = subprocess.run([build._hipcc(), *build.HIPCC_FLAGS, "-S", "--cuda-device-only", str(source), "-o", out],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    kernels = _kernels(out)
    assert len(kernels) == 8   # two kernels, two types, two head sizes
    for name, code in kernels:
        barriers = _under_way_at_barriers(code)
        assert len(barriers) >= 3 and not any(barriers.values()), (name, sorted(barriers.values()))
