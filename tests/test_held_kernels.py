"""A kernel that returns at once where an earlier check failed, and that may count a failed check itself, decides
so for a whole block: read by every thread, the count could change between two waves of a block whose other
waves then go on without what the first one sets up (no GPU needed: the sources)."""
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = open(os.path.join(ROOT, "manifolddmc_amd", "csrc", "mdmc_pipeline.hip")).read()


def functions():
    """name -> (is a kernel, body) of the device functions."""
    out = {}
    for m in re.finditer(r"^(?:template <[^\n]*>\n)?(__global__|__device__)[^;{]*?\b(\w+)\(", SOURCE, re.M):
        at = SOURCE.find("{", m.end())
        depth, end = 1, at + 1
        while depth:
            depth += {"{": 1, "}": -1}.get(SOURCE[end], 0)
            end += 1
        name = m.group(2)
        if m.group(1) == "__global__":
            head = SOURCE[m.start():at]
            name = re.findall(r"\b(k[A-Z]\w*)\(", head)[0]
        out[name] = (m.group(1) == "__global__", SOURCE[at:end])
    return out


def reaches(name, target, fns, seen=()):
    body = fns[name][1]
    if re.search(target, body):
        return True
    called = set(re.findall(r"\b(\w+)\(", body)) & set(fns)
    return any(reaches(c, target, fns, seen + (name,)) for c in called if c not in seen and c != name)


def test_blocks_decide_together():
    fns = functions()
    kernels = [n for n, (kernel, _) in fns.items() if kernel]
    assert len(kernels) > 40 and "kDropVertices" in kernels and "kCompactQuads" in kernels
    held = [n for n in kernels if re.search(r"\b(chainHeld|notYet)\(", fns[n][1])]
    counting = [n for n in held if reaches(n, r"\binvalid\(", fns) and reaches(n, r"__syncthreads", fns)]
    assert "kDropVertices" in counting
    for n in counting:
        for line in fns[n][1].splitlines():
            if re.search(r"\b(chainHeld|notYet)\(", line):
                assert "__syncthreads_or(" in line, (n, line.strip())
