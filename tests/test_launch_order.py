"""What kernels on the second stream may read (source check, no GPU)."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "ie-solver_amd", "csrc")


def _kernels(name):
    src = open(os.path.join(CSRC, name)).read()
    for m in re.finditer(r"__global__[^{]*?\b(k_\w+)\s*\(", src):
        body = src[m.end():]
        end = re.search(r"^}", body, re.M).start()
        yield m.group(1), body[:end]


def test_decouple_goes_by_its_levels_verdict():
    """A level's decouple runs beside the scans of the levels above, which
    write the error word: a workgroup whose waves read it before and after
    such a write would run on with LDS that its first wave never filled."""
    seen = []
    for f in ("rs_decouple.hip", "rs_sweep.hip"):
        for name, body in _kernels(f):
            if name.startswith("k_decouple"):
                seen.append(name)
                assert "pools_ok" not in body and "s.err[" not in body, name
                assert "s.halt[level]" in body, name
    assert sorted(seen) == ["k_decouple", "k_decouple_small", "k_decouple_sweep"]
