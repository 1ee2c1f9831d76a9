"""Every kernel launcher that the native headers declare has a caller in the
C ABI: a path that nothing runs is not kept right by any other test."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "polymer_dns_amd", "csrc")


def read(*ext):
    return "\n".join(open(os.path.join(CSRC, f)).read() for f in sorted(os.listdir(CSRC)) if f.endswith(ext))


def test_every_declared_launcher_is_called():
    declared = set(re.findall(r"\b(launch_\w+)\s*\(", open(os.path.join(CSRC, "kmm_kernels.h")).read()))
    called = set(re.findall(r"\b(launch_\w+)\s*\(", read(".cpp")))
    assert len(declared) > 20
    assert sorted(declared - called) == []
