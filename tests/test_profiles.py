"""The committed profiler summaries are of the present kernels: the names they
list are the ones bench.py looks up."""
import os
import re
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)


def _kernels(name):
    text = open(os.path.join(ROOT, "profiles", name)).read()
    return set(re.findall(r"\| `(k_class[^`]*)` \|", text))


def test_kernel_names():
    import bench
    classes = [(a, b, c, d) for a in range(3) for b in range(a + 1) for c in range(3) for d in range(c + 1)
               if (a, b) >= (c, d)]
    assert len(classes) == 21
    for name in ("jk_c60_631gs_hbm_traffic.md", "jk_classes_c60_631gs_kernel_trace.md",
                 "jk_classes_c60_631gs_sq_counters.md"):
        have = _kernels(name)
        missing = [bench.kernel_name(lq) for lq in classes if bench.kernel_name(lq) not in have]
        assert not missing, (name, missing)


def test_traffic_of_the_dominant_kernel():
    import bench
    b, source = bench.profile_traffic(bench.kernel_name((2, 1, 1, 1)))  # (dp|pp)
    assert source and b > 1e9
