"""Models of one cluster set share the patch search on the CPU."""
import os
import subprocess

from cemc_amd.lattice import FCCSettings
from test_patches import _records

HERE = os.path.dirname(os.path.abspath(__file__))


def test_one_search_per_cluster_set(tmp_path):
    """Four sizes of one set and one of another take two searches; the covers
    are the search's own, from several threads, and a bounded number stays."""
    exe = str(tmp_path / "patch_covers_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", os.path.join(HERE, "patch_covers_check.cpp"), "-o", exe],
                   check=True)
    shells = {2: 4, 3: 2}
    sets = [FCCSettings(size, ["A", "B"], sh) for size, sh in
            [(5, shells), (6, shells), ((5, 6, 9), shells), (12, shells), (6, {2: 3, 3: 1})]]
    lines = ["%d" % len(sets)]
    for st in sets:
        recs = _records(st, 0)
        # sites numbered as they appear, blocks by cluster
        seen, names = {}, {}
        rows = []
        for mem, name, _ in recs:
            ids = [seen.setdefault(c, len(seen)) for c in mem] + [-1] * (3 - len(mem))
            rows.append([len(mem)] + ids + [names.setdefault(name, len(names))])
        lines.append("%d %d 6" % (len(seen), len(recs)))
        lines += [" ".join(str(v) for v in r) for r in rows]
    got = subprocess.run([exe], input="\n".join(lines), capture_output=True, text=True, check=True).stdout
    searches, good, kept, newest = (int(v) for v in got.split())
    assert (searches, good, kept, newest) == (2, 1, 16, 1)
