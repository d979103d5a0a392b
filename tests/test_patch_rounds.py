"""Rounds of the patch kernel (cemc_amd/csrc/ce_patch_kernel.h)."""
import os
import subprocess

import pytest

from cemc_amd.lattice import FCCSettings
from test_patches import _records

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def round_check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("round") / "patch_round_check")
    subprocess.run(["g++", "-O2", "-std=c++17", os.path.join(HERE, "patch_round_check.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("species,shells,size,q", [
    (2, {2: 4, 3: 2}, (5, 6, 7), 6),
    (3, {2: 3, 3: 2, 4: 1}, (5, 5, 5), 5),
    (4, {2: 3, 3: 2}, (5, 5, 5), 4),
])
def test_unfilled_slots_read_inside_their_tables(round_check, species, shells, size, q):
    """A round with fewer moves than slots evaluates swaps of earlier rounds
    as well: no index leaves its patch's table."""
    st = FCCSettings(size, list("ABCD"[:species]), shells)
    recs = _records(st, 0)
    cols = sorted({c for mem, _, _ in recs for c in mem})
    info = st.periodic_descriptor()
    at = {int(c): k for k, c in enumerate(info["cols"])}
    names = sorted({name for _, name, _ in recs})
    lines = ["%d %d %d %d %d %d %d 400" % (*size, species, q, len(cols), len(recs))]
    lines += ["%d %d %d" % tuple(info["col_cells"][at[c]]) for c in cols]
    for mem, name, _ in recs:
        ids = [cols.index(c) for c in mem] + [-1] * (3 - len(mem))
        lines.append(" ".join(str(v) for v in [len(mem)] + ids + [names.index(name)]))
    got = subprocess.run([round_check], input="\n".join(lines), capture_output=True, text=True, check=True).stdout
    n_eval, n_out = (int(v) for v in got.split())
    assert n_eval > 0 and n_out == 0
