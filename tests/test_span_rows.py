"""Binning of triangles without exact masks: the tile rows of
include/srp/device/span_rows.h list every tile with a covered pixel (a host
build of the same header against the reference's sequential walk)."""
import os
import shutil
import subprocess

import pytest

from scene_runner import REPO


def test_rows_list_every_covered_tile(tmp_path):
    cc = shutil.which("gcc") or shutil.which("cc")
    if not cc:
        pytest.skip("no C compiler")
    exe = str(tmp_path / "span_rows_check")
    subprocess.run([cc, "-O2", "-std=c11", "-ffp-contract=off", "-fno-fast-math", "-I", os.path.join(REPO, "include"),
                    os.path.join(REPO, "tests", "native", "span_rows_check.c"), "-lm", "-o", exe], check=True)
    r = subprocess.run([exe, "4000"], stdout=subprocess.PIPE, text=True)
    print(r.stdout)
    assert r.returncode == 0 and r.stdout.startswith("0 missed")
    # and it is worth having: well under the boxes' tiles
    assert float(r.stdout.split(",")[1].split()[0]) < 0.6
