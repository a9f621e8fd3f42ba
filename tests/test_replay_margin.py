"""The replay's jumps keep their margin under an inexact reciprocal, as the
device's is, over walks of every length that draws take (up to 65,536 steps):
a host build of the header's device branch against sequential additions."""
import os
import shutil
import subprocess

import pytest

from scene_runner import REPO


def test_jumps_stay_exact_with_an_inexact_reciprocal(tmp_path):
    cc = shutil.which("gcc") or shutil.which("cc")
    if not cc:
        pytest.skip("no C compiler")
    exe = str(tmp_path / "replay_margin_check")
    subprocess.run([cc, "-O2", "-std=c11", "-ffp-contract=off", "-fno-fast-math", "-I", os.path.join(REPO, "include"),
                    os.path.join(REPO, "tests", "native", "replay_margin_check.c"), "-lm", "-o", exe], check=True)
    r = subprocess.run([exe, "4000"], stdout=subprocess.PIPE, text=True)
    print(r.stdout)
    assert r.returncode == 0 and r.stdout.strip().splitlines()[-1].startswith("0 of ")
