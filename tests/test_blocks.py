"""The block cache of device memory on a simulated card, on the CPU: blocks cut
from larger ones, joined and given back, and what it can serve when the card
is full (tests/blocks_check.cpp)."""
import os
import shutil
import subprocess

import pytest

from .conftest import REPO


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ absent")
    exe = tmp_path_factory.mktemp("blocks") / "blocks_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I" + os.path.join(REPO, "ompmc_amd", "csrc"),
                    os.path.join(REPO, "tests", "blocks_check.cpp"), "-o", str(exe)], check=True)
    return str(exe)


@pytest.mark.parametrize("name", ["cut_join_evict", "full_card", "reusable", "two_devices", "any_order"])
def test_block_cache(check, name):
    r = subprocess.run([check, name], stdout=subprocess.PIPE, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
