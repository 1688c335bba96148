"""bench.py reads counter figures only while the sources that the counted kernels are compiled
from match: the lists name every header of theirs (host logic, no GPU)."""

import os
import re

import pytest

import bench

CSRC = os.path.join(bench.ROOT, "cuda-cvdv_amd", "csrc")


@pytest.mark.parametrize("sources", ["FFT_SOURCES", "BATCH_SOURCES"])
def test_lists_name_every_included_header(sources):
    listed = getattr(bench, sources)
    for name in listed:
        with open(os.path.join(CSRC, name)) as f:
            included = re.findall(r'^#include "([^"/]+)"', f.read(), re.M)
        assert set(included) <= set(listed), name


def test_fft_list_names_the_planner_of_chains():
    """Which kernel runs a transform is decided there."""
    assert "fft_chain.hip" in bench.FFT_SOURCES
