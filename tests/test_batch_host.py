"""Host code of the batched solve (xs_batch_host.cpp) over a simulated HIP
runtime whose streams order nothing that the interface does not promise."""
import os
import subprocess

import pytest

import xsolver_amd

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def create(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("hostsim") / "batch_create")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(HERE, "hostsim"), "-o", exe,
                    os.path.join(HERE, "hostsim", "batch_create.cpp")], check=True)

    def run(late, offsets, bad_row=-1, memory=1 << 40):
        p = subprocess.run([exe, str(late), str(offsets), str(bad_row), str(memory)],
                           capture_output=True, text=True, timeout=60)
        assert p.returncode == 0, p.stderr
        rc, slots, v32 = map(int, p.stdout.split())
        return rc, slots, v32
    return run


@pytest.mark.parametrize("late", [0, 1, 2, 3, 1000])
def test_flags_cleared_before_the_kernels_that_set_them(create, late):
    """The offset counts decide between diagonal slots and CSR, the pivot flag
    between a batch and an error, whenever the null stream gets its turn."""
    assert create(late, 5) == (xsolver_amd.XS_OK, 1, 0)
    assert create(late, 6) == (xsolver_amd.XS_OK, 0, 1)    # slots would drop an entry
    assert create(late, 27) == (xsolver_amd.XS_OK, 0, 1)
    assert create(late, 5, bad_row=1200)[0] == xsolver_amd.XS_ERR_PIVOT


def test_batch_that_fits_without_slots_is_taken(create):
    """Diagonal slots are a second copy of the matrix: where the memory does
    not hold them, the batch runs from its CSR arrays."""
    lo, hi = 0, 1 << 22   # the memory that a batch without slots needs
    while hi - lo > 1:
        mid = (lo + hi) // 2
        lo, hi = (lo, mid) if create(0, 6, memory=mid)[0] == xsolver_amd.XS_OK else (mid, hi)
    assert create(0, 6, memory=lo)[0] == xsolver_amd.XS_ERR_MEMORY
    assert create(0, 5, memory=hi) == (xsolver_amd.XS_OK, 0, 1)
    # room for the FP64 slots (40 bytes a row) but not the FP32 ones as well
    assert create(0, 5, memory=hi + 45 * 3000) == (xsolver_amd.XS_OK, 0, 1)
    assert create(0, 5, memory=hi + 60 * 3000) == (xsolver_amd.XS_OK, 1, 0)
