"""The grid-resident loops (device/resident.hpp and the kernels built on it)
run on the CPU: the emulation (tests/emu/) runs the workgroups of such a launch
side by side, so the loops' index arithmetic, sums, publication, fallback
and the host's decisions about them are checked without a GPU.  With
SFR_EMU_ASAN=1 under AddressSanitizer, as tests/test_emulated_kernels.py."""
import os
import subprocess
import sys

import pytest

from tests.test_emulated_kernels import ASAN, HERE, SLOW, _env, emu_lib  # noqa: F401


def run(lib, group, passes):
    res = subprocess.run([sys.executable, os.path.join(HERE, "emu", "run_resident.py"), lib, group],
                         capture_output=True, text=True, env=_env(), timeout=600 * SLOW)
    print(res.stdout)
    assert res.returncode == 0, res.stdout + res.stderr[-3000:]
    assert "RESIDENT OK" in res.stdout and res.stdout.count("PASS") == passes


@pytest.mark.timeout(700 * SLOW)
def test_resident_loops_match_the_loops_of_kernels(emu_lib):  # noqa: F811
    """PCG, mixed PCG and BiCGSTAB on nine matrices (one to 33 workgroups with rows,
    empty ones among them, odd row counts, 16-bit offsets, escapes, 32-bit
    columns, 2 to 8 slots), and the three batches; that the loops did run
    resident is read from the context's counts."""
    run(emu_lib, "routes", 30)


@pytest.mark.timeout(700 * SLOW)
def test_a_workgroup_that_gives_up_on_the_last_sum(emu_lib):  # noqa: F811
    """One workgroup's wait runs out on a sum that the others see complete and
    end the solve with: its rows of x are not written, so the solve counts
    as stalled, whatever the others recorded."""
    run(emu_lib, "late", 13)


@pytest.mark.timeout(700 * SLOW)
def test_a_stall_seen_while_entering(emu_lib):  # noqa: F811
    """The mark of a launch that has stalled appears while a workgroup is
    entering it: its waves must agree on whether to go on."""
    run(emu_lib, "split", 3)


@pytest.mark.timeout(700 * SLOW)
def test_what_a_stall_costs(emu_lib):  # noqa: F811
    """A stall in one system of a batch ends the batch's resident launches, and
    the context keeps to the loops of kernels for a while."""
    run(emu_lib, "away", 8)


@pytest.mark.timeout(700 * SLOW)
def test_batches_give_the_device_back(emu_lib):  # noqa: F811
    """No resident launch runs past its limit of iterations, single or batched,
    and the next one goes on where it ended."""
    run(emu_lib, "slices", 5)


@pytest.mark.timeout(100 * SLOW)
def test_launches_that_fit_the_device_together(emu_lib):  # noqa: F811
    """The host's count of resident workgroups in flight, an XCD at a time."""
    run(emu_lib, "count", 13)
