"""The partwise kernels' workspace is reserved once for a plan, for the class that
needs most of it: growing it class by class frees and allocates it, and each free
waits for the device.  Checked in the sources."""
import os

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rchem_amd", "csrc")


def test_one_reservation_outside_the_loops():
    with open(os.path.join(CSRC, "rchem_api.cpp")) as fh:
        text = fh.read()
    assert text.count("part_slab_d.ensure(") == 1
    line = next(l for l in text.splitlines() if "part_slab_d.ensure(" in l)
    assert line.startswith("  if (slab > 0)")  # prepare_plan's own level


def test_a_launch_stays_within_it():
    """The grid of every form of the kernel is bounded by the slabs that fit."""
    with open(os.path.join(CSRC, "eri_part.hpp")) as fh:
        text = fh.read()
    launch = text[text.index("hipError_t eri_part_launch(const EriArgs& a"):]
    assert "bytes / eri_part_slab<LA, LB, LC, LD>()" in launch
    calls = [l for l in launch.splitlines() if "return eri_part_launch_rows<" in l]
    assert len(calls) == 3 and all("grid(" in l for l in calls)
