"""The training kernel's elimination over four lanes (lane_lu.hpp): its result
must not depend on the order in which the lanes run between two barriers."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_elimination_does_not_depend_on_the_lanes_order(tmp_path):
    from mole_amd import build

    exe = str(tmp_path / "lane_lu_order")
    subprocess.run([build._hipcc(), "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-ffp-contract=off",
                    os.path.join(HERE, "lane_lu_order.cpp"), "-o", exe], check=True, capture_output=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
