"""The wide Gram-Schmidt update's loads (csrc/trl_sums.h), compiled for the
CPU with every load checked: a basis whose last column ends at its last row is
read inside its bounds at every remainder of rows and columns, with the sums
in their fixed order."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "nutrlan_amd", "csrc")


def test_ragged_rows_stay_in_bounds(tmp_path):
    exe = str(tmp_path / "sums_bounds")
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-I", CSRC,
                    os.path.join(HERE, "sums_bounds.cpp"), "-o", exe], check=True)

    def counts(*args):
        return [int(x) for x in subprocess.run([exe, *args], capture_output=True, text=True, check=True).stdout.split()]

    assert counts() == [0, 0]
    assert counts("whole")[0] > 0  # the check sees a read past the last row
