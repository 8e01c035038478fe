"""Basic scheme: the workgroup that decides to stop runs beside the tiles of an
inverse y pass, so its decision must not reach a word that these tiles test
(waves of one workgroup would disagree on whether to run).  The next z pass
skips its work and makes the decision known to the passes after it (CPU
only: the device code's own predicates, compiled for the host)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def lines(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("probe") / "stop_probe")
    subprocess.check_call([HIPCC, "-std=c++17", "-O1", "--offload-arch=gfx950", "--cuda-host-only", "-o", exe,
                           os.path.join(HERE, "stop_probe.hip")])
    return subprocess.run([exe], capture_output=True, text=True, check=True).stdout.split("\n")


@pytest.mark.parametrize("why,done", [(0, 0), (1, 1), (2, 2), (3, 3)])
def test_deciding_launch_is_not_gated_by_its_decision(lines, why, done):
    before, same, skip_other, after_other, skip_first, after, code = lines[why].split()
    assert before == same == "1111"
    # every workgroup of the next z pass skips, its first thread sets `done`
    assert skip_other == skip_first == str(int(done != 0))
    assert after_other == "1111"
    assert after == ("1111" if done == 0 else "0000")
    assert int(code) == done
