"""Choices of a tuning file that were timed on other tiles: a line for a grid
whose x and y tiles have been narrowed since (lines of 32 and 48 points) is
timed again, one for a grid that keeps its tiles (64) is taken."""
import pytest

from test_gpu_tuning import child

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,taken", [(32, 0), (48, 0), (64, 1)])
def test_line_without_the_narrowed_tiles(tmp_path, n, taken):
    path = tmp_path / "tune.txt"
    child(64, path)
    dev = path.read_text().split()[0]
    path.write_text(f"{dev} {n} {n} {n} 6 6 512 1 1 512 1\n")
    assert child(n, path)["tuning"]["from_tuning_file"] == taken
    # its own choice is there for the next process
    assert child(n, path)["tuning"]["from_tuning_file"] == 1
