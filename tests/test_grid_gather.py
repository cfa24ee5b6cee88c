"""How the workgroups of a KH_GRID_CYCLE launch gather (kh_grid_gather.hpp, host
only): the kernel's own steps run on a model of the control block in every order
they can take (grid_gather_model.cpp), for as many workgroups on the home XCD as
the cycle has parts, for fewer, more and none, with the time limit passing at
any moment or never. Whichever way, exactly the parts work together or one
workgroup alone, every wait ends, and the block is clear for the next launch."""
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    out = tmp_path_factory.mktemp("gather") / "grid_gather_model"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Wextra", f"-I{HERE.parent / 'kutta_amd' / 'csrc'}",
                    "-o", str(out), str(HERE / "grid_gather_model.cpp")], check=True)
    return out


@pytest.mark.parametrize("expires", [1, 0])
@pytest.mark.parametrize("parts,home,away", [(1, 1, 1), (1, 1, 3), (2, 2, 2), (2, 2, 3), (3, 3, 1), (2, 1, 2),
                                             (2, 3, 1), (2, 0, 3)])
def test_every_order_of_the_steps(model, parts, home, away, expires):
    done = subprocess.run([str(model), str(parts), str(home), str(away), str(expires)], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout
    words = done.stdout.replace(",", "").split()
    together, alone = int(words[4]), int(words[6])
    assert (together > 0) == (home == parts)
    assert (alone > 0) == (home != parts or expires == 1)
