"""CPU check of the host's split of the loss partials: also for no rows (a network whose memory could not be had), where a
division by the number of partials ended the process."""
import subprocess
import sys

import pytest

CODE = """
from sfsim_amd import atmosphere as atm
lib = atm.lib()
print(lib._ZN5sfsim20surrogate_loss_slotsEi({rows}), lib._ZN5sfsim20surrogate_loss_partsEi({rows}))
"""


@pytest.mark.parametrize("rows", [0, 1, 16, 17, 64, 8192, 1 << 20])
def test_slots(rows):
    run = subprocess.run([sys.executable, "-c", CODE.format(rows=rows)], capture_output=True, text=True)
    assert run.returncode == 0, run.returncode
    slots, parts = map(int, run.stdout.split())
    assert parts == (rows * 16 + 255) // 256
    assert 1 <= slots <= 256 and slots * parts <= max(1 << 20, parts)
