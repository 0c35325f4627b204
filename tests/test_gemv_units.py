"""The rows that waves of the Q4_K GEMV kernels load, walked on the CPU: inside
their range for every wave of a launch, those without work among them."""
from __future__ import annotations

import os
import subprocess

ORACLE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle")


def test_every_wave_loads_rows_of_its_range():
    subprocess.run(["make", "-s", "-C", ORACLE, "_build/gemv_units_probe"], check=True)
    p = subprocess.run([os.path.join(ORACLE, "_build", "gemv_units_probe")], capture_output=True, text=True)
    assert p.returncode == 0, p.stdout
    assert p.stdout.startswith("walked ")
