"""The coupled V-cycle through the C ABI, on the GPU (tests/native/parity.cpp):
the cycle against the one with separate residual, restriction and prolongation (uniform levels 1, 3, 4
and 5: one to five smoothed levels, with the dense bottom at none, the last or the first coarse one),
and on hierarchies with sliced-ELL copies on several levels;
the greedy aggregation at the edges of its windows and with conflict lists past their slots;
the pressure operator's row runs at the edges of their tiles against sums on the host; the dense
inverse of the coarsest operator at the edges of its blocks; the ILU(0) sweeps where the trailing
colours change path; the contraction of the shape gradient with the boundary modes against the host
loop; pressure solves in FP64 (level 0 coupled and separate) and with the FP32 cycle against the
oracle's, and momentum solves: on both sides of 65,536 rows, up to where the PCG update runs in the
cycle's first launch and a workgroup takes 64 rows, and on 460,672 rows, where a workgroup takes
several runs of 128 or 256 rows."""
import subprocess
from pathlib import Path

import pytest

BIN = Path(__file__).resolve().parent / "native" / "build" / "parity"

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level", [1, 3, 4, 5])
def test_coupled_cycle(level):
    print(f"[case] coupled V-cycle level {level}", flush=True)
    r = subprocess.run([str(BIN), "coupled", str(level)], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0 and "ALL PASSED" in r.stdout, r.stdout[-3000:] + r.stderr[-2000:]


@pytest.mark.parametrize("case", ["copies", "aggregate", "runs", "inverse", "ilutail", "shape"])
def test_tile_edges(case):
    print(f"[case] {case}", flush=True)
    r = subprocess.run([str(BIN), case, "0"], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0 and "ALL PASSED" in r.stdout, r.stdout[-3000:] + r.stderr[-2000:]


@pytest.mark.parametrize("case", ["pcg", "mixed"])
@pytest.mark.parametrize("level", [2, 4, 5])
def test_pressure_solve(case, level):
    print(f"[case] {case} level {level}", flush=True)
    r = subprocess.run([str(BIN), case, str(level)], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0 and "ALL PASSED" in r.stdout, r.stdout[-3000:] + r.stderr[-2000:]


@pytest.mark.parametrize("level", [4, 5])
def test_momentum_solve(level):
    print(f"[case] bicgstab level {level}", flush=True)
    r = subprocess.run([str(BIN), "bicgstab", str(level)], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0 and "ALL PASSED" in r.stdout, r.stdout[-3000:] + r.stderr[-2000:]
