"""The fixed-dt kernels' source run on the CPU with the waves of a workgroup in a chosen order
(wave_model.cpp).  Test infrastructure only."""
from __future__ import annotations

import ctypes as C
import subprocess
from pathlib import Path
from typing import Sequence

import numpy as np

from mcluminescence_amd._abi import DEFAULT_SEED, RunParams, run_array

HERE = Path(__file__).resolve().parent
FLAGS = ["-O1", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-mavx2", "-mfma",
         "-Wno-unknown-pragmas", "-Wno-attributes", f"-I{HERE}"]

# schedules: the waves in turn, or one of them behind or ahead of all others (random: SHUFFLED)
IN_TURN, SHUFFLED = 0, 200


def behind(w: int) -> int:
    return 1 + w


def ahead(w: int) -> int:
    return 100 + w


# where the clusters live
LDS, SCRATCH, SCRATCH_ALL = 0, 1, 2


class Model:
    def __init__(self, out: Path):
        subprocess.run(["g++", *FLAGS, str(HERE / "wave_model.cpp"), "-o", str(out)], check=True)
        self.lib = C.CDLL(str(out))
        self.lib.wm_run_fixed_dt.argtypes = [
            C.POINTER(RunParams), C.c_int, C.c_uint64, C.c_int, C.c_int, C.c_int, C.c_int, C.c_int,
            C.c_int, C.c_double, C.c_int, C.c_uint64, C.c_void_p, C.c_void_p, C.c_void_p, C.c_char_p,
            C.c_int]

    def run(self, runs: Sequence[RunParams], waves: int, *, n_bins: int = 0, form: int = LDS,
            wide: bool = False, persistent: bool = False, holes_per_cell: float = 2.0,
            schedule: int = IN_TURN, schedule_seed: int = 0, seed: int = DEFAULT_SEED):
        """(counts, live electron-steps, work rows, error text)."""
        total = sum(int(r.sims) for r in runs)
        row = n_bins or max(int(r.n_steps) for r in runs)
        counts = np.full((total, row), 0xFFFFFFFF, np.uint32)
        live = np.zeros(total, np.uint64)
        work = np.zeros((total, 4), np.uint64)
        err = C.create_string_buffer(256)
        self.lib.wm_run_fixed_dt(run_array(runs), len(runs), seed, n_bins, row, waves, form, int(wide),
                                 int(persistent), holes_per_cell, schedule, schedule_seed,
                                 counts.ctypes.data, live.ctypes.data, work.ctypes.data, err, len(err))
        return counts, live, work, err.value.decode()
