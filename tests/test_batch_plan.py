"""CPU checks of how batches above one launch are split (csrc/vs_batch.hip): what the kernels assume of the sizes holds
for every vocabulary, stride, type, batch and CU count."""
import random

import numpy as np
import pytest

from volundr_amd import _lib

ROWS, GMAX, LANES, ROUNDS = 128, 64, 512, 16  # rows per launch, workgroups per row, threads, 64-key rounds per wave


def plan(dtype, V, ld, mis, B, ws_rows, cus):
    L = _lib.load()
    out = np.zeros(7, np.int32)
    ws = L.vs_sample_workspace_bytes(1, V) * ws_rows
    _lib.check(L.vs_batch_plan(dtype, V, ld, mis, B, ws, cus, out.ctypes.data), "vs_batch_plan")
    return dict(zip(("rows", "E", "G", "CH", "kcap", "kmax", "nv"), out.tolist()))


@pytest.mark.parametrize("cus", [8, 32, 38, 64, 104, 128, 256, 304])
def test_every_open_row_has_a_workgroup(cus):
    """The resolve kernel runs one workgroup per CU and takes each open row of a launch once: a launch of more rows than
    CUs would leave rows without a result."""
    for B in (2, 20, 64, 65, 100, 128, 129, 500):
        p = plan(_lib.VS_F32, 163840, 163840, 0, B, 64, cus)
        assert 1 <= p["rows"] <= min(B, ROWS, cus), (B, p)


def test_sizes_the_kernels_assume():
    rng = random.Random(5)
    for _ in range(4000):
        dtype = rng.choice([_lib.VS_F32, _lib.VS_BF16, _lib.VS_F16])
        vec = 4 if dtype == _lib.VS_F32 else 8
        V = int(round(8192 * (786432 / 8192) ** rng.random()))
        ld = V + rng.choice([0, 0, 1, 8, 640, rng.randrange(64)])
        mis, B = rng.randrange(vec), rng.randrange(1, 400)
        ws_rows, cus = min(64, rng.choice([64, B])), rng.choice([32, 64, 128, 256, 256, 304])
        p = plan(dtype, V, ld, mis, B, ws_rows, cus)
        span = V + (mis if ld % vec == 0 else vec - 1)
        what = (dtype, V, ld, mis, B, ws_rows, cus, p)
        assert 1 <= p["rows"] <= min(B, cus, ROWS if ws_rows == 64 else ws_rows), what
        assert p["E"] in (16, 32) and 1 <= p["G"] <= GMAX, what
        assert p["CH"] % vec == 0 and p["CH"] <= p["E"] * LANES, what          # a chunk fits its workgroup's registers
        assert (p["G"] - 1) * p["CH"] < span <= p["G"] * p["CH"], what         # every position once, no empty chunk
        assert p["kcap"] % 64 == 0 and 64 <= p["kmax"] <= min(p["kcap"], 256), what  # top lists of 64 always fit
        assert p["kcap"] * p["G"] <= (5120 if p["rows"] > 64 else 8192), what  # the row's list area
        assert -(-p["G"] // 8) * -(-p["kcap"] // 64) <= ROUNDS, what           # the finish kernel's registers
        assert 8 <= p["nv"] <= p["kcap"], what
