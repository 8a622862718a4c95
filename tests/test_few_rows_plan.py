"""Which shapes the exact product sends to its tiles for few rows, against
measured times (holo_few_rows_plan computes the choice without a GPU, for 256
CUs)."""
import ctypes as C

import pytest

F16, Q4_0, Q8_0, Q4_K, Q6_K = 1, 2, 8, 12, 14

# (type, rows, out, in, prepared copy, us on the few-row tiles, us on the 64 x 256 tiles)
MEASURED = [
    (F16, 64, 4096, 4096, 0, 24, 35), (F16, 192, 4096, 4096, 0, 60, 40), (F16, 64, 11008, 4096, 0, 53, 45),
    (F16, 100, 11008, 4096, 0, 92, 65), (F16, 64, 4096, 11008, 0, 52, 82), (F16, 192, 4096, 11008, 0, 132, 82),
    (F16, 256, 1024, 4096, 0, 28, 40), (F16, 512, 4096, 4096, 0, 130, 65), (F16, 512, 500, 2048, 0, 22, 31),
    (Q6_K, 64, 14336, 4096, 1, 40, 45), (Q6_K, 80, 14336, 4096, 1, 67, 59), (Q6_K, 100, 14336, 4096, 1, 68, 59),
    (Q6_K, 192, 14336, 4096, 1, 104, 84), (Q6_K, 100, 14336, 4096, 0, 69, 86), (Q6_K, 100, 4096, 4096, 1, 28, 45),
    (Q6_K, 140, 4096, 11008, 1, 83, 90), (Q6_K, 64, 4096, 14336, 1, 46, 105), (Q6_K, 512, 14336, 4096, 1, 236, 162),
    (Q4_0, 192, 11008, 4128, 0, 74, 106), (Q4_0, 192, 8192, 1056, 0, 25, 23), (Q8_0, 512, 2048, 1056, 0, 23, 21),
    (Q8_0, 256, 4096, 11040, 0, 97, 125), (Q8_0, 1000, 1024, 4128, 0, 67, 57), (Q8_0, 64, 8192, 1056, 0, 12, 16),
    (Q4_0, 64, 4096, 4128, 0, 21, 50), (Q4_0, 512, 11008, 4096, 0, 240, 118)]


@pytest.fixture(scope="module")
def lib():
    import holo_mi355x as h
    return h.load()


@pytest.mark.parametrize("t,M,N,K,prepared,few,tiles", MEASURED)
def test_measured_shapes_run_the_faster_tiles(lib, t, M, N, K, prepared, few, tiles):
    plan = (C.c_int * 4)()
    assert lib.holo_few_rows_plan(t, M, N, K, prepared, plan) == (few < tiles), list(plan)


def test_shapes_that_stay_elsewhere(lib):
    """Two rows, F16 rows too short to keep the GEMVs' precision, K no whole
    blocks or too long, more than 1024 rows, a type without such tiles."""
    plan = (C.c_int * 4)()
    for args in ((Q4_0, 2, 4096, 4096), (F16, 16, 4096, 992), (Q4_K, 16, 4096, 1056), (Q4_0, 16, 4096, 4100),
                 (Q8_0, 16, 4096, 16416), (Q4_0, 1025, 256, 4096), (0, 16, 4096, 4096)):
        assert lib.holo_few_rows_plan(*args, 0, plan) == 0, args
    assert lib.holo_few_rows_plan(F16, 16, 4096, 1024, 0, plan) == 1
