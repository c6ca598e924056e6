"""What the batched calls decide on the host (include/rocrand_batched.h): which batches fit the
no-allocation call's array, and the status of streams that no call takes."""
import ctypes

import pytest

from rocrand_amd import rocrand as R

torch = pytest.importorskip("torch")

S = 131072
TYPE_ERROR, OUT_OF_RANGE = 103, 104


# Batches of MRG32k3a streams whose engines wrap (offset S - 1 or S - 100), cut into one tile
# more each there, and Philox streams: the most of each that the array takes.
@pytest.mark.skipif(torch.cuda.device_count() > 0, reason="the outputs are not device memory: nothing may run")
@pytest.mark.parametrize("rng,kind,offset,n,count", [
    (R.MRG32K3A, R.BATCH_UNIFORM_FLOAT, S - 1, 2, 69904), (R.MRG32K3A, R.BATCH_UNIFORM_FLOAT, S - 100, 255, 69904),
    (R.MRG32K3A, R.BATCH_UNIFORM_FLOAT, S - 100, 300, 59918), (R.MRG32K3A, R.BATCH_NORMAL_FLOAT, S - 1, 600, 59918),
    (R.MRG32K3A, R.BATCH_UNIFORM_FLOAT, S - 100, S, 809), (R.PHILOX4_32_10, R.BATCH_UNIFORM_FLOAT, 0, 16, 51149),
    (R.PHILOX4_32_10, R.BATCH_UNIFORM_FLOAT, 0, 10**6, 12865)])
def test_batches_that_fit_the_no_allocation_array(rng, kind, offset, n, count):
    arr = (R.BatchStream * count)(*[R.BatchStream(rng, kind, i, offset, n, 0.0, 1.0, 0x1004) for i in range(count)])
    assert R.load().rocrand_generate_batched_noalloc(arr, count, None) != OUT_OF_RANGE


@pytest.mark.parametrize("stream,want", [
    ((R.XORWOW, R.BATCH_UINT, 1, 0, 10, 0.0, 1.0, 0x1000), TYPE_ERROR),
    ((R.MRG32K3A, 8, 1, 0, 10, 0.0, 1.0, 0x1000), TYPE_ERROR),
    ((R.PHILOX4_32_10, R.BATCH_UINT, 1, 0, 10, 0.0, 1.0, None), OUT_OF_RANGE),
    ((R.PHILOX4_32_10, R.BATCH_POISSON, 1, 0, 10, 0.0, 1.0, 0x1000), OUT_OF_RANGE),
    ((R.MRG32K3A, R.BATCH_POISSON, 1, 0, 10, float("nan"), 1.0, 0x1000), OUT_OF_RANGE)])
def test_streams_are_checked_before_the_device_is_asked(stream, want):
    """Every call names the stream's fault, also where there is no device."""
    L = R.load()
    arr = (R.BatchStream * 1)(R.BatchStream(*stream))
    plan = ctypes.c_void_p()
    assert L.rocrand_batch_plan_create(ctypes.byref(plan), arr, 1, None) == want
    assert not plan
    assert L.rocrand_generate_batched(arr, 1, None) == want
    assert L.rocrand_generate_batched_noalloc(arr, 1, None) == want
