"""Single products through the staging area that all matrix handles share: with a residual and without, the largest that fit and the first that do not, several threads at once, handles that come and go."""
import ctypes
import gc
import re
import threading

import numpy as np
import pytest

import espresso_amd._lib as lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import espresso_amd.ops as o
    o.init()
    yield o


def matrix(ops, rows, cols, seed):
    w = np.random.default_rng(seed).normal(0, 0.02, (rows, cols)).astype(np.float16)
    return ops.Matrix(lib.FORMAT_F16, w.view(np.uint8), rows, cols), w.astype(np.float64)


def check(m, w, batch, seed, residual):
    rng = np.random.default_rng(seed)
    x = rng.normal(0, 1, (batch, w.shape[1])).astype(np.float16)
    r = rng.normal(0, 1, (batch, w.shape[0])).astype(np.float32) if residual else None
    want = x.astype(np.float64) @ w.T + (0 if r is None else r)
    # exact products, fp32 sums in some order: one rounding per addition, relative to the sum of the magnitudes
    bound = (w.shape[1] + 16) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).T + np.abs(want) + 1)
    assert (np.abs(m.gemv(x, r) - want) <= bound).all(), (batch, residual)


PRODUCTS_BEFORE = 128   # that a program makes before the area is worth its memory


@pytest.fixture()
def area(ops):
    """The area is there for as long as this matrix is."""
    m, _ = matrix(ops, 16, 8, 0)
    for _ in range(PRODUCTS_BEFORE):
        m.gemv(np.zeros((1, 8), np.float16))
    yield m
    m.close()


# 1 MiB of activations is 1024 rows of 512 columns, 4 MiB of results 1024 rows of 1024
@pytest.mark.parametrize("rows,cols,batches", [(24, 8, (1, 2, 5)), (70, 512, (1, 3, 1024, 1025)), (1024, 64, (2, 1024, 1025)), (1023, 72, (7,))])
def test_every_size_takes_its_way(ops, area, rows, cols, batches):
    m, w = matrix(ops, rows, cols, rows)
    for batch in batches:
        for residual in (False, True):
            check(m, w, batch, batch, residual)
    m.close()


@pytest.mark.parametrize("held", [False, True])
def test_threads_and_handles(ops, held, request):
    if held:
        request.getfixturevalue("area")
    failures = []

    def work(seed):
        try:
            for i in range(12):
                m, w = matrix(ops, 64 + 16 * seed, 256, seed)
                for batch in (1, 2, 6, 40):
                    check(m, w, batch, 100 * seed + i, batch % 2 == 0)
                m.close()
        except BaseException as e:   # noqa: BLE001
            failures.append(e)

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures


def test_a_handle_leaves_the_last_error(ops):
    """A matrix that is made and multiplied, whether or not the area comes with it, is no failure: the most recent one stays what it was."""
    m, _ = matrix(ops, 32, 64, 1)
    with pytest.raises(lib.EspressoError, match="layer_product: rows 0"):
        m.layer_product(np.zeros((0, 64), np.float16))
    m.close()
    said = lib.last_error()
    other, w = matrix(ops, 32, 64, 2)
    assert lib.last_error() == said and "layer_product" in said
    for _ in range(PRODUCTS_BEFORE):
        check(other, w, 2, 3, True)
    assert lib.last_error() == said
    other.close()
    assert lib.last_error() == said


def test_the_area_comes_when_products_have_paid_for_it_and_goes_with_the_last_handle(ops):
    """Handles made for a few products cost what they did without the area (21 MiB of device memory, 5 of pinned)."""
    gc.collect()   # handles of other tests
    with open("/proc/self/maps") as f:
        hip = ctypes.CDLL(re.search(r"/\S*libamdhip64\.so\S*", f.read()).group(0))
    free, total = ctypes.c_size_t(), ctypes.c_size_t()

    def held(since):
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return since - free.value

    def mebibytes(since):
        return held(since) / 2 ** 20

    m, w = matrix(ops, 32, 64, 1)
    for _ in range(PRODUCTS_BEFORE + 1):
        check(m, w, 2, 3, True)   # whatever the first products of a process allocate for good
    m.close()
    start = -held(0)
    for _ in range(3):
        m, w = matrix(ops, 32, 64, 1)
        for _ in range(PRODUCTS_BEFORE - 1):
            check(m, w, 2, 3, True)
        assert mebibytes(start) < 16
        m.close()
    a, w = matrix(ops, 32, 64, 1)
    b, _ = matrix(ops, 32, 64, 2)
    for i in range(PRODUCTS_BEFORE):
        assert mebibytes(start) < 16
        check(a, w, (2, 5, 2)[i % 3], 3, True)
    assert mebibytes(start) >= 16
    a.close()
    assert mebibytes(start) >= 16
    b.close()
    assert mebibytes(start) < 16
