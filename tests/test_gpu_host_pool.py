"""Host entry points on device memory kept between calls: growing, shrinking and
alternating sizes and precisions, calls from several threads, a refused call in
between, and a release must leave every result what a fresh call gives."""
import threading

import numpy as np
import pytest

from tests.conftest import rel_l2, wst_case

pytestmark = pytest.mark.gpu

CASES = [(300, 64, 96, 10.0, False), (5000, 250, 128, 5.0, True), (40, 32, 32, 20.0, True), (2000, 128, 500, 3.0, False)]


def _call(cg, k, nx, ny, fov, single):
    m = k["ms"].astype("c8") if single else k["ms"]
    w = k["wgt"].astype("f4") if single else k["wgt"]
    d = k["dirty"].astype("f4") if single else k["dirty"]
    xp, yp = np.radians(fov) / nx, np.radians(fov) / nx
    eps = 1e-5 if single else 1e-9
    img = cg.ms2dirty(k["uvw"], [k["f0"]], m, w, nx, ny, xp, yp, 0, 0, eps, True)
    return img, cg.dirty2ms(k["uvw"], [k["f0"]], d, w, xp, yp, 0, 0, eps, True).ravel()


def test_host_calls_share_nothing(gpu):
    import cugridder_amd as cg
    lib = cg.lib()
    data = [wst_case(n, nx, ny, fov) for n, nx, ny, fov, _ in CASES]
    fresh = []
    for k, (_, nx, ny, fov, single) in zip(data, CASES):
        assert lib.cg_host_release() == 0
        fresh.append(_call(cg, k, nx, ny, fov, single))

    def same(i):
        _, nx, ny, fov, single = CASES[i]
        # FP64 atomics of the 2-D and dense gridders aside, the same sums
        for a, b in zip(_call(cg, data[i], nx, ny, fov, single), fresh[i]):
            assert rel_l2(a, b) < (1e-6 if single else 1e-14)

    for i in (1, 0, 3, 2, 1, 2, 0):
        same(i)
    with pytest.raises(Exception):
        cg.ms2dirty(data[0]["uvw"], [-1.0], data[0]["ms"], None, 64, 96, 1e-3, 1e-3, 0, 0, 1e-9, True)
    same(0)
    failed = []

    def worker(first):
        try:
            for j in range(6):
                same((first + j) % len(CASES))
        except BaseException as e:  # noqa: BLE001
            failed.append(e)

    threads = [threading.Thread(target=worker, args=(t,)) for t in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
    assert lib.cg_host_release() == 0
    same(3)
