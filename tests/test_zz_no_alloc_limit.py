"""The largest launch that the allocation-free batch takes, to the chunk: what
it was refused by when the chunks were in its scratch."""
import ctypes as C

import pytest

from test_zz_no_alloc import _launch, _models

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 20])
def test_no_alloc_limit(n):
    from mocassin_amd import _capi
    f = _capi.load().mc_transport_batch_noalloc
    f.restype = C.c_int
    f.argtypes = [C.POINTER(C.c_void_p), C.c_int32, C.c_void_p, C.c_void_p, C.c_void_p,
                  C.POINTER(_capi.McBatchTuning), C.POINTER(_capi.McCounters), C.c_void_p]
    tuning = {"waves_per_cu": 8, "emit_min": 32, "walk_steps": 8, "chunk": 64}
    up = lambda b: -(-b // 256) * 256
    need = lambda c: 256 + sum(up(b) for b in (216 * n, 96 * n, 8 * (n + 1), 8 * n, 128 * n, 4 * c, 8 * c, 4 * c))
    most = max(c for c in range(523000, 524289) if need(c) <= 8 << 20)
    print("%d models, %d chunks" % (n, most), flush=True)
    models = _models([(7, 1000, 3.e4, 100.)] * n)
    packets = [64] * (n - 1) + [64 * (most - n + 1)]
    try:
        c, _ = _launch(f, models, packets, [0] * n, tuning)
        assert c[-1]["n_flights"] > 0
        with pytest.raises(_capi.McError, match="MC_EINVAL"):
            _launch(f, models, packets[:-1] + [packets[-1] + 64], [0] * n, tuning)
    finally:
        for T in models:
            T.close()
