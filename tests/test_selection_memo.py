"""A thread's remembered choice of a kernel follows every change of the tuning cache and the model, made by any thread."""
import ctypes
import threading

import torchlette_amd as T
from torchlette_amd import _lib as L


def test_a_choice_follows_the_cache_in_every_thread():
    lib = L.load()
    buf = ctypes.create_string_buffer(64)
    ptr = ctypes.cast(buf, ctypes.c_void_p).value
    w = L.QWeight(L.FMT_INT8_GROUPED, 64, 3000, 2048, ptr, ptr)

    def chosen():
        c = L.KernelConfig()
        assert lib.tlhip_selected_config(ctypes.byref(w), L.F16, 1, L.F16, ctypes.byref(c)) == 0
        return c.as_tuple()

    steps, seen = [threading.Barrier(2) for _ in range(8)], []

    def other():
        for i in range(4):
            steps[2 * i].wait(20)
            seen.append(chosen())
            steps[2 * i + 1].wait(20)

    before = T.exportTuningCache()
    winner = L.KernelConfig.of(L.VARIANT_GEMV, 16, 1, 8, 2, 4)
    thread = threading.Thread(target=other)
    try:
        T.clearTuningCache()
        own = chosen()
        assert own != winner.as_tuple()
        thread.start()
        want = []
        for i, change in enumerate((lambda: None, lambda: lib.tlhip_tune_cache_seed(ctypes.byref(w), L.F16, 1, L.F16, ctypes.byref(winner)),
                                    T.clearTuningCache, lambda: T.importTuningCache(seeded))):
            change()
            if i == 1:
                seeded = T.exportTuningCache()
            want.append(chosen())
            steps[2 * i].wait(20)
            steps[2 * i + 1].wait(20)
    finally:
        if thread.ident:
            thread.join(30)
        T.clearTuningCache()
        T.importTuningCache(before)
    assert want == seen == [own, winner.as_tuple(), own, winner.as_tuple()]
