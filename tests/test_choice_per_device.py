"""The default choice for devices of different sizes in one process: nothing of one device's choices may serve the other.
(CPU: the choice alone, no kernel runs.)"""
import ctypes
import threading


class Scratch(ctypes.Structure):
    """w4a16::Scratch."""
    _fields_ = [("ws", ctypes.c_void_p), ("ws_bytes", ctypes.c_size_t), ("cnt", ctypes.c_void_p), ("cnt_len", ctypes.c_int),
                ("epoch", ctypes.c_int), ("cus", ctypes.c_int)]


def test_a_choice_is_kept_for_its_device_only():
    from lmdeploy_amd._lib import lib
    pick, feasible = lib._ZN5w4a169algo_pickEiiiiRKNS_7ScratchEb, lib._ZN5w4a1613algo_feasibleEiiiiRKNS_7ScratchE
    feasible.restype = ctypes.c_bool
    room = {cus: Scratch(None, 64 << 20, None, 1 << 16, 0, cus) for cus in (256, 64)}
    ask = lambda N, T, cus: pick(1, N, T, 4096, ctypes.byref(room[cus]), 0)
    differ = 0
    for N in (1024, 4096, 16384, 22016, 57344):
        for T in (1, 8, 16, 24, 200):
            made = {}
            for cus in (256, 64, 256, 64):
                got, fresh = ask(N, T, cus), []
                assert got >= 0 and feasible(got, N, T, 4096, ctypes.byref(room[cus])), (N, T, cus, got)
                t = threading.Thread(target=lambda: fresh.append(ask(N, T, cus)))     # a thread that has chosen nothing yet
                t.start()
                t.join()
                assert fresh == [got], (N, T, cus, got, fresh)
                made[cus] = got
            differ += made[256] != made[64]
    assert differ > 3, differ
