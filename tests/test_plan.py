"""CPU: the default kernel's plan, which a thread keeps for its last eight
grids, is the one a search finds, and a repeated call does not search again."""
import ctypes as C
import threading
import time

import pytest

mx = pytest.importorskip("mmsp_amd")


class Geom(C.Structure):
    _fields_ = [("dim", C.c_int), ("n", C.c_int * 3), ("b0", C.c_int * 3), ("b1", C.c_int * 3), ("s", C.c_int * 3),
                ("nodes", C.c_int), ("fields", C.c_int), ("w", C.c_double * 3), ("wf", C.c_float * 3), ("vol", C.c_double),
                ("dx", C.c_double * 3)]


class Choice(C.Structure):
    _fields_ = [(n, C.c_int) for n in ("variant", "ty", "tz", "chunk", "opt")]


make_geom = mx.lib._ZN5mmspx9make_geomERK10mmspx_desc
make_geom.restype, make_geom.argtypes = Geom, [C.c_void_p]
default_choice = mx.lib._ZN5mmspx14default_choiceERKNS_4GeomEii
default_choice.restype, default_choice.argtypes = Choice, [C.c_void_p, C.c_int, C.c_int]


def plan(shape, model, precision, fields=1, bc=None):
    """A call without arguments that asks for the plan of this grid."""
    d = mx.make_desc(shape, fields, fields > 1, precision, bc)
    g = make_geom(C.byref(d))
    return lambda: tuple(getattr(default_choice(C.byref(g), d.precision, mx._model(model)), n) for n, _ in Choice._fields_)


N = [(mx.NEUMANN, mx.NEUMANN)] * 3
GRIDS = [((40 + 9 * k, 64, 70 + k), m, p) for k in range(4) for m in ("ac", "ch") for p in ("f64", "f32", "f32ref")]
GRIDS += [((300, 200), m, "f64") for m in ("ac", "ac_noise", "ch_dw", "ch_noise")]
GRIDS += [((300, 200), "ac", "f64", 1, N[:2]), ((40, 64, 70), "ch", "f64", 1, N), ((300, 200), "gg", "f32", 8),
          ((300, 200), "zener", "f32", 4), ((90, 90, 97), "gg", "f64", 8), ((90, 90, 97), "gg", "f64", 4)]


def test_plans_are_those_of_a_search():
    plans = [plan(*g) for g in GRIDS]
    searched = []
    for p in plans:  # a new thread has kept nothing
        t = threading.Thread(target=lambda: searched.append(p()))
        t.start()
        t.join()
    assert len(set(searched)) > 8
    for order in (range(len(plans)), reversed(range(len(plans)))):
        for k in order:
            for _ in range(2):
                assert plans[k]() == searched[k], GRIDS[k]


def test_a_repeated_plan_is_not_searched_for():
    plans = [plan((200 + k, 64, 64), "ac", "f64") for k in range(12)]  # more than are kept

    def best(calls):
        times = []
        for _ in range(50):
            t = time.perf_counter()
            for p in calls:
                p()
            times.append(time.perf_counter() - t)
        return min(times)

    assert best([plans[0]] * 12) < 0.6 * best(plans)
