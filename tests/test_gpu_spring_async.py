"""GPU: spring-chain solves on device memory return before they end, as every solve on
device memory does, and solves of several streams and threads at once do not disturb
one another."""
import ctypes as C
import threading
import time

import numpy as np
import pytest
import torch

import deamd
from deamd import _abi

pytestmark = pytest.mark.gpu
M = deamd.ExplicitRungeKutta


class Device:
    """A solve on device memory, its results in buffers of its own."""

    def __init__(self, method, n, t1, seed, points=0):
        self.sys, y0 = deamd.gen_spring(n, seed=seed)
        put = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
        p = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
        b = _abi.ode_defaults()
        b.family, b.n, b.method = _abi.DE_FAMILY_SPRING_CHAIN, n, method.method_id
        b.t0_scalar, b.tf_scalar, b.h0 = 0.0, t1, method.settings["h0"]
        b.rtol, b.atol, b.max_steps = 1e-6, 1e-9, 10000000
        self.keep = [put(self.sys.params_packed), put(y0)]
        b.params, b.y0 = p(self.keep[0]), p(self.keep[1])
        for name, v, ty in (("sizes", self.sys.sizes, C.c_int32),
                            ("state_offset", self.sys.state_offset, C.c_int64),
                            ("param_offset", self.sys.param_offset, C.c_int64)):
            self.keep.append(put(v))
            setattr(b, name, C.cast(p(self.keep[-1]), C.POINTER(ty)))
        f64 = lambda m: torch.full((m,), float("nan"), dtype=torch.float64, device="cuda")  # noqa: E731
        self.out = {"y_final": f64(len(y0)), "t_final": f64(n)}
        for k in ("accepted", "rejected", "evals"):
            self.out[k] = torch.full((n,), -1, dtype=torch.int64, device="cuda")
        self.out["status"] = torch.full((n,), -1, dtype=torch.int32, device="cuda")
        if points:
            self.keep.append(put(np.linspace(0.0, t1, points)))
            b.n_eval, b.t_eval = points, p(self.keep[-1])
            self.out["dense"] = f64(len(y0) * points)
            self.out["n_dense"] = torch.full((n,), -1, dtype=torch.int32, device="cuda")
        r = _abi.OdeResult()
        for k, v in self.out.items():
            setattr(r, k, p(v))
        self.b, self.r = b, r
        torch.cuda.synchronize()

    def solve(self, stream):
        _abi.check(deamd.lib().de_ode_batch_solve(C.byref(self.b), C.byref(self.r),
                                                  C.c_void_p(stream.cuda_stream)))

    def results(self):
        return {k: v.cpu().numpy().copy() for k, v in self.out.items()}


def same(a, b):
    return all(np.array_equal(a[k], b[k], equal_nan=a[k].dtype.kind == "f") for k in a)


@pytest.mark.parametrize("name,t1", [("rk4", 400.0), ("dop853", 400.0), ("rkf45", 400.0),
                                     ("dopri5", 400.0)])
def test_the_call_returns_before_the_solve_ends(name, t1):
    method = M.rk4(0.02) if name == "rk4" else getattr(M, name)()
    stream = torch.cuda.Stream()
    d = Device(method, 8192, t1, seed=5)
    d.solve(stream)  # streams, shapes, workspace pool
    stream.synchronize()
    first = d.results()
    t0 = time.perf_counter()
    d.solve(stream)
    returned = time.perf_counter() - t0
    ended = torch.cuda.Event()
    ended.record(stream)
    pending = not ended.query()
    stream.synchronize()
    total = time.perf_counter() - t0
    assert pending and returned < 0.5 * total, (returned, total)
    assert (first["status"] == deamd.DE_STATUS_COMPLETE).all() and same(d.results(), first)


def test_solves_of_several_streams_and_threads():
    work = [Device(M.rk4(0.02), 3000, 8.0, 1, points=9), Device(M.dopri5(), 7000, 8.0, 2),
            Device(M.dop853(), 2000, 8.0, 3), Device(M.dopri5(), 500, 8.0, 4, points=5)]
    streams = [torch.cuda.Stream() for _ in work]
    alone = []
    for d, s in zip(work, streams):
        d.solve(s)
        s.synchronize()
        alone.append(d.results())
    for _ in range(3):
        for d in work:
            for v in d.out.values():
                v.fill_(-7)
        torch.cuda.synchronize()
        errors = []

        def caller(d, s):
            try:
                for _ in range(4):
                    d.solve(s)
            except Exception as e:  # noqa: BLE001
                errors.append(e)

        threads = [threading.Thread(target=caller, args=a) for a in zip(work, streams)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        torch.cuda.synchronize()
        assert not errors, errors
        for d, want in zip(work, alone):
            assert same(d.results(), want)
