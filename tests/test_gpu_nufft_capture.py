"""F^H d and F captured into a graph after calls of the same size that took the
separable form: the capture takes the direct sums and finds their workspaces
allocated."""
import ctypes as C

import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_nufft import DIRECT_TOL, _problem

pytestmark = pytest.mark.gpu

CAPTURE_THREAD_LOCAL = 1


def _hip(name, *args):
    """A HIP runtime call, in the runtime that the library is linked against."""
    from impatient import _lib
    st = getattr(_lib.load(), name)(*args)
    assert st == 0, f"{name}: {st}"


@pytest.mark.parametrize("op,nc", [("adjoint", 1), ("adjoint", 2), ("adjoint", 5),
                                   ("adjoint", 32), ("forward", 1), ("forward", 2),
                                   ("forward", 5), ("forward", 17)])
def test_capture_after_a_separable_call(ctx, op, nc):
    """Three replays with the program's own (separable) calls between them, each
    against the separable result before it, on inputs changed in between."""
    from impatient import Context
    from impatient._lib import call, ptr
    N, M = 256, 60000
    p = _problem(N, N, nc, M)
    n = N * N
    r = np.random.default_rng(4)
    own = Context(0)   # its workspaces are what the calls here made
    try:
        def up(v):
            return own.to_device(np.ascontiguousarray(v, np.float32).reshape(-1))
        g = [up(p[k]) for k in ("kx", "ky", "t", "x", "y", "fm")]
        s = [up(p["s"].real), up(p["s"].imag)]
        ni, no = (nc * M, n) if op == "adjoint" else (n, nc * M)
        src = [up(r.standard_normal(ni)) for _ in range(2)]
        out = [own.alloc((no,)) for _ in range(2)]
        opt = [None, None] if op == "adjoint" else []   # phi

        def run():
            call("imp_nudft_" + op, own.h, C.c_int(M), C.c_int(n), C.c_int(nc), ptr(g[0]),
                 ptr(g[1]), None, ptr(g[2]), ptr(g[3]), ptr(g[4]), None, ptr(g[5]), *opt,
                 ptr(src[0]), ptr(src[1]), ptr(s[0]), ptr(s[1]), ptr(out[0]), ptr(out[1]))

        def result():
            own.synchronize()
            v = out[0].get() + 1j * out[1].get()
            for o in out:   # so that a replay which writes nothing is seen
                o.zero()
            return v

        def records():
            tot, k = C.c_double(), C.c_int()
            call("imp_profile_read", own.h, b"nufft_" + op.encode(), C.byref(tot), C.byref(k))
            return k.value
        call("imp_profile_enable", own.h, C.c_int(1))
        call("imp_profile_reset", own.h)
        run()
        want = result()
        assert records() == 1
        call("imp_profile_enable", own.h, C.c_int(0))
        st = C.c_void_p(own.stream())
        graph, ex = C.c_void_p(), C.c_void_p()
        _hip("hipStreamBeginCapture", st, C.c_int(CAPTURE_THREAD_LOCAL))
        try:
            run()
        finally:
            _hip("hipStreamEndCapture", st, C.byref(graph))
        _hip("hipGraphInstantiate", C.byref(ex), graph, None, None, C.c_size_t(0))
        for i in range(3):
            _hip("hipGraphLaunch", ex, st)
            got = result()
            assert rel_l2(got, want) < DIRECT_TOL
            _hip("hipGraphLaunch", ex, st)
            assert np.array_equal(got, result())
            src[0].upload(r.standard_normal(ni))
            run()
            want = result()
        _hip("hipGraphExecDestroy", ex)
        _hip("hipGraphDestroy", graph)
    finally:
        own.close()
