"""Maps and reductions without flags_out inside a stream capture, recorded
before any other call of their kind without flags (their kernels are compiled
by a call that reads its flags), and replayed with eager work and waits in
between; each replay equals the eager result.  A fresh child process, so the
captured call is the first that needs the words of unread flags."""
import os
import subprocess
import sys
import textwrap

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_first_call_without_flags_is_captured():
    code = """
        import ctypes as C
        import os
        import numpy as np
        import phase
        from test_gpu_alias_deep import _Desc, _desc

        class Insn(C.Structure):
            _fields_ = [(n, C.c_uint8) for n in ("op", "dt", "dst", "a", "b", "c")] + [("pad_", C.c_uint16), ("i", C.c_int64)]

        class Prog(C.Structure):
            _fields_ = [(n, C.c_int32) for n in ("n_insn", "n_in", "out_reg", "out_dtype")] + [("insn", Insn * 48)]

        def prog(n_in, out, *insns):
            p = Prog(len(insns), n_in, out, 0)
            for k, t in enumerate(insns):
                p.insn[k] = Insn(*t)
            return p

        phase.init(0)
        lib = C.CDLL(os.path.join(phase.LIB_DIR, "libphhip.so"))
        with open("/proc/self/maps") as f:
            hip = C.CDLL(next(m.split()[-1] for m in f if "libamdhip64.so" in m))
        n = 5000
        h = np.arange(n, dtype=np.int32)
        x, z = phase.NArray.from_numpy(h), phase.NArray.from_numpy(np.zeros(n, np.int32))
        s = phase.NArray.from_numpy(np.zeros(1))
        add = prog(1, 1, (0, 0, 0, 0), (3, 0, 1, 0, 0))   # r1 = x + x, checked
        load = prog(1, 0, (0, 0, 0, 0))
        d = _desc(0, n, [n])
        ins, zin = (C.c_void_p * 1)(x.device_ptr), (C.c_void_p * 1)(z.device_ptr)
        fl, z_ptr, s_ptr = C.c_int32(0), C.c_void_p(z.device_ptr), C.c_void_p(s.device_ptr)

        def both(flags):
            rc = lib.ph_map(C.byref(add), 1, ins, C.byref(d), z_ptr, C.byref(d), flags)
            return rc or lib.ph_reduce(C.byref(load), 1, zin, C.byref(d), -1, 1, 0, s_ptr, None, flags)

        assert both(C.byref(fl)) == 0 and fl.value == 0
        stream, graph, run = C.c_void_p(), C.c_void_p(), C.c_void_p()
        assert lib.ph_get_stream(C.byref(stream)) == 0
        print("capture", flush=True)
        assert hip.hipStreamBeginCapture(stream, 0) == 0
        rc = both(None)
        assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0 and rc == 0, rc
        assert hip.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
        host, total = np.zeros(n, np.int32), C.c_double()
        for k in range(4):
            src = (h * (k + 1) % 1000).astype(np.int32)
            assert lib.ph_h2d(C.c_void_p(x.device_ptr), C.c_void_p(src.ctypes.data), C.c_size_t(4 * n)) == 0
            assert hip.hipGraphLaunch(run, stream) == 0
            assert lib.ph_d2h(C.c_void_p(host.ctypes.data), z_ptr, C.c_size_t(4 * n)) == 0
            assert lib.ph_d2h(C.byref(total), s_ptr, C.c_size_t(8)) == 0
            assert np.array_equal(host, 2 * src) and total.value == 2.0 * src.sum(), k
            assert both(C.byref(fl)) == 0 and fl.value == 0
        print("replayed")
    """
    env = dict(os.environ)
    env["PYTHONPATH"] = os.pathsep.join([os.path.join(ROOT, "ph-core_amd"), os.path.join(ROOT, "tests"),
                                         env.get("PYTHONPATH", "")])
    r = subprocess.run([sys.executable, "-c", textwrap.dedent(code)], env=env, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "replayed" in r.stdout, r.stdout + r.stderr
