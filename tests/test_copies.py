"""The library's host <-> device copies against a runtime that carries every
one of them out as late as it may (tests/native/deferred_hip.cc, on the CPU):
what a copy reads must stay as it was until the wait that covers it. Each test
runs in a process of its own, with freed memory overwritten (MALLOC_PERTURB_)."""
import ctypes
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = os.path.join(ROOT, "tests", "native", "deferred_hip.cc")


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    so = str(tmp_path_factory.mktemp("hip") / "libdeferred_hip.so")
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC",
                        "-fvisibility=hidden", "-Wall", "-o", so, SOURCE],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    return so


def in_child(runtime, name, *args):
    """Runs child_<name> of this file on the deferred runtime."""
    r = subprocess.run(
        [sys.executable, os.path.abspath(__file__), runtime, name] +
        [str(a) for a in args], capture_output=True, text=True, timeout=300,
        cwd=ROOT, env=dict(os.environ, MALLOC_PERTURB_="165"))
    assert r.returncode == 0, r.stdout[-1000:] + r.stderr[-2000:]


@pytest.mark.parametrize("w,h,table_mb,dots,pad", [
    (8, 8, 0, 0, 0), (72, 40, 0, 9, 0), (72, 40, 0, 9, 1),
    (520, 264, 0, 40, 0), (520, 264, 0, 40, 3),
    (72, 40, 17, 0, 0), (72, 40, 17, 9, 0), (520, 264, 17, 40, 3)])
def test_sources_live_until_the_copies_are_done(runtime, w, h, table_mb, dots,
                                                pad):
    in_child(runtime, "upload", w, h, table_mb, dots, pad)


@pytest.mark.parametrize("w,h", [(72, 40), (520, 264)])
def test_sources_of_the_encoder_calls(runtime, w, h):
    in_child(runtime, "encoder", w, h)


# Memory that the runtime knows, as (first plane, planes) of five planes one
# behind the other, of which the library is given 1 to 3; the copies that it
# may take for them.
KNOWN = {"ordinary": (), "one": ((1, 3),), "inside": ((0, 5),),
         "apart": ((1, 1), (2, 1), (3, 1)), "first": ((1, 1), (2, 2)),
         "last": ((1, 2), (3, 1)), "behind": ((2, 2),)}
COPIES = {"ordinary": 1, "one": 1, "inside": 1, "apart": 3, "first": 3,
          "last": 3, "behind": 3}


@pytest.mark.parametrize("known", sorted(KNOWN))
def test_touching_planes(runtime, known):
    """Planes that touch go in one copy where they are one allocation, or none
    that the runtime knows, and else in a copy each."""
    in_child(runtime, "planes", sorted(KNOWN).index(known))


# --- in the child -----------------------------------------------------------

def large_table(fr, mb):
    """The frame with `mb` MB of dequant table (the tail is never addressed)."""
    import numpy as np
    table = np.ones((mb << 20) // 4, np.float32)
    table[:fr.dequant_table.size] = fr.dequant_table
    fr.dequant_table = table


def child_upload(hip, w, h, table_mb, dots, pad):
    """Uploads, a refused one between: nothing waits after either, and no
    source changed while it waited."""
    import numpy as np
    from pik_amd import synth
    from pik_amd.runtime import PikGpuError, Reconstructor
    fr = synth.make_frame(w, h, seed=w + h, num_dots=dots)
    assert len(fr.dots) == dots
    if table_mb:
        large_table(fr, table_mb)
    if pad:
        for name in ("ac", "dc", "quant_field", "ac_strategy"):
            a = getattr(fr, name)
            wide = np.zeros(a.shape[:-1] + (a.shape[-1] + pad,), a.dtype)
            wide[..., :a.shape[-1]] = a
            setattr(fr, name, wide[..., :a.shape[-1]])
    bad = fr.copy()
    bad.quant_field = bad.quant_field.copy()
    bad.quant_field[-1, -1] = 0
    with Reconstructor(0) as rec:
        for f, good in ((fr, True), (bad, False), (fr, True)):
            if good:
                rec.upload(f)
            else:
                with pytest.raises(PikGpuError):
                    rec.upload(f)
            assert hip.deferred_hip_waiting() == 0
            assert hip.deferred_hip_changed() == 0
    assert hip.deferred_hip_copies() > 0


def child_encoder(hip, w, h):
    """Quantizer, adjoint with host pointers and search: nothing waits when
    they return, and no source changed while it waited."""
    import numpy as np
    from pik_amd import synth
    from pik_amd.runtime import Reconstructor
    fr, op = synth.make_opsin_frame(w, h, seed=2, predict=False)
    target = np.zeros((3, h, w), np.float32)
    weight = np.ones(fr.quant_field.shape, np.float32)
    with Reconstructor(0) as rec:
        rec.upload(fr)
        for call in (lambda: rec.quantize(op),
                     lambda: rec.fwd_adj(fr.quant_field.astype(np.float32),
                                         target=target),
                     lambda: rec.search_quant_field(op, target, steps=2,
                                                    weight=weight)):
            before = hip.deferred_hip_copies()
            call()
            assert hip.deferred_hip_copies() > before
            assert hip.deferred_hip_waiting() == 0
            assert hip.deferred_hip_changed() == 0


def child_planes(hip, which):
    import numpy as np
    from pik_amd import abi, synth
    from pik_amd.runtime import Reconstructor
    known = sorted(KNOWN)[which]
    hip.deferred_hip_bytes.restype = ctypes.c_size_t
    hip.deferred_hip_range.argtypes = [ctypes.c_void_p, ctypes.c_size_t]
    hip.deferred_hip_forget.argtypes = [ctypes.c_void_p]

    def copies(call, at, plane):
        """Sizes in planes of the copies of `call` that are planes'."""
        for first, n in KNOWN[known]:
            hip.deferred_hip_range(at + first * plane, n * plane)
        k = hip.deferred_hip_copies()
        call()
        for first, n in KNOWN[known]:
            hip.deferred_hip_forget(at + first * plane)
        return [hip.deferred_hip_bytes(i) // plane
                for i in range(k, hip.deferred_hip_copies())
                if hip.deferred_hip_bytes(i) % plane == 0]

    want = [3] if COPIES[known] == 1 else [1, 1, 1]
    fr = synth.make_frame(520, 264, seed=1)  # AC above 256 KB: copies of it
    ac = np.zeros((5,) + fr.ac.shape[1:], np.int16)
    ac[1:4] = fr.ac
    fr.ac = ac[1:4]
    fc, keep = fr.to_c()
    with Reconstructor(0) as rec:
        def upload():
            rec._check(rec._lib.pikgpu_frame_upload(rec._ctx,
                                                    ctypes.byref(fc)))
        assert copies(upload, ac.ctypes.data, ac[0].nbytes) == want
        planes = (ctypes.c_void_p * 3)(*[a.ctypes.data for a in ac[1:4]])

        def add_pass():
            rec._check(rec._lib.pikgpu_frame_add_pass(
                rec._ctx, planes, ac.shape[2]))
        assert copies(add_pass, ac.ctypes.data, ac[0].nbytes) == want
        rec._check(rec._lib.pikgpu_run(rec._ctx, 0))
        out = np.full((5, 264, 520), 7, np.float32)
        to = (abi.c_float_p * 3)(
            *[a.ctypes.data_as(abi.c_float_p) for a in out[1:4]])

        def download():
            rec._check(rec._lib.pikgpu_download(rec._ctx, to, 520 * 4))
        assert copies(download, out.ctypes.data, out[0].nbytes) == want
        assert np.all(out[1:4] == 0) and np.all(out[::4] == 7)
    # only ordinary memory with an allocation behind it is tried and refused
    assert hip.deferred_hip_refused() == (3 if known == "behind" else 0)
    assert hip.deferred_hip_changed() == 0


if __name__ == "__main__":
    sys.path.insert(0, ROOT)
    HIP = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
    globals()["child_" + sys.argv[2]](HIP, *(int(a) for a in sys.argv[3:]))
