"""Every entry point works on its context's GPU whatever device the calling thread has current: allocations,
launches, events.  The engine's host side runs here on a runtime of two imaginary GPUs (fake_hip.cpp), in a process
of its own; kernels do nothing there, so calls that wait for a kernel's result report a runtime error."""
import ctypes
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
A_EQ_B, TIMING, REUSE_A, REUSE_B, PRUNE = 1, 2, 4, 8, 16


class Params(ctypes.Structure):
    _fields_ = [("M", ctypes.c_int64), ("K", ctypes.c_int64), ("N", ctypes.c_int64), ("tile", ctypes.c_int32),
                ("tau", ctypes.c_float), ("flags", ctypes.c_uint32), ("reserved", ctypes.c_uint32)]


def _child(fake_path, lib_path):
    fake = ctypes.CDLL(fake_path, mode=ctypes.RTLD_GLOBAL)
    fake.fake_wrong.restype = ctypes.c_char_p
    L = ctypes.CDLL(lib_path)
    n, tile, nb = 256, 32, 8
    X = ctypes.create_string_buffer(4 * n * n)          # stands for device and host memory alike
    out = ctypes.create_string_buffer(1 << 20)
    i64, f32, f64, p = ctypes.c_int64, ctypes.c_float, ctypes.c_double, ctypes.byref

    def context(device):
        fake.fake_expect(device)
        fake.fake_thread_device(1 - device)
        h = ctypes.c_void_p()
        assert L.spamm_create(p(h), device) == 0
        assert fake.fake_checked() and not fake.fake_wrong(), "create: %r" % fake.fake_wrong()
        return h

    def call(h, device, name, *args, works=True, rc=0):
        fake.fake_expect(device)
        fake.fake_thread_device(1 - device)
        got = getattr(L, name)(h, *args)
        assert got == rc, (name, got)
        assert not works or fake.fake_checked(), "%s did nothing that could be checked" % name
        assert not fake.fake_wrong(), "%s on device %d: %r" % (name, device, fake.fake_wrong())

    for device in (0, 1):
        for shape in (0, 1):                            # a small C by the kernel of its own, and by gate and GEMM
            # operands converted stage by stage, then a call that finds both resident: every buffer of gate and
            # multiply is new to the context.  A further context per form
            for flags in (REUSE_A | REUSE_B, REUSE_A | REUSE_B | TIMING, REUSE_A, REUSE_B | TIMING, REUSE_B | PRUNE, 0, TIMING, PRUNE,
                          A_EQ_B, A_EQ_B | PRUNE | TIMING):
                h = context(device)
                assert L.spamm_set_option(h, 4, shape) == 0
                for role in (1, 0):
                    call(h, device, "spamm_normmap_f32", role, X, i64(n), i64(n), tile)
                for half in (False, True):
                    call(h, device, "spamm_multiply_f16" if half else "spamm_multiply", p(Params(n, n, n, tile, 0.5, flags, 0)), X, X, X)
                    if flags in (REUSE_B | PRUNE, PRUNE, A_EQ_B | PRUNE | TIMING):
                        break                           # (what a tau-aware call leaves is not for every reuse)
                L.spamm_destroy(h)
            h = context(device)
            assert L.spamm_set_option(h, 4, shape) == 0
            call(h, device, "spamm_multiply_noalloc", p(Params(n, n, n, tile, 0.5, 0, 0)), X, X, X)
            call(h, device, "spamm_set_normmaps", X, X, i64(nb), i64(nb), i64(nb), tile)
            call(h, device, "spamm_gate", f32(0.5))
            call(h, device, "spamm_normmap_f16", 1, X, i64(n), i64(n), tile)
            call(h, device, "spamm_normmap_f16", 0, X, i64(n), i64(n), tile)
            call(h, device, "spamm_gate", f32(0.5))
            call(h, device, "spamm_gemm_gated", X)
            call(h, device, "spamm_get_klist", out)
            call(h, device, "spamm_get_fp16", 0, out)
            call(h, device, "spamm_get_macro_counts", out, None, works=shape == 0)
            call(h, device, "spamm_dropped_bound_tiles", f32(0.5), out)
            call(h, device, "spamm_fill_decay_f32", X, i64(n), i64(n), X, ctypes.c_uint64(1), 1)
            call(h, device, "spamm_dropped_bound", f32(0.5), out, rc=-3)
            call(h, device, "spamm_error_vs_dense_f64", X, i64(0), i64(n), out, rc=-3)
            call(h, device, "spamm_count_kept", f64(0.5), out, None, rc=-3)
            call(h, device, "spamm_tau_for_ratio", f64(0.5), out, None, rc=-3)
            call(h, device, "spamm_tune_bisect", f64(0.5), f64(0.01), 20, out, None, rc=-3)
            L.spamm_destroy(h)
    print("ok")


def test_every_entry_point_works_on_its_contexts_device(tmp_path):
    lib = os.path.join(ROOT, "cuspamm_amd", "libspamm_gfx950.so")
    if not os.path.exists(lib):
        pytest.fail("the engine has not been built")
    fake = os.path.join(str(tmp_path), "fake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "fake_hip.cpp"), "-o", fake], check=True)
    run = subprocess.run([sys.executable, os.path.abspath(__file__), fake, lib], stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                         text=True, timeout=120)
    assert run.returncode == 0 and run.stdout.strip().endswith("ok"), run.stdout[-3000:]


if __name__ == "__main__":
    _child(*sys.argv[1:3])
