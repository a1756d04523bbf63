"""What the engine's host side launches and allocates, on a runtime of imaginary GPUs (fake_hip.cpp): kernels do nothing
there, so a call that waits for a kernel's result reports a runtime error, unless the runtime is told to answer for it.  Each check runs in a process of its own."""
import ctypes
import os
import re
import subprocess
import sys
import time

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
i64, f64, p = ctypes.c_int64, ctypes.c_double, ctypes.byref


class Engine:
    def __init__(self, fake_path, lib_path):
        self.fake = ctypes.CDLL(fake_path, mode=ctypes.RTLD_GLOBAL)
        self.fake.fake_launches.restype = ctypes.c_char_p
        self.fake.fake_held.restype = ctypes.c_size_t
        self.fake.fake_limit.argtypes = [ctypes.c_size_t]
        self.L = ctypes.CDLL(lib_path)

    def context(self):
        h = ctypes.c_void_p()
        assert self.L.spamm_create(p(h), 0) == 0
        return h

    def launches(self):
        """(kernel, workgroups) of each launch since the last look."""
        out = []
        for item in self.fake.fake_launches().decode().split(";")[:-1]:
            name, grid = item.rsplit(" ", 1)
            length, rest = re.match(r"_ZN5spamm(\d+)(\w+)", name).groups()
            out.append((rest[:int(length)], int(grid)))
        return out


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    lib = os.path.join(ROOT, "cuspamm_amd", "libspamm_gfx950.so")
    if not os.path.exists(lib):
        pytest.fail("the engine has not been built")
    fake = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "fake_hip.cpp"), "-o", fake], check=True)

    def run(check, *args):
        done = subprocess.run([sys.executable, os.path.abspath(__file__), fake, lib, check] + [str(a) for a in args], text=True,
                              stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=120)
        assert done.returncode == 0 and done.stdout.strip().endswith("ok"), done.stdout[-3000:]
    return run


def counters_of_the_tau_passes(e, nbM, nbK, nbN):
    h = e.context()
    maps = ctypes.create_string_buffer(4 * max(nbM, nbN) * nbK)
    assert e.L.spamm_set_normmaps(h, maps, maps, i64(nbM), i64(nbK), i64(nbN), 32) == 0
    out = ctypes.c_float()
    e.launches()
    assert e.L.spamm_tau_for_ratio(h, f64(0.5), p(out), None) == -3
    assert e.L.spamm_tune_bisect(h, f64(0.5), f64(0.01), 20, p(out), None) == -3
    seen = set()
    for name, grid in e.launches():
        jb = {"k_tau_hist": 16, "k_tau_tree": 4}.get(name)
        if jb:
            seen.add(name)
            units = nbM * -(-nbN // jb) * -(-nbK // 64)                     # of jb columns and 64 k, dealt to waves in turn
            share = -(-units // (16 * grid)) * 16 * jb * 64
            assert share < 2 ** 32, "%s: %d workgroups of up to %d products" % (name, grid, share)
            assert nbM * nbK * nbN > 2 ** 38 or grid <= 256
    assert seen == {"k_tau_hist", "k_tau_tree"}


# the most products of two norm maps of half a gigabyte or less, and sizes that a multiply has
@pytest.mark.parametrize("shape", [(65535, 1025, 65535), (65535, 1, 65535), (1024, 512, 1024), (64, 33, 64)])
def test_a_workgroup_counts_less_than_32_bits_hold(run, shape):
    """Products that fall into one bin or leaf together -- equal norms -- must not pass its 32-bit counter."""
    run("counters_of_the_tau_passes", *shape)


def resident_operands(e, h, M, K, N, tile):
    X = ctypes.create_string_buffer(16)                                     # (nothing reads them)
    assert e.L.spamm_normmap_f32(h, 1, X, i64(K), i64(N), tile) == 0
    assert e.L.spamm_normmap_f32(h, 0, X, i64(M), i64(K), tile) == 0


def workgroups_of_the_report(e, M, K, N):
    h = e.context()
    resident_operands(e, h, M, K, N, 64)
    out = (ctypes.c_double * 3)()
    e.launches()
    e.L.spamm_error_vs_dense_f64(h, ctypes.create_string_buffer(16), i64(0), i64(M), out)
    grid = dict(e.launches())["k_error_limbs"]
    blocks = (M // 64) * (N // 64)
    # whole groups of at most 8 x 8, no wider than C: less than twice the blocks in the narrower direction's last
    # group, and one round of groups over the XCDs
    assert blocks <= grid <= 2 * blocks + 8 * 64, "%d workgroups for %d blocks" % (grid, blocks)


@pytest.mark.parametrize("shape", [(65536, 1024, 128), (128, 1024, 65536), (16384, 512, 512), (512, 512, 16384), (4096, 512, 512),
                                   (4096, 4096, 4096), (576, 1024, 14592), (1088, 512, 4160), (832, 832, 832)])
def test_the_report_has_a_workgroup_per_block_of_c(run, shape):
    """Of 64 x 64: also where C is narrow, which takes no more of them than the same C the other way round."""
    run("workgroups_of_the_report", *shape)


def product_of_the_report(e, M, K, N, whole):
    h = e.context()
    resident_operands(e, h, M, K, N, 64)
    e.launches()
    e.L.spamm_error_vs_dense_f64(h, ctypes.create_string_buffer(16), i64(0), i64(M), (ctypes.c_double * 3)())
    assert ("k_limbs" in dict(e.launches())) == bool(whole)


@pytest.mark.parametrize("shape", [(1048576, 64, 64), (4096, 64, 4096), (4096, 192, 4096), (65536, 1024, 64), (64, 4096, 131072), (65536, 2048, 128), (512, 256, 512)])
def test_reports_that_the_split_would_make_longer_are_left_in_fp64(run, shape):
    run("product_of_the_report", *shape, 0)


@pytest.mark.parametrize("shape", [(4096, 256, 4096), (512, 512, 512), (1024, 1024, 1024), (64, 4096, 4096), (16384, 512, 512), (4096, 4096, 4096)])
def test_reports_in_whole_numbers(run, shape):
    run("product_of_the_report", *shape, 1)


MIB = 1 << 20


def report(e, h, M):
    e.fake.fake_answer(b"k_error_limbs", 19, 20)
    e.fake.fake_answer(b"k_error_dense", 11, 12)
    e.launches()
    assert e.L.spamm_error_vs_dense_f64(h, ctypes.create_string_buffer(16), i64(0), i64(M), (ctypes.c_double * 3)()) == 0
    return [name for name, _ in e.launches()]


def memory_after_a_report(e, n):
    h = e.context()
    resident_operands(e, h, n, n, n, 64)
    before = e.fake.fake_held()
    assert "k_limbs" in report(e, h, n)
    assert e.fake.fake_held() - before <= 513 * MIB, "%d MiB more than before" % ((e.fake.fake_held() - before) // MIB)


@pytest.mark.parametrize("n", [2048, 8192, 8256, 16384])
def test_a_report_gives_its_scratch_back(run, n):
    run("memory_after_a_report", n)


def multiply_on_a_full_card(e):
    h = e.context()
    resident_operands(e, h, 4096, 4096, 4096, 64)
    e.fake.fake_limit(e.fake.fake_held() + 130 * MIB)
    assert "k_limbs" in report(e, h, 4096)                                  # 128 MiB of scratch, which stay
    X = ctypes.create_string_buffer(16)
    assert e.L.spamm_normmap_f32(h, 1, X, i64(4096), i64(8192), 64) == 0    # needs 64 MiB in the place of 32
    assert e.L.spamm_last_hip_error(h) == 0


def test_scratch_of_a_report_goes_when_a_multiply_finds_no_memory(run):
    run("multiply_on_a_full_card")


def report_on_a_full_card(e):
    h = e.context()
    resident_operands(e, h, 4096, 4096, 4096, 64)
    e.fake.fake_limit(e.fake.fake_held() + MIB)
    assert report(e, h, 4096)[-1] == "k_error_dense"
    assert e.L.spamm_last_hip_error(h) == 0


def test_a_report_without_memory_for_its_scratch_leaves_no_error(run):
    run("report_on_a_full_card")


class Params(ctypes.Structure):
    _fields_ = [("M", i64), ("K", i64), ("N", i64), ("tile", ctypes.c_int32), ("tau", ctypes.c_float), ("flags", ctypes.c_uint32),
                ("reserved", ctypes.c_uint32)]


def multiply_on_a_partition(e, cus):
    e.fake.fake_cus(cus)
    h = e.context()
    X = ctypes.create_string_buffer(16)

    def kernels(eighths, K, tau):
        """Of a C with so many eighths of a unit of 128 x 128 per CU."""
        M, N = 128 * eighths, 128 * (cus // 8)
        e.launches()
        assert e.L.spamm_multiply(h, p(Params(M, K, N, 64, tau, 0, 0)), X, X, X) == 0
        return [name for name, _ in e.launches() if name in ("k_small", "k_small_three", "k_gate", "k_gemm")]

    for tau, most in ((0.5, 48), (0.0, 16)):
        assert kernels(2, 2048, tau) == ["k_small"] and kernels(16, 2048, tau) == ["k_small"]
        if tau:
            assert kernels(20, 2048, tau) == ["k_small_three"] and kernels(24, 16384, tau) == ["k_small_three"]
            assert "k_gate" in kernels(32, 16384, tau) and "k_gate" in kernels(60, 2048, tau)
            for eighths in (27, 32):                # the one round that macro tiles fill: K up to 8192, on either side of it any
                assert kernels(eighths, 8192, tau) == ["k_small_three"]
                assert kernels(eighths, 8256, tau) == ["k_gate", "k_gemm"] and kernels(eighths, 65536, tau) == ["k_gate", "k_gemm"]
            assert kernels(26, 8256, tau) == ["k_small_three"] and kernels(33, 8256, tau) == ["k_small_three"]
        assert "k_gate" in kernels(most + 2, 2048, tau)
        assert ("k_gate" in kernels(most, 2048, tau)) is False


def stages_on_a_partition(e, cus):
    e.fake.fake_cus(cus)
    h = e.context()
    X = ctypes.create_string_buffer(16)

    def kernels(eighths, K, tile, tau=0.5):
        resident_operands(e, h, 128 * eighths, K, 128 * (cus // 8), tile)
        e.launches()
        assert e.L.spamm_gate(h, ctypes.c_float(tau)) == 0 and e.L.spamm_gemm_gated(h, X) == 0
        return [name for name, _ in e.launches() if name in ("k_small", "k_small_three", "k_gate", "k_gemm")]

    apart = ["k_gate", "k_gemm"]
    assert kernels(16, 65536, 64) == ["k_small"] * 2 and kernels(16, 2048, 32, 0.0) == ["k_small"] * 2 and kernels(17, 2048, 32, 0.0) == apart
    for eighths, K, tile in ((26, 8256, 64), (33, 8256, 64), (37, 2048, 32)):          # up to 832 and from 1025 to 1200 units: any K
        assert kernels(eighths, K, tile) == ["k_small_three"] * 2
    assert kernels(38, 2048, 32) == apart
    for eighths in (27, 32):                                                           # the round that macro tiles fill: 64 k tiles, K = 4096
        for K, tile in ((2048, 32), (4096, 64), (4096, 128)):
            assert kernels(eighths, K, tile) == ["k_small_three"] * 2 and kernels(eighths, K + tile, tile) == apart
        assert kernels(eighths, 8192, 128) == apart and kernels(eighths, 65536, 128) == apart


@pytest.mark.parametrize("cus", [256, 128, 64, 32])
def test_lines_of_the_stages_by_the_small_kernel(run, cus):
    """Gate and multiply called apart: the one-launch kernel runs twice, so its lines lie elsewhere than a multiply's."""
    run("stages_on_a_partition", cus)


@pytest.mark.parametrize("cus", [256, 128, 64, 32])
def test_lines_of_the_small_kernel_are_by_work_per_cu(run, cus):
    """A partition of an XCD or a few has its lines where a CU has as much to do as on the whole chip."""
    run("multiply_on_a_partition", cus)


def passes_over_halves(e, tile, n):
    h = e.context()
    memory = ctypes.create_string_buffer(64)
    start = -(-ctypes.addressof(memory) // 16) * 16

    def kernels(call, *args):
        e.launches()
        assert call(h, *args) == 0
        return [name for name, _ in e.launches() if name.startswith("k_normmap")]

    C = ctypes.c_void_p(start)
    for a in range(0, 16, 2):
        A = ctypes.c_void_p(start + a)
        passes = kernels(e.L.spamm_normmap_f16, 0, A, i64(n), i64(n), tile) + kernels(e.L.spamm_normmap_f16, 1, A, i64(n), i64(n), tile)
        square = kernels(e.L.spamm_multiply_f16, p(Params(n, n, n, tile, 0.5, 1, 0)), A, A, C)
        assert passes and square
        for name in passes + square:
            assert a % 4 == 0 or "lean" not in name, (name, a)
        if n * n * 2 <= 32 * MIB:
            assert a % 4 or all("lean" in name for name in passes)
        for b in range(0, 16, 2):
            pair = kernels(e.L.spamm_multiply_f16, p(Params(n, n, n, tile, 0.5, 0, 0)), A, ctypes.c_void_p(start + b), C)
            assert len(pair) == 1
            assert (a % 4 == 0 and b % 4 == 0) or "lean" not in pair[0], (pair, a, b)
            if 2 * n * n * 2 <= 32 * MIB:
                assert a % 4 or b % 4 or "lean" in pair[0]


@pytest.mark.parametrize("n", [256, 1024, 5120])
@pytest.mark.parametrize("tile", [32, 64, 128])
def test_halves_between_two_words_are_not_read_by_buffer_loads(run, tile, n):
    """Buffer loads are of whole 32-bit words: passes that read their input by them take no matrix of halves that begins at an odd half."""
    run("passes_over_halves", tile, n)


def forms_of_the_one_launch_kernel(e, tile):
    h = e.context()
    X = ctypes.create_string_buffer(16)
    for M, N, name, unit in ((1024, 1024, "k_small", 64), (2048, 2048, "k_small", 128), (3072, 3584, "k_small_three", 128)):
        for k_tiles in (1, 63, 64, 65, 128):
            e.launches()
            assert e.L.spamm_multiply(h, p(Params(M, k_tiles * tile, N, tile, 0.5, 0, 0)), X, X, X) == 0
            full = [item.rsplit(" ", 1)[0] for item in e.fake.fake_launches().decode().split(";")[:-1] if "k_small" in item]
            sizes = "ILi%dELi%dE" % (tile, unit)
            word = "_ZN5spamm%d%sENS_8WordArgs%sEE" % (len(name), name, sizes)
            general = "_ZN5spamm%d%s%s" % (len(name), name, sizes if unit == 64 or name == "k_small" else "ILi%dE" % tile)
            assert len(full) == 1 and full[0].startswith(word if k_tiles <= 64 else general), (full, k_tiles)


@pytest.mark.parametrize("tile", [32, 64, 128])
def test_the_list_is_a_register_up_to_one_word_of_k_tiles(run, tile):
    """Both forms of the one-launch kernel go by one name and give the same bits: which of them ran shows in its arguments."""
    run("forms_of_the_one_launch_kernel", tile)


def forms_of_the_gate(e, nbM, nbK, nbN, tile, chunks, few):
    h = e.context()
    maps = ctypes.create_string_buffer(4 * max(nbM, nbN) * nbK)
    assert e.L.spamm_set_normmaps(h, maps, maps, i64(nbM), i64(nbK), i64(nbN), tile) == 0
    e.launches()
    assert e.L.spamm_gate(h, ctypes.c_float(0.5)) == 0
    assert [name for name, _ in e.launches()] == ["k_gate_chunks" if chunks else "k_gate", "k_order_few" if few else "k_order"]


@pytest.mark.parametrize("shape", [(512, 1, 16, 128, 0, 1), (513, 1, 16, 128, 0, 0), (16, 1, 1024, 128, 0, 0), (2048, 2, 64, 32, 0, 1), (2049, 2, 64, 32, 0, 0),
                                   (8, 19392, 8, 32, 0, 1), (8, 19393, 8, 32, 1, 1), (4, 65535, 4, 64, 0, 1), (2, 65535, 2, 128, 0, 1)])
def test_lines_of_gate_and_schedule(run, shape):
    """64 super tiles of C are a wave's lanes; a macro tile's sets of k fill a CU's LDS up to 19392 k tiles of 32, and fit at the others."""
    run("forms_of_the_gate", *shape)


def time_looked_for_a_result(e):
    h = e.context()
    maps = ctypes.create_string_buffer(4 * 64 * 64)
    assert e.L.spamm_set_normmaps(h, maps, maps, i64(64), i64(64), i64(64), 32) == 0
    times = []
    for _ in range(20):
        start = time.perf_counter()
        assert e.L.spamm_count_kept(h, f64(0.5), p(i64()), p(f64())) == -3               # (no kernel writes it: the runtime says the stream has ended)
        times.append(time.perf_counter() - start)
    assert min(times) >= 100e-6, "%.1f us" % (min(times) * 1e6)


def test_a_result_is_looked_for_some_100_us_before_the_stream_is_asked(run):
    """Whatever the core: asking the stream costs 6 us more, and most calls that wait have their result after 10 to 60."""
    run("time_looked_for_a_result")


if __name__ == "__main__":
    globals()[sys.argv[3]](Engine(*sys.argv[1:3]), *map(int, sys.argv[4:]))
    print("ok")
