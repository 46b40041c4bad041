"""The library's host code without a GPU: streams, captures and the choice of
kernels, over a pretended HIP runtime (tests/fake_hip.cpp) that writes the
calls down. Everything here runs on the CPU."""
import os
import shutil
import subprocess

import pytest

import orc

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    if not shutil.which("g++") or not os.path.exists(os.path.join(ROCM, "include", "hip", "hip_runtime_api.h")):
        pytest.skip("no compiler or no HIP headers")
    exe = str(tmp_path_factory.mktemp("fake") / "fake_hip")
    lib = os.path.dirname(orc.HIP_LIB)
    subprocess.run(["g++", "-std=c++17", "-O1", "-rdynamic", "-I", os.path.join(ROCM, "include"),
                    os.path.join(ROOT, "tests", "fake_hip.cpp"), "-o", exe, "-L", lib, "-lorc_hip",
                    f"-Wl,-rpath,{lib}", "-Wl,--allow-shlib-undefined", "-ldl", "-lpthread"], check=True)

    def run(*args):
        r = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stderr
        return r.stdout.splitlines()

    return run


@pytest.mark.parametrize("how", ["race", "race_hip"])
def test_a_capture_begun_by_another_thread_pulls_no_stream_in(fake, how):
    """A thread begins capturing the stream that used the prefill workspace
    last, just as a call on another stream takes the workspace over."""
    fake(how)


def test_workspace_order_around_a_capture(fake):
    fake("order")


def test_init_without_memory_for_the_workspace(fake):
    fake("no_memory")


Q4_K, Q6_K, Q8_0, Q4_0, F16 = 12, 14, 8, 2, 1


@pytest.mark.parametrize("call,prefill", [
    ((Q6_K, 32, 2048, 2048), False), ((Q6_K, 48, 2048, 2048), True), ((Q4_K, 64, 896, 1024), False),
    ((Q4_K, 128, 896, 1024), True), ((Q6_K, 128, 512, 512), False), ((Q6_K, 256, 512, 512), True),
    ((Q4_0, 24, 64, 8192), True), ((F16, 40, 64, 1024), False), ((F16, 48, 64, 1024), True),
    ((Q8_0, 24, 2048, 2048), True), ((Q4_K, 127, 3072, 3072), True), ((Q6_K, 23, 3072, 3072), False)])
def test_small_prompt_calls_take_the_faster_kernels(fake, call, prefill):
    """Both sides of the line between the verify and the prefill kernels."""
    got = any("k_pf" in line for line in fake("gemm", *call))
    assert got == prefill


def test_the_prefill_kernels_tests_reach_them(fake):
    """Cases of the GPU tests that are there for the prefill kernels."""
    import test_gpu_prefill as t

    for qt, nt, n_out, n_in in t.K_CASES + [c for c in t.CASES if c[0] in (Q8_0, Q4_0)]:
        assert any("k_pfI" in line for line in fake("gemm", qt, nt, n_out, n_in)), (qt, nt, n_out, n_in)


@pytest.mark.parametrize("call,split", [
    ((8, 8, 64, 64, 0), False), ((8, 8, 64, 128, 0), False), ((8, 8, 64, 129, 0), True), ((16, 8, 64, 64, 0), False),
    ((16, 8, 64, 65, 0), True), ((32, 8, 64, 8, 56), False), ((32, 8, 64, 9, 50), True), ((14, 2, 64, 4, 0), True),
    ((8, 8, 128, 64, 192), False), ((8, 8, 128, 64, 193), True), ((32, 32, 128, 64, 384), False),
    ((32, 32, 128, 129, 0), True), ((16, 8, 128, 8, 100), False), ((16, 8, 128, 16, 100), True),
    ((24, 8, 128, 8, 50), False), ((24, 8, 128, 24, 0), True), ((28, 4, 128, 1, 0), True)])
def test_short_contexts_take_the_faster_attention(fake, call, split):
    """heads, kv heads, head_dim, tokens, position: both sides of the line."""
    assert any("k_kv_split" in line for line in fake("attn", *call)) == split


@pytest.mark.parametrize("call,ranges", [((F16, 300, 128256, 8192), 2), ((F16, 3000, 128256, 8192), 2),
                                         ((30, 200, 128256, 12288), 3), ((F16, 300, 400000, 8192), 2),
                                         ((F16, 300, 700000, 8192), 0)])
def test_tall_dense_matrices_keep_their_ranges(fake, call, ranges):
    """An F16 or BF16 row is summed in ranges of at most 4096 values however
    much of the workspace their sums take: in chunks of fewer tokens, or (64
    tokens do not fit) by the kernels that need no workspace."""
    got = [int(line.split()[2].split("x")[2]) for line in fake("gemm", *call) if "4k_pfI" in line]
    assert len(got) > 0 if ranges else not got
    assert all(z >= ranges for z in got), got


@pytest.mark.parametrize("call", [(Q8_0, 24, 65535 * 128, 32), (Q8_0, 24, 65535 * 128 + 1, 32), (F16, 300, 9000000, 64),
                                  (Q4_K, 40, 8400000, 256)])
def test_any_number_of_rows_is_taken(fake, call):
    fake("gemm", *call)


def test_the_workspace_holds_32_k_positions(fake):
    """The last pass of a 32768-position prompt of eight 128-wide kv heads, and
    its key ranges over few rows."""
    for call in ((32, 8, 128, 1024, 31744), (32, 8, 128, 40, 32728), (64, 8, 128, 1, 32767)):
        got = fake("attn", *call)
        assert any("k_kv_split" in line for line in got), call
    assert any("k_attn_fa_sum" in line for line in got)


def test_bytes_of_timed_attention_calls(fake):
    fake("prof_bytes")


def test_no_exception_leaves_a_c_entry_point(fake):
    fake("no_host_memory")
