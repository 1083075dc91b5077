"""The host side of the launches that are more than one kernel, on the CPU: tests/host/launch_order.cpp
stands in for the HIP runtime and follows whose data each workspace holds."""
import subprocess
from pathlib import Path

import pytest

HOST = Path(__file__).resolve().parent / "host"


@pytest.fixture(scope="module")
def program(mi, tmp_path_factory):
    exe = tmp_path_factory.mktemp("launch_order") / "launch_order"
    lib = mi._lib.LIB_PATH
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-pthread", str(HOST / "launch_order.cpp"), "-o", str(exe),
                    str(lib), f"-Wl,-rpath,{lib.parent}", "-Wl,-rpath,/opt/rocm/lib", "-Wl,--export-dynamic",
                    "-Wl,--allow-shlib-undefined"], check=True)
    return exe


def run(program, scenario):
    r = subprocess.run([str(program), scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    return r.stdout


@pytest.mark.parametrize("source", ["library", "caller", "static"])
def test_calls_from_several_threads_on_one_stream_keep_their_operands(program, source):
    run(program, "one_stream_" + source)


@pytest.mark.parametrize("other", ["takeover", "takeover_larger", "release_all", "release_one", "table_busy"])
def test_a_workspace_stays_with_a_call_that_is_between_two_launches(program, other):
    run(program, other)


def test_per_thread_streams_do_not_share_a_workspace(program):
    run(program, "per_thread_stream")


def test_a_caller_workspace_on_any_16_byte_boundary_takes_the_copy(program):
    run(program, "caller_alignment")


def test_memory_held_for_copies_is_bounded_and_a_failed_allocation_is_remembered(program):
    run(program, "copy_memory")


def test_a_trace_buffer_has_room_for_every_call_of_its_shape(program):
    run(program, "trace_room")


def test_which_of_its_kernels_a_config_runs(program):
    """A config's deep-ring kernel takes the calls on 16-byte boundaries; 4 bytes off them its own kernel runs (that of
    DEEP_TWIN where it has none)."""
    from h100_gemm_amd import kernel_configs as kc
    ran = {(name, int(a)): kernel for name, a, kernel in (line.split() for line in run(program, "which_kernel").splitlines())}
    deep = [c for c in kc.CONFIGS if c.get("DEEP")]
    assert len(ran) == 2 * len(kc.CONFIGS) and len(deep) == 13
    for c in kc.CONFIGS:
        name = kc.config_name(c)
        assert ("gemm_deep_kernel" in ran[name, 0]) == bool(c.get("DEEP")), name
        if c.get("DEEP"):
            own = ("gemm_mfma16_kernel" if c["KIND"] == "mfma16" else
                   "gemm_shared_ring_kernel" if c.get("SHARED") else "gemm_wavek_kernel")
            assert own in ran[name, 4], (name, ran[name, 4])
