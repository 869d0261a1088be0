"""CPU tests of the device library's host code against a stand-in for the GPU
(fake_device.cpp): what an upload allocates and prepares, what it gives up when
memory runs out, how many threads copy."""
import os
import subprocess

import pytest

from hetegeneous_parallel_programming_amd import _native as nat

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP = os.path.join(ROOT, "hetegeneous_parallel_programming_amd", "csrc", "hip")


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    nat.host()  # libtc_host.so is built
    out = tmp_path_factory.mktemp("fake")
    flags = ["-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + os.path.join(ROOT, "include"),
             "-I" + HIP]
    sources = [os.path.join(HIP, f) for f in ("tc_runtime.cpp", "tc_copy.cpp", "tc_batch.cpp", "tc_server.cpp")]
    sources.append(os.path.join(ROOT, "tests", "fake_device.cpp"))
    jobs = [(subprocess.Popen(["g++", *flags, "-c", s, "-o", str(out / f"{i}.o")], stderr=subprocess.PIPE, text=True))
            for i, s in enumerate(sources)]
    for j in jobs:
        err = j.communicate(timeout=300)[1]
        assert j.returncode == 0, err
    lib = os.path.dirname(nat.HOST_LIB)
    exe = str(out / "fake_device")
    subprocess.run(["g++", *[str(out / f"{i}.o") for i in range(len(sources))], "-L" + lib, "-ltc_host",
                    "-Wl,-rpath," + lib, "-pthread", "-o", exe], check=True, capture_output=True, timeout=300)

    def run(*args):
        p = subprocess.run([exe, *args], capture_output=True, text=True, timeout=120)
        assert p.returncode == 0, p.stdout + p.stderr
        return p.stdout

    return run


def test_one_shot_calls_prepare_for_one_count(fake):
    fake("one_shot")


def test_codes_and_lines_take_no_memory_that_is_needed(fake):
    fake("memory")


def test_which_graphs_get_codes_and_lines(fake):
    fake("choice")


def test_a_plain_count_is_one_launch(fake):
    fake("plain")


def test_clients_share_the_copy_threads(fake):
    fake("clients")


def test_words_of_a_batch(fake):
    fake("batch_words")


def test_batches_with_many_light_rows(fake):
    fake("light")
