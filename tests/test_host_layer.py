"""The C++ host layer's own bookkeeping over a device in host memory (host_double.cpp): what a checkpoint owns, what is waited for,
what is recorded.  The layer's sources are compiled as they are, against the double in place of the HIP library."""
import concurrent.futures
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
HOST = os.path.join(ROOT, "strix-halo-vulkan_amd", "host")


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    d = tmp_path_factory.mktemp("host_double")
    flags = ["-O0", "-std=c++17", "-fPIC", "-I" + os.path.join(ROOT, "include"), "-I" + HOST]
    sources = [os.path.join(HOST, f) for f in ("llm.cpp", "gguf.cpp", "sample.cpp")] + [os.path.join(HERE, "host_double.cpp")]

    def compiled(src):
        obj = str(d / (os.path.basename(src) + ".o"))
        subprocess.check_call([os.environ.get("CXX", "g++")] + flags + ["-c", src, "-o", obj])
        return obj

    with concurrent.futures.ThreadPoolExecutor(4) as ex:
        objs = list(ex.map(compiled, sources))
    lib = str(d / "libhost_double.so")
    subprocess.check_call([os.environ.get("CXX", "g++"), "-shared", "-o", lib] + objs)
    return ctypes.CDLL(lib)


def test_a_copied_checkpoint_keeps_what_it_held(host):
    assert host.double_copied_checkpoint() == 1


def test_a_checkpoint_taken_again_uses_its_memory_again(host):
    assert host.double_own_checkpoint_again() == 1


def test_a_checkpoint_another_graph_restores_is_read_to_the_end_and_not_written(host):
    assert host.double_restored_elsewhere() == 1


def test_a_checkpoint_that_outlives_its_model_keeps_its_carry_alone(host):
    assert host.double_checkpoint_outlives_its_model() == 0


@pytest.mark.parametrize("free_mb,on_device", [(8000, 1), (1100, 1), (1023, 0), (0, 0)])
def test_a_checkpoint_leaves_a_sixteenth_of_the_device_free(host, free_mb, on_device):
    assert host.double_checkpoint_where_free(free_mb) == on_device


def test_cells_of_a_prompt_are_recorded_for_the_counts_that_come_again(host):
    # one to four rows (what the head was staged for) and a full chunk of 64, whatever the prompts' lengths
    assert host.double_recordings_for_cells() == 5
