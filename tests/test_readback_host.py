"""The host half of the staged readback, on the CPU: the library's read_back
called in a child process in which a small stand-in for the HIP runtime is
loaded first, so that its allocations, copies and launches are seen (the
stand-in carries a launch out with memcpy, as the kernel would)."""
import os
import subprocess
import sys
import textwrap

import pytest

from vk_gltf_viewer_amd import _native as N

FAKE = r"""
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
typedef struct { uint32_t x, y, z; } dim3;
unsigned host_flags = 0;
int allocs = 0, frees = 0, copies = 0, launches = 0, busy = 0, news = 0, late = 0;
void* _Znwm(size_t n) { ++news; return malloc(n ? n : 1); }   /* operator new */
int hipHostMalloc(void** p, size_t n, unsigned flags) { ++allocs; host_flags = flags; return posix_memalign(p, 4096, n) ? 2 : 0; }
int hipHostFree(void* p) { ++frees; free(p); return 0; }
int hipPointerGetAttributes(void* a, const void* p) { (void)a; (void)p; return 1; }
int hipGetLastError(void) { return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* st) { (void)kind; (void)st; ++copies; late += busy; memcpy(d, s, n); return 0; }
int hipStreamSynchronize(void* st) { (void)st; busy = 0; return 0; }
int hipStreamQuery(void* st) { (void)st; return busy ? 600 : 0; }
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, void* st) { (void)g; (void)b; (void)sh; (void)st; return 0; }
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, void** st)
{
    dim3 one = { 1, 1, 1 };
    *g = one; *b = one; *sh = 0; *st = 0;
    return 0;
}
int hipLaunchKernel(const void* f, dim3 g, dim3 b, void** args, size_t sh, void* st)
{
    (void)f; (void)g; (void)b; (void)sh; (void)st;
    const uint8_t* src = *(const uint8_t**)args[0];
    uint8_t* stage = *(uint8_t**)args[1];
    size_t bytes = *(size_t*)args[2];
    uint32_t* flags = *(uint32_t**)args[3], epoch = *(uint32_t*)args[4];
    memcpy(stage, src, bytes);
    for (size_t p = 0; p * 16384 < bytes; ++p) flags[p] = epoch;
    ++launches;
    return 0;
}
"""

PROLOGUE = """
import ctypes as C, sys
import numpy as np
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
lib = C.CDLL(sys.argv[2])
read_back = lib._ZN4vkgv9read_backEPvPKvmP12ihipStream_t
read_back.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_void_p]
user = lib._ZN4vkgv14read_back_userEb
user.argtypes, user.restype = [C.c_bool], None
count = lambda name: C.c_int.in_dll(fake, name).value
def setv(name, v): C.c_int.in_dll(fake, name).value = v
buf = np.empty(9 * 2**20 + 64, np.uint8)
src = buf[-buf.ctypes.data % 16:][:9 * 2**20]
src[:] = np.random.default_rng(1).integers(0, 256, len(src), dtype=np.uint8)
def read(n, first=0):
    dst = np.zeros(n, np.uint8)
    assert read_back(dst.ctypes.data, src[first:].ctypes.data, n, None) == 0
    assert np.array_equal(dst, src[first:first + n]), n
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    d = tmp_path_factory.mktemp("fakehip")
    (d / "fake.c").write_text(FAKE)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", str(d / "fake.so"), str(d / "fake.c")], check=True)
    return str(d / "fake.so")


def child(fake, body):
    if not os.path.exists(N.HIP_LIB):
        pytest.skip("the device library is not built")
    r = subprocess.run([sys.executable, "-c", PROLOGUE + textwrap.dedent(body), fake, N.HIP_LIB], capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 0, r.stderr


def test_the_stage_is_coherent_memory(fake):
    """The host reads flags and pieces while the kernel that stores them runs."""
    child(fake, """
        user(True)
        read(4 * 2**20)
        assert count("allocs") == 1 and count("launches") == 2
        assert C.c_uint.in_dll(fake, "host_flags").value & 0x40000000, "hipHostMallocCoherent"
        user(False)
        assert count("frees") == 1
    """)


def test_small_reads_are_staged_only_behind_work(fake):
    """On an idle stream a plain copy is faster below 896 KB."""
    child(fake, """
        user(True)
        for n, busy, launches in ((262144, 0, 0), (917500, 0, 0), (917504, 0, 1), (262144, 1, 1), (262140, 1, 0)):
            setv("busy", busy)
            before = count("launches")
            read(n)
            assert count("launches") - before == launches, (n, busy)
        user(False)
    """)


def test_a_plain_copy_is_not_queued_behind_work(fake):
    """The runtime is slow at that; the stream is waited for first."""
    child(fake, """
        user(True)
        for n in (4, 4096, 65536, 262140):
            setv("busy", 1)
            read(n)
        assert count("copies") == 4 and count("late") == 0
        user(False)
    """)


def test_a_read_allocates_nothing_that_could_throw(fake):
    """No exception can leave the C entry points from here."""
    child(fake, """
        user(True)
        before = count("news")
        for _ in range(3):
            read(2**20)
        assert count("news") == before
        user(False)
    """)


def test_any_size_arrives_whole(fake):
    child(fake, """
        user(True)
        for n in (1, 4, 65540, 262140, 262144, 262148, 2**20 - 4, 2**20, 2**21, 2**21 + 4, 2**22 + 16388, 9 * 2**20):
            setv("busy", 1)
            read(n)
        before = count("launches")
        read(2**21 + 2)          # not whole words: the plain copy
        read(2**21, 8)           # a source off the 16-byte grid: the plain copy
        assert count("launches") == before
        user(False)
        assert count("frees") == count("allocs") == 1
    """)
