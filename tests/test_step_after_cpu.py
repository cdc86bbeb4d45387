"""What ``step_after_kernel`` writes, thread by thread on the CPU: the step inputs, words beside them not.  Which buffers it takes."""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest

STUBS = """
#include <stdint.h>
#include <stddef.h>
#define __device__
#define __global__
#define __forceinline__ inline
#define __shared__ static
#define __launch_bounds__(n)
struct uint4 { uint32_t x, y, z, w; };
static struct { int x; } threadIdx, blockIdx;
static int first_half;   // of the kernel, in front of its barrier; the second run does it again, to no effect, and goes on
#define __syncthreads() do { if (first_half) return; } while (0)
constexpr int kHd = 128;
inline int32_t from_host(const int32_t *p) { return *p; }
"""
RUN = """
extern "C" void run(const int32_t *from, int32_t *to, int words, const int32_t *drafted, int drafts, void *kv, int planes, int slots) {
    for (blockIdx.x = 0; blockIdx.x < kCommitGroups; ++blockIdx.x)
        for (first_half = 1; first_half >= 0; --first_half)
            for (threadIdx.x = 0; threadIdx.x < 256; ++threadIdx.x)
                step_after_kernel(from, to, words, drafted, drafts, (uint4 *)kv, planes, slots);
}
extern "C" int planes_ok(const void *kv, int n_layers, int n_kv, int slots) { return kv_planes_ok(kv, n_layers, n_kv, slots); }
"""


@pytest.fixture(scope="module")
def step_after(tmp_path_factory):
    src = open(os.path.join(os.path.dirname(__file__), "..", "bitmtp_amd", "csrc", "decode_ops.hip")).read()
    body = [re.search(what, src, re.S | re.M).group(0) for what in (
        r"^constexpr int kCommitGroups = .*?$", r"^__device__ __forceinline__ void commit_rows\(.*?^\}",
        r"^__global__ [^\n]*step_after_kernel\(.*?^\}", r"^static bool kv_planes_ok\(.*?^\}")]
    out = tmp_path_factory.mktemp("step_after")
    (out / "t.cpp").write_text(STUBS + "\n".join(body) + RUN)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", str(out / "t.cpp"), "-o", str(out / "t.so")], check=True)
    return ctypes.CDLL(str(out / "t.so"))


@pytest.mark.parametrize("rows", [1, 2, 9, 16, 31, 32])
def test_words_beside_the_inputs_stay(step_after, rows):
    words, slots, planes = 2 + 3 * rows, 40, 4
    gen = np.random.default_rng(rows)
    inputs = gen.integers(0, 1000, words + 3).astype(np.int32)
    drafted = gen.integers(0, 1000, max(rows - 1, 1)).astype(np.int32)
    inputs[-3 - (rows - 1):-3] = -2 ** 31 + np.arange(rows - 1)   # tokens of the draft behind the first one
    inputs[-3:] = (20, 5, 3)
    memory = np.full(words + 300, -7, dtype=np.int32)   # as many words behind the inputs as there are threads
    kv = gen.integers(0, 2 ** 31, (planes, slots, 64)).astype(np.int32)
    want = kv.copy()
    want[:, 5:8] = kv[:, 20:23]
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)   # noqa: E731
    step_after.run(p(inputs), p(memory[20:]), words, p(drafted), len(drafted), p(kv), planes, slots)
    got = memory[20:20 + words]
    assert np.array_equal(got[:words - rows + 1], inputs[:words - rows + 1]) and np.array_equal(got[words - rows + 1:], drafted[:rows - 1])
    assert (memory[:20] == -7).all() and (memory[20 + words:] == -7).all()
    assert np.array_equal(kv, want)


@pytest.mark.parametrize("n_layers,n_kv,slots,ok", [
    (36, 8, 240000, True),            # 4B shape: 2 ** 31 pieces of 16 bytes and more
    (28, 8, 1 << 22, True),           # the longest segment that steps take
    (2 ** 25, 1, 1, True), (2 ** 26, 1, 1, False), (2 ** 20, 2 ** 12, 1, False),   # a row's pieces are counted in 32 bits
    (0, 8, 64, False), (36, 0, 64, False), (36, 8, 0, False)])
def test_buffers_of_any_length_are_taken(step_after, n_layers, n_kv, slots, ok):
    assert step_after.planes_ok(ctypes.c_void_p(64), n_layers, n_kv, slots) == ok
    assert not step_after.planes_ok(None, n_layers, n_kv, slots)


def test_more_pieces_than_are_counted_are_not_committed(step_after):
    """As ``bonsai_kv_commit`` refuses them."""
    words, planes, slots, n = 5, 576, 600000, 233017   # n * planes * 16 just above 2 ** 31
    inputs = np.array([1, 2, 3, 4, 5, 300000, 0, n], dtype=np.int32)
    to, drafted = np.zeros(words, dtype=np.int32), np.zeros(1, dtype=np.int32)
    kv = np.full(4096, 7, dtype=np.int32)             # nothing beside its start would be there
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)   # noqa: E731
    step_after.run(p(inputs), p(to), words, p(drafted), 1, p(kv), planes, slots)
    assert (kv == 7).all() and np.array_equal(to, inputs[:words])
