"""The library's host code without a GPU: sr_api.cpp and sr_full_host.cpp linked with tests/cpp/hip_on_cpu.cpp, where device memory
is host memory and no kernel runs.  What an upload or a launch hands to the kernels is looked at, with allocations that fail."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import opentail.stingray_amd as sa
from opentail.stingray_amd import SamplerContext, SamplingParams

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host") / "libhost_side.so")
    src = [os.path.join(ROOT, "opentail", "stingray_amd", "csrc", f) for f in ("sr_api.cpp", "sr_full_host.cpp")]
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fPIC", "-shared", "-Wl,-Bsymbolic", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-o", out, os.path.join(ROOT, "tests", "cpp", "hip_on_cpu.cpp")] + src, check=True)
    return out


@pytest.fixture()
def ctx(lib, monkeypatch):
    monkeypatch.setattr(sa, "_LIB_PATH", lib)
    monkeypatch.setattr(sa, "_lib", None)
    c = SamplerContext(0, use_torch_stream=False)
    for f in ("cpu_scan_builds", "cpu_stream_waits", "cpu_launches", "cpu_live"):
        getattr(c.L, f).restype = C.c_int64
    c.L.cpu_live.argtypes = [C.c_void_p]
    c.L.cpu_uniforms.restype = C.c_void_p
    yield c
    c.L.cpu_fail(0, 0)
    c.close()


def _launch(ctx, batch, addr=4096, dtype=sa.SR_DTYPE_F32, stride=None):
    ctx._check(ctx.L.sr_sample_launch(ctx.h, batch.h, addr, dtype, stride or batch.vocab, 64, None))


@pytest.mark.parametrize("topk", [0, 40])
def test_uniforms_are_never_read_from_memory_that_was_given_away(ctx, topk):
    """A batch that could not be uploaded with more rows, and then has no pinned memory for that many uniforms."""
    rows, vocab = 5_000, 1_000
    p = [SamplingParams(Temperature=0.8, TopK=topk)]
    u = np.random.default_rng(1).random(20 * rows)
    b = ctx.new_batch().upload(p * rows, vocab, u[:rows])
    _launch(ctx, b)
    assert ctx.L.cpu_live(ctx.L.cpu_uniforms()) >= 8 * rows
    b.set_uniforms(u[:rows])
    _launch(ctx, b)
    assert np.array_equal(np.ctypeslib.as_array((C.c_double * rows).from_address(ctx.L.cpu_uniforms())), u[:rows])
    ctx.L.cpu_fail(1, 1)
    with pytest.raises(RuntimeError):
        ctx._check(ctx.L.sr_batch_upload(b.h, 20 * rows, vocab, b._packed[2] * 20, *[None] * 6, 0, None, u.ctypes.data, 1))
    with pytest.raises(RuntimeError):
        b.set_uniforms(u)
    ctx.L.cpu_fail(0, 0)
    _launch(ctx, b)
    assert ctx.L.cpu_live(ctx.L.cpu_uniforms()) > 0
    # a batch that fails once goes on working
    b.upload(p * rows, vocab, u[:rows])
    b.set_uniforms(u[rows:2 * rows])
    _launch(ctx, b)
    assert np.array_equal(np.ctypeslib.as_array((C.c_double * rows).from_address(ctx.L.cpu_uniforms())), u[rows:2 * rows])
    b.close()
