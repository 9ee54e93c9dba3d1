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
def test_a_batch_whose_upload_failed_is_refused_until_one_succeeds(ctx, topk):
    """A batch that could not be uploaded with more rows names device memory of an older, smaller one: no call launches it or
    gives it uniforms (whose old place may have been given away), and it works again once it has been uploaded."""
    rows, vocab = 5_000, 1_000
    p = [SamplingParams(Temperature=0.8, TopK=topk)]
    u = np.random.default_rng(1).random(20 * rows)
    uniforms = lambda: np.ctypeslib.as_array((C.c_double * rows).from_address(ctx.L.cpu_uniforms()))
    b = ctx.new_batch().upload(p * rows, vocab, u[:rows])
    _launch(ctx, b)
    assert ctx.L.cpu_live(ctx.L.cpu_uniforms()) >= 8 * rows
    b.set_uniforms(u[:rows])
    _launch(ctx, b)
    assert np.array_equal(uniforms(), u[:rows])
    ctx.L.cpu_fail(1, 1)
    with pytest.raises(RuntimeError):
        ctx._check(ctx.L.sr_batch_upload(b.h, 20 * rows, vocab, b._packed[2] * 20, *[None] * 6, 0, None, u.ctypes.data, 1))
    launches = ctx.L.cpu_launches()
    with pytest.raises(ValueError, match="upload"):
        b.set_uniforms(u)
    with pytest.raises(ValueError, match="upload"):
        b.append_tokens(np.full(rows, -1), None)
    ctx.L.cpu_fail(0, 0)
    with pytest.raises(ValueError, match="upload"):
        _launch(ctx, b)
    out = np.zeros(64, dtype=np.float32).ctypes.data
    for call in (lambda: ctx.L.sr_build_distribution_launch(ctx.h, b.h, 4096, 0, vocab, out, vocab, vocab),
                 lambda: ctx.L.sr_sample_with_distribution_launch(ctx.h, b.h, 4096, 0, vocab, out, vocab, vocab, 64),
                 lambda: ctx.L.sr_spec_verify_launch(ctx.h, b.h, 4096, None, None, 0, 64, 64),
                 lambda: ctx.L.sr_resample_rows_launch(ctx.h, b.h, 4096, 0, vocab, np.zeros(1, np.int32).ctypes.data, 1, 64, None)):
        assert call() == sa.SR_ERR_INVALID_ARGUMENT
    assert ctx.L.cpu_launches() == launches
    b.upload(p * rows, vocab, u[:rows])
    b.set_uniforms(u[rows:2 * rows])
    _launch(ctx, b)
    assert np.array_equal(uniforms(), u[rows:2 * rows])
    b.close()


def test_scan_masks_that_could_not_be_made_are_made_by_the_next_launch(ctx):
    vocab = 1_000
    b = ctx.new_batch().upload([SamplingParams(Temperature=0.8, TopK=40)] * 8, vocab, np.full(8, 0.5))
    _launch(ctx, b)
    made = ctx.L.cpu_scan_builds()
    ctx.L.cpu_fail(1, 1)
    with pytest.raises(RuntimeError):  # rows at eight different offsets: eight mask rows instead of one
        _launch(ctx, b, stride=vocab + 1)
    ctx.L.cpu_fail(0, 0)
    assert ctx.L.cpu_scan_builds() == made
    _launch(ctx, b, stride=vocab + 1)
    assert ctx.L.cpu_scan_builds() == made + 1
    assert [ctx.L.cpu_scan_row(r) for r in range(8)] == list(range(8))  # the descriptors that the kernel reads
    b.close()


def test_an_upload_makes_scan_masks_for_the_logits_of_its_own_batch(ctx):
    """Two batches take turns on one context, one with aligned fp32 logits, one with bf16 rows at odd addresses: after each has
    been launched once, no launch builds masks again or waits."""
    p = [SamplingParams(Temperature=0.8, TopK=40)] * 4
    a, b = ctx.new_batch(), ctx.new_batch()
    for step in range(4):
        for batch, vocab, addr, dtype in ((a, 1_000, 4096, sa.SR_DTYPE_F32), (b, 1_001, 4098, sa.SR_DTYPE_BF16)):
            batch.upload(p, vocab, np.full(4, 0.5))
            made, waits = ctx.L.cpu_scan_builds(), ctx.L.cpu_stream_waits()
            _launch(ctx, batch, addr, dtype)
            if step:
                assert (ctx.L.cpu_scan_builds(), ctx.L.cpu_stream_waits()) == (made, waits)
    a.close()
    b.close()
