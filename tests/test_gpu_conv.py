"""GPU parity of qa_conv2d_3x3s2, one conv level of the audio tower's stem
(3x3, stride 2, pad 1, + bias, erf GELU; src/audio_encoder.rs:204-236,
376-447), against the oracle (oracle/qa_oracle_audio.c or_conv3x3s2: f64
accumulation, f32 GELU, one rounding; pinned to torch's conv2d).

Every case calls the product through the C ABI on an MI355X: c_in = 1 takes
the direct kernel (qa_conv.hip), c_in a multiple of 8 >= 64 the implicit GEMM
(qa_gemm.hip with the convolution loader, both tile shapes).

Tolerance: one rounding of an f32 sum (and the f32 GELU): the north star
(max relative error <= 1e-2 with the 1e-3 max|r| floor, MAE <= 1e-3) and
every output above the floor within 1 ulp of the f64-exact oracle.  The stem's
shapes per 100-frame mel chunk: conv1 [128 x 100 x 1] -> [64 x 50 x 480],
conv2 -> [32 x 25 x 480], conv3 -> [16 x 13 x 480] (rows (b, t, f) for
conv_out).  At 300 s (300 chunks) the oracle checks sampled row blocks.
"""
from __future__ import annotations

import ctypes
import os

import numpy as np
import pytest

from conftest import assert_parity

pytestmark = pytest.mark.gpu

F16, BF16 = 0, 1


def _h16(orc, x, dtype):
    return orc.h16_from_f32(np.asarray(x, np.float32), dtype)


def _case(orc, dtype, b, h, w, c_in, c_out, seed, w_std=None):
    rng = np.random.default_rng(seed)
    x = _h16(orc, rng.standard_normal((b, h, w, c_in)), dtype)
    ldw = (9 * c_in + 7) // 8 * 8
    std = w_std if w_std is not None else 1.0 / np.sqrt(9 * c_in)
    wt = np.zeros((c_out, ldw), np.uint16)
    wt[:, :9 * c_in] = _h16(orc, std * rng.standard_normal((c_out, 9 * c_in)), dtype)
    bias = _h16(orc, 0.05 * rng.standard_normal(c_out), dtype)
    return x, wt, bias


def _conv_gpu(ctx, pkg, dtype, x, wt, bias, c_out, flags):
    b, h, w, c_in = x.shape
    ho, wo = (h - 1) // 2 + 1, (w - 1) // 2 + 1
    dx, dw = ctx.to_device(x), ctx.to_device(wt)
    db = ctx.to_device(bias) if bias is not None else None
    dy = ctx.alloc(b * ho * wo * c_out * 2)
    ctx.conv2d_3x3s2(pkg.ConvDesc(dtype=dtype, flags=flags, batch=b, h=h, w=w, c_in=c_in,
                                  c_out=c_out, x=int(dx), weight=int(dw),
                                  bias=int(db) if db is not None else None, y=int(dy)))
    y = ctx.download(dy, (b * ho * wo, c_out))
    for buf in (dx, dw, db, dy):
        if buf is not None:
            buf.free()
    return y


CASES = [
    # b, h, w, c_in, c_out
    (2, 128, 100, 1, 480),   # conv1 of two mel chunks
    (1, 9, 7, 1, 16),        # odd sizes, direct
    (1, 64, 50, 480, 480),   # conv2 of one chunk
    (2, 32, 25, 480, 480),   # conv3 of two chunks
    (1, 13, 11, 64, 40),     # odd sizes, ragged N, implicit
    (3, 6, 5, 128, 136),
]


@pytest.mark.parametrize("dtype", [F16, BF16], ids=["f16", "bf16"])
@pytest.mark.parametrize("b,h,w,c_in,c_out", CASES)
@pytest.mark.parametrize("tmajor", [False, True], ids=["rows_hw", "rows_wh"])
def test_conv(ctx, pkg, orc, dtype, b, h, w, c_in, c_out, tmajor):
    x, wt, bias = _case(orc, dtype, b, h, w, c_in, c_out, b * h * w + c_in)
    flags = pkg.QA_CONV_GELU | (pkg.QA_CONV_TOKEN_MAJOR if tmajor else 0)
    got = _conv_gpu(ctx, pkg, dtype, x, wt, bias, c_out, flags)
    want = orc.conv3x3s2(dtype, x, wt, bias, gelu=True, token_major=tmajor)
    assert_parity(got, want, orc, dtype, ulp_tol=1)


@pytest.mark.parametrize("batch", [900, 901])
def test_conv1_groups(ctx, pkg, orc, batch):
    """Level 1 in two channel groups (5625 blocks of 128 pixels) and with all six
    channel tiles in one block (5632, the last a quarter full): the bits of two
    images' own call, in every place."""
    x, wt, bias = _case(orc, F16, 2, 64, 50, 1, 168, 17)
    want = _conv_gpu(ctx, pkg, F16, x, wt, bias, 168, pkg.QA_CONV_GELU).reshape(2, -1)
    assert_parity(want.reshape(-1, 168), orc.conv3x3s2(F16, x, wt, bias, gelu=True), orc, F16, ulp_tol=1)
    got = _conv_gpu(ctx, pkg, F16, x[np.arange(batch) % 2], wt, bias, 168, pkg.QA_CONV_GELU).reshape(batch, -1)
    assert (got[0::2] == want[0]).all() and (got[1::2] == want[1]).all()


@pytest.mark.parametrize("tile", ["0", "1", "2", "6", "8"],
                         ids=["128x128", "256x128", "128x256", "256x256", "256x160"])
def test_conv_tiles_and_no_activation(ctx, pkg, orc, monkeypatch, tile):
    """Every implicit-GEMM tile shape, without bias and GELU (the plain sum)."""
    monkeypatch.setenv("QA_TILE", tile)
    x, wt, _ = _case(orc, F16, 2, 20, 18, 96, 200, 7)
    got = _conv_gpu(ctx, pkg, F16, x, wt, None, 200, 0)
    want = orc.conv3x3s2(F16, x, wt, None, gelu=False)
    assert_parity(got, want, orc, F16, ulp_tol=1)


@pytest.mark.parametrize("dtype", [F16, BF16], ids=["f16", "bf16"])
@pytest.mark.parametrize("tile,splits", [("0", "2"), ("1", "3"), ("2", "5"), ("6", "2"), ("8", "9")])
@pytest.mark.parametrize("tmajor", [False, True], ids=["rows_hw", "rows_wh"])
def test_conv_split_k(ctx, pkg, orc, monkeypatch, dtype, tile, splits, tmajor):
    """K split over f32 partials and the reduce kernel, on every tile shape
    (taps and channels of a split start inside a tap; 14 stages, uneven splits):
    bias, GELU, both row orders."""
    monkeypatch.setenv("QA_TILE", tile)
    monkeypatch.setenv("QA_SPLITS", splits)
    x, wt, bias = _case(orc, dtype, 2, 20, 18, 96, 200, 7)
    flags = pkg.QA_CONV_GELU | (pkg.QA_CONV_TOKEN_MAJOR if tmajor else 0)
    got = _conv_gpu(ctx, pkg, dtype, x, wt, bias, 200, flags)
    want = orc.conv3x3s2(dtype, x, wt, bias, gelu=True, token_major=tmajor)
    assert_parity(got, want, orc, dtype, ulp_tol=1)
    assert np.array_equal(got, _conv_gpu(ctx, pkg, dtype, x, wt, bias, 200, flags))


SHORT = (2, 32, 25, 480, 480)  # the third level of two chunks: 16 tiles of 128 x 128, which the planner splits in six


def _short(orc, dtype):
    b, h, w, c_in, c_out = SHORT
    return _case(orc, dtype, b, h, w, c_in, c_out, 13)


def _conv_desc(pkg, dtype, x, wt, bias, y):
    b, h, w, c_in, c_out = SHORT
    return pkg.ConvDesc(dtype=dtype, flags=pkg.QA_CONV_GELU, batch=b, h=h, w=w, c_in=c_in, c_out=c_out,
                        x=int(x), weight=int(wt), bias=int(bias), y=int(y))


@pytest.mark.parametrize("dtype", [F16, BF16], ids=["f16", "bf16"])
@pytest.mark.parametrize("tmajor", [False, True], ids=["rows_hw", "rows_wh"])
def test_conv_planner_splits_short_clips(ctx, pkg, orc, monkeypatch, dtype, tmajor):
    """The planner's own split: other bits than the unsplit call's (sums in
    another order), the same in each call, and right."""
    x, wt, bias = _short(orc, dtype)
    flags = pkg.QA_CONV_GELU | (pkg.QA_CONV_TOKEN_MAJOR if tmajor else 0)
    got = _conv_gpu(ctx, pkg, dtype, x, wt, bias, SHORT[-1], flags)
    assert_parity(got, orc.conv3x3s2(dtype, x, wt, bias, gelu=True, token_major=tmajor), orc, dtype, ulp_tol=1)
    assert np.array_equal(got, _conv_gpu(ctx, pkg, dtype, x, wt, bias, SHORT[-1], flags))
    monkeypatch.setenv("QA_SPLITS", "1")
    assert not np.array_equal(got, _conv_gpu(ctx, pkg, dtype, x, wt, bias, SHORT[-1], flags))


def test_conv_captured_runs_unsplit(pkg, orc, monkeypatch):
    """A captured convolution that would be split when eager runs unsplit: every
    replay has the unsplit call's bits, also with eager, split calls between."""
    from hipgraph import Capture
    x, wt, bias = _short(orc, F16)
    want = orc.conv3x3s2(F16, x, wt, bias, gelu=True)
    with pkg.Context(0) as ctx:
        dx, dw, db = ctx.to_device(x), ctx.to_device(wt), ctx.to_device(bias)
        dy, dz = ctx.alloc(want.size * 2), ctx.alloc(want.size * 2)
        monkeypatch.setenv("QA_SPLITS", "1")
        ctx.conv2d_3x3s2(_conv_desc(pkg, F16, dx, dw, db, dz))
        unsplit = ctx.download(dz, want.shape)
        monkeypatch.delenv("QA_SPLITS")
        with Capture(ctx.stream) as cap:
            ctx.conv2d_3x3s2(_conv_desc(pkg, F16, dx, dw, db, dy))
        for _ in range(3):
            ctx.upload(dy, np.zeros(want.shape, np.uint16))
            cap.replay()
            assert np.array_equal(ctx.download(dy, want.shape), unsplit)
            ctx.conv2d_3x3s2(_conv_desc(pkg, F16, dx, dw, db, dz))
            ctx.sync()
        eager = ctx.download(dz, want.shape)
        assert not np.array_equal(eager, unsplit)
        assert_parity(unsplit, want, orc, F16, ulp_tol=1)
        assert_parity(eager, want, orc, F16, ulp_tol=1)
        cap.close()


def test_conv_allocates_nothing(ctx, pkg, monkeypatch):
    """The first split convolution of a context takes no device memory (3 x 2080
    x 480 partials, 12 MB, for ten chunks' third level): the buffer is the
    context's from its creation."""
    from hipgraph import hip

    def free_bytes():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    b, h, w, c_in, c_out = SHORT
    x, wt, bias = ctx.alloc(5 * b * h * w * c_in * 2), ctx.alloc(c_out * 9 * c_in * 2), ctx.alloc(c_out * 2)
    y = ctx.alloc(5 * b * 16 * 13 * c_out * 2)
    desc = _conv_desc(pkg, F16, x, wt, bias, y)
    desc.batch = 5 * b
    ctx.conv2d_3x3s2(desc)  # loads the kernels' code
    ctx.sync()
    with pkg.Context(0) as fresh:
        monkeypatch.setenv("QA_SPLITS", "1")
        fresh.conv2d_3x3s2(desc)  # what a stream's first launch takes, without partials
        fresh.sync()
        monkeypatch.delenv("QA_SPLITS")
        before = free_bytes()
        fresh.conv2d_3x3s2(desc)
        fresh.sync()
        assert free_bytes() == before
    for buf in (x, wt, bias, y):
        buf.free()


def test_conv_leaves_captured_workspace(pkg, orc, monkeypatch):
    """A split convolution keeps its partials apart from the workspace that a
    captured split linear uses: the replays stay right after eager convolutions
    whose partials are larger."""
    from hipgraph import Capture
    rng = np.random.default_rng(11)
    m, n, k = 64, 128, 1024
    a = _h16(orc, rng.standard_normal((m, k)), F16)
    w = _h16(orc, rng.standard_normal((n, k)) * 0.05, F16)
    x, wt, bias = _case(orc, F16, 2, 20, 18, 96, 200, 7)
    conv_want = orc.conv3x3s2(F16, x, wt, bias, gelu=True)
    with pkg.Context(0) as ctx:
        da, dw, dc = ctx.to_device(a), ctx.to_device(w), ctx.alloc(m * n * 2)
        dx, dk, db, dy = ctx.to_device(x), ctx.to_device(wt), ctx.to_device(bias), ctx.alloc(conv_want.size * 2)
        lin = pkg.linear_desc(F16, m, n, k, da, dw, dc)
        conv = pkg.ConvDesc(dtype=F16, flags=pkg.QA_CONV_GELU, batch=2, h=20, w=18, c_in=96, c_out=200,
                            x=int(dx), weight=int(dk), bias=int(db), y=int(dy))
        monkeypatch.setenv("QA_SPLITS", "2")
        ctx.linear(lin)  # grows the workspace
        want = ctx.download(dc, (m, n))
        with Capture(ctx.stream) as cap:
            ctx.linear(lin)
        for splits in ("2", "5", "3"):
            monkeypatch.setenv("QA_SPLITS", splits)
            ctx.conv2d_3x3s2(conv)
            ctx.upload(dc, np.zeros((m, n), np.uint16))
            cap.replay()
            assert np.array_equal(ctx.download(dc, (m, n)), want)
            ctx.conv2d_3x3s2(conv)  # and the replay leaves the partials alone
            assert_parity(ctx.download(dy, conv_want.shape), conv_want, orc, F16, ulp_tol=1)
        cap.close()


def test_conv_stem_at_300_s(ctx, pkg, orc):
    """conv2 over the 300 chunks of 300 s of audio (240 000 output pixels,
    995 GFLOP): the oracle checks the first, a middle and the last block of 64
    output rows."""
    from qwen3_aligner_wgpu_amd import host
    b, h, w, c = 300, 64, 50, 480
    _, wt, bias = _case(orc, F16, 1, 1, 1, c, c, 3)
    x = host.synth_normal(3, 1, (b, h, w, c))  # 921.6 MB, generated in parallel C
    got = _conv_gpu(ctx, pkg, F16, x, wt, bias, c, pkg.QA_CONV_GELU)
    m = got.shape[0]
    for m0 in (0, m // 2 + 17, m - 64):
        want = orc.conv3x3s2(F16, x, wt, bias, gelu=True, rows=(m0, m0 + 64))
        assert_parity(got[m0:m0 + 64], want, orc, F16, ulp_tol=1)


def test_conv_validate(ctx, pkg):
    lib = pkg.lib()
    ok = dict(dtype=F16, flags=pkg.QA_CONV_GELU, batch=1, h=64, w=50, c_in=480, c_out=480,
              x=0x100000, weight=0x200000, bias=None, y=0x300000)
    for kw, code, needle in [(dict(c_in=40), pkg.QA_EUNSUPPORTED, "c_in=40"),
                             (dict(c_in=100), pkg.QA_EUNSUPPORTED, "c_in=100"),
                             (dict(c_out=20), pkg.QA_EINVAL, "multiple of 8"),
                             (dict(flags=8), pkg.QA_EINVAL, "unknown flags"),
                             (dict(x=0x100008), pkg.QA_EINVAL, "aligned"),
                             (dict(h=0), pkg.QA_EINVAL, "bad shape"),
                             (dict(c_in=1, c_out=2048), pkg.QA_EUNSUPPORTED, "c_out=2048"),
                             (dict(batch=1 << 20), pkg.QA_EINVAL, "2 GiB")]:
        d = pkg.ConvDesc(**{**ok, **kw})
        assert lib.qa_conv2d_3x3s2(ctx.handle, ctypes.byref(d)) == code, kw
        assert needle in pkg.last_error(), (kw, pkg.last_error())
