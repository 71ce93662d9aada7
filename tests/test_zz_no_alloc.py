"""mmhip_qmm_dev_noalloc: the batched QMM (batchMatMulUnified's device twin)
with the library's fixed per-device scratch instead of an allocated one.

Its output must equal mmhip_qmm_dev's bit for bit (same kernels, same
inputs) on two calls in a row, the second with a smaller input, so that
nothing left in the shared scratch by the first call leaks into the second
(only Q8_0 rows that end in a partial block use the scratch; the others run in
one launch without it); both are also checked against the oracle's matMulQ8_0 /
dequantize + GEMV (qmm.zig:58-138, inference.zig:1231-1264) at the QMM
tolerance. Inputs beyond the fixed scratch are refused with an error. Captured
calls (HIP graphs) give the eager calls' bits on every replay, as do an MoE
layer's.
"""
import ctypes

import numpy as np
import pytest

import mmhip as mm

pytestmark = pytest.mark.gpu

TOL_QMM = 1e-2


def _run(ctx, fn, w, x, rows, batch, layout):
    dx = mm.DeviceArray.from_numpy(ctx, x)
    dy = mm.DeviceArray(ctx, rows * batch * 4)
    try:
        fn(w, 0, dx, dy, batch, layout)
        ctx.synchronize()
        y = dy.to_numpy(np.float32, rows * batch)
    finally:
        dx.free()
        dy.free()
    return y.reshape(batch, rows) if layout == 0 else y.reshape(rows, batch).T


@pytest.mark.parametrize("fmt", [mm.Q8_0, mm.IQ2_XXS])
@pytest.mark.parametrize("layout", [0, 1])
def test_noalloc_matches_qmm_dev_twice(ctx, orc, fmt, layout):
    rng = np.random.default_rng(900 + fmt + layout)
    cases = [(1536, 2048, 64), (512, 768, 5)]  # the second call is smaller in rows, columns and batch
    for rows, cols, batch in cases:
        raw = mm.make_weight(rng, fmt, rows, cols)
        x = (rng.standard_normal((batch, cols)) * 2.0).astype(np.float32)
        w = ctx.upload(raw, fmt, rows, cols)
        try:
            got = _run(ctx, ctx.qmm_dev_noalloc, w, x, rows, batch, layout)
            ref = _run(ctx, ctx.qmm_dev, w, x, rows, batch, layout)
        finally:
            w.free()
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), (rows, cols, batch)
        cpu = orc.batch_mat_mul_unified(raw, fmt, x, rows, batch, cols).reshape(batch, rows)
        assert mm.max_abs_rel(got, cpu) <= TOL_QMM


@pytest.mark.parametrize("layout", [0, 1])
def test_noalloc_scratch_holds_nothing_over(ctx, orc, layout):
    """Q8_0 rows that end in a partial block, whose digits go through the fixed
    scratch: a call that fills it to the last byte (256 vectors of 8190 columns),
    then smaller ones, each with mmhip_qmm_dev's bits and the oracle's results."""
    rng = np.random.default_rng(940 + layout)
    for rows, cols, batch in [(48, 8190, 256), (100, 1000, 7), (33, 2330, 64), (16, 40, 2)]:
        raw = mm.make_weight(rng, mm.Q8_0, rows, cols)
        x = (rng.standard_normal((batch, cols)) * 2.0).astype(np.float32)
        w = ctx.upload(raw, mm.Q8_0, rows, cols)
        try:
            got = _run(ctx, ctx.qmm_dev_noalloc, w, x, rows, batch, layout)
            ref = _run(ctx, ctx.qmm_dev, w, x, rows, batch, layout)
        finally:
            w.free()
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), (rows, cols, batch)
        cpu = orc.batch_mat_mul_unified(raw, mm.Q8_0, x, rows, batch, cols).reshape(batch, rows)
        assert mm.max_abs_rel(got, cpu) <= 1e-3


def test_noalloc_size_limit(ctx):
    rng = np.random.default_rng(950)
    raw = mm.make_weight(rng, mm.IQ2_XXS, 16, 8448)  # 8448 columns: 256 x 8448 x 2.125 bytes > the scratch
    w = ctx.upload(raw, mm.IQ2_XXS, 16, 8448)
    dx = mm.DeviceArray.from_numpy(ctx, np.zeros((256, 8448), np.float32))
    dy = mm.DeviceArray(ctx, 256 * 16 * 4)
    try:
        with pytest.raises(mm.MmhipError, match="scratch"):
            ctx.qmm_dev_noalloc(w, 0, dx, dy, 256, 0)
        ctx.qmm_dev_noalloc(w, 0, dx, dy, 240, 0)  # 240 x 8448 x 2.125 fits
        ctx.synchronize()
    finally:
        w.free()
        dx.free()
        dy.free()


def test_noalloc_at_the_limit(ctx, orc):
    """256 vectors of 8192 columns fill the scratch exactly."""
    rng = np.random.default_rng(960)
    rows, cols, batch = 48, 8192, 256
    raw = mm.make_weight(rng, mm.Q8_0, rows, cols)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    w = ctx.upload(raw, mm.Q8_0, rows, cols)
    try:
        got = _run(ctx, ctx.qmm_dev_noalloc, w, x, rows, batch, 0)
        ref = _run(ctx, ctx.qmm_dev, w, x, rows, batch, 0)
    finally:
        w.free()
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))


def _put(ctx, d, arr):
    arr = np.ascontiguousarray(arr, dtype=np.float32)
    mm.check(ctx.lib.mmhip_memcpy_h2d(ctx.handle, d.ptr, mm._ptr(arr), arr.nbytes), "mmhip_memcpy_h2d")


class _Graph:
    """A captured sequence of calls on the context's stream (HIP runtime)."""

    def __init__(self, ctx, calls):
        self.hip, self.stream = ctypes.CDLL("libamdhip64.so"), ctypes.c_void_p(ctx.stream)
        graph, self.exe = ctypes.c_void_p(), ctypes.c_void_p()
        self._ok(self.hip.hipStreamBeginCapture(self.stream, 2))  # hipStreamCaptureModeRelaxed
        try:
            calls()
        finally:
            rc = self.hip.hipStreamEndCapture(self.stream, ctypes.byref(graph))
        self._ok(rc)
        self._ok(self.hip.hipGraphInstantiate(ctypes.byref(self.exe), graph, None, None, ctypes.c_size_t(0)))
        self._ok(self.hip.hipGraphDestroy(graph))

    @staticmethod
    def _ok(rc):
        assert rc == 0, f"HIP error {rc}"

    def launch(self):
        self._ok(self.hip.hipGraphLaunch(self.exe, self.stream))

    def free(self):
        self._ok(self.hip.hipGraphExecDestroy(self.exe))


@pytest.mark.parametrize("fmt,cols", [(mm.Q8_0, 1000), (mm.Q8_0, 768), (mm.Q8_0, 2304), (mm.IQ2_XXS, 768)])
def test_noalloc_under_capture(ctx, fmt, cols):
    """A captured call replayed with other vectors each time, eager calls in
    between: every replay gives the eager call's bits (the scratch, the digit
    kernel and the tile kernel)."""
    rng = np.random.default_rng(970 + cols)
    rows, batch = 100, 19
    w = ctx.upload(mm.make_weight(rng, fmt, rows, cols), fmt, rows, cols)
    dx, dy, de = (mm.DeviceArray(ctx, n * 4) for n in (batch * cols, batch * rows, batch * rows))
    g = None
    try:
        _put(ctx, dx, np.zeros((batch, cols)))
        ctx.qmm_dev_noalloc(w, 0, dx, de, batch, 0)  # the kernels are loaded outside the capture
        ctx.synchronize()
        g = _Graph(ctx, lambda: ctx.qmm_dev_noalloc(w, 0, dx, dy, batch, 0))
        for _ in range(4):
            _put(ctx, dx, rng.standard_normal((batch, cols)))
            g.launch()
            ctx.qmm_dev_noalloc(w, 0, dx, de, batch, 0)
            ctx.synchronize()
            a, b = (d.to_numpy(np.uint32, batch * rows) for d in (dy, de))
            assert np.array_equal(a, b)
    finally:
        if g:
            g.free()
        for h in (w, dx, dy, de):
            h.free()


@pytest.mark.parametrize("fmt,t", [(mm.Q8_0, 40), (mm.IQ2_XXS, 40), (mm.Q8_0, 9)])
def test_moe_layer_under_capture(ctx, fmt, t):
    """A captured layer call of several tokens (more than one routing workgroup
    at 40) replayed with other tokens each time: the eager call's bits."""
    rng = np.random.default_rng(980 + fmt + t)
    hidden, inter, E = 512, 256, 12
    layer = mm.MoeLayer(ctx, hidden=hidden, inter=inter, n_experts=E, expert_type=fmt,
                        router=rng.normal(0.0, 0.05, (E, hidden)).astype(np.float32),
                        gate=mm.make_weight(rng, fmt, inter, hidden, E), up=mm.make_weight(rng, fmt, inter, hidden, E),
                        down=mm.make_weight(rng, fmt, hidden, inter, E),
                        shared=tuple(mm.make_weight(rng, fmt, *s) for s in ((inter, hidden), (inter, hidden), (hidden, inter))),
                        shared_inter=inter)
    dx, dy, de = (mm.DeviceArray(ctx, t * hidden * 4) for _ in range(3))
    g = None
    try:
        _put(ctx, dx, np.zeros((t, hidden)))
        layer.ffn_dev(dx, de, t)  # the kernels are loaded outside the capture
        ctx.synchronize()
        g = _Graph(ctx, lambda: layer.ffn_dev(dx, dy, t))
        for _ in range(4):
            _put(ctx, dx, rng.standard_normal((t, hidden)))
            g.launch()
            layer.ffn_dev(dx, de, t)
            ctx.synchronize()
            a, b = (d.to_numpy(np.uint32, t * hidden) for d in (dy, de))
            assert np.array_equal(a, b)
    finally:
        if g:
            g.free()
        layer.free()
        for h in (dx, dy, de):
            h.free()
