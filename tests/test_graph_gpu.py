"""HIP-graph capture through the C ABI (tf_graph_*), and the two device-side
step helpers (tf_gather_indexed, tf_record_step).

A captured sequence of library calls is replayed several times with the
program's own eager work (new inputs uploaded, the outputs read back) and
synchronisations between the replays, and every replay is checked bit for
bit against the same calls run eagerly on the same inputs.  The capture's
rules are checked from the host: a block-cache miss and a synchronising call
during capture fail, the capture then yields no graph, and the context keeps
working; a block allocated during capture and freed while its graph exists
is not handed to other allocations.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from tensors_amd import ops, synth
from tensors_amd._lib import TFError, call, lib
from tests.conftest import assert_bitexact

pytestmark = pytest.mark.gpu


def _end(ctx):
    g = C.c_void_p()
    call("tf_graph_end", ctx.handle, C.byref(g))
    return g


def test_graph_replays_match_eager_calls(ctx):
    B, K, N = 64, 256, 128
    a = ctx.array(synth.normal(1001, (B, K)))
    w = ctx.array(synth.normal(1002, (N, K), std=0.06))
    z, h, c = ctx.empty((B, N)), ctx.empty((B, N)), ctx.empty((N,))
    z2, h2, c2 = ctx.empty((B, N)), ctx.empty((B, N)), ctx.empty((N,))

    def seq(zz, hh, cc):
        ops.gemm(a, w, zz, trans_b=True)
        ops.relu(zz, hh)
        ops.colsum(hh, cc)

    seq(z2, h2, c2)                    # eager once: any workspace is grown now
    ctx.sync()
    call("tf_graph_begin", ctx.handle)
    seq(z, h, c)
    g = _end(ctx)
    try:
        for r in range(4):
            a.upload(synth.normal(1100 + r, (B, K)))      # eager work between replays
            call("tf_graph_launch", ctx.handle, g)
            seq(z2, h2, c2)                               # the same calls, eagerly
            ctx.sync()
            for got, want, what in ((z, z2, "gemm"), (h, h2, "relu"), (c, c2, "colsum")):
                assert_bitexact(got.numpy(), want.numpy(), f"replay {r}: {what}")
    finally:
        call("tf_graph_destroy", g)


def test_capture_without_room_for_partials_runs_without_them():
    """A product that shares tiles between workgroups, or splits K, when run
    eagerly is captured by a fresh context too, which has no room for the
    partial sums: it runs unsplit, and eager products that allocate that room
    afterwards leave the graph valid.  fp32 sums of 100 and bf16 ones of 512
    products: within 512 * 2^-24 of the sum of magnitudes in any order."""
    import tensors_amd as ta
    own = ta.Context(0)
    try:
        a, b = synth.normal(1301, (1500, 100)), synth.normal(1302, (100, 1500))
        h, w = (ta.f32_to_bf16_bits(synth.normal(s, (512, 512))) for s in (1303, 1304))
        da, db, c = own.array(a), own.array(b), own.zeros((1500, 1500))
        dh, dw, z = own.array(h, ta.BF16), own.array(w, ta.BF16), own.zeros((512, 512))

        def seq():
            ops.gemm(da, db, c)
            ops.gemm(dh, dw, z, trans_a=True)

        want = a.astype(np.float64) @ b.astype(np.float64)
        zw = ta.bf16_bits_to_f32(h).astype(np.float64).T @ ta.bf16_bits_to_f32(w).astype(np.float64)
        own.sync()
        call("tf_graph_begin", own.handle)
        seq()
        g = _end(own)
        try:
            for r in range(3):
                call("tf_graph_launch", own.handle, g)
                for got, ref in ((c, want), (z, zw)):
                    assert np.abs(got.numpy() - ref).max() < 1e-4 * np.abs(ref).max(), f"replay {r}"
                seq()                                      # eagerly: the shares are allocated now
        finally:
            call("tf_graph_destroy", g)
    finally:
        del da, db, c, dh, dw, z
        own.close()


def test_relu_bwd_colsum_capture_without_workspace():
    """Rows that do not start on a whole access, in a context that has no
    workspace yet: the capture takes the form that needs none.  dz is exact;
    column sums of 32768 values: within 32768 * 2^-24 of the sum of magnitudes."""
    import tensors_amd as ta
    own = ta.Context(0)
    try:
        rows, cols = 32768, 2
        dy, x = synth.normal(1305, (rows, cols)), synth.normal(1306, (rows, cols))
        ddy, dx, dz, db = own.array(dy), own.array(x), own.zeros((rows, cols)), own.zeros((cols,))
        want = dy * (x > 0)
        own.sync()
        call("tf_graph_begin", own.handle)
        ops.relu_bwd_colsum(ddy, dx, dz, db)
        g = _end(own)
        try:
            for r in range(3):
                call("tf_graph_launch", own.handle, g)
                assert np.array_equal(dz.numpy(), want), f"replay {r}"
                bound = rows * 2.0 ** -24 * np.abs(want).astype(np.float64).sum(0)
                assert (np.abs(db.numpy() - want.astype(np.float64).sum(0)) <= bound).all(), f"replay {r}"
                ops.relu_bwd_colsum(ddy, dx, dz, db)
        finally:
            call("tf_graph_destroy", g)
    finally:
        del ddy, dx, dz, db
        own.close()


def test_layernorm_bwd_beside_a_graph_leaves_it_valid():
    """A LayerNorm backward whose block-per-row form wants more workspace than a
    captured graph found runs beside that graph without moving it.  Sums of
    4096 terms in dx, 256 in dgamma and dbeta: far within 4096 * 2^-24 of the
    largest value."""
    import tensors_amd as ta
    own = ta.Context(0)
    try:
        rows, cols = 256, 4096
        x, dy = synth.normal(1307, (rows, cols)), synth.normal(1308, (rows, cols))
        gamma = synth.normal(1309, (cols,)) + np.float32(1)
        dx_, ddy, dg, db0 = own.array(x), own.array(dy), own.array(gamma), own.zeros((cols,))
        y, mean, rstd = own.zeros((rows, cols)), own.zeros((rows,)), own.zeros((rows,))
        gx, gg, gb = own.zeros((rows, cols)), own.zeros((cols,)), own.zeros((cols,))
        s = own.zeros((cols,))
        ops.colsum(dx_, s)                                  # a workspace of the smallest size
        ops.layernorm_fwd(dx_, dg, db0, y, mean, rstd)
        own.sync()
        call("tf_graph_begin", own.handle)
        ops.colsum(dx_, s)
        g = _end(own)
        try:
            x64, dy64 = x.astype(np.float64), dy.astype(np.float64)
            r = 1 / np.sqrt(x64.var(1, keepdims=True) + 1e-5)
            xh = (x64 - x64.mean(1, keepdims=True)) * r
            d = dy64 * gamma
            want = (r * (d - d.mean(1, keepdims=True) - xh * (d * xh).mean(1, keepdims=True)),
                    (dy64 * xh).sum(0), dy64.sum(0))
            for i in range(2):
                ops.layernorm_bwd(ddy, dx_, dg, mean, rstd, gx, gg, gb)
                for got, ref in zip((gx, gg, gb), want):
                    assert np.abs(got.numpy() - ref).max() <= 4096 * 2.0 ** -24 * np.abs(ref).max()
                call("tf_graph_launch", own.handle, g)
                assert np.abs(s.numpy() - x64.sum(0)).max() <= 256 * 2.0 ** -24 * np.abs(x64).sum(0).max()
        finally:
            call("tf_graph_destroy", g)
    finally:
        del dx_, ddy, dg, db0, y, mean, rstd, gx, gg, gb, s
        own.close()


def test_capture_fails_on_a_cache_miss_and_on_sync(ctx):
    call("tf_graph_begin", ctx.handle)
    p = C.c_void_p()
    with pytest.raises(TFError):
        call("tf_hip_alloc", ctx.handle, C.c_size_t((3 << 30) + 12345), C.byref(p))   # no such cached block
    with pytest.raises(TFError):
        _end(ctx)
    call("tf_graph_begin", ctx.handle)
    with pytest.raises(TFError):
        call("tf_hip_sync", ctx.handle)
    with pytest.raises(TFError):
        _end(ctx)
    # The context is usable afterwards.
    x = ctx.array(synth.normal(1200, (1000,)))
    y = ctx.empty((1000,))
    ops.relu(x, y)
    assert_bitexact(y.numpy(), np.maximum(x.numpy(), 0).astype(np.float32), "relu after failed captures")


def test_gather_and_record_in_a_replayed_graph(ctx):
    n, bytes_ = 3, 4096 * 4 + 8
    srcs = [ctx.array(synth.normal(1300 + i, (bytes_ // 4,))) for i in range(n)]
    table = ctx.array(np.array([s.ptr for s in srcs], np.uint64), np.uint64)
    counter = ctx.array(np.array([0], np.int64))
    dst = ctx.empty((bytes_ // 4,))
    ring = ctx.zeros((8,))
    call("tf_gather_indexed", ctx.handle, dst.ptr, table.ptr, n, counter.ptr, bytes_)
    call("tf_record_step", ctx.handle, dst.ptr, ring.ptr, 8, counter.ptr)     # eager: step 0
    ctx.sync()
    assert_bitexact(dst.numpy(), srcs[0].numpy(), "gather step 0")
    call("tf_graph_begin", ctx.handle)
    call("tf_gather_indexed", ctx.handle, dst.ptr, table.ptr, n, counter.ptr, bytes_)
    call("tf_record_step", ctx.handle, dst.ptr, ring.ptr, 8, counter.ptr)
    g = _end(ctx)
    try:
        for step in range(1, 10):                         # the ring holds 8: later steps only count
            call("tf_graph_launch", ctx.handle, g)
            ctx.sync()
            assert_bitexact(dst.numpy(), srcs[step % n].numpy(), f"gather step {step}")
            assert int(counter.numpy()[0]) == step + 1
    finally:
        call("tf_graph_destroy", g)
    want = np.array([srcs[s % n].numpy()[0] for s in range(8)], np.float32)
    assert_bitexact(ring.numpy(), want, "recorded values")


def test_block_allocated_during_capture_stays_with_its_graph(ctx):
    # A size class no other test uses (2 MB steps above 1 MB: 38.1 MB -> 40 MB).
    n = 10_000_000
    x = ctx.array(synth.normal(1400, (n,)))
    first = ctx.empty((n,))
    first.free()                                   # the cache now holds one block of the class
    call("tf_graph_begin", ctx.handle)
    inside = ctx.empty((n,))                       # served from the cache during capture
    ops.relu(x, inside)
    g = _end(ctx)
    try:
        held = inside.ptr
        inside.free()                              # freed while the graph exists
        other = ctx.empty((n,))
        assert other.ptr != held, "a block the graph writes was handed to another allocation"
        call("tf_hip_fill_f32", ctx.handle, other.ptr, 5.0, n)
        call("tf_graph_launch", ctx.handle, g)     # writes relu(x) into the held block
        ctx.sync()
        assert np.all(other.numpy() == 5.0), "a replay wrote into another allocation's memory"
    finally:
        call("tf_graph_destroy", g)
    other.free()
    ctx.sync()
