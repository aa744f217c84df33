"""agx_trace_rays over its staging paths: one ray, sizes around a wave, a block
and the limit between the pinned and the device staging, a smaller call after a
larger one, and outputs left out; against the staging without allocation.
"""
import ctypes as C
import time

import numpy as np
import pytest

from atrc_amd import capi, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("accel", [capi.ACCEL_ATRC, capi.ACCEL_BVH4, capi.ACCEL_BVH4_WATERTIGHT])
def test_ray_counts(accel):
    s, _, _ = scenes.procedural_spheres(n_spheres=8, subdiv=2, seed=3, extent=12.0)
    s.accel = accel
    desc, keep = s.to_desc()
    with capi.Context(0) as ctx:
        ctx.upload_scene(desc)
        for n in (1, 63, 64, 65, 257, 32767, 32768, 32769, 5, 100_001):
            o, d = scenes.random_rays(((-2, -2, -2), (14, 14, 14)), n, seed=n)
            tmin, tmax = np.full(n, 0.01, np.float32), np.full(n, 40.0, np.float32)
            print(f"[ray sizes] accel {accel}, {n} rays", flush=True)
            for any_hit in (False, True):
                a = ctx.trace_rays(o, d, tmin, tmax, any_hit=any_hit)
                sa = ctx.stats()
                b = ctx.trace_rays(o, d, tmin, tmax, any_hit=any_hit, noalloc=True)
                sb = ctx.stats()
                for k in ("entity",) if any_hit else ("entity", "prim", "t", "u", "v"):
                    np.testing.assert_array_equal(a[k].view(np.uint32), b[k].view(np.uint32))
                for k in ("closest_rays", "shadow_rays", "closest_node_visits", "closest_tri_tests", "closest_hits",
                          "shadow_node_visits", "shadow_tri_tests"):
                    assert sa[k] == sb[k], (n, k)
                assert sa["total_ms"] > 0


@pytest.mark.parametrize("any_hit", [False, True])
def test_staging_without_allocation_at_its_capacity(gpu_ctx, any_hit):
    n = 131072
    _query_scene(gpu_ctx)
    q = _query(n)
    print(f"[ray sizes] {n} rays, any_hit {any_hit}", flush=True)
    a, b = (gpu_ctx.trace_rays(*q, any_hit=any_hit, noalloc=k) for k in (False, True))
    for k in ("entity",) if any_hit else ("entity", "prim", "t", "u", "v"):
        np.testing.assert_array_equal(a[k].view(np.uint32), b[k].view(np.uint32))


@pytest.mark.parametrize("n", [100, 40_000])
def test_outputs_may_be_left_out(gpu_ctx, n):
    s, _, _ = scenes.cornell_box()
    s.accel = capi.ACCEL_BVH4
    desc, keep = s.to_desc()
    gpu_ctx.upload_scene(desc)
    o, d = scenes.random_rays(((0.1, 0.1, 0.1), (5, 5, 5)), n, seed=1)
    tmin, tmax = np.zeros(n, np.float32), np.full(n, np.inf, np.float32)
    full = gpu_ctx.trace_rays(o, d, tmin, tmax)
    ent, t = np.zeros(n, np.int32), np.zeros(n, np.float32)
    f = capi.fptr
    assert gpu_ctx.lib.agx_trace_rays(gpu_ctx.h, f(o), f(d), f(tmin), f(tmax), n, 0, capi.iptr(ent), None, f(t), None,
                                      None) == 0
    np.testing.assert_array_equal(ent, full["entity"])
    np.testing.assert_array_equal(t.view(np.uint32), full["t"].view(np.uint32))


@pytest.mark.parametrize("any_hit", [False, True])
def test_calls_of_several_parts(gpu_ctx, any_hit):
    """A call of more rays than the device staging holds is traced in parts of 2^22:
    the same as the parts asked for one by one."""
    part = 1 << 22
    n = part + 77
    s, _, _ = scenes.cornell_box()
    s.accel = capi.ACCEL_BVH4
    desc, keep = s.to_desc()
    gpu_ctx.upload_scene(desc)
    o, d = scenes.random_rays(((0.1, 0.1, 0.1), (5, 5, 5)), n, seed=2)
    tmin, tmax = np.zeros(n, np.float32), np.full(n, 9.0, np.float32)
    print(f"[ray parts] {n} rays, any_hit {any_hit}", flush=True)
    full = gpu_ctx.trace_rays(o, d, tmin, tmax, any_hit=any_hit)
    st = gpu_ctx.stats()
    assert st["trace_shadow_launches" if any_hit else "trace_closest_launches"] == 2
    tests = 0
    for a, b in ((0, part), (part, n)):
        g = gpu_ctx.trace_rays(o[a:b], d[a:b], tmin[a:b], tmax[a:b], any_hit=any_hit)
        tests += gpu_ctx.stats()["shadow_tri_tests" if any_hit else "closest_tri_tests"]
        for k in ("entity",) if any_hit else ("entity", "prim", "t", "u", "v"):
            np.testing.assert_array_equal(full[k][a:b].view(np.uint32), g[k].view(np.uint32))
    assert tests == st["shadow_tri_tests" if any_hit else "closest_tri_tests"]


@pytest.mark.parametrize("n", [100, 40_000])
def test_queries_do_not_wait_for_the_default_stream(n):
    """A query uses its context's stream alone: it returns while work that another
    library put on the default stream is still running.  Streams share a few hardware
    queues, and one that shares the default stream's waits for it all the same: of eight contexts
    some do not."""
    torch = pytest.importorskip("torch")
    s, _, _ = scenes.cornell_box()
    s.accel = capi.ACCEL_BVH4
    desc, keep = s.to_desc()
    o, d = scenes.random_rays(((0.1, 0.1, 0.1), (5, 5, 5)), n, seed=1)
    tmin, tmax = np.zeros(n, np.float32), np.full(n, np.inf, np.float32)
    x = torch.randn(8192, 8192, device="cuda:0")
    y = torch.empty_like(x)
    torch.mm(x, x, out=y)
    torch.cuda.synchronize()
    ctxs = [capi.Context(0) for _ in range(8)]
    early = 0
    for ctx in ctxs:
        ctx.upload_scene(desc)
        a = ctx.trace_rays(o, d, tmin, tmax)
        torch.cuda.synchronize()
        for _ in range(12):  # some 0.1 s of products of 8 ms
            torch.mm(x, x, out=y)
        end = torch.cuda.Event()
        end.record()
        b = ctx.trace_rays(o, d, tmin, tmax)
        early += not end.query()
        torch.cuda.synchronize()
        for k in a:
            np.testing.assert_array_equal(a[k].view(np.uint32), b[k].view(np.uint32))
    for ctx in ctxs:
        ctx.close()
    print(f"[ray streams] {n} rays: {early} of 8 contexts returned early", flush=True)
    assert early > 0


def _query_scene(ctx):
    s, _, _ = scenes.procedural_spheres(n_spheres=8, subdiv=2, seed=3, extent=12.0)
    s.accel = capi.ACCEL_BVH4
    desc, keep = s.to_desc()
    ctx.upload_scene(desc)


def _query(n):
    o, d = scenes.random_rays(((-2, -2, -2), (14, 14, 14)), n, seed=n)
    return o, d, np.full(n, 0.01, np.float32), np.full(n, 40.0, np.float32)


def test_pinned_staging_grows_with_the_calls():
    """Calls of a new context in an order that takes the staging through its
    sizes: exact powers of two and one more, and the same size until it turns to pinned memory."""
    with capi.Context(0) as ctx:
        _query_scene(ctx)
        for n in (1, 1024, 1025, 2048, 4096, 4097, 4097, 4097, 4097, 4097, 4097, 8192, 8193, 3, 32768, 32768, 32768,
                  32768, 32768, 32768, 20000, 32769, 4096):
            q = _query(n)
            print(f"[ray staging] {n} rays", flush=True)
            for any_hit in (False, True):
                a = ctx.trace_rays(*q, any_hit=any_hit)
                sa = ctx.stats()
                b = ctx.trace_rays(*q, any_hit=any_hit, noalloc=True)
                sb = ctx.stats()
                for k in ("entity",) if any_hit else ("entity", "prim", "t", "u", "v"):
                    np.testing.assert_array_equal(a[k].view(np.uint32), b[k].view(np.uint32))
                for k in ("closest_tri_tests", "shadow_tri_tests", "closest_hits"):
                    assert sa[k] == sb[k], (n, k)


def test_first_call_of_a_context():
    """A context's first call of 32,768 rays, just within the pinned staging's
    range, takes about as long as one of 33,000 through the device staging (the whole buffer
    made in that call took 2.4 times as long)."""
    def first(n):
        q, times, keep = _query(n), [], []
        for _ in range(7):  # contexts stay open: memory that a closed one gave back is cheap to get again
            ctx = capi.Context(0)
            keep.append(ctx)
            _query_scene(ctx)
            t = time.perf_counter()
            ctx.trace_rays(*q)
            times.append(time.perf_counter() - t)
        for ctx in keep:
            ctx.close()
        return sorted(times)[3]

    first(100)
    a, b = first(32768), first(33000)
    print(f"[ray staging] first call: 32768 rays {a * 1e6:.0f} us, 33000 rays {b * 1e6:.0f} us", flush=True)
    assert a < 1.5 * b
