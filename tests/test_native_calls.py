"""The operators' native call path (kea_native: Replays, gemm, quantize): the same results as the Python path, and
everything it does not take left to that path."""
from __future__ import annotations

import sys
import threading

import pytest
import torch

from kea_kernels import _hip, formats, lowbit
from kea_kernels.binary import bits, layer_parts
from kea_kernels.ternary import fused_kernels, runtime

DEV = "cuda"


def _layer(n=260, k=272, parts=2, bias=True):
    g = torch.Generator().manual_seed(n + k)
    codes = bits.pack_signs(torch.where(torch.rand(n, k, generator=g) < 0.5, -1, 1).to(torch.int8))
    scale = torch.rand(n, generator=g) + 0.5
    return layer_parts.LAYERS[parts].prepare(codes, scale, torch.randn(n, generator=g) if bias else None, k, DEV)


def _python_path(monkeypatch):
    """Switches the native path off."""
    monkeypatch.setattr(lowbit, "_native_gemm", lambda *a: False)
    monkeypatch.setattr(lowbit, "_native_quantize", lambda *a: None)


def _inputs(k):
    g = torch.Generator().manual_seed(k)
    x = torch.randn(3, 7, k, generator=g).to(DEV)
    return [x, x[0], x[0, 0], x.half(), x[:, ::2], x[:, :, :].transpose(0, 1), torch.cat([x, x], -1)[..., :k]]


@pytest.mark.gpu
@torch.inference_mode()
def test_replayed_operator_calls_equal_the_first():
    """linear, conv, project and the ternary call on every kind of view: the second (replayed) call gives the first
    (checked) call's bits, shape and strides."""
    layer = _layer()
    norm = torch.nn.LayerNorm(272, device=DEV)
    norm.weight.uniform_(0.5, 1.5)
    for x in _inputs(272):
        calls = [lambda: layer.linear(x), lambda: layer.linear(x, out_dtype=torch.bfloat16)]
        if x.dim() == 3:
            xc = x.transpose(1, 2)
            calls += [lambda: layer.conv(xc), lambda: layer.project(xc, conv=True, components=3, activation="silu")]
        if x.dim() >= 2:
            calls += [lambda: layer.project(x, components=1, norm=norm, input_activation="silu"),
                      lambda: layer.project(x, components=2, activation="silu", norm=norm)]
        for call in calls:
            first, again = call(), call()
            assert torch.equal(first, again) and first.stride() == again.stride() and first.dtype == again.dtype
            assert first.data_ptr() != again.data_ptr()


@pytest.mark.gpu
def test_ternary_calls_replay_and_follow_the_module():
    g = torch.Generator().manual_seed(1)
    codes = formats.pack_ternary(torch.randint(-1, 2, (96, 128), generator=g, dtype=torch.int8))
    mod = runtime.PackedLinear(codes, torch.rand(96, generator=g), 128, mode="x2").to(DEV)
    x = torch.randn(5, 128, generator=g).to(DEV)
    first = mod(x)
    assert torch.equal(first, mod(x))
    xc = x.t().reshape(1, 128, 5).contiguous()
    assert torch.equal(fused_kernels.int8_matmul(xc, mod, True, 2), first.t()[None])
    assert torch.equal(fused_kernels.int8_matmul(xc, mod, True, 2), first.t()[None])
    mod.scale = mod.scale * 2                                    # other weights: the kept calls are dropped
    assert torch.equal(mod(x), 2 * first)


@pytest.mark.gpu
def test_calls_left_to_the_python_path():
    layer = _layer()
    x = torch.randn(4, 272, device=DEV)
    want = layer.linear(x)
    replay = layer.launches.replay
    tag = 8 + layer.PARTS
    assert torch.equal(replay(x, torch.float32, tag), want)
    assert replay(x, torch.float16, tag) is None and replay(x[:2], torch.float32, tag) is None
    assert replay(x, torch.float32, tag + 1) is None and replay(x.cpu(), torch.float32, tag) is None
    assert replay("x", torch.float32, tag) is None and replay(x, "f32", tag) is None and replay(x, torch.float32, None) is None
    g = x.clone().requires_grad_()
    with pytest.raises(RuntimeError, match="inference only"):
        layer.linear(g)
    with torch.no_grad():
        assert torch.equal(layer.linear(g), want)
    assert replay(torch.nn.Parameter(x), torch.float32, tag) is None  # a subclass
    seen = []
    torch.func.vmap(lambda v: seen.append(replay(v, torch.float32, tag)) or v)(torch.stack([x, x]))
    assert seen == [None]
    with torch.inference_mode():
        assert layer.linear(x).is_inference()


@pytest.mark.gpu
@torch.inference_mode()
def test_kept_layouts_are_bounded_and_evicted_oldest_first():
    layer = _layer()
    launches = layer.launches
    xs = [torch.randn(m, 272, device=DEV) for m in range(1, launches.max_entries + 3)]
    outs = [layer.linear(x) for x in xs]
    tag = 8 + layer.PARTS
    assert launches.replay(xs[0], torch.float32, tag) is None and launches.replay(xs[1], torch.float32, tag) is None
    assert all(torch.equal(launches.replay(x, torch.float32, tag), o) for x, o in zip(xs[2:], outs[2:]))
    assert all(torch.equal(layer.linear(x), o) for x, o in zip(xs, outs))


@pytest.mark.gpu
@torch.inference_mode()
def test_side_streams_threads_and_graphs():
    """Launches on the caller's current stream, from several threads at once, and captured."""
    layer = _layer()
    x = torch.randn(64, 272, device=DEV)
    want = layer.linear(x)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        layer.linear(x + 1.0)            # the stream's pool has its blocks
        event = torch.cuda.Event()
        torch.cuda.synchronize()
        torch.cuda._sleep(100_000_000)
        z = x + 1.0                      # on the side stream, behind the wait
        got = layer.linear(z)
        event.record()
    assert not event.query()             # the call went behind the wait on its stream
    torch.cuda.synchronize()
    assert torch.equal(got, layer.linear(x + 1.0))
    bad = []

    def work():
        with torch.inference_mode():
            for m in (64, 32, 64, 16):
                if not torch.equal(layer.linear(x[:m]), want[:m]):
                    bad.append(m)

    threads = [threading.Thread(target=work) for _ in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not bad
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = layer.linear(x)
    for i in range(3):
        x.normal_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, layer.linear(x))


@pytest.mark.gpu
@pytest.mark.parametrize("wbits,parts,group,residual,glu,acc", [(1, 1, 0, False, False, False), (2, 3, 128, False, False, True),
                                                                (1, 2, 0, True, False, False), (2, 1, 0, False, True, False)])
@torch.inference_mode()
def test_native_gemm_and_quantize_equal_the_python_path(monkeypatch, wbits, parts, group, residual, glu, acc):
    from kea_kernels.binary import kernels
    m, n, k = 21, 96, 256
    g = torch.Generator().manual_seed(parts)
    codes = torch.randint(0, 256, (n, k // 8), generator=g, dtype=torch.uint8) if wbits == 1 else \
        formats.pack_ternary(torch.randint(-1, 2, (n, k), generator=g, dtype=torch.int8))
    words = kernels.relayout_codes(codes, k, wbits).to(DEV)
    scale = torch.rand(n, k // group if group else 1, generator=g).half().to(DEV)
    x = torch.randn(m, k, generator=g).to(DEV)
    res = torch.randn(m, n, generator=g).to(DEV) if residual else None
    norm = torch.nn.LayerNorm(k, device=DEV)

    def run():
        q, qs, ldq = lowbit.quantize(x, (0, k, 1, m), m, k, parts, norm=norm, input_activation="silu")
        y = torch.full((m, n // 2 if glu else n), 7.0, device=DEV)
        a = torch.full((parts, m, n), 7, device=DEV, dtype=torch.int32) if acc else None
        lowbit.gemm(wbits, q, qs, words, n, k, scale, None, y, a, ws_group=group, residual=res, residual_factor=0.5, glu=glu)
        return [q, qs, y] + ([a] if acc else [])

    assert lowbit._native_quantize(x, (0, k, 1, m), m, k, parts, norm, "", torch.float32, None) is not None
    native = run()
    _python_path(monkeypatch)
    assert all(torch.equal(a, b) for a, b in zip(native, run()))


@pytest.mark.gpu
@torch.inference_mode()
def test_refused_arguments_raise_as_before():
    layer = _layer()
    q, qs, _ = lowbit.quantize(torch.randn(8, 272, device=DEV), (0, 272, 1, 8), 8, 272, 2)
    y = torch.empty(8, 260, device=DEV)

    def gemm(q=q, qs=qs, words=layer.words, scale=layer.scale, y=y, **kw):
        lowbit.gemm(1, q, qs, words, 260, 272, scale, None, y, None, **kw)

    gemm()
    for bad, message in [(dict(q=q.float()), "int8"), (dict(qs=qs[:1]), "qs must be"), (dict(words=layer.words[:10]), "native words"),
                         (dict(scale=layer.scale[:9]), "weight scales"), (dict(y=y[:4]), "row-major"), (dict(m=9), "exceeds"),
                         (dict(qs=qs.cpu()), "expected cuda"), (dict(y=None), "nothing to compute"),
                         (dict(ws_group=96, scale=torch.ones(260, 3, device=DEV)), "ws_group must be"), (dict(residual=y.half()), "residual must be")]:
        with pytest.raises(ValueError, match=message):
            gemm(**bad)
    for rows, m in [((0, 272, 1, 9), 9), ((0, 273, 1, 8), 8), ((0, 272, 2, 8), 8), ((0, -1, 1, 8), 8), ((272, 272, 1, 0), 8)]:
        with pytest.raises(ValueError):
            lowbit.quantize(torch.randn(8, 272, device=DEV), rows, m, 272, 2)


@pytest.mark.gpu
@torch.inference_mode()
def test_a_norm_without_parameters_or_of_another_length_is_refused_whatever_was_kept():
    layer = _layer()
    x = torch.randn(4, 272, device=DEV)
    w = torch.ones(272, device=DEV)
    norm = torch.nn.LayerNorm(272, device=DEV)
    norm.weight, norm.bias = torch.nn.Parameter(w), torch.nn.Parameter(w)
    short = torch.nn.LayerNorm(272, device=DEV)
    short.weight, short.bias = torch.nn.Parameter(w[:100]), torch.nn.Parameter(w[:100])
    assert short.weight.data_ptr() == norm.weight.data_ptr()
    mod = runtime.PackedLinear(formats.pack_ternary(torch.ones(96, 272, dtype=torch.int8)), torch.ones(96), 272, mode="x1").to(DEV)
    for call in (lambda norm: layer.project(x, components=1, norm=norm), lambda norm: fused_kernels.int8_matmul(x, mod, norm=norm)):
        for _ in range(2):
            assert not torch.equal(call(None), call(norm))
        with pytest.raises(AttributeError):
            call(torch.nn.LayerNorm(272, elementwise_affine=False))
        with pytest.raises(ValueError, match="LayerNorm shape"):
            call(short)


class _Owner:
    """A stand-in for a plan's owner that keeps another one when it is dropped."""

    def __init__(self, dropped=None):
        self.dropped = dropped

    def __del__(self):
        if self.dropped:
            self.dropped()


def _keep(replays, x, owner, need=0):
    replays.keep(x, torch.float32, 1, None, None, 0.0, owner, 0, need, (4, 16), False)


@pytest.mark.gpu
def test_a_failed_allocation_releases_the_owner():
    replays, x, owner = _hip.native().Replays(4), torch.randn(4, 16, device=DEV), _Owner()
    _keep(replays, x, owner, 1 << 60)
    count = sys.getrefcount(owner)
    assert replays.call(x, torch.float32, 1) is None and sys.getrefcount(owner) == count
    del replays
    assert sys.getrefcount(owner) == count - 1


@pytest.mark.gpu
def test_keeping_while_an_owner_is_released_stays_bounded():
    """Releasing an evicted plan may run other code that keeps a layout: the limit holds, and nothing is lost or doubled."""
    replays, xs = _hip.native().Replays(1), [torch.randn(m, 16, device=DEV) for m in (4, 5, 6)]
    inner, outer = _Owner(), _Owner()
    free = sys.getrefcount(inner), sys.getrefcount(outer)
    kept = lambda: (sys.getrefcount(inner) - free[0], sys.getrefcount(outer) - free[1])  # noqa: E731
    _keep(replays, xs[0], _Owner(lambda: _keep(replays, xs[1], inner)))
    _keep(replays, xs[2], outer)                 # evicts the first, whose release keeps `inner`, which evicts `outer`
    assert kept() == (1, 0)
    _keep(replays, xs[2], outer)
    assert kept() == (0, 1)
    del replays
    assert kept() == (0, 0)


def test_the_module_is_bound_and_declines_cpu_tensors():
    native = _hip.native()
    x = torch.randn(2, 16)
    assert native.quantize(x, 0, 16, 1, 2, 2, 16, 1, None, None, 0.0, False, torch.float32, 16) is None
    assert native.Replays(4).call(x, torch.float32, 1) is None
    assert lowbit._native_gemm(1, x, x, x, 16, 16, x, None, x, None, None, False, 0, None, 0, None, 1.0, False) is False
