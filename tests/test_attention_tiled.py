"""The tiled relative-position attention (kea_relpos_attention_tiled) and the calls that reach it: relpos_attention at
129 .. 256 frames and FastConformerEncoder.attention above 256.

Tolerance: a score is two 128-term dot products in FP32 (rounding 2^-24 a step, each operand held to 2^-22 and better),
so it is off by at most about 128 * 2^-23 of the sum of its terms' magnitudes; measured errors are 3e-7 of the output's
largest value, and 2e-6 is the bar of the FP32 kernels."""
from __future__ import annotations

import ctypes
import math

import pytest
import torch

from kea_kernels import _hip, encoder as E

H, DK = 8, 128
D = H * DK


def _inputs(b, t, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(b, t, 3 * D, generator=g) * scale, torch.randn(2 * t - 1, D, generator=g),
            torch.randn(H, DK, generator=g) * 0.1, torch.randn(H, DK, generator=g) * 0.1)


def _reference(qkv, pos, u, v):
    """The definition in FP64: s = ((q + u) k + (q + v) p_{T-1-i+j}) / sqrt(dk), softmax, P V."""
    b, t, _ = qkv.shape
    q, k, vv = (x.transpose(1, 2) for x in qkv.double().view(b, t, 3, H, DK).unbind(2))
    p = pos.double().view(2 * t - 1, H, DK).permute(1, 2, 0)
    i = torch.arange(t)
    band = ((q + v.double()[:, None]) @ p).gather(3, (t - 1 - i[:, None] + i[None]).expand(b, H, t, t))
    a = torch.softmax(((q + u.double()[:, None]) @ k.transpose(2, 3) + band) / math.sqrt(DK), -1)
    return (a @ vv).transpose(1, 2).reshape(b, t, D)


def _tiled(qkv, pos, u, v, ld=3 * D, ldo=D):
    """The C entry on device tensors, into a poisoned output and workspace."""
    L, (b, t, _) = _hip.lib(), qkv.shape
    out = torch.full((b, t, ldo), 7.0, device="cuda")
    need = L.kea_relpos_attention_tiled_workspace(b, t, H)
    ws = torch.full((need,), 255, dtype=torch.uint8, device="cuda")
    _hip.check(L.kea_relpos_attention_tiled(qkv.data_ptr(), ld, pos.data_ptr(), pos.stride(0), u.data_ptr(),
                                            v.data_ptr(), out.data_ptr(), ldo, b, t, H, DK, 1 / math.sqrt(DK),
                                            ws.data_ptr(), need, _hip.stream_handle(out.device)), "tiled")
    return out.cpu()


def _close(got, ref, tol=2e-6):
    assert torch.isfinite(got).all()
    assert float((got.double() - ref).abs().max() / ref.abs().max()) < tol


@pytest.mark.gpu
@pytest.mark.parametrize("b,t", [(1, 1), (2, 15), (1, 32), (2, 63), (1, 64), (3, 65), (1, 97), (1, 128), (2, 129),
                                 (1, 191), (1, 192), (1, 193), (1, 257), (2, 300), (1, 521), (1, 1000)])
def test_every_tile_edge_matches_fp64(b, t):
    x = _inputs(b, t, 31 * b + t)
    _close(_tiled(*(a.cuda() for a in x)), _reference(*x))


@pytest.mark.gpu
@pytest.mark.parametrize("scale_v", [1e-30, 1e-6, 1e6, 1e30])
def test_any_magnitude_of_values(scale_v):
    """Values far outside FP16's range, and a key whose value row is 2^20 times the others'."""
    qkv, pos, u, v = _inputs(1, 200, 5)
    qkv[..., 2 * D:] *= scale_v
    qkv[0, 70, 2 * D:] *= 2.0 ** 20
    qkv[0, 70, D:2 * D] = 0.0
    ref = _reference(qkv, pos, u, v)
    _close(_tiled(*(a.cuda() for a in (qkv, pos, u, v))) / scale_v, ref / scale_v)


def _row_error(got, ref):
    """The largest error of an output row (one query and head) over that row's own largest element."""
    got, ref = (x.double().view(*x.shape[:2], H, DK) for x in (got, ref))
    return float(((got - ref).abs().amax(-1) / ref.abs().amax(-1)).max())


@pytest.mark.gpu
@pytest.mark.parametrize("key", [0, 69, 199])
@pytest.mark.parametrize("power,score", [(12, -60), (20, -60), (40, -60), (100, -200)])
def test_large_values_under_a_suppressed_key(key, power, score):
    """One key of next to no probability whose value row is 2^power times the others': every output row is as accurate,
    for its own size, as FP32 is. (FP32: 200 roundings of 2^-24, of random sign, and scores of size 4 off by 2^-22.)"""
    qkv, pos, u, v = _inputs(1, 200, 7)
    q, k = qkv[..., :D].view(1, 200, H, DK), qkv[..., D:2 * D].view(1, 200, H, DK)
    q[..., 0], k[..., 0], u[:, 0] = 4.0, 0.0, 0.0
    k[:, key] = 0.0
    k[:, key, :, 0] = score * math.sqrt(DK) / 4.0
    qkv[:, key, 2 * D:] *= 2.0 ** power
    assert _row_error(_tiled(*(a.cuda() for a in (qkv, pos, u, v))), _reference(qkv, pos, u, v)) < 2e-6


@pytest.mark.gpu
@pytest.mark.parametrize("key", [0, 69, 199])
@pytest.mark.parametrize("small,large", [(-60, 90), (-100, 120), (-20, 127)])
def test_large_values_under_a_key_without_probability(key, small, large):
    """A key whose probability is zero in FP32 (2^-288) and whose value row is 2^147 to 2^220 times the others': it adds
    nothing to any output, whatever its exponent, so the bar is that of a suppressed key."""
    qkv, pos, u, v = _inputs(1, 200, 18)
    q, k = qkv[..., :D].view(1, 200, H, DK), qkv[..., D:2 * D].view(1, 200, H, DK)
    q[..., 0], k[..., 0], u[:, 0] = 4.0, 0.0, 0.0
    k[:, key] = 0.0
    k[:, key, :, 0] = -200 * math.sqrt(DK) / 4.0
    qkv[..., 2 * D:] *= 2.0 ** small
    qkv[:, key, 2 * D:] = torch.sign(qkv[:, key, 2 * D:]) * 2.0 ** large
    assert _row_error(_tiled(*(a.cuda() for a in (qkv, pos, u, v))), _reference(qkv, pos, u, v)) < 2e-6


@pytest.mark.gpu
@pytest.mark.parametrize("power", [9, 11, 13, 15, 20, 60])
@pytest.mark.parametrize("operand", ["k_row", "k_dim", "q_row", "q_dim", "p_row", "p_dim", "v_element", "v_half"])
def test_rows_and_elements_of_any_size(operand, power):
    """A row 2^power times its neighbours, or a few elements that much larger than the rest of their rows, where the other
    operand is zero: the scores they leave ordinary, and every other element of the output, are as accurate as in FP32
    (the bar of the kernels that serve up to 128 frames, here for each row's own size)."""
    b, t = 1, 150
    qkv, pos, u, v = _inputs(b, t, 14)
    x = {"q": qkv[..., :D], "k": qkv[..., D:2 * D], "v": qkv[..., 2 * D:], "p": pos[None]}
    heads = {name: y.unflatten(-1, (H, DK)) for name, y in x.items()}
    big, want = 2.0 ** power, slice(None)
    if operand in ("k_row", "p_row", "q_row"):      # the row's product: one score far below the others, or an unused row
        heads[operand[0]][:, 70, :, 1:] = 0.0
        heads[operand[0]][:, 70, :, 0] = -big if operand != "q_row" else big
        heads["q"][..., 0] = u[:, 0] = v[:, 0] = 0.0
        if operand == "q_row":
            heads["q"][:, 70, :, 0], heads["k"][..., 0], heads["p"][..., 0] = big, 0.0, 0.0
        else:
            heads["q"][:, :, :, 0] = 1.0
    elif operand in ("k_dim", "p_dim", "q_dim"):    # elements that the other operand has no use for
        heads[operand[0]][..., 5] *= big
        for other in "kp" if operand == "q_dim" else "q":
            heads[other][..., 5] = 0.0
        if operand != "q_dim":
            u[:, 5] = v[:, 5] = 0.0
    elif operand == "v_element":
        heads["v"][:, 70, :, 3] *= big
        want = [d for d in range(DK) if d != 3]
    else:
        heads["v"][:, :, :, 64:] *= big
        want = slice(0, 64)
    got, ref = _tiled(*(a.cuda() for a in (qkv, pos, u, v))), _reference(qkv, pos, u, v)
    assert torch.isfinite(got).all()
    got, ref = (y.double().view(b, t, H, DK)[..., want] for y in (got, ref))
    worst = float(((got - ref).abs().amax(-1) / ref.abs().amax(-1)).max())
    print(operand, power, worst)
    assert worst < 4e-6


@pytest.mark.gpu
@pytest.mark.parametrize("scale_v", [1e-37, 1e-34, 1e36])
def test_values_near_the_ends_of_the_range(scale_v):
    qkv, pos, u, v = _inputs(1, 140, 15)
    qkv[..., 2 * D:] *= scale_v
    assert _row_error(_tiled(*(a.cuda() for a in (qkv, pos, u, v))), _reference(qkv, pos, u, v)) < 2e-6


@pytest.mark.gpu
@pytest.mark.parametrize("b,t", [(1, 1), (2, 15), (1, 33), (3, 65), (2, 129), (1, 193), (2, 300), (1, 521)])
def test_the_fp32_form_at_every_tile_edge(b, t):
    """Half of the heads have keys with an element past the split form's bound that no query uses, so their workgroups run
    the FP32 form."""
    qkv, pos, u, v = _inputs(b, t, 16 + t)
    q, k, _ = (x.view(b, t, H, DK) for x in qkv.split(D, 2))
    k[:, :, ::2, 9] *= 2.0 ** 30
    q[:, :, ::2, 9] = u[::2, 9] = v[::2, 9] = 0.0
    _close(_tiled(*(a.cuda() for a in (qkv, pos, u, v))), _reference(qkv, pos, u, v))


@pytest.mark.gpu
def test_large_scores_and_small_queries():
    """Scores in the hundreds (a sharp softmax) hold the FP32 error of a score, 2^-24 of its terms; tiny queries give
    the mean of the values."""
    qkv, pos, u, v = _inputs(1, 150, 6)
    qkv[..., :2 * D] *= 8.0
    got, ref = _tiled(*(a.cuda() for a in (qkv, pos, u, v))), _reference(qkv, pos, u, v)
    assert float((got.double() - ref).norm() / ref.norm()) < 1e-4
    qkv[..., :D] = 0.0
    u, v = u * 1e-30, v * 1e-30
    _close(_tiled(*(a.cuda() for a in (qkv, pos, u, v))), _reference(qkv, pos, u, v))


@pytest.mark.gpu
def test_row_strides():
    """Rows of a wider matrix: qkv with ld > 3 d, pos with ldp > d, out with ldo > d (columns past d untouched)."""
    qkv, pos, u, v = _inputs(2, 140, 8)
    wide = torch.randn(2, 140, 3 * D + 8)
    wide[..., :3 * D] = qkv
    widep = torch.randn(279, D + 4)
    widep[:, :D] = pos
    got = _tiled(wide.cuda(), widep.cuda()[:, :D], u.cuda(), v.cuda(), ld=3 * D + 8, ldo=D + 4)
    _close(got[..., :D], _reference(qkv, pos, u, v))
    assert bool((got[..., D:] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("where", ["v_inf", "v_nan", "k_inf", "k_nan", "q_inf", "p_inf"])
def test_non_finite_inputs_as_the_formula(where):
    """An infinity or NaN reaches exactly the outputs the FP32 formula gives it to."""
    qkv, pos, u, v = _inputs(2, 300, 9)
    bad = math.inf if where.endswith("inf") else math.nan
    part = {"q": 0, "k": D, "v": 2 * D}
    if where[0] == "p":
        pos[310, 130] = bad
    else:
        qkv[1, 200, part[where[0]] + 130] = bad
    got = _tiled(*(a.cuda() for a in (qkv, pos, u, v)))
    ref = _reference(qkv, pos, u, v).float()
    assert torch.equal(torch.isnan(got), torch.isnan(ref)) and torch.equal(torch.isinf(got), torch.isinf(ref))
    fine = torch.isfinite(ref)
    assert float((got - ref)[fine].abs().max()) < 2e-6 * float(ref[fine].abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("where,row", [("v", 4290), ("k", 4170), ("v", 4230)])
def test_infinities_past_the_64th_key_block(where, row):
    """More key blocks than a wave looks over: the block that holds the infinity is seen by one wave other than the first."""
    t, L = 4300, _hip.lib()
    g = torch.Generator().manual_seed(12)
    qkv, pos = torch.randn(1, t, 3 * DK, generator=g), torch.randn(2 * t - 1, DK, generator=g)
    u, v = torch.randn(1, DK, generator=g) * 0.1, torch.randn(1, DK, generator=g) * 0.1
    qkv[0, row, {"k": DK, "v": 2 * DK}[where] + 3] = math.inf
    dev = [a.cuda() for a in (qkv, pos, u, v)]
    out = torch.full((1, t, DK), 7.0, device="cuda")
    ws = torch.empty(L.kea_relpos_attention_tiled_workspace(1, t, 1), dtype=torch.uint8, device="cuda")
    _hip.check(L.kea_relpos_attention_tiled(dev[0].data_ptr(), 3 * DK, dev[1].data_ptr(), DK, dev[2].data_ptr(),
                                            dev[3].data_ptr(), out.data_ptr(), DK, 1, t, 1, DK, 1 / math.sqrt(DK),
                                            ws.data_ptr(), ws.numel(), _hip.stream_handle(out.device)), "tiled")
    got, rows = out[0].cpu(), torch.tensor([0, 63, 64, 2000, 4299])      # (the reference: a few queries of each kind)
    q, k, vv = qkv[0].double().split(DK, 1)
    j = torch.arange(t)
    for i in rows.tolist():
        s = ((q[i] + u[0].double()) * k).sum(1) + ((q[i] + v[0].double()) * pos[t - 1 - i + j].double()).sum(1)
        p = torch.softmax(s / math.sqrt(DK), 0)
        ref = (p[:, None] * vv).sum(0).float()
        fine = torch.isfinite(ref)
        assert torch.equal(torch.isnan(got[i]), torch.isnan(ref)) and torch.equal(torch.isinf(got[i]), torch.isinf(ref))
        assert not fine.any() or float((got[i] - ref)[fine].abs().max()) < 1e-5 * float(ref[fine].abs().max())


@pytest.mark.gpu
def test_layer_attention_routes(monkeypatch):
    """FastConformerEncoder.attention above 256 frames: the tiled kernel for plain FP32 tensors, the PyTorch form for
    what only it takes, the same values either way; relpos_attention still refuses more than 256 frames."""
    model = E.FastConformerEncoder(E.synthetic_weights(E.EncoderConfig(layers=1)), E.EncoderConfig(layers=1))
    x = _inputs(2, 270, 10)
    qkv, pos, u, v = (a.cuda() for a in x)
    calls = []
    tiled = E._attention_tiled
    monkeypatch.setattr(E, "_attention_tiled", lambda *a: calls.append(1) or tiled(*a))
    ref = _reference(*x)
    _close(model.attention(qkv, pos, u, v).cpu(), ref)
    assert calls == [1]
    wide = torch.cat([qkv, qkv], -1)
    _close(model.attention(wide[..., :3 * D], pos, u, v).cpu(), ref)     # a row stride of 6 d
    assert calls == [1, 1]
    off = torch.cat([torch.zeros(2 * D + 1, device="cuda"), qkv.flatten()])[2 * D + 1:].view_as(qkv)
    _close(model.attention(off, pos, u, v).cpu(), ref, 1e-5)                   # misaligned
    _close(model.attention(qkv, pos.t().contiguous().t(), u, v).cpu(), ref, 1e-5)
    g = qkv.clone().requires_grad_()
    out = model.attention(g, pos, u, v)                                        # recorded by autograd
    assert out.requires_grad
    _close(out.detach().cpu(), ref, 1e-5)
    with torch.no_grad():
        _close(model.attention(g, pos, u, v).cpu(), ref)
    assert calls == [1, 1, 1]
    batched = torch.func.vmap(lambda q: model.attention(q, pos, u, v))(torch.stack([qkv, 2 * qkv]))
    _close(batched[0].cpu(), ref, 1e-5)
    class Watching(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Watching():                                                           # a mode that may rewrite operators
        _close(model.attention(qkv, pos, u, v).cpu(), ref, 1e-5)
    with pytest.raises((ValueError, RuntimeError)):
        model.attention(qkv.double(), pos, u, v)                               # mixed types: PyTorch refuses
    assert calls == [1, 1, 1]
    with pytest.raises(ValueError, match="256 frames"):
        E.relpos_attention(qkv, pos, u, v, H)
    with torch.device("cuda"):                                                 # a default device is no such mode
        _close(model.attention(qkv, pos, u, v).cpu(), ref)
    assert calls == [1, 1, 1, 1]


@pytest.mark.gpu
def test_scratch_is_bounded_whatever_the_batch():
    """300 clips, 0.94 GB of workspace in one call, with the bound lowered: the scratch stays below it, the bits are a
    single clip's; an empty batch allocates nothing to speak of."""
    b, t, bound = 300, 130, 64 << 20
    qkv = torch.randn(b, t, 3 * D, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    _, pos, u, v = (a.cuda() for a in _inputs(1, t, 17))
    want = [E.relpos_attention(qkv[i:i + 1], pos, u, v, H) for i in (0, 1, 157, 299)]
    torch.cuda.synchronize()
    keep, E.ATTENTION_SCRATCH = getattr(E, "ATTENTION_SCRATCH", None), bound
    try:
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        got = E.relpos_attention(qkv, pos, u, v, H)
        peak = torch.cuda.max_memory_allocated() - before - got.numel() * 4
    finally:
        E.ATTENTION_SCRATCH = keep
    assert peak <= bound + 512
    assert all(torch.equal(got[i], w[0]) for i, w in zip((0, 1, 157, 299), want))
    assert E.relpos_attention(qkv[:0], pos, u, v, H).shape == (0, t, D)


@pytest.mark.gpu
def test_graph_replays_equal_eager():
    """Captured with its workspace from the graph's pool; every replay equals the eager result on new inputs."""
    qkv, pos, u, v = (a.cuda() for a in _inputs(1, 200, 11))
    E.relpos_attention(qkv, pos, u, v, H)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        out = E.relpos_attention(qkv, pos, u, v, H)
    for seed in range(3):
        qkv.copy_(_inputs(1, 200, 20 + seed)[0].cuda())
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, E.relpos_attention(qkv, pos, u, v, H))


def test_refusals_before_any_launch():
    L = _hip.lib()
    need = L.kea_relpos_attention_tiled_workspace(1, 300, 8)
    assert need > 0 and need % 16 == 0
    assert L.kea_relpos_attention_tiled_workspace(0, 300, 8) == 0 == L.kea_relpos_attention_tiled_workspace(1, 0, 8)
    assert L.kea_relpos_attention_tiled_workspace(1, 65535 * 64 + 1, 1) == 0
    q = ctypes.c_void_p(0x1000)

    def call(x=q, ld=3072, ldp=1024, ldo=1024, t=300, dk=128, ws=q, nbytes=need):
        return L.kea_relpos_attention_tiled(x, ld, q, ldp, q, q, q, ldo, 1, t, 8, dk, 1.0, ws, nbytes, None)

    assert call(dk=64) == -1 and call(t=0) == -1 and call(ld=3068) == -1 and call(ldp=1020) == -1 and call(x=None) == -1
    assert call(x=ctypes.c_void_p(0x1004)) == -2 and call(ldo=1026) == -2 and call(ws=ctypes.c_void_p(0x1008)) == -2
    assert call(nbytes=need - 1) == -4 and call(ws=None) == -4
    assert L.kea_relpos_attention_tiled(q, 3072, q, 1024, q, q, q, 1024, 0, 300, 8, 128, 1.0, q, need, None) == 0
