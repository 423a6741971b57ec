"""The split-FP16 subsampling (kea_subsample_stage1 / stage2 / out) against FP64 at the edges of its tiles: single frames, output
rows that end inside a tile of four, several clips; infinities and NaN take the plain FP32 sums of the general kernels."""
import math

import pytest
import torch
import torch.nn.functional as F

from kea_kernels import encoder as E

FRAMES = [1, 2, 3, 5, 8, 13, 16, 17, 31, 32, 33, 36, 37, 63, 65, 129, 257, 1000]


def model():
    cfg = E.EncoderConfig(layers=1)
    return E.FastConformerEncoder(E.synthetic_weights(cfg, seed=4), cfg, "cuda", parts=1)


def exact(enc, feats):
    s, c = {k: v.double().cpu() for k, v in enc.sub.items()}, enc.cfg.sub_channels
    x = feats.double().cpu().transpose(1, 2).unsqueeze(1)
    x = F.relu(F.conv2d(x, s["conv.0.weight"], s["conv.0.bias"], stride=2, padding=1))
    for i in (2, 5):
        x = F.conv2d(x, s[f"conv.{i}.weight"], s[f"conv.{i}.bias"], stride=2, padding=1, groups=c)
        x = F.relu(F.conv2d(x, s[f"conv.{i + 1}.weight"], s[f"conv.{i + 1}.bias"]))
    b, _, t, f = x.shape
    return F.linear(x.transpose(1, 2).reshape(b, t, c * f), s["out.weight"], s["out.bias"]) * math.sqrt(enc.cfg.d_model)


def general(enc, feats):
    split, enc._sub_split = enc._sub_split, None
    try:
        return enc._subsample_fused(feats)
    finally:
        enc._sub_split = split


@pytest.mark.parametrize("n,k", [(16, 32), (256, 256)])
def test_split_weights_hold_fp32(n, k):
    """hi + lo is the weight to 2^-22 of itself or 2^-39 of its row's largest, and the fragments are a permutation."""
    g = torch.Generator().manual_seed(n)
    w = torch.randn(n, k, generator=g) * torch.exp(3 * torch.randn(n, k, generator=g)) * 2.0 ** torch.randint(-80, 80, (n, 1), generator=g)
    hi, lo, m = E._split_f16(w)
    back = (hi.double() + lo.double()) * m.double()[:, None]
    bound = torch.maximum(w.double().abs() * 2.0**-22, w.double().abs().amax(1, keepdim=True) * 2.0**-39)
    assert bool(((back - w.double()).abs() <= bound).all())
    f = E._fragments([hi, lo])
    i, ks, gq = 5, k // 32 - 1, 3
    assert torch.equal(f[0, ks, 1, gq, i], lo[i, 32 * ks + 8 * gq:32 * ks + 8 * gq + 8])
    assert torch.equal(f.reshape(-1).view(torch.int16).sort()[0],
                       torch.cat([hi, lo]).reshape(-1).view(torch.int16).sort()[0])


@pytest.mark.parametrize("change,taken", [(None, True), ("inf", False), ("nan", False), ("tiny_row", False), ("zero_row", True),
                                          ("bias", False), ("channels", False), ("huge", False), ("large_first", False),
                                          ("large_second", False), ("wide_row", False), ("wide_out", False),
                                          ("wide_channels", False), ("wide_second", False), ("wide_last", False)])
def test_models_that_are_taken(change, taken):
    """What has no split form, or is of another size, stays on the general kernels."""
    cfg = E.EncoderConfig(layers=1, sub_channels=128 if change == "channels" else 256)
    p = "encoder.pre_encode."
    s = {k[len(p):]: v.float().clone() for k, v in E.synthetic_weights(cfg, seed=4).items() if k.startswith(p)}
    if change in ("inf", "nan"):
        s["conv.3.weight"].view(-1)[7] = float(change)
    elif change in ("tiny_row", "zero_row"):
        s["conv.0.weight"][5] = 1e-10 if change == "tiny_row" else 0.0
    elif change in ("wide_channels", "wide_second", "wide_last"):
        if change == "wide_channels":                # (each layer within its own range)
            s["conv.0.weight"][11] *= 2.0**5
        s[{"wide_channels": "conv.2.weight", "wide_second": "conv.5.weight", "wide_last": "conv.6.weight"}[change]][11] *= (
            2.0**12 if change == "wide_channels" else 2.0**17)
    elif change in ("wide_row", "wide_out"):
        s["conv.3.weight" if change == "wide_row" else "out.weight"][7, 7] = 2.0**18
    elif change == "huge":
        s["out.weight"][7, 7] = 2.0**81
    elif change in ("large_first", "large_second"):
        s["conv.0.weight" if change == "large_first" else "conv.2.weight"][7] = 1e4
    elif change == "bias":
        s["conv.0.bias"][9] = 1e5
    assert (E._SplitSubsampling.prepare(s, cfg) is not None) == taken


@pytest.mark.gpu
@pytest.mark.parametrize("b,frames", [(1 + i % 3, t) for i, t in enumerate(FRAMES)])
@torch.inference_mode()
def test_matches_exact(b, frames):
    """FP32 accuracy: every operand is held to 2^-22 and sums are FP32, so the root mean square error is no larger than
    the general kernels', and no element is off by more than the 1e-5 of the largest output that those are held to."""
    enc = model()
    assert enc._sub_split is not None
    feats = torch.randn(b, 128, frames, generator=torch.Generator().manual_seed(frames)).cuda()
    want, got, old = exact(enc, feats), enc.subsample(feats).double().cpu(), general(enc, feats).double().cpu()
    assert got.shape == want.shape == old.shape
    top = float(want.abs().max())
    rms, rms_old = ((got - want).square().mean().sqrt() / top, (old - want).square().mean().sqrt() / top)
    print(b, frames, float(rms), float(rms_old), float((got - want).abs().max()) / top)
    assert float((got - want).abs().max()) < 1e-5 * top and rms <= rms_old


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1e-30, 1e-6, 1e6, 1e30])
@torch.inference_mode()
def test_any_magnitude(scale):
    """Power-of-two scales per tile and position: accuracy does not depend on the size of the features."""
    enc = model()
    feats = (torch.randn(2, 128, 50, generator=torch.Generator().manual_seed(1)) * scale).cuda()
    want, got = exact(enc, feats), enc.subsample(feats).double().cpu()
    assert float((got - want).abs().max() / want.abs().max()) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("value", [float("inf"), -float("inf"), float("nan"), 3e38])
@torch.inference_mode()
def test_special_values_as_general(value):
    """An infinite, NaN or near-overflow feature gives what the general kernels give: the same elements finite, and those
    close; the rest the same kind."""
    enc = model()
    feats = torch.randn(2, 128, 200, generator=torch.Generator().manual_seed(2)).cuda()
    feats[1, 77, 90] = value
    got, want = enc.subsample(feats), general(enc, feats)
    assert torch.equal(got[0], enc.subsample(feats[:1])[0])
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    ok = torch.isfinite(want)
    assert float((got[ok] - want[ok]).abs().max()) <= 1e-5 * float(want[ok].abs().max())


def _row_error(got, want):
    """The largest error of an output row (one frame of one clip) over that row's own largest element."""
    return float(((got - want).abs().amax(-1) / want.abs().amax(-1)).max())


@pytest.mark.gpu
@pytest.mark.parametrize("mel,frame", [(0, 86), (77, 88), (127, 90)])
@pytest.mark.parametrize("power", [10, 16, 24, 40, 100])
@torch.inference_mode()
def test_a_large_feature_is_seen_by_its_own_rows_only(mel, frame, power):
    """One feature 2^power times the others: every output row is as accurate, for its own size, as the general kernels'
    (the rows of the same tile that do not see it among them), and those rows hold the bits of a clip without it up to FP32
    rounding."""
    enc = model()
    feats = torch.randn(2, 128, 200, generator=torch.Generator().manual_seed(3)).cuda()
    plain = enc.subsample(feats).double().cpu()
    feats[1, mel, frame] *= 2.0**power
    want, got, old = exact(enc, feats), enc.subsample(feats).double().cpu(), general(enc, feats).double().cpu()
    print(mel, frame, power, _row_error(got, want), _row_error(old, want))
    assert _row_error(got, want) <= 2 * _row_error(old, want)
    away = (8 * torch.arange(25) - frame).abs() > 7           # an output frame t sees 8 t - 7 .. 8 t + 7
    assert _row_error(got[1, away], plain[1, away]) < 4e-6


@pytest.mark.gpu
@torch.inference_mode()
def test_features_of_mixed_sizes():
    """Frames and mel bands whose sizes differ by up to 2^40, zeros between them."""
    enc = model()
    g = torch.Generator().manual_seed(4)
    feats = torch.randn(2, 128, 130, generator=g) * 2.0 ** torch.randint(-20, 20, (2, 128, 130), generator=g)
    feats[0, :, :31] *= 2.0**40
    feats[0, 40:90] *= 2.0**-30
    feats[1] *= (torch.rand(128, 130, generator=g) < 0.1)
    feats = feats.cuda()
    want, got, old = exact(enc, feats), enc.subsample(feats).double().cpu(), general(enc, feats).double().cpu()
    print(_row_error(got, want), _row_error(old, want))
    assert _row_error(got, want) <= 2 * _row_error(old, want)


@pytest.mark.gpu
@pytest.mark.parametrize("key", ["conv.0.weight", "conv.0.bias", "conv.2.weight", "conv.3.weight", "conv.3.bias", "conv.5.weight",
                                 "conv.6.weight", "out.weight", "out.bias"])
@pytest.mark.parametrize("how", ["in place", "replaced"])
@pytest.mark.parametrize("inference", [False, True])
def test_changed_weights_are_seen(key, how, inference):
    """The call after a change to a weight uses it in every operand made from it, as a new model does."""
    with torch.inference_mode(inference):
        enc, feats = model(), torch.randn(1, 128, 40, generator=torch.Generator().manual_seed(6)).cuda()
        before = enc.subsample(feats)
        if how == "in place":
            enc.sub[key].mul_(1.5)
        else:
            enc.sub[key] = enc.sub[key] * 1.5
        got, want = enc.subsample(feats).double().cpu(), exact(enc, feats)
        assert not torch.equal(got, before.double().cpu())
        assert float((got - want).abs().max() / want.abs().max()) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("key", ["conv.0.weight", "conv.3.weight", "conv.5.bias", "out.weight"])
def test_assigned_data_is_seen(key):
    """`tensor.data = other` leaves the tensor and its count of changes what they were."""
    enc, feats = model(), torch.randn(1, 128, 40, generator=torch.Generator().manual_seed(16)).cuda()
    enc.subsample(feats)
    for factor in (1.5, 0.5):                  # (the second may get the memory of the first)
        enc.sub[key].data = enc.sub[key].detach() * factor
        got, want = enc.subsample(feats).double().cpu(), exact(enc, feats)
        assert float((got - want).abs().max() / want.abs().max()) < 1e-5


@pytest.mark.gpu
@torch.inference_mode()
def test_weights_changed_into_what_is_not_taken_and_back():
    enc, feats = model(), torch.randn(1, 128, 40, generator=torch.Generator().manual_seed(7)).cuda()
    first = enc.subsample(feats)
    kept = enc.sub["conv.0.weight"].clone()
    enc.sub["conv.0.weight"][5] = 1e-12
    want = exact(enc, feats)
    assert float((enc.subsample(feats).double().cpu() - want).abs().max() / want.abs().max()) < 1e-5
    enc.sub["conv.0.weight"].copy_(kept)
    assert float((enc.subsample(feats) - first).abs().max() / first.abs().max()) < 1e-5


@pytest.mark.gpu
@torch.inference_mode()
def test_graphs_follow_changed_weights():
    """An EncoderGraph uses the weights of the moment, also where they leave the split kernels; a graph captured by the
    caller reads the same buffers before and after a change."""
    enc = model()
    graph, audio = E.EncoderGraph(enc, 1, 16000), torch.randn(1, 16000, generator=torch.Generator().manual_seed(13)).cuda()
    feats, own = enc.pre(audio), torch.cuda.CUDAGraph()
    enc.subsample(feats)
    torch.cuda.synchronize()
    with torch.cuda.graph(own):
        out = enc.subsample(feats)
    for change in (lambda s: s["conv.3.weight"].mul_(1.5), lambda s: s["out.bias"].add_(1.0),
                   lambda s: s.update({"conv.6.weight": s["conv.6.weight"].clone().mul_(0.5)})):
        before = graph(audio).clone()
        with torch.inference_mode(False):
            change(enc.sub)
        after = graph(audio).clone()
        assert not torch.equal(before, after) and torch.equal(after, enc(audio)) and torch.equal(graph.replay(), after)
        junk = [torch.full((1 << 20,), 7.0, device="cuda") for _ in range(20)]   # (what was freed meanwhile is overwritten)
        own.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, enc.subsample(feats))
        del junk
    kept = out.clone()
    enc.sub["conv.0.weight"][5] = 1e-12                                          # the general kernels from here on
    assert torch.equal(graph(audio), enc(audio)) and enc._sub_split is None
    own.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, kept)


@pytest.mark.gpu
@torch.inference_mode()
def test_weights_at_any_address():
    """Weights that are views into one buffer, off the alignment that the kernels' vector loads need."""
    cfg = E.EncoderConfig(layers=1)
    w = E.synthetic_weights(cfg, seed=4)
    p = "encoder.pre_encode."
    flat = torch.cat([torch.zeros(1)] + [w[k].flatten().float() for k in w if k.startswith(p)]).cuda()
    at = 1
    for k in [k for k in w if k.startswith(p)]:
        w[k] = flat[at:at + w[k].numel()].view(w[k].shape)
        at += w[k].numel()
    feats = torch.randn(1, 128, 40, generator=torch.Generator().manual_seed(8)).cuda()
    assert torch.equal(E.FastConformerEncoder(w, cfg, "cuda", parts=1).subsample(feats), model().subsample(feats))


@pytest.mark.gpu
@torch.inference_mode()
def test_capture_after_a_change():
    """A capture cannot lay the weights out: it takes the general kernels, and replays give their results."""
    enc, feats = model(), torch.randn(2, 128, 64, generator=torch.Generator().manual_seed(9)).cuda()
    enc.subsample(feats)
    general(enc, feats)                       # (their libraries are set up before the capture)
    enc.sub["conv.3.weight"].mul_(0.5)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = enc.subsample(feats)
    for seed in range(3):
        feats.copy_(torch.randn(2, 128, 64, generator=torch.Generator().manual_seed(20 + seed)))
        graph.replay()
        torch.cuda.synchronize()
        want = exact(enc, feats)
        assert float((out.double().cpu() - want).abs().max() / want.abs().max()) < 1e-5


@pytest.mark.gpu
@torch.inference_mode()
def test_scales_whose_product_leaves_the_range():
    """Small values through small weights, the result still a normal number (and made ordinary by the next layer)."""
    enc = model()
    for key, power in [("conv.2.weight", -20), ("conv.3.weight", -54), ("conv.5.weight", 60), ("conv.6.weight", 59)]:
        enc.sub[key].mul_(2.0**power)
    for i in (0, 2, 3, 5, 6):
        enc.sub[f"conv.{i}.bias"].zero_()
    feats = torch.randn(1, 128, 40, generator=torch.Generator().manual_seed(10)).cuda() * 2.0**-45
    want, got, old = exact(enc, feats), enc.subsample(feats).double().cpu(), general(enc, feats).double().cpu()
    print(_row_error(got, want), _row_error(old, want))
    assert _row_error(got, want) <= 2 * _row_error(old, want)


@pytest.mark.gpu
@pytest.mark.parametrize("size", [0.0, 2.0**-48, 2.0**-20, 1.0])
@torch.inference_mode()
def test_small_weights_of_both_first_convolutions(size):
    """Ordinary biases through a depthwise convolution of small weights, where the first convolution's are small too: the
    units that the first kernel holds them in leave the product what it is, whatever the features."""
    enc = model()
    for key, power in [("conv.0.weight", -26), ("conv.2.weight", -34), ("conv.3.weight", 36)]:
        enc.sub[key].mul_(2.0**power)
    enc.sub["conv.2.bias"].zero_()
    enc.sub["conv.0.bias"].abs_().add_(0.25)
    assert enc._current_split() is not None
    feats = torch.randn(2, 128, 40, generator=torch.Generator().manual_seed(14)).cuda() * size
    want, got, old = exact(enc, feats), enc.subsample(feats).double().cpu(), general(enc, feats).double().cpu()
    print(size, _row_error(got, want), _row_error(old, want))
    assert _row_error(got, want) <= 2 * _row_error(old, want)


@pytest.mark.gpu
@pytest.mark.parametrize("small,large", [("conv.3", "conv.5"), ("conv.6", "out")])
@torch.inference_mode()
def test_a_layer_of_weights_below_the_split_form(small, large):
    """Weights that a split row's scale does not reach, made up for by the next layer's."""
    enc = model()
    enc.sub[small + ".weight"].mul_(2.0**-108)
    for layer in (small, "conv.5", "conv.6", "out"):
        enc.sub[layer + ".bias"].zero_()
    enc.sub[large + ".weight"].mul_(2.0**76)
    feats = torch.randn(1, 128, 40, generator=torch.Generator().manual_seed(15)).cuda() * 2.0**12
    want, got, old = exact(enc, feats), enc.subsample(feats).double().cpu(), general(enc, feats).double().cpu()
    print(_row_error(got, want), _row_error(old, want))
    assert _row_error(got, want) <= 2 * _row_error(old, want)


@pytest.mark.gpu
@torch.inference_mode()
def test_a_large_weight_of_a_dead_channel():
    """A weight 2^24 times the others of its row for an input that is always zero: what the others give is as accurate as
    with the general kernels."""
    enc = model()
    enc.sub["conv.5.weight"][3], enc.sub["conv.5.bias"][3] = 0.0, 0.0
    enc.sub["conv.6.weight"][:, 3] *= 2.0**24
    feats = torch.randn(1, 128, 40, generator=torch.Generator().manual_seed(11)).cuda()
    want, got, old = exact(enc, feats), enc.subsample(feats).double().cpu(), general(enc, feats).double().cpu()
    print(_row_error(got, want), _row_error(old, want))
    assert _row_error(got, want) <= 2 * _row_error(old, want)


@pytest.mark.gpu
@pytest.mark.parametrize("large,reader", [("conv.2", "conv.3"), ("conv.5", "conv.6"), ("conv.6", "out")])
@torch.inference_mode()
def test_a_large_channel_that_is_not_read(large, reader):
    enc = model()
    enc.sub[large + ".weight"][3] *= 2.0**24
    w = enc.sub[reader + ".weight"]
    (w[:, 3] if reader != "out" else w.view(-1, 256, 16)[:, 3]).zero_()
    feats = torch.randn(1, 128, 40, generator=torch.Generator().manual_seed(12)).cuda()
    want, got, old = exact(enc, feats), enc.subsample(feats).double().cpu(), general(enc, feats).double().cpu()
    print(_row_error(got, want), _row_error(old, want))
    assert _row_error(got, want) <= 2 * _row_error(old, want)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n", [(1, 128), (127, 256), (128, 1024), (129, 128), (1000, 1024), (2100, 1024), (4000, 1024),
                                 (17000, 256)])
@torch.inference_mode()
def test_output_linear_slices(m, n):
    """kea_subsample_out over its K slices (16 to 1) and row remainders; a row with an infinity gives the exact kinds.
    A sum is a chain of at most 3 * 4096 / 64 FP32 matrix products and 16 additions, each off by at most 2^-24 of a partial
    sum, and the operands are held to 2^-22: 216 * 2^-24 of the sum of the magnitudes bounds an element. The root mean
    square error is no larger than that of the FP32 product the kernel stands for."""
    from kea_kernels import _hip
    g = torch.Generator().manual_seed(m + n)
    x, w = torch.randn(m, 4096, generator=g).cuda().relu(), torch.randn(n, 4096, generator=g).cuda()
    bias = torch.randn(n, generator=g).cuda()
    xh, xl, xs = E._split_f16(x)
    planes = torch.stack([xh, xl], 1).contiguous()
    planes[m // 2, 0, 5], planes[m // 2, 1, 5], xs[m // 2] = float("inf"), 0.0, float("inf")
    wh, wl, wm = E._split_f16(w)
    frags = E._fragments([wh, wl])
    plain = w.view(n, 16, 256).transpose(1, 2).contiguous()  # (channel, frequency)
    L = _hip.lib()
    space = torch.empty(L.kea_subsample_out_workspace(m, n), device="cuda", dtype=torch.uint8)
    y = torch.full((m, n), float("nan"), device="cuda")
    args = [planes.data_ptr(), xs.data_ptr(), m, n, frags.data_ptr(), wm.data_ptr(), plain.data_ptr(), 1.0, bias.data_ptr(),
            y.data_ptr(), space.data_ptr(), space.numel(), _hip.stream_handle(y.device)]
    _hip.check(L.kea_subsample_out(*args), "kea_subsample_out")
    want, size = x.double() @ w.double().t() + bias.double(), x.double() @ w.double().abs().t() + bias.double().abs()
    old = x @ w.t() + bias
    rows = torch.arange(m, device="cuda") != m // 2
    assert bool(((y - want).abs() <= 216 * 2.0**-24 * size)[rows].all())
    print(m, n, *(float((z - want)[rows].square().mean().sqrt()) for z in (y, old)))
    assert m == 1 or (y - want)[rows].square().mean() <= (old - want)[rows].square().mean()
    assert torch.equal(y[m // 2], torch.sign(w[:, 5]) * float("inf"))
    if space.numel():
        assert L.kea_subsample_out(*args[:11], space.numel() - 1, args[12]) == -4
    assert L.kea_subsample_out(*args[:3], 100, *args[4:]) == -1
