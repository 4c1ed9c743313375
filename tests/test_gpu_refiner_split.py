"""The native refiner's own convolutions (brovisionml_amd/csrc/refiner_conv.hip:
split-half matrix products at fp32 precision) against the float64 restatement
(oracle/refiner.py), where their tiling, their scales and their fp32 path can
go wrong: grids around the tile sizes, one-pixel grids, hidden states far from
unit scale, maps and weights of opposite scales, single values beyond a split
map's scale, a uv map beyond it, an infinity or a NaN in the decoder's maps or
in a weight.  The bars are those of tests/test_gpu_refiner_native.py, or four
times what plain fp32 convolutions show on the same inputs; non-finite values
give the restatement's NaN pattern and its values elsewhere."""
from __future__ import annotations

import numpy as np
import pytest

from brovisionml_amd import refiner as rf, workloads as wl
from oracle import refiner as oref
from tests import refiner_pins as pins

pytestmark = pytest.mark.gpu
TOL_RESULT, TOL_COARSE = 5e-6, 1e-4


def run(H, W, fov, seed, change=lambda maps: None, change_weights=lambda w: None,
        change_both=lambda maps, w: None):
    """(native result, coarse), (restatement's result, coarse)."""
    import torch
    print(f"[gpu] refiner {H}x{W} fov {fov}", flush=True)
    weights = rf.random_weights(seed)
    maps = [a.copy() for a in pins.inputs(H, W, seed)]
    change(maps)
    change_weights(weights)
    change_both(maps, weights)
    intr = wl.intrins_from_fov(8 * H, 8 * W, fov)
    dec = rf.DecoderOutput(*(torch.from_numpy(a)[None].to("cuda:0") for a in maps))
    out, coarse = rf.NativeRefiner(weights).forward(dec, intr, 8 * H, 8 * W, coarse=True)
    torch.cuda.synchronize()
    want = []
    with np.errstate(all="ignore"):
        oref.refine_forward(weights, *maps, intr, wl.scaled_intrinsics(intr, H, W, 8 * H, 8 * W),
                            wl.build_ray8(intr, H, W, 8 * H, 8 * W).reshape(3, H, W),
                            rf.uv_map(intr, H, W, 8 * H, 8 * W), trace=want, nthreads=16)
    return ((out.cpu().numpy()[0].astype(np.float64), coarse.cpu().numpy().astype(np.float64)),
            (want[-1][1], np.stack([c.reshape(3, H, W) for c, _ in want])))


def check(got, want, grow=1.0):
    """grow: how much larger the convolutions' sums, and so their rounding,
    are than for maps of unit scale (at most the maps' own scale)."""
    for g, w, tol in ((got[0], want[0], TOL_RESULT), (got[1], want[1], TOL_COARSE)):
        assert np.array_equal(np.isnan(g), np.isnan(w))
        err = np.nanmax(np.abs(g - w), initial=0.0)
        print(f"    max-abs {err:.3e}, {np.isnan(w).mean():.3f} NaN", flush=True)
        assert err <= grow * tol


# (max-abs, rms) of result and coarse that convolutions in plain fp32 matrix
# products (csrc/conv.hip) show against the restatement, at most, over the
# inputs of the tests that use them: a pixel with a small xy pair amplifies its
# heads' rounding, so the rms says more.  The bars are four times these.
FP32_LINES = {(32, 128): ((1.51e-6, 1.10e-7), (6.46e-5, 4.4e-7)),
              (52, 80): ((3.10e-6, 2.03e-7), (2.01e-5, 3.8e-7)),
              (68, 96): ((2.38e-6, 2.19e-7), (5.70e-5, 5.2e-7)),
              (52, 128): ((1.75e-5, 1.12e-6), (1.02e-4, 1.74e-6))}
FP32_INFINITE = ((1.44e-5, 4.7e-7), (7.44e-4, 3.4e-6))
FP32_SPREAD = ((2.24e-5, 4.9e-7), (4.46e-4, 1.03e-6))
FP32_HEAD = ((8.46e-6, 3.7e-7), (5.59e-5, 7.4e-7))
FP32_SCALE = ((3.72e-6, 4.7e-7), (1.83e-5, 1.0e-6))
FP32_WIDE = {179.8: ((1.44e-5, 1.12e-6), (5.58e-5, 1.71e-6)),
             179.99: ((3.12e-5, 1.75e-6), (3.11e-5, 1.08e-6)),
             179.999: ((8.33e-5, 3.32e-6), (3.36e-5, 1.85e-6))}


def check_fp32(got, want, fp32):
    for g, w, (mx, rms) in zip(got, want, fp32):
        assert np.array_equal(np.isnan(g), np.isnan(w))
        d = np.abs(g - w)[~np.isnan(w)]
        print(f"    max-abs {d.max(initial=0.0):.3e}, rms {np.sqrt((d ** 2).sum() / max(1, d.size)):.3e}, "
              f"{np.isnan(w).mean():.3f} NaN", flush=True)
        assert d.max(initial=0.0) <= 4 * mx
        assert (d ** 2).sum() <= (4 * rms) ** 2 * d.size


@pytest.mark.parametrize("H,W", [(1, 1), (1, 33), (2, 16), (3, 17), (4, 15), (9, 31), (8, 48),
                                 (17, 65), (129, 161),
                                 # either side of a choice of tile: 48, 73, 110, 128 of 16 x 4
                                 (45, 64), (45, 65), (72, 64), (73, 64), (40, 161), (41, 161),
                                 (62, 128), (63, 129)])
def test_grids(cuda, H, W):
    check(*run(H, W, 60.0, H + W))


@pytest.mark.parametrize("H,W", [(32, 128), (52, 80), (68, 96), (52, 128)])
def test_grids_at_lines(cuda, H, W):
    """64 and 65 tiles of 16 x 4, and 102 and 104.  (52 x 128's maps are the
    ill-conditioned ones.)"""
    check_fp32(*run(H, W, 60.0, H + W), FP32_LINES[(H, W)])


@pytest.mark.parametrize("H,W", [(64, 256), (65, 257), (160, 256), (161, 249)])
def test_large_grids(cuda, H, W):
    """Either side of 256 and of 640 tiles.  Of these 16,000 to 40,000 pixels a
    few have an xy pair so small that it amplifies the heads' rounding:
    convolutions in plain fp32 matrix products differ from the restatement by
    up to 1.61e-5 (result) and 2.44e-4 (coarse) on these same inputs, the split
    products by 6.1e-6 and 2.2e-4, so the bars here are 4 times those of the
    smaller grids."""
    check(*run(H, W, 60.0, H + W), grow=4.0)


@pytest.mark.parametrize("scale", [1e-6, 30.0])
def test_hidden_scale(cuda, scale):
    def change(maps):
        maps[2] *= np.float32(scale)
    check_fp32(*run(13, 24, 60.0, 31, change), FP32_SCALE)


@pytest.mark.parametrize("fov", [179.8, 179.99, 179.999])
def test_wide_field_of_view(cuda, fov):
    """u reaches 572 and 11,459, which the maps' scales take, and 114,592, past the
    largest scale beside these weights."""
    check_fp32(*run(13, 24, fov, 37), FP32_WIDE[fov])


@pytest.mark.parametrize("which,value", [(2, np.nan), (2, np.inf), (1, -np.inf), (1, np.nan)])
def test_non_finite(cuda, which, value):
    def change(maps):
        maps[which][7, 10, 3] = value
    check(*run(20, 70, 60.0, 41, change))


def test_non_finite_medium(cuda):
    """A row through the fp32 products beside split ones, four rows a wave."""
    def change(maps):
        maps[2][7, 10, 3] = np.inf
    check(*run(62, 97, 60.0, 43, change))


INFINITE = [
    ("gru.convz.weight", (5, 90, 2, 2)), ("gru.convz.weight", (5, 129, 2, 2)),
    ("gru.convr.weight", (17, 3, 2, 2)), ("gru.convq.weight", (5, 9, 2, 2)),
    ("gru.convq.weight", (63, 64, 2, 2)), ("gru.convq.weight", (9, 20, 0, 4)),
    ("xy_head.0.weight", (3, 7, 1, 1)), ("angle_head.2.weight", (0, 63, 0, 0)),
    ("up_prob_head.0.weight", (8, 65, 1, 1)), ("prob_head.4.weight", (24, 1, 0, 0))]


@pytest.mark.parametrize("H,W,name,at", [(20, 70, *i) for i in INFINITE] +
                         [(62, 97, *i) for i in INFINITE if "gru" in i[0]] +
                         [(161, 256, *i) for i in INFINITE[1:6:2]])
def test_infinite_weight(cuda, H, W, name, at):
    """One infinite weight beside finite maps, in each part of each layer: it
    saturates (or makes NaN) what it reaches and no more.  (At the centre tap
    no padding zero meets it; the one in a corner makes NaN at the border,
    which spreads.)"""
    def change(w):
        w[name][at] = np.inf
    check_fp32(*run(H, W, 60.0, 41, change_weights=change), FP32_INFINITE)


# One large value in a feature (1) or hidden (2) map: grids of all sets of
# tiles, magnitudes on both sides of the split form's range, and the hidden
# map's first row, whose windows reach over the border.
OUTLIERS = [(16, 80, which, at, v) for which in (1, 2) for at in ((7, 10, 0),)
            for v in (3e3, 6e4, 1e5, 1e7, -1e10, 1e18, 1e30)]
OUTLIERS += [(H, W, which, (33, 0, 40), v) for H, W in ((60, 64), (60, 80), (62, 97), (161, 256))
             for which, v in ((1, 1e10), (2, -1e7))]


@pytest.mark.parametrize("H,W,which,at,value", OUTLIERS)
def test_outlier(cuda, H, W, which, at, value):
    """A finite value far above the rest of its map costs no other pixel its
    precision."""
    def change(maps):
        maps[which][at] = value
    check_fp32(*run(H, W, 60.0, 41, change), FP32_SPREAD)


# Spreads that one scale a map cannot hold: a channel far above the others with
# weights as far below theirs, a region far below the rest that large weights
# bring back, a map far from unit scale throughout.
def big_channel(maps, w):
    maps[1][9] *= np.float32(1e9)
    for g in "zrq":
        w[f"gru.conv{g}.weight"][:, 64 + 9] *= np.float32(1e-9)


def dim_region(maps, w):
    one = maps[1][5].copy()
    maps[1][:, :, :30] = 0
    maps[1][:, :, 30:] *= np.float32(1e-9)
    maps[1][5, :, :30], maps[1][5, :, 30:] = one[:, :30], 0
    for g in "zrq":
        w[f"gru.conv{g}.weight"][:, np.r_[64:69, 70:128]] *= np.float32(1e9)


def large_features(maps, w):
    maps[1] *= np.float32(1e9)
    for g in "zrq":
        w[f"gru.conv{g}.weight"][:, 64:128] *= np.float32(1e-9)


def large_head_weights(maps, w):
    for g in "zr":
        w[f"gru.conv{g}.weight"] *= np.float32(0.01)
    w["gru.convq.weight"] *= np.float32(1e-6)
    w["gru.convq.bias"] *= np.float32(1e-6)
    maps[2] *= np.float32(1e-6)
    for h in ("prob", "xy", "angle", "up_prob"):
        w[f"{h}_head.0.weight"][:, :64] *= np.float32(1e6)


@pytest.mark.parametrize("spread", [big_channel, dim_region, large_features, large_head_weights],
                         ids=lambda f: f.__name__)
@pytest.mark.parametrize("H,W", [(20, 70), (62, 97), (161, 256)])
def test_spread(cuda, H, W, spread):
    """What weights and maps of opposite scales give."""
    check_fp32(*run(H, W, 60.0, 41, change_both=spread), FP32_SPREAD)


# One activation of a head far above the others, which the next layer's zero (or
# as small) weights leave out, and one weight far above the others of its row, on
# an activation as small.
def first_activation(w, h):
    w[h + ".0.bias"][3] = 1e10
    w[h + ".2.weight"][:, 3] = 0


def second_activation(w, h):
    w[h + ".2.bias"][9] = 1e9
    w[h + ".4.weight"][:, 9] *= np.float32(1e-9)


def one_weight(w, h):
    w[h + ".0.weight"][5] *= np.float32(1e-10)
    w[h + ".0.bias"][5] *= np.float32(1e-10)
    w[h + ".2.weight"][:, 5] *= np.float32(1e10)


@pytest.mark.parametrize("spread", [first_activation, second_activation, one_weight],
                         ids=lambda f: f.__name__)
@pytest.mark.parametrize("head", ["prob_head", "xy_head", "angle_head", "up_prob_head"])
@pytest.mark.parametrize("H,W", [(20, 70), (62, 97)])
def test_head_spread(cuda, H, W, head, spread):
    check_fp32(*run(H, W, 60.0, 41, change_weights=lambda w: spread(w, head)), FP32_HEAD)


def test_captured_forward_takes_each_maps_path(cuda):
    """A forward captured on ordinary maps and replayed on maps with an outlier,
    an infinity and ordinary ones again gives each the eager forward's bits."""
    import torch
    H, W = 45, 64
    print(f"[gpu] refiner {H}x{W} captured", flush=True)
    model = rf.NativeRefiner(rf.random_weights(5))
    intr = wl.intrins_from_fov(8 * H, 8 * W, 60.0)
    dec = rf.DecoderOutput(*(torch.from_numpy(a)[None].to("cuda:0") for a in pins.inputs(H, W, 5)))
    ordinary = (dec.feature.clone(), dec.hidden.clone())
    out = torch.empty((1, 3, 8 * H, 8 * W), device="cuda:0")
    model.forward(dec, intr, 8 * H, 8 * W, out=out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        model.forward(dec, intr, 8 * H, 8 * W, out=out)
    for feature, hidden in ((0.0, 0.0), (0.0, 1e10), (np.inf, 0.0), (0.0, 0.0), (1e7, np.inf)):
        dec.feature.copy_(ordinary[0])
        dec.hidden.copy_(ordinary[1])
        if feature:
            dec.feature[0, 3, 20, 30] = feature
        if hidden:
            dec.hidden[0, 7, 10, 3] = hidden
        want = model.forward(dec, intr, 8 * H, 8 * W)
        out.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int32), want.view(torch.int32))


@pytest.mark.parametrize("H,W", [(13, 19), (62, 97), (161, 249)])
@pytest.mark.parametrize("pad_t,pad_l,cut_h,cut_w", [(0, 0, 0, 4), (5, 3, 11, 6), (8, 4, 9, 8),
                                                     (7, 0, 7, 1)])
def test_crop_is_a_slice(cuda, H, W, pad_t, pad_l, cut_h, cut_w):
    """The crop the upsample writes (16-byte or single stores) has the whole
    result's bits, into an `out` of any alignment, and coarse maps asked for
    change neither."""
    import torch
    print(f"[gpu] refiner {H}x{W} crop {pad_t} {pad_l} {cut_h} {cut_w}", flush=True)
    intr = wl.intrins_from_fov(8 * H, 8 * W, 60.0)
    model = rf.NativeRefiner(rf.random_weights(3))
    dec = rf.DecoderOutput(*(torch.from_numpy(a)[None].to("cuda:0") for a in pins.inputs(H, W, 3)))
    whole = model.forward(dec, intr, 8 * H, 8 * W)
    crop = rf.Crop(orig_h=8 * H - cut_h, orig_w=8 * W - cut_w, pad_t=pad_t, pad_l=pad_l)
    want = whole[:, :, pad_t:pad_t + crop.orig_h, pad_l:pad_l + crop.orig_w]
    for shift in (0, 1):
        flat = torch.full((3 * crop.orig_h * crop.orig_w + 8,), 7.0, device="cuda:0")
        out = flat[shift:shift + 3 * crop.orig_h * crop.orig_w].view(1, 3, crop.orig_h, crop.orig_w)
        got, _ = model.forward(dec, intr, 8 * H, 8 * W, crop=crop, coarse=True, out=out)
        assert torch.equal(got, want)
        assert bool((flat[:shift] == 7.0).all()) and bool((flat[shift + out.numel():] == 7.0).all())
