"""The LDS-streamed conv GEMM (csrc/conv_stream.hip) against the oracle, at the
edges of its tiles: ragged pixel and column tiles, a K that ends inside a
stage, taps outside the image, stages that cross taps, channel views, output
rows that are only 8-byte aligned (16 bit, N4 % 8 == 4), and every tile the
plan picks. Tolerances are those of the kernels it stands beside: fp32 sums of
at most 25 x 256 products (relative 1e-4), 16-bit storage with fp32 sums (two
roundings of the result against the stored inputs)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover - the gpu marker keeps these off CPU runs
    pytest.skip("no GPU", allow_module_level=True)

from tests import gpu_util as G  # noqa: E402

F32, F16, BF16 = 0, 1, 2
V = G.conv.Variant
BAR = {F32: 1e-4, F16: 2e-3, BF16: 8e-3}


def check(name, r, dt):
    err = G.rel_err(r.got, r.want_r)
    print(f"{name} dt{dt} {r.plan}: max_rel_err={err:.3e}", flush=True)
    assert not np.isnan(np.asarray(r.got)).any(), name
    assert err <= BAR[dt], (name, err)


# (h, w, cin, cout, n), act, residual, (bm, bn) of the 16-bit plan (None: 64 x 64
# in the place of a direct kernel, at most 64 outputs)
PW = [((23, 37, 32, 96, 3), "relu", False, (64, 64)),        # one unit a lane half, 40 pixels in the last tile
      ((21, 37, 72, 100, 3), "hardswish", True, (64, 64)),   # K ends inside a stage; 8-byte output rows
      ((24, 30, 328, 132, 3), "relu6", True, (64, 64)),      # stages of 8 units, 41 units
      ((200, 331, 48, 128, 1), "none", True, (128, 128)),
      ((200, 331, 40, 68, 1), "relu", False, (128, 96)),
      ((200, 331, 64, 184, 1), "sigmoid", False, (128, 64)),
      ((40, 72, 128, 40, 1), "relu", True, None),            # in place of the 16x16-block launch
      ((181, 182, 40, 44, 1), "none", False, None),          # in place of the direct kernel
      ((257, 257, 96, 20, 1), "relu", True, None)]           # in place of the one-tap launch


@pytest.mark.parametrize("dt", [F32, F16, BF16], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("case", PW, ids=lambda c: "x".join(map(str, c[0])))
def test_pointwise(case, dt):
    (h, w, cin, cout, n), act, res, tile = case
    r = G.run_pw(h, w, cin, cout, act, res, dt, 9100 + cin, n=n)
    if dt != F32 and tile:
        assert (r.plan.variant, r.plan.bm, r.plan.bn) == (V.TILE, *tile), r.plan
    elif dt != F32:
        assert r.plan.variant == V.DIRECT and r.plan.ws_bytes == 0, r.plan
        assert r.plan.grid == -(-n * h * w // 64), r.plan
    check(f"pw {case}", r, dt)


# ih, iw, cin, cout, k, s, d, pad, act, residual, n
IG = [(23, 31, 64, 100, 3, 1, 1, (1, 1, 1, 1), "relu", True, 5),
      (41, 37, 32, 96, 3, 2, 1, (0, 1, 1, 0), "hardswish", False, 6),      # 4 units a tap: a stage is a tap
      (40, 50, 40, 72, 5, 1, 1, (2, 2, 2, 2), "none", False, 2),           # 5 units a tap: stages cross taps
      (33, 47, 72, 68, 3, 1, 2, (2, 2, 2, 2), "relu6", True, 3),           # dilated
      (30, 40, 36, 80, 2, 1, 1, (0, 0, 0, 0), "relu", False, 4),           # an odd kg count, few pixels: the tiled GEMM
      (45, 83, 48, 128, 3, 1, 1, (1, 1, 1, 1), "relu", True, 18),          # 128 x 128 tiles, a ragged last one
      (45, 83, 32, 96, 3, 1, 1, (1, 1, 1, 1), "none", False, 18),          # 128 x 96
      (45, 83, 32, 176, 3, 2, 1, (1, 1, 1, 1), "relu", False, 60),         # 128 x 64
      (33, 47, 64, 64, 3, 1, 1, (1, 1, 1, 1), "relu", True, 11),           # in place of the direct kernel
      (65, 64, 64, 36, 3, 1, 1, (1, 1, 1, 1), "relu", False, 17),          # the same above 65536 pixels, 16 bit
      # fp32 only, odd kg counts: a K tail, stages that cross taps, dilated with a stride
      (60, 80, 36, 80, 2, 1, 1, (0, 0, 0, 0), "relu", False, 10),
      (45, 83, 20, 96, 5, 1, 1, (2, 2, 2, 2), "none", True, 18),
      (45, 83, 36, 68, 3, 2, 2, (2, 2, 2, 2), "relu6", True, 60)]
# their tiles at fp32 and at 16 bit (in the direct kernel's place a wavefront's);
# None: another kernel runs the call (fp32 with a split K, a few pixels, an odd kg count)
IG_TILES = [(None, (64, 64)), (None, (64, 64)), (None, (64, 64)), (None, (64, 64)), (None, None),
            ((128, 128),) * 2, ((128, 96),) * 2, ((128, 64),) * 2, ((32, 32),) * 2, (None, (32, 32)),
            ((64, 64), None), ((128, 96), None), ((64, 64), None)]


@pytest.mark.parametrize("dt", [F32, F16, BF16], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("case", IG, ids=lambda c: "x".join(map(str, c[:7])))
def test_igemm(case, dt):
    ih, iw, cin, cout, k, s, d, pad, act, res, n = case
    r = G.run_igemm(ih, iw, cin, cout, k, s, pad, act, res, dt, 9300 + cin, n=n, d=d)
    tile = IG_TILES[IG.index(case)][dt != F32]
    if tile == (32, 32):
        assert r.plan.grid == -(-n * ih * iw // 64), r.plan
    assert ((r.plan.bm, r.plan.bn) == tile and r.plan.splitk == 1) if tile else r.plan.bm != 64, r.plan
    check(f"igemm {case}", r, dt)


# ih, iw, cin, cout, s, d, pad, n: 1x1 convs through the KxK entry, past the
# split-K kernel's block limit; only the last reads input pixel m for output m
ONE_TAP = [(97, 101, 64, 68, 2, 1, (0, 0, 0, 0), 5),
           (66, 61, 48, 100, 1, 1, (0, 1, 1, 0), 4),
           (65, 63, 48, 100, 1, 1, (0, 0, 2, 0), 4),  # rows below the image only
           (65, 63, 48, 100, 1, 2, (0, 0, 0, 1), 4),  # columns right of it only
           (64, 64, 40, 72, 1, 1, (1, 0, 0, 1), 4),   # as many outputs as inputs, shifted
           (199, 187, 328, 96, 3, 1, (2, 1, 0, 2), 3),  # stages of 8 units, pixels with no input
           (65, 63, 72, 100, 1, 1, (0, 0, 0, 0), 4)]


@pytest.mark.parametrize("dt", [F32, F16, BF16], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("case", ONE_TAP, ids=lambda c: "x".join(map(str, c[:6])))
def test_one_tap_with_stride_and_padding(case, dt):
    ih, iw, cin, cout, s, d, pad, n = case
    r = G.run_igemm(ih, iw, cin, cout, 1, s, pad, "none", False, dt, 9350 + cin, n=n, d=d)
    assert r.plan.bm == 64 or dt == F32, r.plan  # (fp32 sums the tiled GEMM splits stay there)
    check(f"1x1 {case}", r, dt)


@pytest.mark.parametrize("dt", [F32, F16], ids=["f32", "f16"])
def test_igemm_channel_view(dt):
    """Channels 8..71 of an 88-channel input: the pixel stride and offset of a
    view, with neighbours' channels right beside what is read."""
    ih, iw, full, c0, c, cout = 37, 41, 88, 8, 64, 96
    op = G.orc.conv2d(c, cout, k=3, s=1, pad=[1, 1, 1, 1], act="relu")
    xf, wts, b = G.stream(9400, ih * iw * full, cout * c * 9, cout)
    xs = xf.reshape(ih * iw, full)[:, c0:c0 + c].ravel().copy()
    want = G.rounded_ref(op, ih, iw, xs, wts, b, None, dt, dt, 1) if dt else G.orc.conv2d_ref(op, ih, iw, xs, wts, b, None)
    wp, _ = G.orc.pack_weights_conv(wts, cout, c, 3, 3, 4, dt)
    spec = G.conv.ConvIgemmSpec(ih=ih, iw=iw, cin=c, cout=cout, k=3, pad=(1, 1, 1, 1), act=G.ACT["relu"],
                                dt=G.conv.DType(dt), srcs=[G.conv.SrcView(c=c, stride_c=full, c_off=c0)])
    yd = G.poisoned(ih * iw * cout, dt)
    spec.run([G.dev(G.orc.pack_nhwc(xf, 1, ih, iw, full, dt))], G.dev(wp), G.dev(G.orc.pack_bias(b, cout, dt)), None, yd)
    torch.cuda.synchronize()
    err = G.rel_err(G.orc.unpack_nhwc(G.host(yd, dt), 1, ih, iw, cout, dt), want)
    print(f"igemm view dt{dt} {spec.plan()}: {err:.3e}", flush=True)
    assert err <= BAR[dt], err


@pytest.mark.parametrize("dt", [F16, BF16], ids=["f16", "bf16"])
def test_streamed_equals_the_tiled_gemm(dt):
    """K runs in the tiled GEMM's order (unit pairs, stages of either depth),
    so a call the plan streams equals the forced tiled GEMM bit for bit."""
    for (h, w, cin, cout, n), seed in [((21, 37, 192, 256, 4), 9501), ((40, 72, 48, 64, 16), 9502)]:
        xs = G.stream(seed, n * h * w * cin, cout * cin, cout, n * h * w * cout)
        a = G.run_pw(h, w, cin, cout, "relu", True, dt, seed, n=n, xs=xs, refs=False)
        b = G.run_pw(h, w, cin, cout, "relu", True, dt, seed, n=n, xs=xs, refs=False, variant=1)
        assert np.array_equal(np.asarray(a.got), np.asarray(b.got)), (h, w, cin, cout)


def test_infinities_stay_in_their_pixel():
    """Rows past a tile's last pixel, columns past N4 and the K tail are zeros
    in both operands: an infinity in one pixel reaches that pixel's outputs and
    no other (0 x inf would be a NaN elsewhere)."""
    h, w, cin, cout = 50, 61, 72, 100
    x, wts, b = G.stream(9601, h * w * cin, cout * cin, cout)
    x = x.copy()
    p = 63 * cin  # the last pixel of the first 64-pixel tile
    x[p:p + cin] = np.inf
    wts = np.abs(wts) + np.float32(0.1)
    r = G.run_pw(h, w, cin, cout, "none", False, F16, 0, xs=(x, wts, b, None), refs=False)
    got = np.asarray(r.got).reshape(h * w, cout)
    assert np.isposinf(got[63]).all()
    assert np.isfinite(np.delete(got, 63, 0)).all()
