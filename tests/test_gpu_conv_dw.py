"""The depthwise strip kernel (csrc/conv_dw.hip) against the oracle, for every
strip length its rule picks on a 256-CU device: ragged strips, workgroups that
span several images, rows and columns outside the image, 8-byte channel
vectors. Tolerances as for the other depthwise tests: fp32 sums of at most 25
products (relative 1e-4), 16-bit storage with fp32 sums (two roundings of the
result against the stored inputs)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover - the gpu marker keeps these off CPU runs
    pytest.skip("no GPU", allow_module_level=True)

from tests import gpu_util as G  # noqa: E402

F32, F16, BF16 = 0, 1, 2
BAR = {F32: 1e-4, F16: 2e-3, BF16: 8e-3}

# ih, iw, c, k, s, pad, n: strips of 4, 2 and 1 pixels with 8-channel vectors
# at 16 bit, and with 4-channel ones (c = 44)
CASES = [(150, 147, 64, 3, 1, [1, 1, 1, 1], 3),
         (75, 111, 64, 3, 1, [1, 1, 1, 1], 2),
         (9, 7, 8, 3, 1, [1, 1, 1, 1], 5),       # a workgroup over several images
         (33, 35, 16, 3, 2, [0, 1, 1, 0], 3),
         (93, 91, 64, 5, 1, [2, 2, 2, 2], 1),
         (181, 183, 64, 5, 2, [2, 2, 2, 2], 1),
         (5, 6, 24, 5, 1, [2, 2, 2, 2], 5),
         (5, 6, 24, 5, 2, [2, 2, 2, 2], 5),
         (90, 89, 44, 3, 1, [1, 1, 1, 1], 3),
         (90, 89, 44, 5, 1, [2, 2, 2, 2], 3),
         (180, 179, 44, 3, 2, [1, 1, 1, 1], 3),
         (180, 179, 44, 5, 2, [2, 2, 2, 2], 3),
         (90, 89, 44, 5, 1, [2, 2, 2, 2], 6),    # fp32: strips of 8
         (77, 79, 44, 3, 1, [1, 1, 1, 1], 1),
         (77, 79, 44, 5, 1, [2, 2, 2, 2], 1),
         (155, 157, 44, 5, 2, [2, 2, 2, 2], 1),
         (3, 4, 12, 5, 1, [4, 4, 4, 4], 7),      # output rows and columns with no tap in the image
         (1, 1, 4, 3, 2, [1, 1, 1, 1], 300)]


@pytest.mark.parametrize("dt", [F32, F16, BF16], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:5] + c[6:])))
def test_dw_strips(case, dt):
    ih, iw, c, k, s, pad, n = case
    r = G.run_dw(ih, iw, c, k, s, "hardswish" if c == 16 else "relu", c % 3 == 2, dt, 9000 + ih, pad=pad, n=n)
    err = G.rel_err(r.got, r.want_r)
    print(f"dw {case} dt{dt}: max_rel_err={err:.3e}", flush=True)
    assert not np.isnan(np.asarray(r.got)).any()
    assert err <= BAR[dt], err


@pytest.mark.parametrize("hw", [(12, 14), (96, 93)], ids=["one_pixel", "strips"])
@pytest.mark.parametrize("dt", [G.conv.DType.F32, G.conv.DType.F16], ids=["f32", "f16"])
def test_rows_outside_add_nothing(dt, hw):
    """A kernel row outside the image adds nothing, infinite weights or not:
    with the first row's weights infinite, output row 0 stays what it is
    without that row."""
    h, w = hw
    c, k = 64, 5
    rng = np.random.default_rng(9)
    wts = rng.standard_normal((c, 1, k, k)).astype(np.float32)
    op = G.conv.ConvOp(ih=h, iw=w, cin=c, cout=c, kh=k, kw=k, sh=1, sw=1, pad=(2,) * 4, groups=c, dt=dt, n=1)
    tdt = torch.float32 if dt == G.conv.DType.F32 else torch.float16
    x = torch.from_numpy(rng.standard_normal((1, h, w, c)).astype(np.float32)).to("cuda", tdt)
    out = []
    for first in (0.0, np.inf):
        wts[:, :, 0] = first
        p = G.conv.pack_weights_dw(wts.ravel(), c, k, k, dt)
        p = torch.from_numpy(p.view(np.int16) if p.dtype == np.uint16 else p).to("cuda")
        b = G.conv.pack_bias(np.zeros(c, np.float32), c, dt)
        b = torch.from_numpy(b.view(np.int16) if b.dtype == np.uint16 else b).to("cuda")
        y = torch.full((1, h, w, c), float("nan"), device="cuda", dtype=tdt)
        op.run(x, p, b, None, y)
        out.append(y[:, 0].float().cpu())
    assert torch.isfinite(out[0][:, 2:-2]).all()
    assert torch.equal(out[0][:, 2:-2], out[1][:, 2:-2])
