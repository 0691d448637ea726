"""The KxK conv whose workgroups split K over their wavefronts
(csrc/conv_ksplit.hip), and short pointwise calls on the pointwise one, against the oracle, at the edges of its blocks: ragged
pixel and channel blocks, taps outside the image, units past a part, (tap,
step) pairs that do not divide by the wavefronts, two input parts, and both
sides of its block limit. Tolerances are those of the kernels it stands beside:
fp32 sums of at most 25 x 256 products (relative 1e-4), 16-bit storage with
fp32 sums (two roundings of the result against the stored inputs)."""
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover - the gpu marker keeps these off CPU runs
    pytest.skip("no GPU", allow_module_level=True)

from tests import gpu_util as G  # noqa: E402

F32, F16, BF16 = 0, 1, 2
BAR = {F32: 1e-4, F16: 2e-3, BF16: 8e-3}

# ih, iw, cin, cout, k, s, d, pad, act, residual, n
CASES = [(40, 72, 72, 32, 3, 1, 1, (1, 1, 1, 1), "relu", True, 1),      # one tap a wavefront, 5 steps at fp32
         (23, 31, 16, 20, 3, 2, 1, (1, 1, 1, 1), "none", True, 1),      # ragged blocks of pixels and channels
         (11, 13, 8, 4, 3, 1, 1, (1, 1, 1, 1), "hardswish", False, 3),  # one unit of four a step at 16 bit
         (10, 18, 256, 100, 3, 1, 1, (1, 1, 1, 1), "relu", False, 2),   # past the direct kernel's channels
         (10, 18, 40, 72, 5, 2, 1, (2, 2, 2, 2), "relu6", True, 1),     # 25 taps over 9 wavefronts
         (9, 12, 24, 36, 2, 1, 1, (0, 1, 1, 0), "sigmoid", False, 2),   # 4 taps: some wavefronts have none
         (20, 21, 48, 24, 3, 1, 2, (2, 2, 2, 2), "relu", True, 2),      # dilated
         (5, 4, 16, 16, 3, 1, 1, (3, 3, 3, 3), "none", False, 1),       # pixels with no tap in the image
         (41, 50, 36, 64, 3, 1, 1, (1, 1, 1, 1), "relu", False, 1),     # fp32 only: an odd kg count
         (64, 64, 32, 32, 3, 1, 1, (1, 1, 1, 1), "relu", False, 1),     # 512 blocks: 16 bit's limit
         (64, 65, 32, 32, 3, 1, 1, (1, 1, 1, 1), "relu", False, 1),     # past it
         (64, 64, 32, 64, 3, 1, 1, (1, 1, 1, 1), "relu", True, 1)]      # 1024: fp32's


def check(name, err, dt):
    print(f"{name} dt{dt}: max_rel_err={err:.3e}", flush=True)
    assert err <= BAR[dt], (name, err)


CUS = torch.cuda.get_device_properties(0).multi_processor_count


@pytest.mark.parametrize("dt", [F32, F16, BF16], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:7])))
def test_igemm(case, dt):
    ih, iw, cin, cout, k, s, d, pad, act, res, n = case
    r = G.run_igemm(ih, iw, cin, cout, k, s, pad, act, res, dt, 9700 + cin, n=n, d=d)
    oh, ow = G.orc.out_hw(G.orc.conv2d(cin, cout, k=k, s=s, pad=list(pad), dil=d), ih, iw)
    blocks = -(-n * oh * ow // 16) * -(-cout // 16)
    here = blocks <= CUS * (4 if dt == F32 else 2) and (dt == F32 or cin % 8 == 0)
    assert ((r.plan.bm, r.plan.bn, r.plan.grid) == (16, 16, blocks)) == here, (blocks, r.plan)
    assert not np.isnan(np.asarray(r.got)).any(), case
    check(f"igemm {case}", G.rel_err(r.got, r.want_r), dt)


# h, w, cin, cout, n: pointwise calls of the tiled GEMM's that the one-dispatch
# split-K kernel runs
PW = [(1, 1, 4, 80, 1), (10, 18, 48, 192, 1), (7, 5, 44, 144, 3), (23, 31, 60, 112, 2), (32, 64, 8, 768, 1),
      (32, 64, 12, 784, 1)]  # both sides of 24 blocks a CU of 256


@pytest.mark.parametrize("dt", [F32, F16, BF16], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("case", PW, ids=lambda c: "x".join(map(str, c)))
def test_pointwise_short_k(case, dt):
    h, w, cin, cout, n = case
    r = G.run_pw(h, w, cin, cout, "relu6", True, dt, 9850 + cin, n=n)
    assert ((r.plan.bm, r.plan.bn) == (16, 16)) == (-(-n * h * w // 16) * (cout // 16) <= 24 * CUS), r.plan
    assert not np.isnan(np.asarray(r.got)).any(), case
    check(f"pw {case} {r.plan}", G.rel_err(r.got, r.want_r), dt)


# h, w, cin, cout; on 16 x 16 blocks at fp32 and at 16 bit
PW_LONGER = [((45, 40, 96, 576), (True, True)), ((45, 40, 320, 576), (True, True)),
             ((45, 40, 324, 576), (False, False)), ((32, 64, 128, 768), (True, False))]


@pytest.mark.skipif(CUS != 256, reason="the limits are multiples of the CUs")
@pytest.mark.parametrize("dt", [F32, F16, BF16], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("case", PW_LONGER, ids=lambda c: "x".join(map(str, c[0])))
def test_pointwise_longer_k(case, dt):
    (h, w, cin, cout), here = case
    r = G.run_pw(h, w, cin, cout, "relu", False, dt, 9870 + cin)
    assert (r.plan.bm == 16) == here[dt != F32], r.plan
    check(f"pw {case[0]} {r.plan}", G.rel_err(r.got, r.want_r), dt)


@pytest.mark.parametrize("dt", [F32, F16], ids=["f32", "f16"])
def test_two_parts(dt):
    """A concat read: 24 channels of a 40-channel tensor, then 16 plain ones."""
    ih, iw, c0, c1, cout = 21, 37, 24, 16, 36
    op = G.orc.conv2d(c0 + c1, cout, k=3, s=1, pad=[1, 1, 1, 1], act="relu")
    xa, xb, wts, b = G.stream(9801, ih * iw * 40, ih * iw * c1, cout * (c0 + c1) * 9, cout)
    x = np.concatenate([xa.reshape(ih * iw, 40)[:, 8:8 + c0], xb.reshape(ih * iw, c1)], 1).ravel().copy()
    want = G.rounded_ref(op, ih, iw, x, wts, b, None, dt, dt, 1) if dt else G.orc.conv2d_ref(op, ih, iw, x, wts, b, None)
    wp, _ = G.orc.pack_weights_conv(wts, cout, c0 + c1, 3, 3, 4, dt)
    spec = G.conv.ConvIgemmSpec(ih=ih, iw=iw, cin=c0 + c1, cout=cout, k=3, pad=(1, 1, 1, 1), act=G.ACT["relu"],
                                dt=G.conv.DType(dt), srcs=[G.conv.SrcView(c=c0, stride_c=40, c_off=8),
                                                           G.conv.SrcView(c=c1, stride_c=c1, c_off=0)])
    assert spec.plan().bm == 16
    yd = G.poisoned(ih * iw * cout, dt)
    spec.run([G.dev(G.orc.pack_nhwc(xa, 1, ih, iw, 40, dt)), G.dev(G.orc.pack_nhwc(xb, 1, ih, iw, c1, dt))], G.dev(wp),
             G.dev(G.orc.pack_bias(b, cout, dt)), None, yd)
    torch.cuda.synchronize()
    check("two parts", G.rel_err(G.orc.unpack_nhwc(G.host(yd, dt), 1, ih, iw, cout, dt), want), dt)


def test_infinities_stay_in_their_taps():
    """Missing pixels, taps and units are zeros in both operands: an infinite
    pixel reaches the outputs whose taps touch it and no other."""
    h, w, c, cout = 9, 11, 24, 20
    rng = np.random.default_rng(9901)
    wts = (np.abs(rng.standard_normal((cout, c, 3, 3))) + 0.1).astype(np.float32)
    x = torch.from_numpy(rng.standard_normal((1, h, w, c)).astype(np.float32)).cuda()
    x[0, 0, 0] = float("inf")
    op = G.conv.ConvOp(ih=h, iw=w, cin=c, cout=cout, kh=3, kw=3, pad=(1,) * 4)
    assert op.plan().bm == 16
    p, _ = G.conv.pack_weights_conv(wts.ravel(), cout, c, 3, 3, 4, G.conv.DType.F32)
    b = G.conv.pack_bias(np.zeros(cout, np.float32), cout, G.conv.DType.F32)
    y = torch.full((1, h, w, cout), float("nan"), device="cuda")
    op.run(x, torch.from_numpy(p).cuda(), torch.from_numpy(b).cuda(), None, y)
    got = y[0].cpu()
    assert torch.isposinf(got[:2, :2]).all()
    got[:2, :2] = 0
    assert torch.isfinite(got).all()


NO_SPLIT_PROBE = """
import sys
sys.path.insert(0, %r)
import numpy as np
from tests import gpu_util as G
for dt in (0, 1, 2):
    for cin, cout in ((128, 128), (64, 64)):
        xs = [G.run_igemm(9, 16, cin, cout, 3, 1, [1] * 4, "relu", True, dt, 9950, splitk=k, refs=False).got for k in (0, 1)]
        print(int(np.array_equal(*map(np.asarray, xs))), end=" ")
"""


def test_no_split_override_keeps_k_whole():
    """Under AIH_IGEMM_NO_SPLIT=1 (read once per process) a call of few pixels
    sums K whole: the bits of the forced split of 1. Without it the sums are
    those of nine wavefronts, and the bits differ."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    got = []
    for v in ("1", ""):
        r = subprocess.run([sys.executable, "-c", NO_SPLIT_PROBE % root], capture_output=True, text=True, timeout=100,
                           env=dict(os.environ, AIH_IGEMM_NO_SPLIT=v))
        assert r.returncode == 0, r.stderr
        got.append(r.stdout.split())
    assert got[0] == ["1"] * 6, got
    assert got[1][0] == "0", got
