"""The 3x3 direct kernel (csrc/conv_igemm_direct.hip: weights in LDS,
activations straight into MFMA registers) against the oracle, in calls that run
it: beyond the 16 x 16 blocks of the kernel for few pixels and where the
LDS-streamed GEMM does not stand in (two parts; fewer than four 16-byte units a
tap; fp32 with at most 32 outputs; from 65536 pixels). Two parts, channel views,
stride, dilation, asymmetric padding, odd unit counts, ragged blocks of pixels
and columns, the largest K. Tolerances are those of the kernels beside it: fp32
sums of at most 9 x 160 products (relative 1e-4), 16-bit storage with fp32 sums
(two roundings of the result against the stored inputs)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover - the gpu marker keeps these off CPU runs
    pytest.skip("no GPU", allow_module_level=True)

from tests import gpu_util as G  # noqa: E402

F32, F16, BF16 = 0, 1, 2
BAR = {F32: 1e-4, F16: 2e-3, BF16: 8e-3}
CUS = torch.cuda.get_device_properties(0).multi_processor_count
pytestmark = [pytestmark, pytest.mark.skipif(CUS != 256, reason="the limits are multiples of the CUs")]

# ih, iw, cin or parts, cout, s, d, pad, act, residual, n
CASES = [(93, 91, [32, 24], 32, 1, 1, (1, 1, 1, 1), "relu", True, 1),
         (261, 257, [16, 8], 12, 2, 1, (0, 1, 1, 0), "none", True, 1),
         (95, 89, [48, 24], 28, 1, 2, (2, 2, 2, 2), "relu", False, 1),
         (97, 87, 16, 20, 1, 2, (2, 2, 2, 2), "sigmoid", False, 1),
         (150, 147, 40, 48, 1, 1, (1, 1, 1, 1), "relu6", True, 3),
         (513, 515, 32, 64, 2, 1, (0, 1, 1, 0), "hardswish", True, 1),
         (182, 181, 80, 32, 1, 1, (1, 1, 1, 1), "hardswish", True, 2),
         (256, 257, 160, 24, 1, 1, (1, 1, 1, 1), "relu", True, 1)]  # 16 bit only: 10 steps a tap


def runs_direct(plan, m):
    """The direct kernel's launch: eight wavefronts of 32-pixel blocks a workgroup, at most one a CU."""
    return plan.variant == G.conv.Variant.DIRECT and plan.bm == 32 and plan.grid == min(CUS, -(-m // 256)) and \
        plan.grid != -(-m // 64)


@pytest.mark.parametrize("dt", [F32, F16, BF16], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:6])))
def test_igemm_direct_kernel(case, dt):
    ih, iw, cin, cout, s, d, pad, act, res, n = case
    if cin == 160 and dt == F32:
        cin = 20  # fp32: 80 channels at most, and an odd kg count
    parts = cin if isinstance(cin, list) else None
    r = G.run_igemm(ih, iw, sum(parts) if parts else cin, cout, 3, s, pad, act, res, dt, 9200 + cout, n=n, d=d,
                    parts=parts)
    oh, ow = ((v + p - 2 * d - 1) // s + 1 for v, p in ((ih, pad[0] + pad[2]), (iw, pad[1] + pad[3])))
    assert runs_direct(r.plan, n * oh * ow), r.plan
    err = G.rel_err(r.got, r.want_r)
    print(f"igemm direct {case} dt{dt} {r.plan}: max_rel_err={err:.3e}", flush=True)
    assert not np.isnan(np.asarray(r.got)).any()
    assert err <= BAR[dt], err


@pytest.mark.parametrize("dt", [F32, F16], ids=["f32", "f16"])
def test_igemm_direct_kernel_channel_view(dt):
    """Channels 8..31 of a 48-channel tensor: the view's pixel stride and
    offset, with neighbours' channels right beside what is read."""
    ih, iw, full, c0, c, cout = 95, 89, 48, 8, 24, 20
    op = G.orc.conv2d(c, cout, k=3, s=1, pad=[1, 1, 1, 1], act="relu")
    xf, wts, b = G.stream(9290, ih * iw * full, cout * c * 9, cout)
    xs = xf.reshape(ih * iw, full)[:, c0:c0 + c].ravel().copy()
    want = G.rounded_ref(op, ih, iw, xs, wts, b, None, dt, dt, 1) if dt else G.orc.conv2d_ref(op, ih, iw, xs, wts, b, None)
    wp, _ = G.orc.pack_weights_conv(wts, cout, c, 3, 3, 4, dt)
    spec = G.conv.ConvIgemmSpec(ih=ih, iw=iw, cin=c, cout=cout, k=3, pad=(1, 1, 1, 1), act=G.ACT["relu"],
                                dt=G.conv.DType(dt), srcs=[G.conv.SrcView(c=c, stride_c=full, c_off=c0)])
    assert runs_direct(spec.plan(), ih * iw), spec.plan()
    yd = G.poisoned(ih * iw * cout, dt)
    spec.run([G.dev(G.orc.pack_nhwc(xf, 1, ih, iw, full, dt))], G.dev(wp), G.dev(G.orc.pack_bias(b, cout, dt)), None, yd)
    torch.cuda.synchronize()
    err = G.rel_err(G.orc.unpack_nhwc(G.host(yd, dt), 1, ih, iw, cout, dt), want)
    print(f"igemm direct view dt{dt}: {err:.3e}", flush=True)
    assert err <= BAR[dt], err
