"""The transposed conv's one-window kernel (k_conv_up) at the sizes where its
tiling can go wrong, against torch's conv_transpose1d in float64 over the
f16-rounded operands: |got - ref| <= 2^-13 sum |w h| + 2^-22 |ref| (f32 sums
of exact f16 products in any order)."""
import pytest
import torch

from chatterbox_amdvulkan_amd import cbxops as C

pytestmark = pytest.mark.gpu


def ref_conv(h, w, s):
    ci, co, K = w.shape
    T = h.shape[0]
    y = torch.zeros(((T - 1) * s + K, co), dtype=torch.float64, device=h.device)
    for j in range(K):
        y[j:j + (T - 1) * s + 1:s] += h @ w[:, :, j].contiguous()
    return y


# C_in, C_out, stride, K, pad, T: the upsamplers where the kernel starts to be
# taken, a tile's edges, long inputs (64-step tiles), phases of unequal taps
# (K % stride), of none (K < stride), uneven padding, tiles that do not fill
# the last group of waves; and sizes on the other side of the line
@pytest.mark.parametrize("ci,co,s,K,pad,T", [
    (128, 64, 3, 7, 2, 2752), (128, 64, 3, 7, 2, 2753), (128, 64, 3, 7, 2, 2783), (128, 64, 3, 7, 2, 20001),
    (256, 128, 5, 11, 3, 832), (256, 128, 5, 11, 3, 863), (256, 128, 5, 11, 3, 4001), (128, 96, 2, 3, 0, 2761),
    (256, 64, 3, 5, 1, 2770), (128, 32, 4, 2, 0, 4100), (128, 32, 3, 1, 0, 5600), (128, 64, 5, 3, 1, 1700),
    (128, 32, 2, 7, 5, 8200), (128, 64, 3, 7, 2, 1), (128, 64, 3, 7, 2, 33), (512, 256, 8, 16, 4, 500), (192, 64, 3, 5, 1, 2770),
    (64, 32, 2, 4, 1, 9000)])
@pytest.mark.parametrize("leaky", [True, False])
def test_transposed(cbx, ci, co, s, K, pad, T, leaky):
    g = torch.Generator(device="cuda")
    g.manual_seed(ci + co + K + T)
    x = torch.randn((2, T, ci), generator=g, device="cuda")
    w = torch.randn((ci, co, K), generator=g, device="cuda") * (ci * K / s) ** -0.5
    b = torch.randn((co,), generator=g, device="cuda") * 0.1
    cw = C.Conv1dWeights(w, transpose_stride=s)
    pro = C.CONV_PRO_LEAKY_RELU if leaky else C.CONV_PRO_NONE
    try:
        for bias in (b, None):
            y = C.conv_transpose1d(x, cw, pad, pro, slope=0.1, bias=bias)
            torch.cuda.synchronize()
            for n in range(2):
                h = torch.where(x[n] > 0, x[n], x[n] * 0.1) if leaky else x[n]
                h, w16 = h.half().double(), w.half().double()
                ref, mag = ref_conv(h, w16, s), ref_conv(h.abs(), w16.abs(), s)
                ref, mag = (t[pad:t.shape[0] - pad] for t in (ref, mag))
                if bias is not None:
                    ref = ref + b.double()
                    mag = mag + b.abs().double()
                d = (y[n].double() - ref).abs()
                assert y[n].shape == ref.shape and torch.isfinite(y[n]).all()
                assert not (d > 2.0 ** -13 * mag + 2.0 ** -22 * ref.abs()).any()
            one = C.conv_transpose1d(x[1], cw, pad, pro, slope=0.1, bias=bias)   # rows of one item
            assert torch.allclose(one, y[1], rtol=1e-4, atol=1e-5)
    finally:
        cw.close()
