"""The GELU of the fused inference layers: the function itself, value by value, and
inference against the training forward, which evaluates it with erff."""
import numpy as np
import pytest
from scipy.special import ndtr

import tara_amd as T
from oracle import fno_ref as F
from test_gpu_fno import _blocks, _fields

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def test_gelu_values():
    """A field of +-1 (scale 1 exactly) through a network that does nothing but the
    projection: the prediction is om + 1024 gelu(b1 +- w1), b1 any float.

    Bar: 4e-8 of Phi, the bound the fit states, times |x|, and the float32 roundings on
    the way out (1 - q, the product, the sum with om: half an ulp each, doubled)."""
    n = 8
    cfg = F.Config(n, 2, 1, 2, 1)
    net = T.FNO(n, 2, 1, 2, 1, max_batch=1)
    om = np.ones((1, n, n), np.float32)
    om[:, ::2] = -1.0
    d_om, out = torch.from_numpy(om).cuda(), torch.empty((1, n, n), dtype=torch.float32, device="cuda")
    rng = np.random.default_rng(4)
    worst = 0.0
    b1s = np.concatenate([np.linspace(-7.5, 7.5, 301), rng.uniform(-1e-2, 1e-2, 40), [-6.5, 6.5, 0.0, 30.0, -30.0]])
    for b1 in b1s.astype(np.float32):
        p = np.zeros(net.nparams, np.float32)
        b = _blocks(cfg, p)
        b["wl"][0], b["w"][0] = 1.0, 1.0  # the first channel only
        b["w1"][0], b["b1"][0], b["w2"][0] = 0.25, b1, 1024.0
        net.set_params(p)
        net.forward(1, d_om, out)
        got = out.cpu().numpy()[0]
        for s in (-1.0, 1.0):
            x = float(np.float32(np.float32(0.25 * s) + b1))
            want = x * ndtr(x)
            vals = got[om[0] == s].astype(np.float64)
            assert (vals == vals[0]).all()
            err = abs((vals[0] - s) / 1024.0 - want)
            bar = 4e-8 * abs(x) + 6 * 2.0 ** -24 * abs(want) + 2.0 ** -23 / 1024
            worst = max(worst, err / bar)
            assert err <= bar, (x, err, bar)
    print(f"gelu: worst error {worst:.2f} of the bar")
    net.close()


@pytest.mark.parametrize("n,width,mx,my,layers,nb", [(64, 32, 8, 8, 2, 2), (128, 48, 12, 8, 4, 2)])
def test_inference_vs_training_forward(n, width, mx, my, layers, nb):
    """The loss of the training forward against that of the inference's prediction.

    Bar: 2e-4 relative.  The two GELUs differ by about 1e-7 of a value, which moves its
    rounding to bfloat16 (spacing 2^-8) in one of 4e4 values; a flip is half a spacing,
    so activations differ by 1e-5 in L2, and the prediction's increment by a few times
    that after several layers."""
    cfg = F.Config(n, width, mx, my, layers)
    net = T.FNO(n, width, mx, my, layers, max_batch=nb, seed=2)
    p = net.get_params()
    rng = np.random.default_rng(width)
    b = _blocks(cfg, p)
    b["w2"][:] = rng.standard_normal(b["w2"].size) * 0.3
    for k in ("bl", "b", "b1", "b2"):
        b[k][:] = rng.standard_normal(b[k].size) * 0.1
    net.set_params(p)
    om, tgt = _fields(n, nb, seed=n)
    d_om, d_tgt = torch.from_numpy(om).cuda(), torch.from_numpy(tgt).cuda()
    out = torch.empty_like(d_om)
    net.forward(nb, d_om, out)
    loss, _ = net.grads(nb, d_om, d_tgt)
    net.close()
    d = out.cpu().numpy().astype(np.float64) - tgt
    want = np.mean(np.sqrt((d ** 2).sum((1, 2))) / np.sqrt((tgt.astype(np.float64) ** 2).sum((1, 2))))
    print(f"loss: training {loss:.8f} inference {want:.8f}")
    assert abs(loss - want) < 2e-4 * want
