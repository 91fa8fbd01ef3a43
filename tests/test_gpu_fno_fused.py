"""The fused bfloat16 layers of the FNO at the edges of their shapes: widths that
fill, cross or leave part of a 32-channel tile, rows that end inside a 16- or
32-pixel step, 2 MX not a multiple of 8, one layer (first and last at once), one
wavefront's worth of pixels up to the widest row, and shapes just past what they
take (which run on the separate products): prediction, loss and gradient against
the float64 oracle, and inference against the training forward on one handle.

Bar: 2e-2 relative L2, the bfloat16 bar of the other network tests (operands
rounded at 2^-9, a handful of products one after another); increments 3e-2."""
import numpy as np
import pytest

import tara_amd as T
from oracle import fno_ref as F
from test_gpu_fno import _fields, _rel

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SHAPES = [  # n, width, mx, my, layers, batch
    (8, 5, 2, 4, 1, 2),
    (40, 24, 5, 6, 2, 3),
    (72, 33, 16, 8, 2, 1),
    (104, 32, 7, 10, 3, 2),
    (136, 64, 12, 6, 1, 1),
    (256, 48, 16, 4, 2, 1),
    (264, 16, 4, 4, 2, 1),   # row too wide to fuse
    (64, 72, 4, 4, 2, 1),    # width too large
    (64, 16, 17, 4, 2, 1),   # too many modes
]


@pytest.mark.parametrize("n,width,mx,my,layers,nb", SHAPES)
def test_fused_layers_vs_oracle(n, width, mx, my, layers, nb):
    print(f"fused fno n={n} width={width} modes={mx}x{my} layers={layers} batch={nb}", flush=True)
    cfg = F.Config(n, width, mx, my, layers)
    rng = np.random.default_rng(n + width)
    net = T.FNO(n, width, mx, my, layers, max_batch=nb + 1, seed=5)
    p = net.get_params()
    o = 0
    for name, shape in cfg.sizes():  # a trained-looking network, no zero biases
        k = int(np.prod(shape))
        if name == "w2":
            p[o:o + k] = rng.standard_normal(k) * 0.3
        elif name in ("bl", "b", "b1", "b2"):
            p[o:o + k] = rng.standard_normal(k) * 0.1
        o += k
    net.set_params(p)
    om, tgt = _fields(n, nb, seed=n)
    d_om, d_tgt = torch.from_numpy(om).cuda(), torch.from_numpy(tgt).cuda()
    out = torch.full_like(d_om, float("nan"))
    net.forward(nb, d_om, out)
    pred, lref, gref = F.run(cfg, p.astype(np.float64), om, tgt)
    got = out.cpu().numpy()
    assert _rel(got, pred) < 2e-2
    assert _rel(got - om, pred - om) < 3e-2
    loss, g = net.grads(nb, d_om, d_tgt)
    assert abs(loss - lref) < 2e-2 * max(lref, 1e-3)
    assert _rel(g, gref) < 2e-2
    again = torch.empty_like(out)
    net.forward(nb, d_om, again)  # the training pass in between leaves nothing behind
    assert torch.equal(out, again)
    net.close()
