"""The padded weight copies of the fused layers follow the parameters: after training
steps and after set_params, inference gives the bits of a new network with these
parameters, at widths that fill and leave part of a 32-channel tile, for one to five
layers."""
import numpy as np
import pytest

import tara_amd as T
from test_gpu_fno import _fields

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n,width,mx,my,layers,nb", [(16, 2, 2, 4, 1, 2), (32, 31, 4, 6, 3, 1), (32, 32, 4, 8, 2, 2),
                                                     (40, 33, 5, 4, 5, 2), (64, 64, 6, 8, 4, 1)])
def test_inference_follows_parameters(n, width, mx, my, layers, nb):
    print(f"refresh n={n} width={width} layers={layers}", flush=True)
    om, tgt = _fields(n, nb, seed=n)
    d_om, d_tgt = torch.from_numpy(om).cuda(), torch.from_numpy(tgt).cuda()
    net = T.FNO(n, width, mx, my, layers, max_batch=nb, seed=1)
    out, want = torch.empty_like(d_om), torch.empty_like(d_om)
    seen = []
    for k in range(3):
        if k == 1:
            for _ in range(2):
                net.train_step(nb, d_om, d_tgt, 1e-2)
        elif k == 2:
            p = np.random.default_rng(7).standard_normal(net.nparams).astype(np.float32) * 0.1
            net.set_params(p)
        net.forward(nb, d_om, out)
        fresh = T.FNO(n, width, mx, my, layers, max_batch=nb, seed=9)
        fresh.set_params(net.get_params())
        fresh.forward(nb, d_om, want)
        assert torch.isfinite(out).all()
        assert torch.equal(out, want), k
        seen.append(out.clone())
        fresh.close()
    assert not torch.equal(seen[0], seen[1]) and not torch.equal(seen[1], seen[2])
    net.close()
