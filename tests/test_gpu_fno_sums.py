"""The learned step's column and split-K sums at the edges of their blocks."""
import numpy as np
import pytest

import g4mi
import fno_reference as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ngrid,batch,width,hidden", [(17, 1, 8, 16), (33, 3, 8, 16), (151, 6, 8, 16), (40, 2, 24, 40)])
def test_fno_gradient_sums(ngrid, batch, width, hidden):
    """Fewer rows than the column sums' blocks, a remainder in every lane and
    the eight-row passes (16 channels at 151^2 x 6), channel counts that do
    not divide a block, against float64 autograd: the bounds of the
    gradient test (BF16 products; relative L2 5 %, cosine 0.998)."""
    sh = dict(ngrid=ngrid, width=width, modes=8, layers=1, hidden=hidden)
    f = g4mi.Fno(max_batch=batch, seed=4, **sh)
    rng = np.random.default_rng(ngrid)
    p = f.get_params().astype(np.float64)
    for name, o, n in f.param_blocks():
        if name.startswith("R"):
            p[o:o + n] = rng.normal(size=n) * 0.3
        elif name.startswith("b"):
            p[o:o + n] = rng.normal(size=n) * 0.1
    f.set_params(p.astype(np.float32))
    inp = rng.normal(size=(batch, ngrid * ngrid, 4)).astype(np.float32)
    # a target off the output's mean: the bias sums do not cancel
    tgt = (rng.normal(size=(batch, ngrid * ngrid, 2)) + 3).astype(np.float32)
    _, g = f.loss_grad(inp, tgt)
    _, rg, _ = R.loss_and_grad(p, inp, tgt, ngrid, width, 8, 1, hidden)
    for name, o, n in f.param_blocks():
        a, b = g[o:o + n].astype(np.float64), rg[o:o + n]
        e = np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)
        cos = float(a @ b / max(np.linalg.norm(a) * np.linalg.norm(b), 1e-300))
        print(f"  {ngrid}^2 x {batch}, {name}: {e:.2e} {cos:.6f}", flush=True)
        assert e < 5e-2 and cos > 0.998, name
    f.close()
