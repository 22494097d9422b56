"""Host arrays to the device and back through the context's pinned buffer
(two halves of 524,288 doubles): what is put comes back bit for bit, for one
transfer that fits, for one that ends just at and just past a half, and for
several that share or overrun it, in natural and reverse Cuthill-McKee order
(rows in another order than the caller's) and in both host layouts."""
import numpy as np
import pytest

from tests.helpers import require_lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rcm", [False, True])
@pytest.mark.parametrize("dims", [(1, 1, 1), (5, 4, 3), (64, 64, 42), (64, 64, 43), (128, 64, 64), (61, 87, 83)])
def test_state_round_trip(dims, rcm):
    fvk = require_lib()
    print("host transfers:", dims, "rcm", rcm, flush=True)
    m = fvk.Mesh.box(*dims, jitter=0.0, seed=1)
    ctx = fvk.grd_solv(m, rcm=rcm)
    fl = fvk.Flow(ctx, fvk.flow_cfg())
    rng = np.random.default_rng(sum(dims))
    want = dict(u_cell=rng.standard_normal((m.n_vol, 3)), u_bnd=rng.standard_normal((m.n_bf, 3)),
                p=rng.standard_normal(m.n_vol), dpdx=rng.standard_normal((m.n_vol, 3)),
                spd=rng.standard_normal(m.n_fce))
    for _ in range(2):  # the buffer's halves change roles between the calls
        fl.set_state(**want)
        got = fl.state()
        for k, v in want.items():
            assert np.array_equal(got[k], v), k
    # column-major residuals: with not_r0 the array comes back as it went
    r = rng.standard_normal((m.n_vol, 3))
    back = r.copy()
    norm = fvk.solv_res(ctx, None, back, not_r0=True)
    assert np.array_equal(back, r)
    # sums of n terms in another order: (n - 1) rounding errors of half an ulp at most
    assert np.all(np.abs(norm - np.abs(r).sum(0)) <= m.n_vol * np.finfo(float).eps * np.abs(r).sum(0))
    ctx.destroy()
