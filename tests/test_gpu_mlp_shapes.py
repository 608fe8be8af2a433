"""The cost model's fused passes at other shapes than the tuner's: rows that do
not fill a workgroup's block, more blocks than workgroups, and networks whose
weights do not fit in LDS.  Against the numpy reference in float64; the
tolerances are those of the tuner's network (float32 sums of up to 256 terms, a
gradient relative to the largest of its layer)."""
import ctypes

import numpy as np
import pytest

from dedispersion_amd import load
from dedispersion_amd._lib import check
from oracle import mlp

pytestmark = pytest.mark.gpu

CASES = [((12, 64, 3), n) for n in (1, 15, 16, 17, 8209)] + [((5, 7, 1), 33), ((3, 100, 1), 40), ((20, 90, 3), 37),
                                                            ((256, 256, 2), 21), ((1, 1, 8), 5), ((30, 130, 1), 2051)]


@pytest.mark.parametrize("shape,n", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_fused_passes(torch_cuda, shape, n):
    torch = torch_cuda
    lib = load()
    h = ctypes.c_void_p()
    check(lib.dd_mlp_create(ctypes.byref(h), *shape))
    try:
        count = mlp.param_count(*shape)
        rng = np.random.default_rng(n + shape[1])
        p = np.zeros(count, dtype=np.float32)
        for w, a, b, bo in mlp.layout(*shape):
            p[w:w + a * b] = rng.standard_normal(a * b) * np.sqrt(2.0 / a)
            p[bo:bo + b] = rng.standard_normal(b) * 0.1
        x = rng.standard_normal((n, shape[0])).astype(np.float32)
        t = rng.standard_normal(n).astype(np.float32)
        check(lib.dd_mlp_set_params(h, p.ctypes.data_as(ctypes.POINTER(ctypes.c_float))))
        dx, dt = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
        dy, dl, dg = (torch.full((k,), 7.0, dtype=torch.float32, device="cuda") for k in (n, 1, count))
        check(lib.dd_mlp_forward(h, dx.data_ptr(), n, dy.data_ptr(), None))
        check(lib.dd_mlp_loss_grad(h, dx.data_ptr(), dt.data_ptr(), n, dl.data_ptr(), dg.data_ptr(), None))
        want_y, _ = mlp.forward(p.astype(np.float64), x.astype(np.float64), *shape)
        loss, grad = mlp.loss_grad(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64), *shape)
        assert np.max(np.abs(dy.cpu().numpy() - want_y)) <= 1e-5 * max(1.0, np.max(np.abs(want_y)))
        assert abs(float(dl[0]) - loss) <= 1e-5 * max(1.0, loss)
        g = dg.cpu().numpy()
        for w, a, b, bo in mlp.layout(*shape):
            for lo, hi in ((w, w + a * b), (bo, bo + b)):
                scale = max(np.max(np.abs(grad[lo:hi])), 1e-12)
                assert np.max(np.abs(g[lo:hi] - grad[lo:hi])) <= 2e-4 * scale, (lo, hi)
    finally:
        lib.dd_mlp_destroy(h)
