"""The cost model's passes where their blocks of rows could show: an output inside
the input, parameters that are not finite, wide networks over few rows and narrow
ones over many.  Against the numpy reference in float64, with the tolerances of the
tuner's network."""
import ctypes

import numpy as np
import pytest

from dedispersion_amd import load
from dedispersion_amd._lib import check
from oracle import mlp

pytestmark = pytest.mark.gpu


def network(shape, seed):
    """A network and its parameters."""
    lib = load()
    h = ctypes.c_void_p()
    check(lib.dd_mlp_create(ctypes.byref(h), *shape))
    rng = np.random.default_rng(seed)
    p = np.zeros(mlp.param_count(*shape), dtype=np.float32)
    for w, a, b, bo in mlp.layout(*shape):
        p[w:w + a * b] = rng.standard_normal(a * b) * np.sqrt(2.0 / a)
        p[bo:bo + b] = rng.standard_normal(b) * 0.1
    return lib, h, p, rng


def set_params(lib, h, p):
    check(lib.dd_mlp_set_params(h, p.ctypes.data_as(ctypes.POINTER(ctypes.c_float))))


@pytest.mark.parametrize("at", ["first", "middle", "last", "across"])
@pytest.mark.parametrize("shape,n", [((12, 64, 3), 60000), ((3, 100, 1), 4001), ((1, 5, 1), 70000), ((20, 90, 3), 9001)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_output_inside_the_input(torch_cuda, shape, n, at):
    torch = torch_cuda
    lib, h, p, rng = network(shape, n)
    try:
        set_params(lib, h, p)
        x = torch.from_numpy(rng.standard_normal(n * shape[0]).astype(np.float32)).cuda()
        want = torch.empty(n, device="cuda")
        check(lib.dd_mlp_forward(h, x.data_ptr(), n, want.data_ptr(), None))
        room = torch.zeros(n * shape[0] + n, device="cuda")  # the input and, past it, space for one of the outputs
        room[:n * shape[0]] = x
        start = {"first": 0, "middle": n * (shape[0] // 2), "last": n * (shape[0] - 1),
                 "across": n * shape[0] - n // 2}[at]
        check(lib.dd_mlp_forward(h, room.data_ptr(), n, room[start:].data_ptr(), None))
        assert torch.equal(room[start:start + n], want)
        y, _ = mlp.forward(p.astype(np.float64), x.cpu().numpy().reshape(n, -1).astype(np.float64), *shape)
        assert np.max(np.abs(want.cpu().numpy() - y)) <= 1e-5 * max(1.0, np.max(np.abs(y)))
    finally:
        lib.dd_mlp_destroy(h)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 35])
@pytest.mark.parametrize("shape", [(3, 16, 1), (4, 12, 3), (5, 130, 1)], ids=lambda v: "x".join(map(str, v)))
@pytest.mark.parametrize("where", ["bias", "weight"])
def test_parameters_that_are_not_finite(torch_cuda, where, shape, n):
    """A unit of the first layer that is +inf for every row: what the gradient's
    elements are -- finite, an infinity or NaN -- is what the sums over the n rows
    give, whatever fills a block of rows past them."""
    torch = torch_cuda
    lib, h, p, rng = network(shape, n)
    try:
        # all positive, so that no sum meets infinities of both signs
        x = np.abs(rng.standard_normal((n, shape[0]))).astype(np.float32) + 0.5
        t = rng.standard_normal(n).astype(np.float32)
        p = np.abs(p) + np.float32(0.01)
        w, a, b, bo = mlp.layout(*shape)[0]
        if where == "bias":
            p[bo + 2] = np.inf
        else:
            p[w + 2] = np.inf  # input 0 to unit 2
        set_params(lib, h, p)
        dx, dt = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
        dl, dg = (torch.full((k,), 7.0, dtype=torch.float32, device="cuda") for k in (1, p.size))
        check(lib.dd_mlp_loss_grad(h, dx.data_ptr(), dt.data_ptr(), n, dl.data_ptr(), dg.data_ptr(), None))
        with np.errstate(all="ignore"):
            loss, want = mlp.loss_grad(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64), *shape)
        got = dg.cpu().numpy()
        assert np.isinf(want).any() and np.array_equal(np.isnan(got), np.isnan(want))
        assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)].astype(np.float32))
        assert np.isinf(loss) and float(dl[0]) == loss
    finally:
        lib.dd_mlp_destroy(h)


# networks whose weights are read a few columns at a time: widths on both sides of
# whole blocks of columns and of a workgroup's threads, and rows of one to three blocks
@pytest.mark.parametrize("shape,n", [((9, 95, 4), 5), ((9, 96, 4), 4), ((9, 97, 4), 3), ((2, 129, 2), 12), ((256, 255, 2), 6),
                                     ((256, 256, 8), 9), ((33, 160, 5), 1), ((256, 200, 3), 2053)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_wide_networks(torch_cuda, shape, n):
    torch = torch_cuda
    lib, h, p, rng = network(shape, n)
    try:
        x = rng.standard_normal((n, shape[0])).astype(np.float32)
        t = rng.standard_normal(n).astype(np.float32)
        set_params(lib, h, p)
        dx, dt = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
        dl, dg = (torch.full((k,), 7.0, dtype=torch.float32, device="cuda") for k in (1, p.size))
        check(lib.dd_mlp_loss_grad(h, dx.data_ptr(), dt.data_ptr(), n, dl.data_ptr(), dg.data_ptr(), None))
        loss, grad = mlp.loss_grad(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64), *shape)
        assert abs(float(dl[0]) - loss) <= 1e-5 * max(1.0, loss)
        g = dg.cpu().numpy()
        for w, a, b, bo in mlp.layout(*shape):
            for lo, hi in ((w, w + a * b), (bo, bo + b)):
                scale = max(np.max(np.abs(grad[lo:hi])), 1e-12)
                assert np.max(np.abs(g[lo:hi] - grad[lo:hi])) <= 2e-4 * scale, (lo, hi)
    finally:
        lib.dd_mlp_destroy(h)


def test_largest_network_takes_bounded_memory(torch_cuda):
    """The partial gradients of 256 x 256 x 8 over 2880 rows: at most 512 MiB."""
    torch = torch_cuda
    shape, n = (256, 256, 8), 2880
    lib, h, p, rng = network(shape, n)
    try:
        set_params(lib, h, p)
        dx, dt, dl, dg = (torch.zeros(k, dtype=torch.float32, device="cuda") for k in (n * shape[0], n, 1, p.size))
        torch.cuda.synchronize()
        free, _ = torch.cuda.mem_get_info()
        check(lib.dd_mlp_loss_grad(h, dx.data_ptr(), dt.data_ptr(), n, dl.data_ptr(), dg.data_ptr(), None))
        torch.cuda.synchronize()
        assert free - torch.cuda.mem_get_info()[0] <= (512 << 20) + (4 << 20)  # and the allocator's granularity
    finally:
        lib.dd_mlp_destroy(h)


# narrow networks over many rows, whose blocks have 64 rows from 65536 rows on, on both
# sides of that line and of whole blocks; a wide input whose weights fit in LDS beside
# the gradient's rows but not beside the forward pass's
@pytest.mark.parametrize("shape,n", [((1, 1, 1), 65535), ((1, 1, 1), 65536), ((5, 8, 1), 65599), ((63, 16, 8), 65601),
                                     ((12, 17, 2), 65540), ((256, 8, 1), 65602), ((254, 3, 2), 66001), ((256, 16, 1), 65537),
                                     ((256, 39, 1), 50)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_forward_blocks(torch_cuda, shape, n):
    torch = torch_cuda
    lib, h, p, rng = network(shape, n)
    try:
        x = rng.standard_normal((n, shape[0])).astype(np.float32)
        set_params(lib, h, p)
        dx = torch.from_numpy(x).cuda()
        dy = torch.full((n + 64,), 7.0, dtype=torch.float32, device="cuda")
        check(lib.dd_mlp_forward(h, dx.data_ptr(), n, dy.data_ptr(), None))
        want, _ = mlp.forward(p.astype(np.float64), x.astype(np.float64), *shape)
        got = dy.cpu().numpy()
        assert np.max(np.abs(got[:n] - want)) <= 1e-5 * max(1.0, np.max(np.abs(want)))
        assert np.all(got[n:] == 7.0)
    finally:
        lib.dd_mlp_destroy(h)
