"""The staged float row sums (rows kept as four shifted copies, read four samples
at a time) against the oracle, bit for bit (the same additions in the same order:
no tolerance), where they can go wrong: every tile shape, offsets of every residue
modulo four, samples and DMs that end inside a tile, unpadded rows and windows at
the input's end, an output that is not at 16 bytes, rows that do not fill a group,
more rows than are listed at a time, and shapes whose groups LDS cuts short."""
import numpy as np
import pytest

import oracle
from dedispersion_amd import DD_SINGLE_STEP, DD_STEP_ONE, DD_STEP_TWO, Conf, Plan, workloads
from tests import fused
from tests.conftest import host_threads
from tests.gpu_helpers import compare_rows, stream_of, zapped_flags

pytestmark = pytest.mark.gpu

SHAPES = [Conf(64, t1, i0, i1, u, 1) for t1, u in ((8, 16), (3, 5)) for i0 in (4, 8, 16) for i1 in (1, 2, 4, 8)]
CASES = [
    # channels, zapped, samples, dms, step, padding, conf, offset of the output
    *[(70, (4, 69), 1100, 41, 0.9, 0, c, 0) for c in SHAPES],
    *[(33, (), s, 19, 0.9, 0, Conf(64, 4, 4, 4, 4, 1), 0) for s in (1, 3, 255, 256, 257)],
    *[(60, tuple(range(z)), 520, 9, 0.7, 128, Conf(64, 2, 8, 4, 4, 1), 1) for z in (0, 1, 3, 59, 60)],
    (2100, (5,), 300, 12, 0.5, 128, Conf(64, 4, 4, 2, 16, 1), 0),
    (2049, (), 300, 12, 0.5, 0, Conf(64, 8, 16, 8, 16, 1), 0),
    (64, (), 700, 64, 6.0, 0, Conf(64, 8, 8, 2, 16, 1), 0),
    (64, (), 700, 64, 0.5, 128, None, 0),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v) for v in (
    c[0], len(c[1]), *c[2:6], "default" if c[6] is None else (c[6].threads_d1, c[6].items_d0, c[6].items_d1, c[6].unroll),
    c[7])).replace(" ", ""))
def test_single_step(torch_cuda, case):
    torch = torch_cuda
    channels, zapped, samples, dms, step, padding, conf, offset = case
    w = workloads.tiny(channels=channels, samples=samples, dms=dms, step=step, beams=2, sbeams=2, min_freq=1250.0,
                       bandwidth=300.0 / channels, zapped=zapped, seed=11)
    plan = Plan(w.obs, padding, input_bits=32)
    flags = zapped_flags(plan, zapped)
    plan.set_zapped_channels(flags)
    if conf is not None:
        plan.set_conf(DD_SINGLE_STEP, conf)
    orc = oracle.Oracle(w.obs, padding, threads=host_threads(), input_bits=32)
    z = plan.sizes
    rng = np.random.default_rng(channels + samples)
    host = (rng.standard_normal(z.input_elements) * 10.0 ** rng.integers(-3, 6, z.input_elements)).astype(np.float32)
    d_in = torch.from_numpy(host).cuda()
    room = torch.full((z.output_elements + offset,), -1.0, dtype=torch.float32, device="cuda")
    d_out = room[offset:]
    plan.dedisperse_f32(d_in.data_ptr(), d_out.data_ptr(), stream=stream_of(torch))
    want = orc.dedispersion(host, flags)
    got = d_out.cpu().numpy().reshape(want.shape)
    compare_rows(got, want, samples, f"{case}")
    assert np.all(got[..., samples:] == -1.0)


@pytest.mark.parametrize("padding", [128, 0], ids=["pad128", "unpadded"])
@pytest.mark.parametrize("conf", [None, Conf(64, 8, 4, 1, 3, 1), Conf(64, 3, 8, 2, 8, 1), Conf(64, 8, 16, 8, 16, 1)],
                         ids=lambda c: "default" if c is None else f"t{c.threads_d1}i{c.items_d0}x{c.items_d1}")
def test_two_step(torch_cuda, conf, padding):
    torch = torch_cuda
    w = workloads.tiny(channels=90, samples=1027, dms=19, step=0.9, first=1.1, subbands=6, coarse=5, coarse_step=17.1,
                       coarse_first=2.7, beams=2, sbeams=3, min_freq=1300.0, bandwidth=1.0, zapped=(0, 15, 16, 50), seed=12)
    plan = Plan(w.obs, padding, input_bits=32)
    orc = oracle.Oracle(w.obs, padding, threads=host_threads(), input_bits=32)
    flags = zapped_flags(plan, w.zapped)
    plan.set_zapped_channels(flags)
    if conf is not None:
        plan.set_conf(DD_STEP_ONE, conf)
        plan.set_conf(DD_STEP_TWO, conf)
    z = plan.sizes
    host = (np.random.default_rng(13).standard_normal(z.sub_input_elements) * 1000.0).astype(np.float32)
    d_in = torch.from_numpy(host).cuda()
    d_mid = torch.full((z.intermediate_elements,), -1.0, dtype=torch.float32, device="cuda")
    d_out = torch.full((z.sub_output_elements,), -1.0, dtype=torch.float32, device="cuda")
    s = stream_of(torch)
    plan.step_one_f32(d_in.data_ptr(), d_mid.data_ptr(), stream=s)
    plan.step_two(d_mid.data_ptr(), d_out.data_ptr(), stream=s)
    want_mid = orc.step_one(host, flags)
    mid = d_mid.cpu().numpy().reshape(want_mid.shape)
    compare_rows(mid, want_mid, z.nr_samples_subbanding, f"step one, {conf}")
    want = orc.step_two(mid.ravel())
    compare_rows(d_out.cpu().numpy().reshape(want.shape), want, w.obs.nr_samples_per_batch, f"step two, {conf}")
