"""The matrix-core form of the byte row sums against the oracle, bit for bit
(integer sums: no tolerance), where it can go wrong: rows that do not fill sets
of four, tiles and rows that end inside a block of 128 samples, shift spreads on
both sides of one window and over several, DMs that end inside a wavefront, packed
samples, unpadded rows and windows at the input's end, extreme samples, and an
input that is not at a dword (the vector form)."""
import numpy as np
import pytest

import oracle
from dedispersion_amd import DD_SINGLE_STEP, Conf, Plan, workloads
from tests.conftest import host_threads
from tests.gpu_helpers import compare_rows, stream_of, zapped_flags
from tests.packing import pack_rows, random_values

pytestmark = pytest.mark.gpu

BIG, MID, SMALL, TINY = (Conf(64, 8, 16, 8, 16, 1), Conf(64, 4, 8, 8, 5, 1), Conf(64, 4, 16, 4, 8, 1),
                         Conf(64, 1, 4, 4, 2, 1))
CASES = [
    # channels, zapped, samples, dms, step, bits, padding, conf, fill, offset
    *[(72, tuple(range(1, 1 + k)), 1024, 64, 0.5, 8, 128, BIG, None, 0) for k in range(5)],  # 72 - k rows
    *[(70, (), s, 37, 0.5, 8, 0, BIG, None, 0) for s in (1, 127, 129, 1023, 1025, 2100)],
    *[(66, (3,), 700, 33, 0.4, 8, 128, c, None, 0) for c in (MID, SMALL, TINY)],
    # spreads over a wavefront's eight DMs of the lowest channel: 15, 17, 18, 25, 49 and 60 samples
    *[(300, (), 900, 40, step, 8, 128, BIG, None, 0) for step in (0.80, 0.905, 0.96, 1.3, 2.6, 3.2)],
    (300, (), 900, 40, 3.2, 8, 128, MID, None, 0),
    *[(130, (7, 8), 1500, 40, 0.5, bits, pad, c, None, 0) for bits in (1, 2, 4) for pad in (0, 128) for c in (BIG, SMALL)],
    *[(300, (5,), 600, 24, 0.5, 8, 128, BIG, fill, 0) for fill in (0, 255)],
    (80, (), 640, 24, 0.5, 8, 128, BIG, None, 1),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v) for v in (c[0] - len(c[1]), *c[2:7], c[7].threads_d1,
                                                                              c[7].items_d0, c[7].items_d1, c[8], c[9])))
def test_matrix_form(torch_cuda, case):
    torch = torch_cuda
    channels, zapped, samples, dms, step, bits, padding, conf, fill, offset = case
    w = workloads.tiny(channels=channels, samples=samples, dms=dms, step=step, beams=2, sbeams=2, min_freq=1250.0,
                       bandwidth=300.0 / channels, zapped=zapped, seed=7)
    plan = Plan(w.obs, padding, input_bits=bits)
    flags = zapped_flags(plan, zapped)
    plan.set_zapped_channels(flags)
    plan.set_conf(DD_SINGLE_STEP, conf)
    orc = oracle.Oracle(w.obs, padding, threads=host_threads(), input_bits=bits)
    z = plan.sizes
    values = random_values(np.random.default_rng(samples + dms), 2 * channels, z.nr_dispersed_samples, bits)
    if fill is not None:
        values[:] = fill
    host = pack_rows(values, bits, z.in_pitch).ravel()
    room = torch.zeros(host.size + offset, dtype=torch.uint8, device="cuda")
    d_in = room[offset:]
    d_in.copy_(torch.from_numpy(host))
    d_out = torch.full((z.output_elements,), -1.0, dtype=torch.float32, device="cuda")
    plan.dedisperse(d_in.data_ptr(), d_out.data_ptr(), stream=stream_of(torch))
    want = orc.dedispersion(host, flags)
    got = d_out.cpu().numpy().reshape(want.shape)
    compare_rows(got, want, samples, f"{case}")
    assert np.all(got[..., samples:] == -1.0)
