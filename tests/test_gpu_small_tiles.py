"""The vector byte kernel's smallest tiles, whose rows are taken four at a time,
against the oracle, bit for bit: row counts and rows per barrier that leave one to
three rows over, one and two DMs per wavefront, packed rows, and more rows than one
16-bit accumulation takes."""
import numpy as np
import pytest

import oracle
from dedispersion_amd import DD_SINGLE_STEP, Conf, Plan, workloads
from tests.conftest import host_threads
from tests.gpu_helpers import compare_rows, stream_of, zapped_flags
from tests.packing import pack_rows, random_values

pytestmark = pytest.mark.gpu

CASES = [*[(c, 2, i0, i1, u, 8) for c in (1, 3, 4, 5, 7, 22) for i0, i1, u in ((4, 2, 4), (4, 1, 3), (8, 1, 4))],
         *[(41, 8, 4, 2, u, bits) for u in (7, 16) for bits in (1, 2, 4, 8)],
         (600, 8, 4, 2, 16, 8), (600, 8, 8, 1, 15, 8)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v) for v in c))
def test_small_tiles(torch_cuda, case):
    torch = torch_cuda
    channels, t1, i0, i1, unroll, bits = case
    w = workloads.tiny(channels=channels, samples=530, dms=21, step=0.6, beams=1, sbeams=1, min_freq=1250.0,
                       bandwidth=300.0 / channels, seed=51)
    plan = Plan(w.obs, 0, input_bits=bits)
    flags = zapped_flags(plan, ())
    plan.set_conf(DD_SINGLE_STEP, Conf(64, t1, i0, i1, unroll, 1))
    orc = oracle.Oracle(w.obs, 0, threads=host_threads(), input_bits=bits)
    z = plan.sizes
    host = pack_rows(random_values(np.random.default_rng(52), channels, z.nr_dispersed_samples, bits), bits,
                     z.in_pitch).ravel()
    d_in = torch.from_numpy(host).cuda()
    d_out = torch.full((z.output_elements,), -1.0, dtype=torch.float32, device="cuda")
    plan.dedisperse(d_in.data_ptr(), d_out.data_ptr(), stream=stream_of(torch))
    want = orc.dedispersion(host, flags)
    compare_rows(d_out.cpu().numpy().reshape(want.shape), want, 530, f"{case}")
