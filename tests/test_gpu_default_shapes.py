"""Plans without a caller's configuration take shapes that follow their sizes: the
results equal the oracle's bit for bit on both sides of each line of the rule
(rows, DMs and workgroups), and a caller's configuration stays through what sets
the shapes again."""
import numpy as np
import pytest

import oracle
from dedispersion_amd import DD_SINGLE_STEP, DD_STEP_ONE, DD_STEP_TWO, Conf, Plan, workloads
from tests.conftest import host_threads
from tests.gpu_helpers import compare_rows, stream_of, zapped_flags
from tests.packing import pack_rows, random_values

pytestmark = pytest.mark.gpu

CASES = [
    # channels, samples, dms, beams, step, bits
    *[(72, 700, 40, 1, 0.4, bits) for bits in (1, 2, 4, 8)],
    (40, 700, 40, 1, 0.4, 8),      # rows for the vector form
    (72, 700, 40, 1, 6.0, 8),      # windows for the vector form
    (72, 4100, 260, 9, 0.4, 8),    # several workgroups per compute unit
    (66, 33000, 512, 2, 0.2, 8),   # the largest tiles
    (72, 700, 40, 1, 40.0, 8),     # row windows near LDS's size
    (64, 1, 1, 1, 0.4, 8),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v) for v in c))
def test_single_step(torch_cuda, case):
    torch = torch_cuda
    channels, samples, dms, beams, step, bits = case
    w = workloads.tiny(channels=channels, samples=samples, dms=dms, step=step, beams=beams, sbeams=beams, min_freq=1250.0,
                       bandwidth=300.0 / channels, zapped=(3,), seed=21)
    plan = Plan(w.obs, 128, input_bits=bits)
    flags = zapped_flags(plan, (3,))
    plan.set_zapped_channels(flags)
    orc = oracle.Oracle(w.obs, 128, threads=host_threads(), input_bits=bits)
    z = plan.sizes
    host = pack_rows(random_values(np.random.default_rng(22), beams * channels, z.nr_dispersed_samples, bits), bits,
                     z.in_pitch).ravel()
    d_in = torch.from_numpy(host).cuda()
    d_out = torch.full((z.output_elements,), -1.0, dtype=torch.float32, device="cuda")
    plan.dedisperse(d_in.data_ptr(), d_out.data_ptr(), stream=stream_of(torch))
    want = orc.dedispersion(host, flags)
    compare_rows(d_out.cpu().numpy().reshape(want.shape), want, samples, f"{case}")


@pytest.mark.parametrize("bits", [8, 32])
@pytest.mark.parametrize("coarse,fine", [(3, 5), (20, 17), (70, 33)])
def test_two_step(torch_cuda, coarse, fine, bits):
    torch = torch_cuda
    for per_subband in (8, 64):
        w = workloads.tiny(channels=2 * per_subband, samples=600, dms=fine, step=0.5, subbands=2, coarse=coarse,
                           coarse_step=0.5 * fine, min_freq=1300.0, bandwidth=100.0 / per_subband, seed=23)
        plan = Plan(w.obs, 128, input_bits=bits)
        orc = oracle.Oracle(w.obs, 128, threads=host_threads(), input_bits=bits)
        flags = zapped_flags(plan, ())
        z = plan.sizes
        rng = np.random.default_rng(24)
        host = (rng.integers(0, 256, z.sub_input_elements, dtype=np.uint8) if bits == 8 else
                rng.standard_normal(z.sub_input_elements).astype(np.float32))
        d_in = torch.from_numpy(host).cuda()
        d_mid = torch.full((z.intermediate_elements,), -1.0, dtype=torch.float32, device="cuda")
        d_out = torch.full((z.sub_output_elements,), -1.0, dtype=torch.float32, device="cuda")
        s = stream_of(torch)
        (plan.step_one if bits == 8 else plan.step_one_f32)(d_in.data_ptr(), d_mid.data_ptr(), stream=s)
        plan.step_two(d_mid.data_ptr(), d_out.data_ptr(), stream=s)
        want_mid = orc.step_one(host, flags)
        mid = d_mid.cpu().numpy().reshape(want_mid.shape)
        compare_rows(mid, want_mid, z.nr_samples_subbanding, "step one")
        want = orc.step_two(mid.ravel())
        compare_rows(d_out.cpu().numpy().reshape(want.shape), want, 600, "step two")


def test_callers_configuration_stays(torch_cuda):
    w = workloads.tiny(channels=64, samples=300, dms=8, step=0.5, subbands=4, coarse=4, coarse_step=4.0, seed=25)
    plan = Plan(w.obs, 128)
    conf = Conf(64, 2, 4, 2, 3, 1)
    for mode in (DD_SINGLE_STEP, DD_STEP_ONE, DD_STEP_TWO):
        plan.set_conf(mode, conf)
    plan.set_shifts(shifts=np.zeros(64, dtype=np.float32))
    for mode in (DD_SINGLE_STEP, DD_STEP_ONE, DD_STEP_TWO):
        assert plan.get_conf(mode) == conf
