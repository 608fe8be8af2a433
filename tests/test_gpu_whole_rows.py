"""The compact batch's step two with a tile's rows whole in LDS against the oracle,
bit for bit (integer sums: no tolerance), where it can go wrong: row counts that do
not fill fours, sums that allow four, two or one row to be added as 16-bit pairs,
samples and DMs that end inside a tile, unpadded rows and windows at the input's end,
runs of several sample tiles, and rows that LDS has no room for (the general kernel)."""
import numpy as np
import pytest

from dedispersion_amd import DD_STEP_TWO, Batch, Conf, workloads
from tests.gpu_helpers import stream_of
from tests.test_gpu_batch import Jobs

pytestmark = pytest.mark.gpu

CASES = [
    # subbands, channels per subband, samples, fine DMs, coarse DMs, step, padding, shape
    *[(s, 3, 700, 19, 3, 0.7, 0, (8, 8, 4)) for s in (1, 2, 3, 4, 5, 31, 33, 66)],
    *[(5, c, 700, 19, 3, 0.3, 0, (8, 8, 4)) for c in (64, 65, 128, 129, 257)],
    *[(6, 2, s, 33, 2, 0.7, pad, (8, 4, 4)) for s in (1, 2, 255, 257, 1027) for pad in (0, 128)],
    *[(7, 2, 1100, 9, 2, 0.7, 128, shape) for shape in ((8, 16, 4), (3, 8, 2), (1, 4, 8), (2, 16, 1))],
    (60, 2, 1100, 64, 2, 4.0, 0, (8, 16, 8)),  # row windows that no uint16 kernel takes: floats, beside the batch
    (60, 2, 1100, 64, 2, 0.2, 0, (8, 16, 8)),  # rows that LDS has no room for
    (2, 2, 8200, 32, 513, 0.5, 0, (8, 8, 4)),  # two tiles per run, the last run cut short
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v) for v in c).replace(" ", ""))
def test_whole_rows(torch_cuda, case):
    subbands, per, samples, fine, coarse, step, padding, (t1, i0, i1) = case
    w = workloads.tiny(channels=subbands * per, samples=samples, dms=fine, step=step, subbands=subbands, coarse=coarse,
                       coarse_step=0.5, beams=2 if coarse < 100 else 1, sbeams=2 if coarse < 100 else 1, min_freq=1300.0,
                       bandwidth=300.0 / (subbands * per), zapped=(1,), seed=41)
    jobs = Jobs(torch_cuda, [w], padding=padding)
    batch = Batch()
    batch.add_two_step(jobs.plans[0], jobs.inputs[0].data_ptr(), jobs.mids[0].data_ptr(), jobs.outs[0].data_ptr())
    batch.set_compact_intermediate(True)
    batch.set_conf(DD_STEP_TWO, Conf(64, t1, i0, i1, 2, 1))
    jobs.reset()
    batch.run(stream=stream_of(torch_cuda))
    compact = 255 * per <= 65535 and step < 4.0
    jobs.check(f"{case}", compact=compact)
    out = jobs.outs[0].cpu().numpy().reshape(jobs.want_out[0].shape)
    assert np.all(out[..., samples:] == -1.0)
