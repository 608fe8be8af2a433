"""Which form of a kernel runs, and that each gives the oracle's sums bit for bit
(integer sums: no tolerance).  Every case names the form it is meant for and fails
where another runs: the matrix form of the byte row sums at the edges of its sets of
four rows, of its blocks of samples and of its windows, over packed rows, and its
fallback for input that is not at a dword; batches whose jobs agree on a form,
disagree, or cannot take it, in the persistent and in the chunked launches."""
import numpy as np
import pytest

import oracle
from dedispersion_amd import DD_SINGLE_STEP, DD_STEP_ONE, DD_STEP_TWO, Batch, Conf, DDError, Plan, workloads
from tests.conftest import host_threads
from tests.gpu_helpers import compare_rows, stream_of, zapped_flags
from tests.packing import pack_rows, random_values

pytestmark = pytest.mark.gpu

BIG, MID, SMALL, TINY = (Conf(64, 8, 16, 8, 16, 1), Conf(64, 4, 8, 8, 8, 1), Conf(64, 4, 16, 4, 8, 1),
                         Conf(64, 8, 4, 4, 16, 1))


def beam(channels, samples, dms, step, zapped=(), bits=8, padding=128, offset=0, beams=1, seed=7, subbands=1, coarse=0,
         coarse_step=0.0):
    """One job: its plan, its input `offset` bytes past a dword, its buffers and the oracle's results."""
    import torch

    w = workloads.tiny(channels=channels, samples=samples, dms=dms, step=step, beams=beams, sbeams=beams, min_freq=1250.0,
                       bandwidth=300.0 / channels, zapped=zapped, seed=seed, subbands=subbands, coarse=coarse,
                       coarse_step=coarse_step)
    plan = Plan(w.obs, padding, input_bits=bits)
    flags = zapped_flags(plan, zapped)
    plan.set_zapped_channels(flags)
    orc = oracle.Oracle(w.obs, padding, threads=host_threads(), input_bits=bits)
    z = plan.sizes
    pitch, length = (z.sub_in_pitch, z.nr_dispersed_samples_subbanding) if coarse else (z.in_pitch, z.nr_dispersed_samples)
    host = pack_rows(random_values(np.random.default_rng(seed + samples), beams * channels, length, bits), bits, pitch).ravel()
    room = torch.zeros(host.size + offset, dtype=torch.uint8, device="cuda")
    room[offset:].copy_(torch.from_numpy(host))
    mid = torch.full((max(z.intermediate_elements, 1),), -1.0, dtype=torch.float32, device="cuda")
    out = torch.full((z.sub_output_elements if coarse else z.output_elements,), -1.0, dtype=torch.float32, device="cuda")
    want = orc.step_two(orc.step_one(host, flags).ravel()) if coarse else orc.dedispersion(host, flags)
    return {"plan": plan, "input": room[offset:], "room": room, "mid": mid, "out": out, "want": want, "samples": samples,
            "two_step": bool(coarse)}


def verify(job, what):
    got = job["out"].cpu().numpy().reshape(job["want"].shape)
    compare_rows(got, job["want"], job["samples"], what)
    assert np.all(got[..., job["samples"]:] == -1.0)


# channels, zapped, samples, dms, step, bits, padding, conf, several windows per row
MATRIX = [
    *[(72, tuple(range(1, 1 + k)), 1024, 64, 0.12, 8, 128, BIG, False) for k in range(5)],  # 72 - k rows
    *[(70, (), s, 37, 0.12, 8, 0, BIG, False) for s in (1, 127, 129, 1023, 1025, 2100)],
    *[(66, (3,), 700, 33, 0.1, 8, 128, c, False) for c in (MID, SMALL, TINY)],
    # spreads over a wavefront's eight DMs of the lowest channel: one window takes 17 and 7 + 8
    *[(300, (), 900, 40, step, 8, 128, BIG, step > 0.22) for step in (0.19, 0.215, 0.23, 0.32, 0.4)],
    (300, (9,), 900, 37, 0.4, 8, 0, Conf(64, 4, 16, 8, 8, 1), True),
    *[(130, (7, 8), 1500, 40, 0.12, bits, pad, c, False) for bits in (1, 2, 4) for pad in (0, 128) for c in (BIG, SMALL)],
    *[(300, (7,), 1500, 40, 0.35, bits, 0, BIG, True) for bits in (1, 2, 4)],
]


@pytest.mark.parametrize("case", MATRIX, ids=lambda c: "-".join(str(v) for v in (c[0] - len(c[1]), *c[2:7], c[7].threads_d1,
                                                                               c[7].items_d0, c[7].items_d1)))
def test_matrix(torch_cuda, case):
    channels, zapped, samples, dms, step, bits, padding, conf, wide = case
    job = beam(channels, samples, dms, step, zapped, bits, padding, beams=2)
    job["plan"].set_conf(DD_SINGLE_STEP, conf)
    info = job["plan"].launch_info(DD_SINGLE_STEP)
    assert info["form"] == "matrix" and info["many_windows"] == wide, info
    job["plan"].dedisperse(job["input"].data_ptr(), job["out"].data_ptr(), stream=stream_of(torch_cuda))
    verify(job, f"{case}")


@pytest.mark.parametrize("offset", [0, 1, 2, 3])
@pytest.mark.parametrize("two_step", [False, True])
def test_input_off_a_dword(torch_cuda, two_step, offset):
    """The same call at and past a dword: the matrix form, and the vector form."""
    job = beam(160, 640, 24, 0.12, offset=offset, **(dict(subbands=2, coarse=16, coarse_step=0.1) if two_step else {}))
    mode = DD_STEP_ONE if two_step else DD_SINGLE_STEP
    batch = Batch()
    add(batch, job)
    batch.set_conf(mode, MID)
    assert batch.launch_info(mode)["form"] == ("staged" if offset else "matrix")
    batch.run(stream=stream_of(torch_cuda))
    verify(job, f"batch, {offset}")
    job["out"].fill_(-1.0)
    plan = job["plan"]
    plan.set_conf(mode, MID)
    assert plan.launch_info(mode)["form"] == "matrix"  # of input at a dword
    if two_step:
        plan.step_one(job["input"].data_ptr(), job["mid"].data_ptr(), stream=stream_of(torch_cuda))
        plan.step_two(job["mid"].data_ptr(), job["out"].data_ptr(), stream=stream_of(torch_cuda))
    else:
        plan.dedisperse(job["input"].data_ptr(), job["out"].data_ptr(), stream=stream_of(torch_cuda))
    verify(job, f"plan, {offset}")


def add(batch, job):
    if job["two_step"]:
        batch.add_two_step(job["plan"], job["input"].data_ptr(), job["mid"].data_ptr(), job["out"].data_ptr(), keep=(job,))
    else:
        batch.add_single_step(job["plan"], job["input"].data_ptr(), job["out"].data_ptr(), keep=(job,))


NARROW = dict(channels=300, samples=2100, dms=70, step=0.1)  # one window per row
SEVERAL = dict(channels=300, samples=900, dms=40, step=0.35)  # ... more for some
SPREAD = dict(channels=300, samples=900, dms=40, step=1.3)  # the vector form's
FEW = dict(channels=40, samples=900, dms=40, step=0.1)  # too few rows for the matrix form


def two(j, subbands=3, coarse=24):
    """A job in two steps whose coarse DMs have the steps, and whose subbands the rows, of a single-step job."""
    return dict(j, channels=j["channels"] * subbands, dms=7, step=0.3, subbands=subbands, coarse=coarse,
                coarse_step=j["step"] * (subbands if j["step"] > 1.0 else 1))


SINGLE_BATCHES = [
    ("one", [NARROW], "matrix", False),
    ("agree", [NARROW, dict(NARROW, zapped=(5,), samples=333), dict(NARROW, beams=2, dms=9)], "matrix", False),
    ("several windows", [NARROW, SEVERAL], "matrix", True),
    ("packed with bytes", [NARROW, dict(NARROW, bits=2, padding=0), dict(SEVERAL, bits=1), dict(NARROW, bits=4)], "matrix", True),
    ("mostly matrix", [dict(NARROW, samples=9000), SPREAD], "matrix", True),
    ("mostly vector", [NARROW, dict(SPREAD, samples=30000)], "staged", False),
    ("half vector", [dict(NARROW, samples=3000, dms=64), dict(SPREAD, samples=3000, dms=64, step=2.0)], "staged", False),
    ("few rows", [FEW, FEW], "staged", False),
    ("one off a dword", [dict(NARROW, samples=9000), dict(NARROW, offset=1)], "staged", False),
    ("packed, one off a dword", [dict(NARROW, bits=2), dict(NARROW, bits=2, offset=3, samples=70)], "staged", False),
]


@pytest.mark.parametrize("case", SINGLE_BATCHES, ids=lambda c: c[0])
def test_single_step_batch(torch_cuda, case):
    name, shapes, form, wide = case
    jobs = [beam(**s, seed=20 + k) for k, s in enumerate(shapes)]
    batch = Batch()
    for j in jobs:
        add(batch, j)
    info = batch.launch_info(DD_SINGLE_STEP)
    assert info["form"] == form and info["many_windows"] == wide, info
    for graph in (False, True):
        for j in jobs:
            j["out"].fill_(-1.0)
        batch.run(use_graph=graph, stream=stream_of(torch_cuda))
        for k, j in enumerate(jobs):
            verify(j, f"{name}, graph {graph}, job {k}")


@pytest.mark.parametrize("chunks", [0, 2])
@pytest.mark.parametrize("compact", [True, False])
@pytest.mark.parametrize("case", [c for c in SINGLE_BATCHES if c[0] not in ("few rows", "mostly vector", "half vector")], ids=lambda c: c[0])
def test_two_step_batch(torch_cuda, case, compact, chunks):
    """Step one in the persistent launch and in the chunks' lists, as floats and as uint16 sums."""
    name, shapes, form, wide = case
    shapes = [dict(two(s), samples=min(s["samples"], 3000), zapped=s.get("zapped", (1,)), seed=40 + k)
              for k, s in enumerate(shapes)]
    if compact:  # 257 live channels per subband are the most whose sums fit 16 bits
        shapes = [dict(s, channels=3 * 250) for s in shapes]
    jobs = [beam(**s) for s in shapes]
    batch = Batch()
    for j in jobs:
        add(batch, j)
    batch.set_compact_intermediate(compact)
    batch.set_pipeline(chunks)
    assert batch.info()["compact_intermediate"] == int(compact)
    info = batch.launch_info(DD_STEP_ONE)
    assert info["form"] == form, info
    for graph in (False, True):
        for j in jobs:
            j["out"].fill_(-1.0)
        batch.run(use_graph=graph, stream=stream_of(torch_cuda))
        for k, j in enumerate(jobs):
            verify(j, f"{name}, chunks {chunks}, graph {graph}, job {k}")


def test_queries_refuse_what_cannot_run(torch_cuda):
    job = beam(64, 100, 8, 0.5)
    with pytest.raises(DDError):
        job["plan"].launch_info(DD_SINGLE_STEP, Conf(32, 4, 4, 4, 4, 1))
    with pytest.raises(DDError):
        job["plan"].launch_info(DD_STEP_TWO)
    batch = Batch()
    add(batch, job)
    batch.launch_info(DD_SINGLE_STEP)
    with pytest.raises(DDError):
        batch.launch_info(DD_STEP_TWO)


# subbands, channels per subband, samples, fine DMs, coarse DMs, step, shape, form, tiles per run
STEP_TWO = [
    (31, 3, 700, 19, 3, 0.2, Conf(64, 8, 8, 4, 2, 1), "whole", 1),
    (33, 3, 700, 19, 3, 0.7, Conf(64, 8, 4, 4, 2, 1), "whole", 1),
    (33, 3, 700, 19, 3, 0.7, Conf(64, 8, 8, 4, 2, 1), "staged", 1),  # rows that two workgroups' LDS has no room for
    (60, 3, 700, 19, 3, 0.2, Conf(64, 8, 4, 2, 2, 1), "whole", 1),
    (5, 257, 700, 19, 3, 0.3, Conf(64, 8, 8, 4, 2, 1), "whole", 1),
    (7, 2, 1100, 9, 2, 0.7, Conf(64, 2, 16, 1, 2, 1), "whole", 1),
    (60, 2, 1100, 64, 2, 0.2, Conf(64, 8, 16, 8, 2, 1), "staged", 1),
    (2, 2, 8200, 32, 600, 0.5, Conf(64, 8, 8, 4, 2, 1), "whole", 2),   # the last run cut short
]


@pytest.mark.parametrize("chunks", [0, 2])
@pytest.mark.parametrize("case", STEP_TWO, ids=lambda c: "-".join(str(v) for v in (*c[:6], c[6].items_d0)))
def test_whole_rows(torch_cuda, case, chunks):
    subbands, per, samples, fine, coarse, step, conf, form, run = case
    job = beam(subbands * per, samples, fine, step, (1,), subbands=subbands, coarse=coarse, coarse_step=0.05)
    batch = Batch()
    add(batch, job)
    batch.set_conf(DD_STEP_TWO, conf)
    batch.set_pipeline(chunks)
    info = batch.launch_info(DD_STEP_TWO)
    assert info["form"] == form and info["tiles_per_run"] == run, info
    batch.run(stream=stream_of(torch_cuda))
    verify(job, f"{case}")


@pytest.mark.parametrize("chunks", [0, 2])
@pytest.mark.parametrize("several", ["all have room", "one has none"])
def test_whole_rows_of_several_jobs(torch_cuda, several, chunks):
    """One step-two kernel for the batch: whole rows only where every job's fit."""
    shapes = [(16, 700, 32, 3), (5, 2100, 9, 4), (16 if several == "all have room" else 90, 1030, 33, 2)]
    jobs = [beam(s * 4, samples, fine, 0.3, (2,), subbands=s, coarse=coarse, coarse_step=2.0, seed=60 + k)
            for k, (s, samples, fine, coarse) in enumerate(shapes)]
    batch = Batch()
    for j in jobs:
        add(batch, j)
    batch.set_pipeline(chunks)
    assert batch.launch_info(DD_STEP_TWO)["form"] == ("whole" if several == "all have room" else "staged")
    batch.run(stream=stream_of(torch_cuda))
    for k, j in enumerate(jobs):
        verify(j, f"{several}, chunks {chunks}, job {k}")


# channels, dms, shape, the form, its rows per barrier: sets of four rows per barrier and
# enough work between two barriers for the matrix form, else the vector form, whose
# row list takes half the LDS
ROWS_PER_BARRIER = [
    *[(160, 64, Conf(64, t1, i0, i1, u, 1), "staged", u) for t1, i0, i1 in ((8, 16, 8), (4, 8, 4), (1, 4, 8)) for u in (1, 2)],
    (160, 64, Conf(64, 8, 16, 8, 3, 1), "staged", 3),
    (160, 64, Conf(64, 8, 16, 8, 4, 1), "matrix", 4),
    (160, 64, Conf(64, 8, 8, 8, 4, 1), "staged", 4),
    (160, 64, Conf(64, 8, 8, 8, 8, 1), "matrix", 8),
    (160, 64, Conf(64, 8, 4, 4, 8, 1), "staged", 8),
    (160, 64, Conf(64, 8, 4, 4, 16, 1), "matrix", 16),
    (160, 64, Conf(64, 4, 4, 4, 8, 1), "matrix", 8),
    (160, 64, Conf(64, 2, 8, 4, 4, 1), "matrix", 4),
    (160, 64, Conf(64, 2, 4, 4, 4, 1), "staged", 4),
    (9000, 64, Conf(64, 8, 16, 8, 16, 1), "matrix", 4),  # as many as fit
    (9400, 64, Conf(64, 8, 16, 8, 16, 1), "staged", None),
    (9650, 64, Conf(64, 8, 8, 8, 16, 1), "staged", None),
    (9750, 64, None, "staged", None),
]


@pytest.mark.parametrize("case", ROWS_PER_BARRIER, ids=lambda c: "-".join(str(v) for v in (
    *c[:2], "default" if c[2] is None else (c[2].threads_d1, c[2].items_d0, c[2].items_d1, c[2].unroll))).replace(" ", ""))
def test_rows_per_barrier(torch_cuda, case):
    channels, dms, conf, form, rows = case
    job = beam(channels, 300, dms, 0.1, (3,))
    if conf is not None:
        job["plan"].set_conf(DD_SINGLE_STEP, conf)
    info = job["plan"].launch_info(DD_SINGLE_STEP)
    assert info["form"] == form and (info["rows_per_barrier"] == rows if rows else info["rows_per_barrier"] >= 4), info
    job["plan"].dedisperse(job["input"].data_ptr(), job["out"].data_ptr(), stream=stream_of(torch_cuda))
    verify(job, f"{case}")


# channels, dms, samples, step, bits: plans whose row windows the pipeline cannot take in
# the shape of their sizes, and the form that their own configuration runs
WIDE_WINDOWS = [(73, 961, 15484, 6.13, 32, "groups"), (64, 500, 8000, 12.0, 32, "groups"),
                (61, 53, 16745, 11.6, 32, "direct"), (73, 961, 15484, 0.2, 32, "staged")]


@pytest.mark.parametrize("case", WIDE_WINDOWS, ids=lambda c: "-".join(map(str, c)))
def test_default_shape_of_wide_windows(torch_cuda, case):
    channels, dms, samples, step, bits, form = case
    w = workloads.tiny(channels=channels, samples=samples, dms=dms, step=step, min_freq=1250.0, bandwidth=300.0 / channels)
    plan = Plan(w.obs, 128, input_bits=bits)
    assert plan.launch_info(DD_SINGLE_STEP)["form"] == form


# subbands, coarse DMs, fine DMs, samples, the default's form and tile (samples per lane, DMs
# per wavefront): one group of rows up to 16 subbands, more go through the pipeline
DEFAULT_STEP_TWO = [
    (1, 3, 7, 700, "groups", 4, 1), (2, 40, 8, 2300, "groups", 8, 1), (3, 2, 9, 1100, "groups", 4, 2),
    (16, 30, 16, 2600, "groups", 8, 2), (16, 2, 33, 520, "groups", 4, 2), (4, 260, 17, 900, "groups", 8, 4),
    (17, 2, 9, 700, "staged", 4, 2), (17, 3, 33, 700, "staged", 4, 8), (18, 2, 41, 700, "staged", 4, 4),
    (17, 180, 45, 1300, "staged", 8, 8), (20, 530, 41, 500, "staged", 8, 8),
]


@pytest.mark.parametrize("case", DEFAULT_STEP_TWO, ids=lambda c: "-".join(map(str, c)))
def test_default_shape_of_step_two(torch_cuda, case):
    subbands, coarse, fine, samples, form, items_d0, items_d1 = case
    job = beam(subbands * 2, samples, fine, 0.4, subbands=subbands, coarse=coarse, coarse_step=0.1)
    plan = job["plan"]
    conf = plan.get_conf(DD_STEP_TWO)
    assert plan.launch_info(DD_STEP_TWO)["form"] == form and (conf.items_d0, conf.items_d1) == (items_d0, items_d1), conf
    plan.step_one(job["input"].data_ptr(), job["mid"].data_ptr(), stream=stream_of(torch_cuda))
    plan.step_two(job["mid"].data_ptr(), job["out"].data_ptr(), stream=stream_of(torch_cuda))
    verify(job, f"{case}")


# channels per subband, subbands, coarse DMs, samples, the default's tile: wavefronts, samples
# per lane, DMs per wavefront
DEFAULT_STEP_ONE = [
    (3, 128, 2, 7905, 4, 16, 4), (3, 16, 2, 7905, 8, 8, 2), (5, 128, 2, 7905, 8, 8, 2), (4, 128, 33, 8300, 4, 16, 8),
    (8, 8, 89, 2746, 8, 8, 4), (5, 128, 68, 9521, 4, 16, 8), (5, 128, 96, 4200, 4, 16, 8), (5, 128, 97, 4200, 8, 16, 8),
]


@pytest.mark.parametrize("case", DEFAULT_STEP_ONE, ids=lambda c: "-".join(map(str, c)))
def test_default_shape_of_step_one(torch_cuda, case):
    per, subbands, coarse, samples, waves, items_d0, items_d1 = case
    job = beam(subbands * per, samples, 1, 0.0, subbands=subbands, coarse=coarse, coarse_step=0.1)
    plan = job["plan"]
    conf = plan.get_conf(DD_STEP_ONE)
    assert (conf.threads_d1, conf.items_d0, conf.items_d1) == (waves, items_d0, items_d1), conf
    plan.step_one(job["input"].data_ptr(), job["mid"].data_ptr(), stream=stream_of(torch_cuda))
    plan.step_two(job["mid"].data_ptr(), job["out"].data_ptr(), stream=stream_of(torch_cuda))
    verify(job, f"{case}")


@pytest.mark.parametrize("tables", ["formula", "rising", "zero"])
@pytest.mark.parametrize("first,step", [(0.0, 0.7), (40.0, 0.3), (3.0, 0.0)])
def test_largest_shift(torch_cuda, tables, first, step):
    """The sizes' largest shifts are those of the integer tables, also where step one's
    delays relative to a subband's top channel are negative (a table that rises)."""
    w = workloads.tiny(channels=24, samples=100, dms=9, step=step, first=first, subbands=4, coarse=7, coarse_step=2.5,
                       coarse_first=first)
    plan = Plan(w.obs, 128)
    if tables != "formula":
        a, b = plan.get_shifts()
        a[:24] = np.linspace(0.1, 3.0, 24) if tables == "rising" else 0.0
        b[:4] = np.linspace(0.1, 3.0, 4) if tables == "rising" else 0.0
        plan.set_shifts(a, b)
    z = plan.sizes
    for mode, largest in ((DD_SINGLE_STEP, z.max_shift), (DD_STEP_ONE, z.max_shift_step_one), (DD_STEP_TWO, z.max_shift_step_two)):
        table = plan.get_integer_shifts(mode)
        assert largest == table.max()
        assert np.all(np.diff(table.astype(np.int64), axis=1) >= 0)


# float rows: channels, samples, dms, shape, copies of a row in LDS.  One copy where
# workgroups of few DMs share the compute units, four elsewhere
FLOAT_SINGLE = [
    *[(37, 20001, 1000, Conf(64, *s, 1), 1) for s in ((1, 4, 1, 2), (1, 16, 4, 2), (2, 8, 4, 3), (4, 8, 2, 8), (2, 4, 8, 4),
                                                      (8, 8, 1, 16), (4, 4, 4, 5), (8, 4, 2, 7), (1, 8, 8, 1))],
    (37, 20001, 1000, Conf(64, 8, 16, 1, 4, 1), 4), (37, 20001, 1000, Conf(64, 1, 16, 8, 2, 1), 4),
    (37, 20001, 1000, Conf(64, 4, 4, 8, 4, 1), 4),
    (37, 3001, 70, Conf(64, 1, 4, 4, 2, 1), 4), (37, 3001, 70, Conf(64, 8, 8, 1, 4, 1), 4),
]


@pytest.mark.parametrize("padding", [0, 128])
@pytest.mark.parametrize("case", FLOAT_SINGLE, ids=lambda c: "-".join(map(str, (*c[:3], c[3].threads_d1, c[3].items_d0,
                                                                               c[3].items_d1, c[3].unroll))))
def test_copies_of_float_rows(torch_cuda, case, padding):
    """Additions in the oracle's order: no tolerance."""
    torch = torch_cuda
    channels, samples, dms, conf, copies = case
    w = workloads.tiny(channels=channels, samples=samples, dms=dms, step=0.05, min_freq=1250.0, bandwidth=300.0 / channels,
                       zapped=(0, 9), seed=13)
    plan = Plan(w.obs, padding, input_bits=32)
    flags = zapped_flags(plan, w.zapped)
    plan.set_zapped_channels(flags)
    plan.set_conf(DD_SINGLE_STEP, conf)
    info = plan.launch_info(DD_SINGLE_STEP)
    assert info["form"] == "staged" and info["copies"] == copies, info
    z = plan.sizes
    host = (np.random.default_rng(3).standard_normal(z.input_elements) * 100.0).astype(np.float32)
    d_in = torch.from_numpy(host).cuda()
    d_out = torch.full((z.output_elements,), -1.0, dtype=torch.float32, device="cuda")
    plan.dedisperse_f32(d_in.data_ptr(), d_out.data_ptr(), stream=stream_of(torch))
    want = oracle.Oracle(w.obs, padding, threads=host_threads(), input_bits=32).dedispersion(host, flags)
    got = d_out.cpu().numpy().reshape(want.shape)
    compare_rows(got, want, samples, f"{case}")
    assert np.all(got[..., samples:] == -1.0)


@pytest.mark.parametrize("chunks", [0, 2])
@pytest.mark.parametrize("case", ["large", "small", "together large", "large and small"])
def test_copies_of_a_batch(torch_cuda, case, chunks):
    """One form for all jobs of a batch, by their tiles together."""
    big = dict(channels=40, samples=4000, dms=9, step=0.3, subbands=5, coarse=90, coarse_step=0.2, zapped=(2,))
    small = dict(big, samples=600, coarse=7)
    jobs = {"large": [big], "small": [small], "together large": [dict(small, coarse=40 + k, seed=k) for k in range(9)],
            "large and small": [small, big, dict(small, beams=2)]}[case]
    jobs = [beam(**j) for j in jobs]
    batch = Batch()
    for j in jobs:
        add(batch, j)
    batch.set_compact_intermediate(False)
    batch.set_pipeline(chunks)
    batch.set_conf(DD_STEP_TWO, Conf(64, 2, 4, 2, 3, 1))
    info = batch.launch_info(DD_STEP_TWO)
    assert info["form"] == "staged" and info["copies"] == (4 if case == "small" else 1), info
    assert batch.info()["solo_jobs"] == 0
    for graph in (False, True):
        for j in jobs:
            j["out"].fill_(-1.0)
        batch.run(use_graph=graph, stream=stream_of(torch_cuda))
        for k, j in enumerate(jobs):
            verify(j, f"{case}, chunks {chunks}, graph {graph}, job {k}")


# plans of wide windows: channels per subband, subbands, coarse DMs, samples, their step, and the default's tile
WIDE_STEP_ONE = [(44, 32, 33, 9000, 60.0, 8, 16, 4), (44, 32, 33, 9000, 1.0, 8, 8, 4), (44, 32, 33, 2000, 60.0, 8, 8, 4),
                 (44, 8, 33, 17000, 60.0, 8, 8, 2), (20, 4, 40, 9000, 60.0, 8, 8, 2)]


@pytest.mark.parametrize("case", WIDE_STEP_ONE, ids=lambda c: "-".join(map(str, c)))
def test_default_shape_of_wide_step_one(torch_cuda, case):
    per, subbands, coarse, samples, step, waves, items_d0, items_d1 = case
    job = beam(subbands * per, samples, 1, 0.0, subbands=subbands, coarse=coarse, coarse_step=step)
    plan = job["plan"]
    conf = plan.get_conf(DD_STEP_ONE)
    assert (conf.threads_d1, conf.items_d0, conf.items_d1) == (waves, items_d0, items_d1), conf
    plan.step_one(job["input"].data_ptr(), job["mid"].data_ptr(), stream=stream_of(torch_cuda))
    plan.step_two(job["mid"].data_ptr(), job["out"].data_ptr(), stream=stream_of(torch_cuda))
    verify(job, f"{case}")


def test_default_shape_of_wide_step_two(torch_cuda):
    """Windows that the pipeline does not take: the shape of one group."""
    w = workloads.tiny(channels=64, samples=12288, dms=20, step=3.0, subbands=32, coarse=100, coarse_step=60.0,
                       min_freq=1250.0, bandwidth=300.0 / 64)
    plan = Plan(w.obs, 128)
    conf = plan.get_conf(DD_STEP_TWO)
    assert plan.launch_info(DD_STEP_TWO)["form"] == "groups" and (conf.threads_d1, conf.items_d0, conf.items_d1) == (8, 8, 4)


# jobs (subbands, their step), the form of the batch that asks for the paired step two, its rows
PAIRED = [
    ("all pairs", [(16, 0.1), (6, 0.05)], "pairs", 8), ("one is odd", [(16, 0.1), (5, 0.05)], "pairs", 8),
    ("many subbands", [(16, 0.1), (66, 0.05)], "pairs", 8),
    ("one spreads too far", [(16, 0.1), (16, 1.0)], "whole", 4), ("one has no room", [(16, 1.0), (90, 0.05)], "staged", 4),
]


@pytest.mark.parametrize("chunks", [0, 2])
@pytest.mark.parametrize("case", PAIRED, ids=lambda c: c[0])
def test_paired_step_two_and_what_stands_in(torch_cuda, case, chunks):
    """Where a job cannot take the paired step two, the batch runs what it would without asking."""
    name, shapes, form, rows = case
    jobs = [beam(s * 2, 900, 19, step, (1,), subbands=s, coarse=3, coarse_step=2.0, seed=80 + k)
            for k, (s, step) in enumerate(shapes)]
    forms = []
    for paired in (False, True):
        batch = Batch()
        for j in jobs:
            add(batch, j)
            j["out"].fill_(-1.0)
        batch.set_paired_step_two(paired)
        batch.set_pipeline(chunks)
        forms.append((batch.launch_info(DD_STEP_TWO)["form"], batch.get_conf(DD_STEP_TWO).unroll))
        assert batch.info()["paired_step_two"] == (paired and form == "pairs")
        batch.run(stream=stream_of(torch_cuda))
        for k, j in enumerate(jobs):
            verify(j, f"{name}, paired {paired}, chunks {chunks}, job {k}")
    assert forms[1] == (form, rows) and (form == "pairs" or forms[0] == forms[1])


@pytest.mark.parametrize("two_step", [False, True])
def test_matrix_batch_with_lds_to_the_last_byte(torch_cuda, two_step):
    """A row list that fills LDS beside the rows per barrier: the persistent kernel's
    claim slot has its room too, whatever the number of channels."""
    mode = DD_STEP_ONE if two_step else DD_SINGLE_STEP
    limit = 160 * 1024

    def plan_of(channels):
        w = workloads.tiny(channels=channels, samples=300, dms=1 if two_step else 8, step=0.01, min_freq=1250.0,
                           bandwidth=300.0 / channels, coarse=8 if two_step else 0, coarse_step=0.01)
        return Plan(w.obs, 128)

    conf = Conf(64, 4, 16, 8, 8, 1)
    base = plan_of(6000).launch_info(mode, conf)
    assert base["form"] == "matrix" and base["rows_per_barrier"] == 8
    channels = 6000 + (limit - base["lds_bytes"]) // 16  # 16 bytes per channel
    rows = set()
    for c in range(channels - 2, channels + 3):
        plan = plan_of(c)
        info = plan.launch_info(mode, conf)
        assert info["form"] == "matrix" and info["lds_bytes"] <= limit - 16, (c, info)
        rows.add(info["rows_per_barrier"])
        z = plan.sizes
        buffers = [torch_cuda.zeros(max(n, 1), dtype=d, device="cuda") for n, d in (
            (max(z.input_elements, z.sub_input_elements), torch_cuda.uint8), (z.intermediate_elements, torch_cuda.float32),
            (max(z.output_elements, z.sub_output_elements), torch_cuda.float32))]
        batch = Batch()
        if two_step:
            batch.add_two_step(plan, *(b.data_ptr() for b in buffers))
        else:
            batch.add_single_step(plan, buffers[0].data_ptr(), buffers[2].data_ptr())
        assert batch.launch_info(mode)["form"] == "matrix"
        batch.run(stream=stream_of(torch_cuda))
    assert rows == {7, 8}
    torch_cuda.cuda.synchronize()
