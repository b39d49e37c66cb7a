"""Equivalent-offset migration on the GPU (ktm_eom_*) against the oracle's
restatement of EOM.c csp(): fold and the evaluated-sample count bit for bit,
the gathers to FP32 rounding (the double atan of the taper, EOM.c:1291, may
differ from the C library's in its last bit), per job and for all jobs, on a
line and on a rotated 3-D CSP grid, the post filter (EOM.c:1386-1413), the
job-local entry points, the image<job>.su records (EOM.c:1346-1537) and the
csp(job_id) shim end to end."""
import os

import numpy as np
import pytest
import torch

import oracle
from random_amd import surveys
from random_amd.eom import EomConfig, EomPlan

pytestmark = pytest.mark.gpu


def rel_l2(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def line_case():
    sv = surveys.line2d(nshots=6, nrecv_side=12, ns=501, ncols=80, col_dx=12.5, nscat=4,
                        x0=400.0, t0_range=(0.2, 1.5))
    cfg = EomConfig(ox=0.0, oy=0.0, angle_e_to_n=0.0, oxcsp=0.0, oycsp=0.0, excsp=1500.0,
                    eycsp=0.0, scale_xy=0.01, dcsp_x=12.5, dcsp_y=0.0, dh=25.0, nh=32,
                    aperture=800.0, jobs_x=3, jobs_y=1, ntblock=50, velocity_start=2000.0,
                    velocity_end=2000.0)
    return sv, cfg, surveys.traces_numpy(sv)


def test_eom_line_matches_oracle(cuda):
    print("case: EOM line vs oracle", flush=True)
    sv, cfg, tr = line_case()
    plan = EomPlan(cfg, sv.ns, sv.dt)
    d_tr, d_co = torch.from_numpy(tr).to(cuda), torch.from_numpy(sv.coords).to(cuda)
    csp, fold, n = plan.migrate(d_tr, d_co)
    c0, f0, n0 = oracle.eom_all(cfg, sv.ns, np.float32(sv.dt), tr, sv.coords, cfg.velocity(sv.ns))
    c, f = csp.cpu().numpy(), fold.cpu().numpy()
    same = float(np.mean(c.view(np.uint32) == c0.view(np.uint32)))
    print(f"  evaluated {n} (oracle {n0}); gathers relL2 {rel_l2(c, c0):.2e}, bit-identical "
          f"fraction {same:.8f}; fold cells differing {np.sum(f != f0)}")
    assert n == n0
    assert np.array_equal(f, f0)
    assert rel_l2(c, c0) <= 1e-6
    # one job: its slab equals the oracle's job, the rest stays at the reset value
    job = 1
    cj, fj, nj = plan.migrate(d_tr, d_co, job=job)
    oc, of, on = oracle.eom_job(cfg, sv.ns, np.float32(sv.dt), job, tr, sv.coords,
                                cfg.velocity(sv.ns))
    nx = plan.setup["nx"]
    cj, fj = cj.cpu().numpy(), fj.cpu().numpy()
    assert nj == on
    assert np.array_equal(fj[job * nx:(job + 1) * nx], of)
    assert rel_l2(cj[job * nx:(job + 1) * nx], oc) <= 1e-6
    rest = np.ones(cj.shape[0], bool)
    rest[job * nx:(job + 1) * nx] = False
    assert not cj[rest].any() and np.all(fj[rest] == 1.0)


def test_eom_rotated_grid_matches_oracle(cuda):
    print("case: EOM rotated 3-D CSP grid vs oracle", flush=True)
    sv = surveys.area3d(ntr=400, ns=301, ncols=16, extent=700.0, max_offset=900.0, nscat=3)
    tr = surveys.traces_numpy(sv)
    # header words are metres + 5000; a rotated survey frame with its own origin
    cfg = EomConfig(ox=4900.0, oy=5100.0, angle_e_to_n=12.0, oxcsp=5000.0, oycsp=5000.0,
                    excsp=5400.0, eycsp=5300.0, scale_xy=1.0, dcsp_x=25.0, dcsp_y=30.0, dh=20.0,
                    nh=24, aperture=500.0, jobs_x=2, jobs_y=3, ntblock=128,
                    velocity_start=1800.0, velocity_end=1800.0)
    plan = EomPlan(cfg, sv.ns, sv.dt)
    csp, fold, n = plan.migrate(torch.from_numpy(tr).to(cuda), torch.from_numpy(sv.coords).to(cuda))
    c0, f0, n0 = oracle.eom_all(cfg, sv.ns, np.float32(sv.dt), tr, sv.coords, cfg.velocity(sv.ns))
    c, f = csp.cpu().numpy(), fold.cpu().numpy()
    same = float(np.mean(c.view(np.uint32) == c0.view(np.uint32)))
    print(f"  evaluated {n} (oracle {n0}); gathers relL2 {rel_l2(c, c0):.2e}, bit-identical "
          f"fraction {same:.8f}")
    assert n == n0 and n > 0
    assert np.array_equal(f, f0)
    assert rel_l2(c, c0) <= 1e-6


def test_eom_post_matches_oracle(cuda):
    print("case: EOM post filter vs oracle", flush=True)
    sv, cfg, tr = line_case()
    plan = EomPlan(cfg, sv.ns, sv.dt)
    csp, fold, _ = plan.migrate(torch.from_numpy(tr).to(cuda), torch.from_numpy(sv.coords).to(cuda))
    out = plan.post(csp, fold).cpu().numpy()
    lp, rr = oracle.eom_filters(cfg, sv.ns, np.float32(sv.dt))
    ref = oracle.eom_post(csp.cpu().numpy(), fold.cpu().numpy(), np.float32(sv.dt), lp, rr)
    e = rel_l2(out, ref)
    print(f"  post relL2 {e:.2e}")
    assert e <= 1e-6


def test_eom_job_gathers_and_records(cuda):
    """The job-local entry points (the arrays of csp(job_id)): gathers equal
    to the full volume's slab bit for bit and to the oracle's job, the post
    filter, and the image<job>.su bytes against the oracle's writer fed the
    same post-filtered gathers.  excsp = 1480 leaves the last slab one CSP
    short, so its records stop early (EOM.c:1417)."""
    print("case: EOM job-local gathers, post and records", flush=True)
    sv, cfg, tr = line_case()
    cfg = cfg.replace(excsp=1480.0)
    plan = EomPlan(cfg, sv.ns, sv.dt)
    assert (plan.setup["Nx"], plan.setup["nx"]) == (119, 40)
    d_tr, d_co = torch.from_numpy(tr).to(cuda), torch.from_numpy(sv.coords).to(cuda)
    full, ffold, _ = plan.migrate(d_tr, d_co)
    lp, rr = oracle.eom_filters(cfg, sv.ns, np.float32(sv.dt))
    nx, rec = plan.setup["nx"], 240 + 4 * sv.ns
    for job in range(plan.setup["no_job"]):
        cj, fj, nj = plan.job_migrate(d_tr, d_co, job)
        assert torch.equal(cj, full[job * nx:(job + 1) * nx])
        assert torch.equal(fj, ffold[job * nx:(job + 1) * nx])
        oc, of, on = oracle.eom_job(cfg, sv.ns, np.float32(sv.dt), job, tr, sv.coords,
                                    cfg.velocity(sv.ns))
        assert nj == on and np.array_equal(fj.cpu().numpy(), of)
        assert rel_l2(cj.cpu().numpy(), oc) <= 1e-6
        pj = plan.job_post(cj, fj)
        ref = oracle.eom_post(cj.cpu().numpy(), fj.cpu().numpy(), np.float32(sv.dt), lp, rr)
        assert rel_l2(pj.cpu().numpy(), ref) <= 1e-6
        data = plan.job_records(pj, job)
        want = oracle.eom_job_records(cfg, sv.ns, np.float32(sv.dt), job, pj.cpu().numpy())
        print(f"  job {job}: {len(data) // rec} records")
        assert len(data) == len(want) == (39 if job == 2 else 40) * cfg.nh * rec
        assert data == want


def test_eom_records_rotated_2d_jobs(cuda):
    """Record bytes on a rotated 3-D CSP grid with 2 x 3 job slabs (cdpx/cdpy
    from the rotated CSP position, cdp/iline numbering, the record-count
    prefix rule) for random post-filtered gathers."""
    print("case: EOM records, rotated 2 x 3 job grid", flush=True)
    cfg = EomConfig(ox=4900.0, oy=5100.0, angle_e_to_n=12.0, oxcsp=5000.0, oycsp=5000.0,
                    excsp=5400.0, eycsp=5300.0, scale_xy=1.0, dcsp_x=25.0, dcsp_y=30.0, dh=20.0,
                    nh=5, aperture=500.0, jobs_x=2, jobs_y=3, ntblock=128,
                    velocity_start=1800.0, velocity_end=1800.0)
    ns, dt = 97, np.float32(0.002)
    plan = EomPlan(cfg, ns, dt)
    rng = np.random.default_rng(11)
    counts = []
    for job in range(plan.setup["no_job"]):
        post = rng.standard_normal(plan.job_shape).astype(np.float32)
        data = plan.job_records(torch.from_numpy(post).to(cuda), job)
        assert data == oracle.eom_job_records(cfg, ns, dt, job, post)
        counts.append(len(data) // (240 + 4 * ns))
    print(f"  records per job {counts}")
    nrec = plan.setup["nx"] * plan.setup["ny"] * cfg.nh
    total = plan.setup["Nx"] * plan.setup["Ny"] * cfg.nh
    assert counts == [min(nrec, max(0, total - nrec * j)) for j in range(6)]


def test_eom_csp_shim_files(cuda, tmp_path):
    """csp(job_id) end to end: an IBM SEG-Y line read in blocks of ntblock,
    image<job>.su against the oracle's csp() restatement (headers byte for
    byte, samples to FP32 rounding) and the header files."""
    from test_gpu_shim import write_input
    import ctypes as C
    from random_amd import _lib
    print("case: csp(job) shim, 3 jobs, IBM input", flush=True)
    sv, cfg, tr = line_case()
    cfg = cfg.replace(excsp=1480.0, ntblock=70)    # several blocks, the last one short
    path = str(tmp_path / "in.sgy")
    write_input(path, sv, tr)
    raw = np.fromfile(path, np.uint8)[3600:].reshape(sv.ntr, 240 + 4 * sv.ns)[:, 240:]
    tr_ibm = oracle.ibm_to_float(raw.ravel()).reshape(sv.ntr, sv.ns)
    dt = np.float32(sv.dt)
    lp, rr = oracle.eom_filters(cfg, sv.ns, dt)
    L = _lib.lib()
    c = cfg.to_c()
    img_dir = str(tmp_path / "image_dir")
    _lib.check(L.ktm_eom_globals_init(C.byref(c), path.encode(), img_dir.encode()),
               "ktm_eom_globals_init")
    rec = 240 + 4 * sv.ns
    try:
        g = oracle.eom_grid(cfg)
        for job in range(g.no_job):
            L.csp(job)
            assert L.ktm_eom_last_status() == 0
            data = open(os.path.join(img_dir, f"image{job}.su"), "rb").read()
            oc, of, _ = oracle.eom_job(cfg, sv.ns, dt, job, tr_ibm, sv.coords, cfg.velocity(sv.ns))
            want = oracle.eom_job_records(cfg, sv.ns, dt, job, oracle.eom_post(oc, of, dt, lp, rr))
            assert len(data) == len(want)
            got = np.frombuffer(data, np.uint8).reshape(-1, rec)
            ref = np.frombuffer(want, np.uint8).reshape(-1, rec)
            assert np.array_equal(got[:, :240], ref[:, :240])
            x = got[:, 240:].copy().view(">f4").astype(np.float64)
            y = ref[:, 240:].copy().view(">f4").astype(np.float64)
            e = np.linalg.norm(x - y) / max(np.linalg.norm(y), 1e-300)
            print(f"  job {job}: {len(got)} records, samples relL2 {e:.2e}")
            assert e <= 1e-5
        fh = oracle.eom_file_header(sv.ns, dt)
        assert open(os.path.join(img_dir, "ebdic_header.bin"), "rb").read() == fh[:3200]
        assert open(os.path.join(img_dir, "binary_header.bin"), "rb").read() == fh[3200:]
        L.csp(g.no_job)   # a job that does not exist is an error, not an exit
        assert L.ktm_eom_last_status() == _lib.KTM_ERR_ARG
    finally:
        L.ktm_eom_globals_free()


@pytest.mark.parametrize("ns", [1001, 4097, 7000])
def test_eom_post_long_traces(cuda, ns):
    """The post filter with 4 gather traces per workgroup (short traces), one
    per workgroup with g in LDS (4097) and with g read from global memory
    (7000 samples), against the oracle's DFT path."""
    print(f"case: EOM post filter at ns={ns}", flush=True)
    cfg = EomConfig(ox=0.0, oy=0.0, angle_e_to_n=0.0, oxcsp=0.0, oycsp=0.0, excsp=50.0,
                    eycsp=0.0, dcsp_x=12.5, dh=25.0, nh=3, jobs_x=1, jobs_y=1)
    dt = np.float32(0.002)
    plan = EomPlan(cfg, ns, dt)
    g = torch.Generator(device=cuda).manual_seed(ns)
    csp = torch.randn(plan.shape, generator=g, device=cuda)
    fold = torch.randint(1, 30, plan.shape, generator=g, device=cuda).float()
    out = plan.post(csp, fold).cpu().numpy()
    lp, rr = oracle.eom_filters(cfg, ns, dt)
    ref = oracle.eom_post(csp.cpu().numpy()[:2], fold.cpu().numpy()[:2], dt, lp, rr)
    e = rel_l2(out[:2], ref)
    print(f"  relL2 {e:.2e}", flush=True)
    assert e <= 1e-6


@pytest.mark.parametrize("nh", [32, 200, 201, 400])
@pytest.mark.parametrize("ns", [40, 64, 65, 192, 193, 256, 257, 300, 511, 513, 751])
def test_eom_workgroups_of_one_and_of_four_waves(cuda, ns, nh):
    """Sample and bin counts on both sides of every change between workgroups of
    64 samples and of 256, with more traces than either gates at once."""
    print(f"case: EOM line, {ns} samples, {nh} bins", flush=True)
    sv = surveys.line2d(nshots=14, nrecv_side=20, ns=ns, ncols=80, col_dx=12.5, nscat=4, x0=400.0,
                        t0_range=(0.01, 0.1))
    _, cfg, _ = line_case()
    cfg.velocity_start = cfg.velocity_end = 6000.0
    cfg.nh, cfg.dh = nh, 800.0 / nh
    tr = np.random.default_rng(ns).standard_normal((sv.ntr, ns)).astype(np.float32)
    plan = EomPlan(cfg, ns, sv.dt)
    csp, fold, n = plan.migrate(torch.from_numpy(tr).to(cuda), torch.from_numpy(sv.coords).to(cuda),
                                block=600)
    c0, f0, n0 = oracle.eom_all(cfg, ns, np.float32(sv.dt), tr, sv.coords, cfg.velocity(ns))
    c = csp.cpu().numpy()
    print(f"  evaluated {n} (oracle {n0}); gathers relL2 {rel_l2(c, c0):.2e}", flush=True)
    assert n == n0
    assert np.array_equal(fold.cpu().numpy(), f0)
    assert rel_l2(c, c0) <= 1e-6
    assert ns < 64 or np.abs(c0).max() > 0


@pytest.mark.parametrize("ns,base", [(192, 1400), (256, 1050)])
def test_eom_gathers_beyond_32_bit_offsets(cuda, ns, base):
    """A CSP of more than 2^30 samples, its bins of 2^-12 m beyond 4 GiB: the
    same sums as in a plan whose first bin lies there (shifting by a whole number
    of bins is exact for a width of a power of two)."""
    width = 2.0 ** -12
    shift = int(base / width)
    bins = (1 << 30) // ns + 400_000
    assert 4 * shift * ns > 2 ** 32 and bins > shift
    print(f"case: {bins} bins x {ns} samples, 200 traces", flush=True)
    rng = np.random.default_rng(ns)
    coords = np.zeros((200, 4), np.int32)
    cmp = rng.uniform(base - 60.0, base + 60.0, 200)
    coords[:, 0] = np.round(100.0 * (cmp - 150.0))
    coords[:, 2] = np.round(100.0 * (cmp + 150.0))
    tr = torch.from_numpy(rng.standard_normal((200, ns)).astype(np.float32)).to(cuda)
    co = torch.from_numpy(coords).to(cuda)
    out = []
    for oh, nh in ((0, bins), (base, bins - shift)):
        cfg = EomConfig(ox=0.0, oy=0.0, angle_e_to_n=0.0, oxcsp=0.0, oycsp=0.0, excsp=0.0, eycsp=0.0,
                        scale_xy=0.01, dcsp_x=12.5, dcsp_y=0.0, dh=width, nh=nh, oh=oh, aperture=2500.0,
                        jobs_x=1, jobs_y=1, ntblock=1000, velocity_start=9000.0, velocity_end=9000.0)
        plan = EomPlan(cfg, ns, 0.004)
        csp, fold, n = plan.migrate(tr, co)
        out.append((csp.reshape(nh, ns)[nh - (bins - shift):], fold.reshape(nh, ns)[nh - (bins - shift):], n))
    (c0, f0, n0), (c1, f1, n1) = out
    assert n0 == n1 > 0
    assert bool((f1[1:-1] != 1.0).any()) and bool(c1[1:-1].any())
    assert torch.equal(c0[1:-1], c1[1:-1]) and torch.equal(f0[1:-1], f1[1:-1])
