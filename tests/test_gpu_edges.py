"""Edge cases of the migration path on the GPU against the CPU oracle: every
kernel variant (the sample-count boundaries where the per-column lane layout
changes, from the smallest plan, ns = 4, to the largest, ns = 6144), empty
blocks, blocks with no trace in aperture, offset classes with traces outside
[0, nh), a one-column image, the plan's size limits, and the adjoint of every
variant, and the post-stack filter and its transpose for long traces (the
traces-per-workgroup and kernel-in-LDS choices of ktm_poststack)."""
import numpy as np
import pytest
import torch

import oracle
from random_amd import KtmError, _lib, surveys
from random_amd.ktm import Plan
from random_amd.lsm import Operator, dot_test

pytestmark = pytest.mark.gpu

# sample counts on both sides of capacities of the lane layouts of
# ktm_migrate_block (64 K W samples of K per lane and W waves per column), for
# the 40-column line here and a 4104-column one; LANES below names a size for
# every layout
NS_CASES = [4, 63, 512, 513, 1024, 1025, 1536, 1537, 2048, 2049, 3072, 3073, 4096, 4097, 6144]


def small_line(ns, **kw):
    dt = 0.004
    t1 = max(0.02, 0.8 * ns * dt)
    # shots from x = 100 m, so the 40 columns of 6.25 m from 0 straddle the
    # CMPs and even a 4-sample trace reaches the image
    args = dict(nshots=3, nrecv_side=10, ns=ns, ncols=40, nscat=3, jobs_x=2, x0=100.0,
                t0_range=(min(0.01, t1 / 2), t1))
    args.update(kw)
    return surveys.line2d(**args)


def bitexact_case(sv, tr, cuda, block=None):
    km_o, fold_o, n_o = oracle.migrate(sv.cfg, sv.ns, sv.dt, tr, sv.coords, sv.vel)
    plan = Plan(sv.cfg, sv.ns, sv.dt, sv.vel)
    km, fold, n = plan.migrate(torch.from_numpy(tr).to(cuda), torch.from_numpy(sv.coords).to(cuda),
                               block=block)
    km, fold = km.cpu().numpy(), fold.cpu().numpy()
    same = float(np.mean(km.view(np.uint32) == km_o.view(np.uint32)))
    print(f"  contributions {n} (oracle {n_o}); bit-identical fraction {same:.8f}", flush=True)
    assert n == n_o
    assert np.array_equal(fold, fold_o)
    assert same == 1.0
    return plan, km, fold, n


@pytest.mark.parametrize("ns", NS_CASES)
def test_every_kernel_variant_bitexact(cuda, ns):
    print(f"case: variant at ns={ns}, 60 traces, 40 columns, 2 jobs", flush=True)
    sv = small_line(ns)
    tr = surveys.traces_numpy(sv)
    assert np.abs(tr).max() > 0
    _, km, _, n = bitexact_case(sv, tr, cuda, block=25)
    assert n > 0 and np.abs(km).max() > 0


@pytest.mark.parametrize("ns", [63, 512, 513, 1024])
def test_wide_image_layouts_bitexact(cuda, ns):
    """A 4104-column line (more than two workgroups per CU at 8 samples per
    lane) keeps the default layouts below 1025 samples."""
    print(f"case: wide-image variant at ns={ns}, 60 traces, 4104 columns, 2 jobs", flush=True)
    sv = small_line(ns, ncols=4104)
    tr = surveys.traces_numpy(sv)
    _, km, _, n = bitexact_case(sv, tr, cuda, block=25)
    assert n > 0 and np.abs(km).max() > 0


@pytest.mark.parametrize("ns", [4, 513, 1537, 2049, 3072, 4097, 6144])
def test_adjoint_of_every_variant(cuda, ns):
    print(f"case: dot test at ns={ns}", flush=True)
    sv = small_line(ns)
    plan = Plan(sv.cfg, sv.ns, sv.dt, sv.vel)
    op = Operator(plan, torch.from_numpy(sv.coords).to(cuda))
    g = torch.Generator(device=cuda).manual_seed(ns)
    d = torch.randn((sv.ntr, sv.ns), generator=g, device=cuda)
    m = torch.randn(plan.image_shape, generator=g, device=cuda)
    lhs, rhs, rel = dot_test(op, d, m)
    print(f"  rel {rel:.2e}", flush=True)
    assert rel <= 1e-5


def test_empty_and_out_of_aperture_blocks(cuda):
    print("case: empty block, block with no trace in aperture", flush=True)
    sv = small_line(301)
    tr = surveys.traces_numpy(sv)
    plan = Plan(sv.cfg, sv.ns, sv.dt, sv.vel)
    km, fold, _ = plan.new_image(device=cuda)
    counter = torch.zeros(1, dtype=torch.int64, device=cuda)
    d_tr = torch.from_numpy(tr).to(cuda)
    # an empty block is a no-op
    prepared, geom = plan.prep(d_tr[:0], torch.zeros((0, 4), dtype=torch.int32, device=cuda))
    plan.migrate_block(prepared, geom, km, fold, counter=counter)
    # traces 1000 km down the line: no column within the 2000 m aperture
    far = sv.coords.copy()
    far[:, 0] += 100_000_000
    far[:, 2] += 100_000_000
    prepared, geom = plan.prep(d_tr, torch.from_numpy(far).to(cuda))
    plan.migrate_block(prepared, geom, km, fold, counter=counter)
    torch.cuda.synchronize()
    assert int(counter.item()) == 0
    assert not km.any() and bool((fold == 1.0).all())
    km_o, fold_o, n_o = oracle.migrate(sv.cfg, sv.ns, sv.dt, tr, far, sv.vel)
    assert n_o == 0 and not km_o.any()


def test_offset_classes_with_traces_outside(cuda):
    """nh = 3 classes of 100 m on a split spread up to 375 m: classes 0-2 are
    filled, the traces of class 3 are skipped (Kirchhoff.c:1387)."""
    print("case: offset classes, nh=3, traces beyond the last class", flush=True)
    sv = small_line(401, nshots=4, nrecv_side=30, nh=3, oh=0.0, dh=100.0)
    tr = surveys.traces_numpy(sv)
    _, geo_off = oracle.trace_geometry(sv.cfg, sv.coords)
    assert set(np.unique(geo_off)) >= {0, 1, 2, 3}
    plan, km, fold, _ = bitexact_case(sv, tr, cuda, block=100)
    assert plan.image_shape[2] == 3
    for h in range(3):
        assert np.abs(km[:, :, h]).max() > 0


def test_one_column_image(cuda):
    print("case: one image column, two traces", flush=True)
    sv = small_line(257, nshots=1, nrecv_side=1, ncols=1, jobs_x=1)
    tr = surveys.traces_numpy(sv)
    assert tr.shape[0] == 2
    plan, km, _, n = bitexact_case(sv, tr, cuda)
    assert plan.image_shape[:2] == (1, 1)


def test_plan_size_limits(cuda):
    sv = small_line(64)
    for ns in (3, 6145):
        with pytest.raises(KtmError) as e:
            Plan(sv.cfg, ns, sv.dt, np.ones((sv.cfg.nvel_ilines, 1, ns), np.float32) * 2000.0)
        assert e.value.status == _lib.KTM_ERR_UNSUPPORTED


@pytest.mark.parametrize("ns", [37, 128, 200, 300, 512, 700, 1500, 2000])
def test_poststack_many_traces(cuda, ns):
    """Several transforms per wave (N = 256 to 1024), several waves per transform
    and several workgroups, the last one partly filled: 61 traces of one image
    against an FFT in double of the same single-precision differences.  The
    result is rounded to float once, so its distance is at most 2^-24 of its
    norm, plus the double transforms' own error (below 1e-13)."""
    print(f"case: post-stack of 61 traces at ns={ns}", flush=True)
    sv = small_line(ns, ncols=61, jobs_x=1)
    plan = Plan(sv.cfg, sv.ns, sv.dt, sv.vel)
    g = torch.Generator(device=cuda).manual_seed(ns)
    km = torch.randn(plan.image_shape, generator=g, device=cuda)
    fold = torch.randint(1, 40, plan.image_shape, generator=g, device=cuda).float()
    out = plan.poststack(km, fold).cpu().numpy().reshape(-1, ns)
    _, aa = oracle.alias_filter(sv.cfg, sv.ns, sv.dt)
    k, f = km.cpu().numpy().reshape(-1, ns), fold.cpu().numpy().reshape(-1, ns)
    dt = np.float32(sv.dt)
    d = np.zeros((k.shape[0], ns))
    d[:, 1:] = -dt * np.arange(1, ns, dtype=np.float32) * (k[:, 1:] - k[:, :-1]) * dt / f[:, 1:]
    ref = np.fft.ifft(np.fft.fft(d, axis=-1) * aa.astype(np.float64), axis=-1).real
    ref[:, 0] = 0.0
    assert k.shape[0] == 61
    r = float(np.linalg.norm(out - ref) / np.linalg.norm(ref))
    print(f"  relL2 {r:.2e}", flush=True)
    assert r <= 2.0 ** -24 + 1e-13


@pytest.mark.parametrize("ns", [4, 128, 129, 512, 1024, 1025, 1536, 1537, 2048, 2049, 4096, 4097,
                                6144])
def test_poststack_long_traces(cuda, ns):
    """Forward against the oracle's DFT path and the dot test of the
    transpose on both sides of every transform length of the FFT form
    (N = 256 up to 128 samples, 512 from 129, 1024, 2048, 3072 from 1025 to
    1536 (radix 16 x 16 x 12), 4096 from 1537 to 2048, 8192 from 2049 to
    4096) and of the switch to the FP64 matrix product beyond 4096 samples;
    8 image traces at even ns, 7 at odd ns (the last transform then carries
    one trace)."""
    print(f"case: post-stack and transpose at ns={ns}", flush=True)
    sv = small_line(ns, ncols=7 if ns % 2 else 8, jobs_x=1)
    plan = Plan(sv.cfg, sv.ns, sv.dt, sv.vel)
    g = torch.Generator(device=cuda).manual_seed(ns + 1)
    km = torch.randn(plan.image_shape, generator=g, device=cuda)
    img = torch.randn(plan.image_shape, generator=g, device=cuda)
    fold = torch.randint(1, 40, plan.image_shape, generator=g, device=cuda).float()
    out = plan.poststack(km, fold).cpu().numpy()
    tm, aa = oracle.alias_filter(sv.cfg, sv.ns, sv.dt)
    ref = oracle.poststack(km.cpu().numpy(), fold.cpu().numpy(), sv.dt, aa)
    r = float(np.linalg.norm(out - ref) / np.linalg.norm(ref))
    skm = plan.poststack(km, fold).double().ravel()
    lhs = float(torch.dot(skm, img.double().ravel()))
    rhs = float(torch.dot(km.double().ravel(), plan.poststack_adjoint(img, fold).double().ravel()))
    rel = abs(lhs - rhs) / abs(lhs)
    # the outputs are rounded to float, so the difference is ~1e-7 of the
    # Cauchy-Schwarz scale over sqrt(n); relative to <S km, img> unless that
    # product is below 1 % of the scale by chance
    scale = float(torch.linalg.vector_norm(skm) * torch.linalg.vector_norm(img.double()))
    print(f"  forward relL2 vs oracle {r:.2e}; transpose dot rel {rel:.2e}, "
          f"|<S km, i>| / scale {abs(lhs) / scale:.2e}", flush=True)
    assert r <= 1e-6
    assert abs(lhs - rhs) <= 1e-6 * max(abs(lhs), 1e-2 * scale)


@pytest.mark.parametrize("ns", [4097, 6144])
def test_compensated_and_16bit_long_traces(cuda, ns):
    """The Kahan and BF16 variants of the long-trace layouts against the FP64
    oracle (same traveltime index, FP64 data path)."""
    from random_amd import ACCUM_KAHAN, PREP_CLOSED, TRACE_BF16, TRACE_F32
    print(f"case: Kahan FP32 and BF16 at ns={ns}", flush=True)
    sv = small_line(ns)
    tr = surveys.traces_numpy(sv)
    km64, fold64, n64 = oracle.migrate(sv.cfg, sv.ns, sv.dt, tr, sv.coords, sv.vel,
                                       mode=oracle.FP64_DATA)
    plan = Plan(sv.cfg, sv.ns, sv.dt, sv.vel)
    d_tr, d_co = torch.from_numpy(tr).to(cuda), torch.from_numpy(sv.coords).to(cuda)
    for dtype, tol in ((TRACE_F32, 1e-6), (TRACE_BF16, 3e-3)):
        km, fold, n = plan.migrate(d_tr, d_co, mode=PREP_CLOSED, dtype=dtype, accum=ACCUM_KAHAN,
                                   block=25)
        r = float(np.linalg.norm(km.cpu().numpy() - km64) / np.linalg.norm(km64))
        print(f"  dtype {dtype}: relL2 vs FP64 {r:.2e}", flush=True)
        assert n == n64 and np.array_equal(fold.cpu().numpy(), fold64.astype(np.float32))
        assert r <= tol


@pytest.mark.parametrize("ns", [301, 1003, 1500, 2047, 2600, 3500, 5000])
@pytest.mark.parametrize("ntr", [1, 3, 5, 64, 67, 69, 133, 515, 1089])
def test_trace_list_and_ring_boundaries_bitexact(cuda, ns, ntr):
    """Trace counts around the steps of the trace stream of every lane layout
    (rows staged 2 or 4 at a time, gates 64 at a time, blocks of 512 or 1024
    traces filtered into the list), with every third trace outside the
    offset classes and zero-offset traces on a column (q < 1 at t = 0)."""
    print(f"case: {ntr} traces x {ns} samples", flush=True)
    sv = small_line(ns, nshots=55, nrecv_side=10, ncols=9, jobs_x=1, nh=1, dh=110.0)
    co = sv.coords[np.random.default_rng(ntr).permutation(sv.ntr)[:ntr]].copy()
    co[::4, 2] = co[::4, 0] = 625 * (1 + np.arange(co[::4].shape[0]) % 7)
    sv.coords = co
    tr = np.random.default_rng(ns).standard_normal((ntr, ns)).astype(np.float32)
    bitexact_case(sv, tr, cuda)


def test_prepared_rows_at_any_float(cuda):
    """Prepared rows that start 4 bytes past a 16-byte boundary migrate to the
    same bits as aligned ones."""
    print("case: prepared rows 4 bytes past a 16-byte boundary", flush=True)
    sv = small_line(700)
    plan = Plan(sv.cfg, sv.ns, sv.dt, sv.vel)
    tr = torch.from_numpy(surveys.traces_numpy(sv)).to(cuda)
    prepared, geom = plan.prep(tr, torch.from_numpy(sv.coords).to(cuda))
    km, fold, _ = plan.new_image(device=cuda)
    plan.migrate_block(prepared, geom, km, fold)
    odd = torch.empty(prepared.numel() + 1, device=cuda)[1:].view_as(prepared)
    odd.copy_(prepared)
    assert odd.data_ptr() % 16 == 4
    km2, fold2, _ = plan.new_image(device=cuda)
    plan.migrate_block(odd, geom, km2, fold2)
    assert bool(km.any()) and torch.equal(km, km2) and torch.equal(fold, fold2)


# both sides of the remaining capacities of the lane layouts by samples per lane
# and waves per column (2, 4, 6, 8, 10 or 12 x 64 x 1, 2, 4 or 8); the
# 4104-column image takes wide lanes, the 40-column one narrow ones
LAYOUT_NS = [256, 257, 384, 385, 640, 641, 768, 769, 1280, 1281, 2560, 2561, 5120, 5121]


@pytest.mark.parametrize("ncols", [40, 4104])
@pytest.mark.parametrize("ns", LAYOUT_NS)
def test_lane_layout_boundaries_bitexact(cuda, ns, ncols):
    print(f"case: ns={ns}, 60 traces, {ncols} columns", flush=True)
    sv = small_line(ns, ncols=ncols)
    tr = surveys.traces_numpy(sv)
    _, km, _, n = bitexact_case(sv, tr, cuda, block=43)
    assert n > 0 and np.abs(km).max() > 0


@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("ns", LAYOUT_NS)
def test_adjoint_at_lane_layout_boundaries(cuda, ns, fast):
    print(f"case: dot test at ns={ns}, fast={fast}", flush=True)
    sv = small_line(ns)
    plan = Plan(sv.cfg, sv.ns, sv.dt, sv.vel)
    op = Operator(plan, torch.from_numpy(sv.coords).to(cuda), fast=fast)
    g = torch.Generator(device=cuda).manual_seed(ns)
    d = torch.randn((sv.ntr, sv.ns), generator=g, device=cuda)
    m = torch.randn(plan.image_shape, generator=g, device=cuda)
    lhs, rhs, rel = dot_test(op, d, m)
    print(f"  rel {rel:.2e}", flush=True)
    assert rel <= 1e-5


@pytest.mark.parametrize("ns", [200, 380, 500, 630, 700, 1000, 2000])
@pytest.mark.parametrize("ntr", [7, 8, 9, 63, 71, 72, 73])
def test_chunks_of_eight_rows_bitexact(cuda, ns, ntr):
    """Trace counts around chunks of eight staged rows and the 64 traces whose
    gates are evaluated at once, the last chunk short, for small images and for
    offset classes that fill the widest lanes."""
    for nh, ncols in ((1, 9), (600, 9)):
        print(f"case: {ntr} traces x {ns} samples, {ncols} columns x {nh} classes", flush=True)
        sv = small_line(ns, nshots=8, nrecv_side=10, ncols=ncols, jobs_x=1, nh=nh, dh=900.0 if nh == 1 else 100.0)
        sv.coords = sv.coords[np.random.default_rng(ntr).permutation(sv.ntr)[:ntr]].copy()
        tr = np.random.default_rng(ns).standard_normal((ntr, ns)).astype(np.float32)
        bitexact_case(sv, tr, cuda)


@pytest.mark.parametrize("kahan", [False, True])
@pytest.mark.parametrize("ns", [63, 301, 700, 1100, 1500, 2000, 2600, 5000])
def test_traces_without_a_position_add_nothing(cuda, ns, kahan):
    """A trace whose source or receiver position is NaN or infinite (in a
    geometry that the caller made, with a CMP in reach) has no traveltime: the
    reference arithmetic gives NaN or infinity, never an index below ns.  Image
    and fold are those of the other traces."""
    print(f"case: traces without a position, ns={ns}, kahan={kahan}", flush=True)
    sv = small_line(ns, jobs_x=1)
    plan = Plan(sv.cfg, sv.ns, sv.dt, sv.vel)
    tr = torch.from_numpy(surveys.traces_numpy(sv)).to(cuda)
    kw = dict(mode=_lib.PREP_CLOSED, accum=_lib.ACCUM_KAHAN) if kahan else {}
    prepared, geom = plan.prep(tr, torch.from_numpy(sv.coords).to(cuda), kw.get("mode", 0))
    without = torch.arange(sv.ntr, device=cuda) % 4 == 1
    bad = geom.clone()
    for i in torch.nonzero(without).flatten().tolist():
        bad[i, i // 4 % 4] = float("nan") if i % 8 == 1 else float("inf")
    out = []
    for p, g in ((prepared, bad), (prepared[~without].contiguous(), geom[~without].contiguous())):
        km, fold, comp = plan.new_image(kahan=kahan, device=cuda)
        plan.migrate_block(p, g, km, fold, comp, **kw)
        out.append((km, fold))
    assert bool(out[1][0].any())
    assert torch.equal(out[0][1], out[1][1])
    if kahan:      # other sets of traces between the compensated steps
        assert float((out[0][0] - out[1][0]).norm() / out[1][0].norm()) <= 1e-6
    else:
        assert torch.equal(out[0][0], out[1][0])


# (samples, columns) of every lane layout of ktm_migrate_block, as
# test_host_launches.py finds them taken
LANES = [(200, 300), (384, 4200), (512, 40), (512, 1600), (512, 4200), (640, 4200), (768, 1600),
         (768, 4200), (1024, 40), (1024, 700), (1024, 4200), (1280, 4200), (1536, 40), (1536, 4200),
         (2048, 1000), (2048, 40), (2560, 1000), (3072, 1000), (4096, 1000), (4096, 40), (5120, 1000),
         (6144, 1000), (6144, 40)]


@pytest.mark.parametrize("ns,ncols", LANES)
def test_trace_counts_in_every_lane_layout_bitexact(cuda, ns, ncols):
    """Trace counts around the chunks of rows (2, 4 or 8), the windows (4, 8 or
    16 traces), the 64 traces whose gates are evaluated at once and the blocks
    filtered into the list (512 or 1024), the last ones for few columns, at the
    last sample count of the layout."""
    sv = small_line(ns, nshots=55, nrecv_side=10, ncols=ncols, jobs_x=1, nh=1, dh=110.0, aperture=400.0)
    coords = sv.coords[np.random.default_rng(ns).permutation(sv.ntr)]
    coords[::4, 2] = coords[::4, 0] = 625 * (1 + np.arange(coords[::4].shape[0]) % 7)
    tr = np.random.default_rng(ncols).standard_normal((sv.ntr, ns)).astype(np.float32)
    for ntr in [1, 3, 9, 17, 66, 73, 131] + ([515, 1089] if ncols == 40 else []):
        print(f"case: {ntr} traces x {ns} samples, {ncols} columns", flush=True)
        sv.coords = np.ascontiguousarray(coords[:ntr])
        bitexact_case(sv, tr[:ntr].copy(), cuda)


def test_velocities_whose_inverse_square_overflows(cuda):
    """Zero-offset traces on a column of a velocity of 1e-20 m/s (1/(v dt)^2
    overflows in FP32, the reference's 0 / v^2 does not): the reference's index,
    T = t, in every sample."""
    print("case: zero-offset traces, velocities down to 1e-20 m/s", flush=True)
    sv = small_line(301, ncols=1, jobs_x=1)
    sv.coords[:, 0::2] = 0
    sv.vel[..., 1::3] = 1.0e-20
    tr = np.random.default_rng(1).standard_normal((sv.ntr, sv.ns)).astype(np.float32)
    _, km, _, n = bitexact_case(sv, tr, cuda)
    assert n > 0 and (km[..., 1::3] != 0).any()
