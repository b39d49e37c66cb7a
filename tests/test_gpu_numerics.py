"""The numerical assumptions behind the fast traveltime path of k_migrate.

The kernel computes q = dsr/dt with FMA and the hardware square root on
radicands pre-scaled by 1/dt^2, and falls back to the reference arithmetic of
Kirchhoff.c:1381-1384 whenever an integer lies within 4.8e-7 (q + 1) of q.
That is exact only if |q_fast - q_ref| <= 4.8e-7 (q_ref + 1), which rests on
v_sqrt_f32 being within one ulp.  Both facts are checked here.
"""
import ctypes as C
import math

import numpy as np
import pytest
import torch

from random_amd import _lib

pytestmark = pytest.mark.gpu

EPS = 4.8e-7   # the kernel's tolerance of its fast form (8 x 2^-24; bound 7 x 2^-24)


def _p(t):
    return C.c_void_p(t.data_ptr())


def ulp_diff(a, b):
    ia = a.view(np.int32).astype(np.int64)
    ib = b.view(np.int32).astype(np.int64)
    return np.abs(ia - ib)


def test_hw_sqrt_within_one_ulp_exhaustive(cuda):
    # every float in [1, 4): sqrt(4^k x) = 2^k sqrt(x), so this covers every
    # mantissa of both exponent parities
    print("case: v_sqrt_f32 on all 2^24 floats of [1, 4)", flush=True)
    x = np.arange(1 << 24, dtype=np.int64) + np.float32(1.0).view(np.int32)
    x = x.astype(np.int32).view(np.float32)
    assert x[0] == 1.0 and x[-1] < 4.0 and x[-1] > 3.99
    d_x = torch.from_numpy(x).to(cuda)
    out = torch.empty_like(d_x)
    _lib.check(_lib.lib().ktm_selftest_sqrt(_p(d_x), x.size, _p(out), None), "selftest_sqrt")
    hw = out.cpu().numpy()
    ref = np.sqrt(x)  # correctly rounded
    u = ulp_diff(hw, ref)
    print(f"  max ulp error {u.max()}, fraction not correctly rounded {np.mean(u > 0):.3e}")
    assert u.max() <= 1


def _run_traveltime(cuda, inp, dt, ns):
    d_in = torch.from_numpy(np.ascontiguousarray(inp, np.float32)).to(cuda)
    n = inp.shape[0]
    qf = torch.empty(n, dtype=torch.float32, device=cuda)
    qr = torch.empty_like(qf)
    tk = torch.empty(n, dtype=torch.int32, device=cuda)
    tr = torch.empty_like(tk)
    _lib.check(_lib.lib().ktm_selftest_traveltime(_p(d_in), n, dt, ns, _p(qf), _p(qr), _p(tk),
                                                  _p(tr), None), "selftest_traveltime")
    return qf.cpu().numpy(), qr.cpu().numpy(), tk.cpu().numpy(), tr.cpu().numpy()


def test_fast_traveltime_bound_and_index(cuda):
    print("case: fast vs reference traveltime, 2^24 random samples", flush=True)
    rng = np.random.default_rng(7)
    n = 1 << 24
    dt = np.float32(0.004)
    ns = 1500
    t = rng.integers(0, ns, n)
    d = rng.uniform(0.0, 8000.0, (n, 2)) ** 2
    v = rng.uniform(1400.0, 5000.0, n).astype(np.float32)
    inp = np.stack([d[:, 0], d[:, 1], t, v * v], axis=1).astype(np.float32)
    qf, qr, tk, tr = _run_traveltime(cuda, inp, dt, ns)
    err = np.abs(qf.astype(np.float64) - qr) / (qr.astype(np.float64) + 1.0)
    near = np.abs(qr - np.rint(qr)) <= EPS * (qr + 1.0)
    print(f"  max |q_fast - q_ref| / (q_ref + 1) = {err.max():.3e} (bound {EPS}); "
          f"{near.sum()} samples within the bound of an integer; T mismatches {np.sum(tk != tr)}")
    assert err.max() <= EPS
    assert np.array_equal(tk, tr)
    # the T the kernel keeps is floor of the reference quotient
    ref_T = np.where(qr < ns, np.floor(qr), ns).astype(np.int32)
    assert np.array_equal(tr, ref_T)


def test_fast_traveltime_near_integers(cuda):
    """Samples constructed to land within ~1e-5 samples of an integer (the
    cases the fallback exists for): the kernel's index equals the
    reference's on all of them."""
    print("case: fast vs reference traveltime, 2^22 near-integer samples", flush=True)
    rng = np.random.default_rng(11)
    n = 1 << 22
    dt = np.float32(0.004)
    ns = 1500
    t = rng.integers(0, ns, n)
    t2 = 0.25 * t * t * np.float64(dt) ** 2
    v = rng.uniform(1400.0, 5000.0, n).astype(np.float32)
    v2 = (v * v).astype(np.float64)
    d1 = rng.uniform(0.0, 4000.0, n) ** 2
    s1 = np.sqrt(t2 + d1 / v2)
    target = np.floor(2.0 * s1 / np.float64(dt)) + rng.integers(1, 400, n) + rng.uniform(-1e-5, 1e-5, n)
    rest = target * np.float64(dt) - s1
    d2 = (rest * rest - t2) * v2
    ok = (rest > 0) & (d2 >= 0)
    inp = np.stack([d1[ok], d2[ok], t[ok], v2[ok]], axis=1).astype(np.float32)
    qf, qr, tk, tr = _run_traveltime(cuda, inp, dt, ns)
    dist = np.abs(qr - np.rint(qr))
    err = np.abs(qf.astype(np.float64) - qr) / (qr.astype(np.float64) + 1.0)
    print(f"  {ok.sum()} samples, {np.sum(dist < 1e-4)} within 1e-4 of an integer, "
          f"max rel err {err.max():.3e}, T mismatches {np.sum(tk != tr)}")
    assert np.sum(dist < 1e-4) > ok.sum() // 4
    assert err.max() <= EPS
    assert np.array_equal(tk, tr)


@pytest.mark.parametrize("ns", [4, 63, 501, 1500, 3001, 6144])
def test_limited_traveltime_bound_and_index(cuda, ns):
    """The migration's own form, in units of ns + 1/2 and limited to 1, within
    the same bound; a limited sample is past the trace."""
    print(f"case: limited fast form vs reference traveltime, 2^22 samples, ns={ns}", flush=True)
    rng = np.random.default_rng(ns)
    n = 1 << 22
    dt = np.float32(0.004)
    t = rng.integers(0, ns, n)
    reach = 3000.0 * dt * ns
    d = (reach * rng.uniform(0.0, 1.0, (n, 2)) ** 2) ** 2
    d[: n // 16] = 0.0
    v = rng.uniform(1400.0, 5000.0, n).astype(np.float32)
    inp = np.ascontiguousarray(np.stack([d[:, 0], d[:, 1], t, v * v], axis=1), np.float32)
    _, qr, tk, tr = _run_traveltime(cuda, inp, dt, ns)
    q = torch.empty(n, dtype=torch.float64, device=cuda)
    _lib.check(_lib.lib().ktm_selftest_limited(_p(torch.from_numpy(inp).to(cuda)), n, dt, ns, _p(q),
                                               None), "selftest_limited")
    q = q.cpu().numpy()
    at_limit = q == ns + 0.5
    err = np.abs(q - qr)[~at_limit] / (qr.astype(np.float64) + 1.0)[~at_limit]
    print(f"  max |q - q_ref| / (q_ref + 1) = {err.max():.3e} (bound {EPS}); {at_limit.sum()} at the "
          f"limit; T mismatches {np.sum(tk != tr)}", flush=True)
    assert 0 < at_limit.sum() < n // 2
    assert err.max() <= EPS
    assert (qr[at_limit] > ns).all()
    assert np.array_equal(tk, tr)


def test_eom_taper_and_square_root_round_as_the_reference(cuda):
    """EOM.c:1286-1292: the taper's series and its switch to the full double
    expression (at |d| = 3.2 ms, and where the sum and its error bound round
    apart), and the float square root down to the subnormals.  The device's double
    arctangent and the C library's may be two ulps apart, 1.1e-16 of the sum,
    whose float has an ulp of 8e-8 times its value 1.27e-4 / |d| for d < -1: were
    all of them that far apart, 10 of these 10^6 floats would differ; 30 may, by
    one ulp."""
    rng = np.random.default_rng(3)
    edge = np.float32(0.0032).view(np.int32) + np.arange(-4000, 4001, dtype=np.int32)
    d = np.concatenate([edge.astype(np.int32).view(np.float32), [0.0, 1e-30, 0.00319, 0.0033],
                        10.0 ** rng.uniform(-9.0, 1.4, 490_000)]).astype(np.float32)
    d = np.concatenate([d, -d])
    x = np.concatenate([[0.0, 2.0 ** -149, 2.0 ** -126, 2.0 ** -97, 2.0 ** -96, 2.0 ** -95, 1.0, 2.0, 3e38],
                        2.0 ** rng.uniform(-149.0, 127.0, d.size - 200_009),
                        rng.integers(1, 1 << 20, 100_000).astype(np.float64) ** 2,
                        rng.uniform(0.0, 1e8, 100_000)]).astype(np.float32)
    assert d.size == x.size
    print(f"case: taper and square root of {d.size} floats", flush=True)
    d_d, d_x = torch.from_numpy(d).to(cuda), torch.from_numpy(x).to(cuda)
    taper, root = torch.empty_like(d_d), torch.empty_like(d_x)
    _lib.check(_lib.lib().ktm_selftest_eom(_p(d_d), _p(d_x), d.size, _p(taper), _p(root), None),
               "selftest_eom")
    z = (200.0 * d.astype(np.float64) / 0.080).tolist()
    want = np.array([0.5 + math.atan(v) / 3.14159265359 for v in z]).astype(np.float32)
    u = ulp_diff(taper.cpu().numpy(), want)
    print(f"  taper: {np.sum(u > 0)} differ, by {u.max()} ulp", flush=True)
    assert u.max() <= 1 and np.sum(u > 0) <= 30
    assert np.array_equal(root.cpu().numpy().view(np.int32), np.sqrt(x).view(np.int32))
