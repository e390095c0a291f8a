"""GPU parity of the volume-rendering targets against the CPU oracle.

Integer outputs (sample counts, offsets, validity, ray indices, cells, bitfields,
Morton codes, early-stop counts, termination flags) must match bit for bit.  The
f32 outputs follow the oracle's rounding convention and are compared bit for bit
as well; the oracle's own f32-vs-float64 error bounds live in test_oracle_pins.py.
"""
import numpy as np
import pytest
import torch

import oracle
from jaxngp_amd import volrend
from tests.helpers import blob_bitfield, integrate_inputs, march_inputs, near_far_np

pytestmark = pytest.mark.gpu


def T(a, dev, dtype=None):
    t = torch.from_numpy(np.ascontiguousarray(a))
    if dtype is not None:
        t = t.to(dtype)
    return t.to(dev)


def U(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a, np.uint32)).to(dev)


def N(t):
    return t.cpu().numpy()


def test_morton_round_trip_all_cells(dev):
    G = 128
    idx = np.arange(G ** 3, dtype=np.uint32)
    xyz = volrend.morton3d_invert(U(idx, dev))
    np.testing.assert_array_equal(N(xyz), oracle.morton3d_invert(idx))
    back = volrend.morton3d(xyz)
    np.testing.assert_array_equal(N(back), idx)
    rnd = np.random.default_rng(0).integers(0, 2 ** 32, 100000, dtype=np.uint64).astype(np.uint32)
    np.testing.assert_array_equal(N(volrend.morton3d_invert(U(rnd, dev))), oracle.morton3d_invert(rnd))
    xyz_r = np.random.default_rng(1).integers(0, 2 ** 32, (50000, 3), dtype=np.uint64).astype(np.uint32)
    np.testing.assert_array_equal(N(volrend.morton3d(U(xyz_r, dev))), oracle.morton3d(xyz_r))


@pytest.mark.parametrize("n_bits", [8, 64 * 8, 128 ** 3, 2 * 128 ** 3 + 8])
def test_packbits(dev, rng, n_bits):
    dens = rng.normal(size=n_bits).astype(np.float32)
    thr = rng.normal(size=n_bits).astype(np.float32)
    mask, bits = volrend.packbits(T(thr, dev), T(dens, dev))
    m_o, b_o = oracle.packbits(thr, dens)
    np.testing.assert_array_equal(N(mask), m_o)
    np.testing.assert_array_equal(N(bits), b_o)
    mask, bits = volrend.packbits(0.1, T(dens, dev))
    np.testing.assert_array_equal(N(bits), oracle.packbits(np.float32(0.1), dens)[1])


def _march_both(dev, S, diag, K, G, bound, portion, o, d, t0, t1, noise, bits):
    got = volrend.march_rays(S, diag, K, G, bound, portion, T(o, dev), T(d, dev), T(t0, dev), T(t1, dev),
                             T(noise, dev), T(bits, dev))
    want = oracle.march_rays(S, diag, K, G, bound, portion, o, d, t0, t1, noise, bits)
    return got, want


def _assert_march_equal(got, want):
    measured, valid, ns, start, idcs, xyzs, dirs, dss, z = got
    assert int(N(measured.view(torch.int32))) == int(want["measured"])
    np.testing.assert_array_equal(N(valid), want["ray_is_valid"])
    np.testing.assert_array_equal(N(ns), want["rays_n_samples"])
    np.testing.assert_array_equal(N(start), want["rays_sample_startidx"])
    np.testing.assert_array_equal(N(idcs), want["idcs"])
    np.testing.assert_array_equal(N(xyzs), want["xyzs"])
    np.testing.assert_array_equal(N(dirs), want["dirs"])
    np.testing.assert_array_equal(N(dss), want["dss"])
    np.testing.assert_array_equal(N(z), want["z_vals"])


@pytest.mark.parametrize("case", [
    dict(n=2048, S=2 ** 20, K=1, G=128, bound=1.0, portion=0.0),
    dict(n=4096, S=20000, K=1, G=128, bound=1.0, portion=0.0),      # buffer fills mid-batch
    dict(n=777, S=1, K=1, G=128, bound=1.0, portion=0.0),           # tiny buffer
    dict(n=1500, S=2 ** 19, K=2, G=64, bound=2.0, portion=1 / 256),  # cascades + growing steps
    dict(n=1000, S=2 ** 19, K=1, G=32, bound=1.0, portion=0.0),
    dict(n=1200, S=2 ** 19, K=3, G=64, bound=3.0, portion=1 / 256),  # last cascade's bound 3: not a power of two
])
def test_march_rays_bit_exact(dev, case):
    rng = np.random.default_rng(case["n"])
    o, d, t0, t1, noise, bits, _ = march_inputs(rng, case["n"], bound=case["bound"], G=case["G"], K=case["K"])
    t1[::17] = t0[::17]  # some invalid rays
    got, want = _march_both(dev, case["S"], 1024, case["K"], case["G"], case["bound"], case["portion"], o, d, t0, t1,
                            noise, bits)
    _assert_march_equal(got, want)


def test_march_rays_fill_in_later_launches(dev):
    """Rays are counted in ray-ordered launches (2048, 16384, 131072, the rest); a
    later launch first adds the earlier launches' parked block totals.  A sparse
    field over 2^18 rays, with buffer sizes the oracle's own cumulative counts put
    inside the third launch, inside the fourth, and past every ray (no fill)."""
    rng = np.random.default_rng(77)
    n = 2 ** 18
    o, d, t0, t1, noise, bits, _ = march_inputs(rng, n)
    bits = bits & rng.integers(0, 256, bits.shape, dtype=np.uint8) & rng.integers(0, 256, bits.shape,
                                                                                    dtype=np.uint8)
    full = oracle.march_rays(2 ** 23, 1024, 1, 128, 1.0, 0.0, o, d, t0, t1, noise, bits)
    cum = np.cumsum(full["rays_n_samples"].astype(np.int64))
    assert cum[-1] > 0
    for S in (int(cum[60000]) + 1, int(cum[200000]) + 1, int(cum[-1]) + 1000):
        got, want = _march_both(dev, S, 1024, 1, 128, 1.0, 0.0, o, d, t0, t1, noise, bits)
        _assert_march_equal(got, want)


@pytest.mark.parametrize("dist", [3.0e4, 1.0e5])
def test_march_rays_far_origins(dev, dist):
    """Origins far outside the box: at t ~ 3e4 a step of 2*sqrt(3)/1024 rounds to one
    ulp of t (the visited t differ from t0 + k*ds); at t ~ 1e5 it rounds to zero, so
    t + ds == t: occupied cells then repeat the same sample up to the step cap
    (diagonal_n_steps * bound) and empty cells end the ray (the reference loops
    forever there; the skip ends it instead)."""
    rng = np.random.default_rng(int(dist))
    n = 300
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    target = rng.uniform(-0.5, 0.5, (n, 3))
    o = (target - d * dist).astype(np.float32)
    d = d.astype(np.float32)
    t0, t1 = near_far_np(o, d, 1.0)
    noise = rng.uniform(0, 1, n).astype(np.float32)
    bits, _ = blob_bitfield(rng, G=128, K=1)
    if dist > 5e4:
        bits[: bits.size // 2] = 255  # occupied cells where the stalled rays start
    got, want = _march_both(dev, 2 ** 20, 1024, 1, 128, 1.0, 0.0, o, d, t0, t1, noise, bits)
    _assert_march_equal(got, want)
    assert int(want["measured"]) > 0


def test_march_rays_full_and_empty_fields(dev, rng):
    o, d, t0, t1, noise, _, _ = march_inputs(rng, 3000)
    for fill in (0, 255):
        bits = np.full(128 ** 3 // 8, fill, np.uint8)
        got, want = _march_both(dev, 2 ** 20, 1024, 1, 128, 1.0, 0.0, o, d, t0, t1, noise, bits)
        _assert_march_equal(got, want)


def test_march_rays_zero_rays(dev):
    z = np.zeros((0, 3), np.float32)
    e = np.zeros(0, np.float32)
    bits = np.full(128 ** 3 // 8, 255, np.uint8)
    measured, valid, ns, start, idcs, xyzs, dirs, dss, zz = volrend.march_rays(
        64, 1024, 1, 128, 1.0, 0.0, T(z, dev), T(z, dev), T(e, dev), T(e, dev), T(e, dev), T(bits, dev))
    assert int(N(measured.view(torch.int32))) == 0 and not N(xyzs).any() and not N(idcs.view(torch.int32)).any()


def test_march_rays_reference_batch_shape(dev):
    """Training batch at the reference convention n_rays = total_samples = 2^18."""
    rng = np.random.default_rng(2024)
    n = 2 ** 18
    o, d, t0, t1, noise, bits, _ = march_inputs(rng, n)
    got, want = _march_both(dev, n, 1024, 1, 128, 1.0, 0.0, o, d, t0, t1, noise, bits)
    _assert_march_equal(got, want)
    # size-independent properties: ranges tile [0, measured) in ray order
    ns = N(got[2]).astype(np.int64)
    st = N(got[3]).astype(np.int64)
    v = ns > 0
    assert (st[v][1:] == (st[v] + ns[v])[:-1]).all()
    assert int(ns.sum()) == int(N(got[0].view(torch.int32)))


def test_march_rays_inference_bit_exact(dev):
    rng = np.random.default_rng(99)
    n_total, n_slots, cap = 5000, 1024, 8
    o, d, t0, t1, _, bits, _ = march_inputs(rng, n_total)
    t1[::13] = t0[::13] - 0.1  # t_end < t_start rays
    ts = t0.copy()
    term = np.ones(n_slots, bool)
    idx = np.zeros(n_slots, np.uint32)
    nri = np.zeros(1, np.uint32)
    ts_dev = T(ts, dev)
    term_dev, idx_dev, nri_dev = T(term, dev), U(idx, dev), U(nri, dev)
    for it in range(12):
        got = volrend.march_rays_inference(1024, 1, 128, cap, 1.0, 0.0, T(o, dev), T(d, dev), ts_dev, T(t1, dev),
                                           T(bits, dev), nri_dev, term_dev, idx_dev)
        want = oracle.march_rays_inference(1024, 1, 128, cap, 1.0, 0.0, o, d, ts, t1, bits, nri, term, idx)
        nxt, gidx, gns, gts, gx, gds, gz = got
        assert int(N(nxt.view(torch.int32))[0]) == int(want["next_ray_index"])
        np.testing.assert_array_equal(N(gidx), want["indices"])
        np.testing.assert_array_equal(N(gns), want["n_samples"])
        np.testing.assert_array_equal(N(gx), want["xyzs"])
        np.testing.assert_array_equal(N(gds), want["dss"])
        np.testing.assert_array_equal(N(gz), want["z_vals"])
        # host-side update as the reference wrapper does (t_starts.at[indices].set)
        keep = want["indices"] < n_total
        ts[want["indices"][keep]] = want["t_starts_out"][keep]
        np.testing.assert_array_equal(N(gts), ts)
        nri = np.array([want["next_ray_index"]], np.uint32)
        idx = want["indices"]
        term = (want["n_samples"] < cap) | (rng.uniform(size=n_slots) < 0.3)
        ts_dev, nri_dev, idx_dev, term_dev = gts, nxt, gidx, T(term, dev)


def _crossing_rays(rng, n, G, kind):
    """Rays towards [-1, 1]^3, through grid planes (`axis`: along an axis on a plane, with zeros of
    either sign; `graze`: nearly so), from inside it, or long ones that cross t = 4."""
    d = rng.normal(size=(n, 3))
    o = rng.uniform(-0.95, 0.95, (n, 3))
    if kind in ("axis", "graze"):
        d = np.where(rng.random((n, 3)) < 0.5, -0.0, 0.0) if kind == "axis" else rng.normal(size=(n, 3)) * 1e-4
        d[np.arange(n), rng.integers(0, 3, n)] = np.where(rng.random(n) < 0.5, -1.0, 1.0)
        o = rng.integers(0, G + 1, (n, 3)) * (2.0 / G) - 1.0 - 2.0 * d
    elif kind == "far":
        o = o * 0.7 - 4.0 * d / np.linalg.norm(d, axis=1, keepdims=True)
    d = d / np.linalg.norm(d, axis=1, keepdims=True)
    return o.astype(np.float32), d.astype(np.float32)


@pytest.mark.parametrize("G, diag, bound", [(4, 64, 1.0), (64, 1024, 1.0), (128, 333, 2.0)])
@pytest.mark.parametrize("kind", ["axis", "graze", "inside", "far"])
def test_march_rays_inference_constant_step_one_cascade(dev, kind, G, diag, bound):
    """The one-cascade constant-step march (whole empty blocks skipped, skips in one step)
    against the step-by-step oracle, every output bit for bit: blocks partly filled, blocks
    of one cell, empty space between them."""
    rng = np.random.default_rng([G, len(kind)])
    n, cap = 1500, 8
    o, d = _crossing_rays(rng, n, G, kind)
    t0 = rng.uniform(0.0, 1.0, n).astype(np.float32)
    t1 = (t0 + rng.uniform(0.0, 5.5, n)).astype(np.float32)
    filled = rng.random(G ** 3 // 64) < 0.3  # blocks: 64 cells in Morton order
    filled[0] = True
    bits = np.packbits(np.repeat(filled, 64) & (rng.random(G ** 3) < 0.7), bitorder="little")
    term, idx, nri, ts = np.ones(n, bool), np.zeros(n, np.uint32), np.zeros(1, np.uint32), t0.copy()
    for it in range(3):
        want = oracle.march_rays_inference(diag, 1, G, cap, bound, 0.0, o, d, ts, t1, bits, nri, term, idx)
        got = volrend.march_rays_inference(diag, 1, G, cap, bound, 0.0, T(o, dev), T(d, dev), T(ts, dev), T(t1, dev),
                                           T(bits, dev), U(nri, dev), T(term, dev), U(idx, dev))
        _, _, gns, gts, gx, gds, gz = got
        keep = want["indices"] < n
        ts[want["indices"][keep]] = want["t_starts_out"][keep]
        for g, w in ((gns, want["n_samples"]), (gx, want["xyzs"]), (gds, want["dss"]), (gz, want["z_vals"]), (gts, ts)):
            np.testing.assert_array_equal(N(g), w)
        assert it > 0 or want["n_samples"].any()
        nri, idx, term = np.array([want["next_ray_index"]], np.uint32), want["indices"], np.zeros(n, bool)


@pytest.mark.parametrize("G, diag, bound, portion", [(4, 64, 1.0, 0.0), (64, 1024, 1.0, 0.0), (128, 333, 0.7, 0.0),
                                                     (128, 512, 3.0, 1 / 256)])
@pytest.mark.parametrize("kind", ["axis", "graze", "inside", "far"])
def test_march_rays_one_cascade_edges(dev, kind, G, diag, bound, portion):
    """The walk that crosses stretches of empty cells at once against the step-by-step oracle,
    every output bit for bit, on rays along and through planes of the grid; samples enough for
    several rounds of rays, the last of them partial, and for a buffer that fills."""
    rng = np.random.default_rng([G, len(kind), diag])
    n = 9003
    o, d = _crossing_rays(rng, n, G, kind)
    o *= np.float32(bound)
    t0 = rng.uniform(0.0, 1.0, n).astype(np.float32)
    t1 = (t0 + rng.uniform(0.0, 5.5, n)).astype(np.float32)
    noise = rng.uniform(0, 1, n).astype(np.float32)
    filled = rng.random(G ** 3 // 64) < 0.3  # blocks: 64 cells in Morton order
    filled[0] = True
    bits = np.packbits(np.repeat(filled, 64) & (rng.random(G ** 3) < 0.7), bitorder="little")
    for total in (1 << 14, 1 << 21):
        got, want = _march_both(dev, total, diag, 1, G, bound, portion, o, d, t0, t1, noise, bits)
        _assert_march_equal(got, want)


@pytest.mark.parametrize("n, offset", [(1, 0), (1023, 0), (1025, 0), (3000, 1), (1 << 19, 0), ((1 << 19) + 1, 0)])
def test_slot_assignment_in_one_launch_or_three(dev, n, offset):
    """Terminated slots take the next ray indices in slot order, whichever way they are counted:
    within a block, over blocks, from unaligned flags, up to the one-launch limit and past it."""
    rng = np.random.default_rng(n)
    flags = rng.random(n + offset) < 0.4
    term = T(flags, dev)[offset:]
    idx = rng.integers(0, 1000, n).astype(np.uint32)
    rays = torch.zeros(4, 3, device=dev)
    empty = torch.ones(4, device=dev)  # t_end < t_start: nothing is marched
    out = volrend.march_rays_inference(64, 1, 4, 1, 1.0, 0.0, rays, rays + 1, empty, empty - 1,
                                       torch.zeros(8, dtype=torch.uint8, device=dev), U(np.array([7], np.uint32), dev), term, U(idx, dev))
    want = np.where(flags[offset:], 7 + np.cumsum(flags[offset:]) - 1, idx)
    np.testing.assert_array_equal(N(out[1]), want.astype(np.uint32))
    assert int(N(out[0].view(torch.int32))[0]) == 7 + int(flags[offset:].sum())


def test_integrate_rays_bit_exact_and_backward(dev):
    rng = np.random.default_rng(5)
    start, ns, bgs, dss, z, drgbs = integrate_inputs(rng, 4096, 200)
    m_o, rgbd_o, op_o = oracle.integrate_rays(start, ns, bgs, dss, z, drgbs)
    drgbs_t = T(drgbs, dev).requires_grad_(True)
    bgs_t = T(bgs, dev).requires_grad_(True)
    z_t = T(z, dev).requires_grad_(True)
    m, rgbd, op = volrend.integrate_rays(0.3, U(start, dev), U(ns, dev), bgs_t, T(dss, dev), z_t, drgbs_t)
    assert int(N(m.view(torch.int32))) == int(m_o)
    np.testing.assert_array_equal(N(rgbd.detach()), rgbd_o)
    np.testing.assert_array_equal(N(op.detach()), op_o)
    g = rng.normal(size=(4096, 4)).astype(np.float32)
    rgbd.backward(T(g, dev))
    dbg_o, dz_o, dd_o = oracle.integrate_rays_backward(0.3, start, ns, bgs, dss, z, drgbs, rgbd_o, op_o, g)
    np.testing.assert_array_equal(N(bgs_t.grad), dbg_o)
    np.testing.assert_array_equal(N(z_t.grad), dz_o)
    np.testing.assert_array_equal(N(drgbs_t.grad), dd_o)


def test_integrate_rays_near_plane_and_broadcast_bg(dev):
    rng = np.random.default_rng(6)
    start, ns, bgs, dss, z, drgbs = integrate_inputs(rng, 500, 40)
    z = (z - 2.6).astype(np.float32)  # samples before the near plane and z < 1
    drgbs_t = T(drgbs, dev).requires_grad_(True)
    m, rgbd, op = volrend.integrate_rays(0.3, U(start, dev), U(ns, dev), [1.0, 1.0, 1.0], T(dss, dev), T(z, dev),
                                         drgbs_t)
    m_o, rgbd_o, op_o = oracle.integrate_rays(start, ns, np.ones(3, np.float32), dss, z, drgbs)
    np.testing.assert_array_equal(N(rgbd.detach()), rgbd_o)
    g = rng.normal(size=(500, 4)).astype(np.float32)
    rgbd.backward(T(g, dev))
    _, _, dd_o = oracle.integrate_rays_backward(0.3, start, ns, np.ones((500, 3), np.float32), dss, z, drgbs, rgbd_o,
                                                op_o, g)
    np.testing.assert_array_equal(N(drgbs_t.grad), dd_o)


def test_integrate_rays_2pow20_samples_properties(dev):
    """Integrator workload at 2^20 samples (1024 rays x 1024 samples): opacity in [0,1], measured <= S, and
    the f32 result within float64 error on a subset."""
    rng = np.random.default_rng(8)
    n_rays, m = 1024, 1024
    ns = np.full(n_rays, m, np.uint32)
    start = (np.arange(n_rays) * m).astype(np.uint32)
    S = n_rays * m
    dss = np.full(S, 2 * 1.7320508 / 1024, np.float32)
    z = np.tile(3.0 + np.arange(m, dtype=np.float32) * dss[0], n_rays).astype(np.float32)
    sig = np.log1p(np.exp(rng.normal(0, 2, S))).astype(np.float32)
    drgbs = np.concatenate([sig[:, None], rng.uniform(0, 1, (S, 3)).astype(np.float32)], 1)
    bgs = rng.uniform(0, 1, (n_rays, 3)).astype(np.float32)
    mm, rgbd, op = volrend.integrate_rays(0.3, U(start, dev), U(ns, dev), T(bgs, dev), T(dss, dev), T(z, dev),
                                          T(drgbs, dev))
    m_o, rgbd_o, op_o = oracle.integrate_rays(start, ns, bgs, dss, z, drgbs)
    assert int(N(mm.view(torch.int32))) == int(m_o) <= S
    np.testing.assert_array_equal(N(rgbd), rgbd_o)
    sub = np.arange(0, n_rays, 37)
    rgbd64, op64, _ = oracle.integrate_rays64(start[sub], ns[sub], bgs[sub], dss, z, drgbs)
    np.testing.assert_allclose(N(rgbd)[sub], rgbd64, rtol=1e-4, atol=2e-5)


def _c2_inputs(rng, n_rays, counts):
    """The differentiation workload: rays of `counts` samples, densities softplus(N(0,2)),
    rgb and bg U[0,1], ds = 2 sqrt(3) / 1024, z = 3 + k ds."""
    ns = np.asarray(counts, np.uint32)
    start = np.zeros(n_rays, np.uint32)
    start[1:] = np.cumsum(ns)[:-1]
    S = int(ns.sum())
    ds = np.float32(2 * 1.7320508075688772 / 1024)
    dss = np.full(S, ds, np.float32)
    k = np.arange(S) - np.repeat(start.astype(np.int64), ns)
    z = (np.float32(3) + k.astype(np.float32) * ds).astype(np.float32)
    sig = np.log1p(np.exp(rng.normal(0, 2, S))).astype(np.float32)
    drgbs = np.concatenate([sig[:, None], rng.uniform(0, 1, (S, 3)).astype(np.float32)], 1)
    bgs = rng.uniform(0, 1, (n_rays, 3)).astype(np.float32)
    return start, ns, bgs, dss, z, drgbs


@pytest.mark.parametrize("n_rays,max_samples,full", [(4096, 1024, False), (1024, 1024, True)])
def test_integrate_rays_backward_differentiation_workload(dev, n_rays, max_samples, full):
    """4096 rays x U{1..1024} samples (seed 4; 2,119,089 samples), and 1024 full rays
    (2^20 samples): forward and the reference VJP (dbg, dz, ddrgbs) bit for bit
    against the oracle."""
    rng = np.random.default_rng(4)
    counts = np.full(n_rays, max_samples) if full else rng.integers(1, max_samples + 1, n_rays)
    start, ns, bgs, dss, z, drgbs = _c2_inputs(rng, n_rays, counts)
    print(f"integrate c2: rays={n_rays} samples={int(ns.sum())}", flush=True)
    m_o, rgbd_o, op_o = oracle.integrate_rays(start, ns, bgs, dss, z, drgbs)
    drgbs_t = T(drgbs, dev).requires_grad_(True)
    bgs_t = T(bgs, dev).requires_grad_(True)
    z_t = T(z, dev).requires_grad_(True)
    m, rgbd, op = volrend.integrate_rays(0.3, U(start, dev), U(ns, dev), bgs_t, T(dss, dev), z_t, drgbs_t)
    assert int(N(m.view(torch.int32))) == int(m_o)
    np.testing.assert_array_equal(N(rgbd.detach()), rgbd_o)
    np.testing.assert_array_equal(N(op.detach()), op_o)
    # at these densities no ray reaches T <= 1e-4 within 1024 samples (opacity <= 0.981):
    # every ray keeps its background term; test_integrate_rays_bit_exact_and_backward
    # covers terminated rays
    assert (op_o < 1 - 1e-4).all() and op_o.max() > 0.9
    g = rng.normal(size=(n_rays, 4)).astype(np.float32)
    rgbd.backward(T(g, dev))
    dbg_o, dz_o, dd_o = oracle.integrate_rays_backward(0.3, start, ns, bgs, dss, z, drgbs, rgbd_o, op_o, g)
    np.testing.assert_array_equal(N(bgs_t.grad), dbg_o)
    np.testing.assert_array_equal(N(z_t.grad), dz_o)
    np.testing.assert_array_equal(N(drgbs_t.grad), dd_o)


def test_integrate_rays_inference_bit_exact(dev):
    rng = np.random.default_rng(11)
    n_total, n, cap = 3000, 512, 8
    rays_bg = rng.uniform(0, 1, (n_total, 3)).astype(np.float32)
    rays_rgbd = rng.uniform(0, 0.5, (n_total, 4)).astype(np.float32)
    rays_T = rng.uniform(0, 1, n_total).astype(np.float32)
    rays_T[::7] = 5e-5
    idx = rng.choice(n_total + 100, n, replace=False).astype(np.uint32)
    ns = rng.integers(0, cap + 1, n).astype(np.uint32)
    dss = rng.uniform(0.001, 0.05, (n, cap)).astype(np.float32)
    z = rng.uniform(2, 5, (n, cap)).astype(np.float32)
    drgbs = np.concatenate([rng.uniform(0, 80, (n, cap, 1)), rng.uniform(0, 1, (n, cap, 3))], 2).astype(np.float32)
    cnt, term, rgbd, Tn = volrend.integrate_rays_inference(T(rays_bg, dev), T(rays_rgbd, dev), T(rays_T, dev),
                                                           U(ns, dev), U(idx, dev), T(dss, dev), T(z, dev),
                                                           T(drgbs, dev))
    c_o, t_o, rgbd_o, T_o = oracle.integrate_rays_inference(rays_bg, rays_rgbd, rays_T, ns, idx, dss, z, drgbs)
    assert int(N(cnt.view(torch.int32))) == int(c_o)
    np.testing.assert_array_equal(N(term), t_o)
    keep = idx < n_total
    want_rgbd = rays_rgbd.copy()
    want_T = rays_T.copy()
    want_rgbd[idx[keep]] = rgbd_o[keep]
    want_T[idx[keep]] = T_o[keep]
    np.testing.assert_array_equal(N(rgbd), want_rgbd)
    np.testing.assert_array_equal(N(Tn), want_T)


@pytest.mark.parametrize("n, cap", [((1 << 14) - 1, 1), (1 << 14, 1), ((3 << 14) - 1, 3), ((3 << 14) + 1, 3), (257, 70)])
def test_integrate_rays_inference_both_workgroup_sizes(dev, n, cap):
    """Both sides of the line between workgroups of 256 and 1,024 threads, with a part of a
    workgroup at the end, bit for bit against the oracle; the terminated rays are counted."""
    rng = np.random.default_rng(n)
    n_total = 2 * n
    ns = rng.integers(0, cap + 1, n).astype(np.uint32)
    idx = rng.permutation(n_total + n // 2)[:n].astype(np.uint32)  # some past the last ray
    bg = rng.uniform(0, 1, (n_total, 3)).astype(np.float32)
    rgbd = rng.uniform(0, 1, (n_total, 4)).astype(np.float32)
    trans = rng.uniform(0.0002, 1, n_total).astype(np.float32)
    dss = np.full((n, cap), 0.01, np.float32)
    z = rng.uniform(1, 2, (n, cap)).astype(np.float32)
    drgbs = rng.uniform(0, 1, (n, cap, 4)).astype(np.float32)
    drgbs[..., 0] *= rng.choice([1.0, 1000.0], (n, 1)).astype(np.float32)
    got = volrend.integrate_rays_inference(T(bg, dev), T(rgbd, dev), T(trans, dev), U(ns, dev), U(idx, dev), T(dss, dev),
                                           T(z, dev), T(drgbs, dev))
    cnt, term, rgbd_o, T_o = oracle.integrate_rays_inference(bg, rgbd, trans, ns, idx, dss, z, drgbs)
    assert int(N(got[0].view(torch.int32))) == int(cnt)
    np.testing.assert_array_equal(N(got[1]), term)
    keep = idx < n_total
    rgbd[idx[keep]], trans[idx[keep]] = rgbd_o[keep], T_o[keep]
    np.testing.assert_array_equal(N(got[2]), rgbd)
    np.testing.assert_array_equal(N(got[3]), trans)
