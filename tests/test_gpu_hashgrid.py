"""GPU parity of the hash-grid encoder (forward and table gradient).

Forward: bit-exact against the oracle's f32 restatement (same vertex indices,
weights and summation order), and within |a-b| <= 1e-5 * max(|b|, 1e-4) of the
float64 transcription (the tolerance of the encoder workload: hash indices exact,
encodings within 1e-5 relative of FP64).
Backward: within 1e-5 of the float64 scatter-add, relative to the sum of the
absolute contributions of each row (the kernels merge runs in f32 and sum the
rest in any order); rows no point touches are exactly 0 (a touched row may
cancel to 0 within the tolerance).
"""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from jaxngp_amd.encoders import HashGridEncoder

pytestmark = pytest.mark.gpu


def _c_forward(enc_mod, pos, table, bound=1.0):
    lv = enc_mod.levels
    N, L, F = pos.shape[0], enc_mod.L, enc_mod.F
    out = np.zeros((N, L * F), np.float32)
    scales = np.asarray(lv.scales, np.float32)
    res = np.asarray(lv.resolutions, np.uint32)
    offs = np.asarray(lv.offsets, np.uint32)
    P = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    pos = np.ascontiguousarray(pos, np.float32)
    table = np.ascontiguousarray(table, np.float32)
    oracle.lib().oracle_hashgrid_fwd(ctypes.c_uint32(N), ctypes.c_uint32(L), ctypes.c_uint32(F),
                                     ctypes.c_uint32(enc_mod.T), ctypes.c_uint32(lv.first_hash_level),
                                     ctypes.c_uint32(lv.n_rows), ctypes.c_float(bound), P(scales), P(res), P(offs),
                                     P(pos), P(table), P(out))
    return out


def _c_backward(enc_mod, pos, g, bound=1.0):
    lv = enc_mod.levels
    N, L, F = pos.shape[0], enc_mod.L, enc_mod.F
    out = np.zeros((lv.n_rows, F), np.float64)
    scales = np.asarray(lv.scales, np.float32)
    res = np.asarray(lv.resolutions, np.uint32)
    offs = np.asarray(lv.offsets, np.uint32)
    P = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    oracle.lib().oracle_hashgrid_bwd(ctypes.c_uint32(N), ctypes.c_uint32(L), ctypes.c_uint32(F),
                                     ctypes.c_uint32(enc_mod.T), ctypes.c_uint32(lv.first_hash_level),
                                     ctypes.c_uint32(lv.n_rows), ctypes.c_float(bound), P(scales), P(res), P(offs),
                                     P(np.ascontiguousarray(pos, np.float32)), P(np.ascontiguousarray(g, np.float32)),
                                     P(out))
    return out


CONFIGS = {
    "l16_t2e19": dict(L=16, T=2 ** 19, F=2, N_min=16, N_max=2048),
    "proposal": dict(L=5, T=2 ** 17, F=2, N_min=16, N_max=512),
    "small_f4": dict(L=8, T=2 ** 12, F=4, N_min=4, N_max=64),
    "f1_dense_only": dict(L=3, T=2 ** 20, F=1, N_min=8, N_max=32),
    "f8": dict(L=4, T=2 ** 14, F=8, N_min=16, N_max=256),
    # dense levels of up to 4.1 M rows: a vertex on a level's upper face addresses up
    # to res^2 + res rows (~26 k) past the level, several 8192-row slices into the next
    "dense_overflow": dict(L=4, T=2 ** 22, F=2, N_min=64, N_max=160),
}


@pytest.mark.parametrize("name", list(CONFIGS))
def test_hashgrid_forward_backward(dev, name):
    cfg = CONFIGS[name]
    rng = np.random.default_rng(0)
    g_gen = torch.Generator(device="cpu").manual_seed(1)
    enc = HashGridEncoder(**cfg, generator=g_gen).to(dev)
    N = 40000
    pos = rng.uniform(-1, 1, (N, 3)).astype(np.float32)
    pos[:4] = [[-1, -1, -1], [1, 1, 1], [0, 0, 0], [0.999999, -0.999999, 0.5]]
    table = enc.table.detach().cpu().numpy()
    pos_t = torch.from_numpy(pos).to(dev)
    out, tv = enc(pos_t, 1.0)
    assert tv == 0.0
    got = out.detach().cpu().numpy()
    np.testing.assert_array_equal(got, _c_forward(enc, pos, table))
    lv = oracle.hashgrid_levels(cfg["L"], cfg["T"], cfg["N_min"], cfg["N_max"])
    want64 = oracle.hashgrid_forward64(pos[:8000], table, 1.0, lv, cfg["T"])
    assert (np.abs(got[:8000] - want64) <= 1e-5 * np.maximum(np.abs(want64), 1e-4)).all()
    g = rng.normal(size=got.shape).astype(np.float32)
    out.backward(torch.from_numpy(g).to(dev))
    dt = enc.table.grad.detach().cpu().numpy().astype(np.float64)
    want = _c_backward(enc, pos, g)
    absw = _c_backward(enc, pos, np.abs(g))
    assert (dt[absw == 0] == 0).all()  # rows no point touches stay exactly 0
    assert (np.abs(dt - want) <= 1e-5 * absw + 1e-30).all()


def test_hashgrid_encoder_workload_full_size(dev):
    """Encoder workload: N = 2^18 points, L=16, F=2, T=2^19, table U(-1e-4, 1e-4)."""
    rng = np.random.default_rng(0)
    enc = HashGridEncoder(**CONFIGS["l16_t2e19"], generator=torch.Generator().manual_seed(1)).to(dev)
    assert enc.levels.n_rows == 6098120 and enc.levels.first_hash_level == 5
    N = 2 ** 18
    xyz = rng.uniform(0, 1, (N, 3)).astype(np.float32)
    pos = (xyz * np.float32(2) - np.float32(1)).astype(np.float32)
    out, _ = enc(torch.from_numpy(pos).to(dev), 1.0)
    got = out.detach().cpu().numpy()
    np.testing.assert_array_equal(got, _c_forward(enc, pos, enc.table.detach().cpu().numpy()))
    g = np.random.default_rng(2).normal(size=(N, 32)).astype(np.float32)
    out.backward(torch.from_numpy(g).to(dev))
    dt = enc.table.grad.detach().cpu().numpy().astype(np.float64)
    want = _c_backward(enc, pos, g)
    absw = _c_backward(enc, pos, np.abs(g))
    assert (dt[absw == 0] == 0).all()  # rows no point touches stay exactly 0
    assert (np.abs(dt - want) <= 1e-5 * absw + 1e-30).all()


def test_hashgrid_fp16_table(dev):
    rng = np.random.default_rng(3)
    enc = HashGridEncoder(**CONFIGS["proposal"], param_dtype=torch.float16,
                          generator=torch.Generator().manual_seed(4)).to(dev)
    with torch.no_grad():
        enc.table.copy_(torch.from_numpy(rng.uniform(-1, 1, tuple(enc.table.shape)).astype(np.float16)))
    pos = rng.uniform(-1, 1, (20000, 3)).astype(np.float32)
    out, _ = enc(torch.from_numpy(pos).to(dev), 1.0)
    table32 = enc.table.detach().float().cpu().numpy()
    np.testing.assert_array_equal(out.detach().cpu().numpy(), _c_forward(enc, pos, table32))


def test_level_major_layout_matches_point_major(dev):
    """The level-major [L, N, F] path (XCD-affine kernels) gives the point-major
    encodings transposed, and the same table gradient from the transposed cotangent."""
    from jaxngp_amd import _lib
    rng = np.random.default_rng(9)
    enc = HashGridEncoder(**CONFIGS["l16_t2e19"], generator=torch.Generator().manual_seed(1)).to(dev)
    with torch.no_grad():
        enc.table.uniform_(-1, 1)
    N = 30001
    pos = torch.from_numpy(rng.uniform(-1, 1, (N, 3)).astype(np.float32)).to(dev)
    L, F = 16, 2
    pm = torch.empty(N, L * F, device=dev)
    lm = torch.empty(L, N, F, device=dev)
    t = enc.table.detach()
    _lib.call("hashgrid_encode", [pos, t, pm], enc.descriptor(N, 1.0))
    _lib.call("hashgrid_encode", [pos, t, lm], enc.descriptor(N, 1.0, _lib.ENC_LEVEL_MAJOR))
    torch.testing.assert_close(lm.permute(1, 0, 2).reshape(N, L * F), pm, rtol=0, atol=0)
    g = torch.from_numpy(rng.normal(size=(N, L * F)).astype(np.float32)).to(dev)
    g_lm = g.reshape(N, L, F).permute(1, 0, 2).contiguous()
    d1 = torch.empty_like(t)
    d2 = torch.empty_like(t)
    for d, gg, layout in ((d1, g, _lib.ENC_POINT_MAJOR), (d2, g_lm, _lib.ENC_LEVEL_MAJOR)):
        desc = enc.descriptor(N, 1.0, layout)
        ws = torch.empty(_lib.hashgrid_backward_workspace_bytes(desc), dtype=torch.uint8, device=dev)
        _lib.call("hashgrid_encode_backward", [pos, gg, d, ws], desc)
    want = _c_backward(enc, pos.cpu().numpy(), g.cpu().numpy())
    absw = _c_backward(enc, pos.cpu().numpy(), np.abs(g.cpu().numpy()))
    for d in (d1, d2):
        dt = d.cpu().numpy().astype(np.float64)
        assert (dt[absw == 0] == 0).all()  # rows no point touches stay exactly 0
        assert (np.abs(dt - want) <= 1e-5 * absw + 1e-30).all()


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("T,N", [(2 ** 19, 1), (2 ** 14, 513), (1000, 1025), (999, 511), (2 ** 19, 32769)])
def test_grouped_rows_match_row_by_row_and_staged(dev, T, N, half):
    """The grouped gather (16-byte aligned tables of whole groups), the row-by-row gather
    (the same table a row past alignment, and T = 999, whose row count is odd) and the
    staged point-major output are bit-exact against the oracle."""
    from jaxngp_amd import _lib
    rng = np.random.default_rng(T + N)
    enc = HashGridEncoder(L=16, T=T, F=2, N_min=16, N_max=2048, param_dtype=torch.float16 if half else torch.float32,
                          generator=torch.Generator().manual_seed(1)).to(dev)
    n_rows = enc.levels.n_rows
    buf = torch.empty(n_rows + 1, 2, dtype=enc.table.dtype, device=dev).uniform_(-1, 1)
    shifted = buf[1:]
    table = shifted.clone()
    assert table.data_ptr() % 16 == 0 and shifted.data_ptr() % 16 != 0
    pos_np = rng.uniform(-1, 1, (N, 3)).astype(np.float32)
    pos_np[0] = 1.0  # the upper corner: dense vertices past their level
    pos = torch.from_numpy(pos_np).to(dev)
    want = _c_forward(enc, pos_np, table.float().cpu().numpy())
    for t in (table, shifted):
        for layout in (_lib.ENC_POINT_MAJOR, _lib.ENC_LEVEL_MAJOR):
            out = torch.empty(16, N, 2, device=dev)
            _lib.call("hashgrid_encode", [pos, t, out], enc.descriptor(N, 1.0, layout))
            got = out.permute(1, 0, 2).reshape(N, 32) if layout == _lib.ENC_LEVEL_MAJOR else out.reshape(N, 32)
            np.testing.assert_array_equal(got.cpu().numpy(), want)
        out, ws = torch.empty(N, 32, device=dev), torch.empty(N, 32, device=dev)
        _lib.call("hashgrid_encode_staged", [pos, t, out, ws], enc.descriptor(N, 1.0))
        np.testing.assert_array_equal(out.cpu().numpy(), want)


@pytest.mark.parametrize("L, T, F, N, half", [
    (2, 2 ** 14, 2, 4097, False), (5, 2 ** 15, 1, 4096, False), (6, 2 ** 15, 2, 8193, True), (7, 2 ** 14, 4, 1, False),
    (11, 2 ** 15, 2, 2049, False), (12, 2 ** 15, 2, 1025, False), (8, 2 ** 15, 4, 4095, True), (16, 2 ** 14, 8, 777, False),
    # levels of more than two L2s: neighbouring lanes take a point's levels from n F = 2^17 on
    (3, 2 ** 21, 2, 2 ** 16 - 1, False), (3, 2 ** 21, 2, 2 ** 16, False), (3, 2 ** 19, 8, 2 ** 14 + 5, False),
    (3, 2 ** 22, 4, 2 ** 15 + 1, True), (3, 2 ** 22, 1, 2 ** 17 + 1, False)])
def test_forward_over_the_ways_levels_are_dealt(dev, L, T, F, N, half):
    """One, two and four sets of levels over the XCDs, a last set that is not full, one block
    and several, and large levels: both layouts and the staged output, bit for bit."""
    from jaxngp_amd import _lib
    enc = HashGridEncoder(L=L, T=T, F=F, N_min=16, N_max=512, param_dtype=torch.float16 if half else torch.float32,
                          generator=torch.Generator().manual_seed(1)).to(dev)
    with torch.no_grad():
        enc.table.uniform_(-1, 1)
    pos_np = np.random.default_rng(N).uniform(-1, 1, (N, 3)).astype(np.float32)
    pos = torch.from_numpy(pos_np).to(dev)
    table = enc.table.detach()
    want = _c_forward(enc, pos_np, table.float().cpu().numpy())
    for layout in (_lib.ENC_POINT_MAJOR, _lib.ENC_LEVEL_MAJOR):
        out = torch.empty(L * N * F, device=dev)
        _lib.call("hashgrid_encode", [pos, table, out], enc.descriptor(N, 1.0, layout))
        got = out.view(L, N, F).permute(1, 0, 2) if layout == _lib.ENC_LEVEL_MAJOR else out
        np.testing.assert_array_equal(got.reshape(N, L * F).cpu().numpy(), want)
    if F in (2, 4):
        out, ws = torch.empty(N, L * F, device=dev), torch.empty(N, L * F, device=dev)
        _lib.call("hashgrid_encode_staged", [pos, table, out, ws], enc.descriptor(N, 1.0))
        np.testing.assert_array_equal(out.cpu().numpy(), want)


@pytest.mark.parametrize("F, half", [(2, False), (4, True)])
def test_staged_forward_in_pieces(dev, F, half):
    """More points than the workspace of the staged forward takes at once: two whole pieces and
    a rest of one point, with nothing written past the workspace, bit for bit as point by point."""
    from jaxngp_amd import _lib
    piece = _lib.ENCODE_STAGE_POINTS
    N, L = 2 * piece + 1, 3
    enc = HashGridEncoder(L=L, T=2 ** 12, F=F, N_min=8, N_max=64, param_dtype=torch.float16 if half else torch.float32,
                          generator=torch.Generator().manual_seed(1)).to(dev)
    pos = torch.rand(N, 3, generator=torch.Generator(device=dev).manual_seed(2), device=dev) * 2 - 1
    out, want = torch.empty(N, L * F, device=dev), torch.empty(N, L * F, device=dev)
    ws = torch.full((L * piece * F + 64,), 7.0, device=dev)
    _lib.call("hashgrid_encode_staged", [pos, enc.table.detach(), out, ws], enc.descriptor(N, 1.0))
    _lib.call("hashgrid_encode", [pos, enc.table.detach(), want], enc.descriptor(N, 1.0))
    assert torch.equal(out, want)
    assert (ws[L * piece * F:] == 7.0).all()


def _backward_raw(enc, pos_t, g_t):
    from jaxngp_amd import _lib
    N = pos_t.shape[0]
    desc = enc.descriptor(N, 1.0)
    ws = torch.empty(_lib.hashgrid_backward_workspace_bytes(desc), dtype=torch.uint8, device=pos_t.device)
    d = torch.empty(tuple(enc.table.shape), dtype=torch.float32, device=pos_t.device)  # the gradient is f32
    _lib.call("hashgrid_encode_backward", [pos_t, g_t, d, ws], desc)
    return d


@pytest.mark.parametrize("cfg,half", [
    (CONFIGS["l16_t2e19"], False), (CONFIGS["l16_t2e19"], True),
    (dict(L=16, T=2 ** 19, F=1, N_min=16, N_max=2048), False),
    (dict(L=2, T=2 ** 23, F=2, N_min=150, N_max=160), False),  # slices of 64 KiB, level 0 reaches 1,824
    (dict(L=3, T=2 ** 23, F=2, N_min=150, N_max=200), True),  # of 128 KiB, level 1 reaches 1,025
])
@pytest.mark.parametrize("N", [16, 2048, 20000])
def test_backward_of_points_outside_the_box(dev, cfg, half, N):
    """Points outside [-bound, bound] read rows modulo T, any of the T from a dense level's
    offset on, and their gradient goes to the rows that they read: past the upper corner
    against the oracle (the bound of test_hashgrid_forward_backward; for f16 half an ulp more of
    each entry, of which a row has at most 8 N, and of the row), past the lower one, where the
    oracle's conversion of negative coordinates is undefined, as the adjoint of the forward."""
    enc = HashGridEncoder(**cfg, param_dtype=torch.float16 if half else torch.float32,
                          generator=torch.Generator().manual_seed(1)).to(dev)
    rng = np.random.default_rng(N)
    LF = cfg["L"] * cfg["F"]
    g = rng.normal(size=(N, LF)).astype(np.float32)
    far = rng.choice([1.0, 1.05, 1.3, 1.5, 40.0], (N, 1))
    pos = (rng.uniform(0.9, 1, (N, 3)) * far).astype(np.float32)

    def table_grad(p, up):
        enc.table.grad = None
        out, _ = enc(torch.from_numpy(p).to(dev), 1.0)
        out.backward(torch.from_numpy(up).to(dev))
        return out.detach().cpu().double().numpy(), enc.table.grad.detach().cpu().double().numpy()

    _, got = table_grad(pos, g)
    want, absw = _c_backward(enc, pos, g), _c_backward(enc, pos, np.abs(g))
    assert (got[absw == 0] == 0).all()
    tol = 1e-5 * absw + 1e-30
    if half:
        tol += 2.0 ** -11 * (absw + np.abs(want)) + 8 * N * 2.0 ** -25
    assert (np.abs(got - want) <= tol).all()
    if not half:
        out, d = table_grad(-pos, g)
        _, dabs = table_grad(-pos, np.abs(g))
        t = enc.table.detach().cpu().double().numpy()
        assert abs((out * g).sum() - (d * t).sum()) <= 2e-5 * (dabs * np.abs(t)).sum()


@pytest.mark.parametrize("kind,N", [("random", 1), ("ray", 63), ("one_cell", 64), ("ray", 65), ("ray", 513),
                                    ("random", 1025), ("one_cell", 5000), ("random", 30000)])
def test_backward_item_and_run_edges(dev, kind, N):
    """Sizes around a wavefront, a phase and an item of the one-pass table gradient; all
    points in one cell (runs as long as the wavefront, few rows, several parts a slice)
    and none sharing a cell.  The bound of test_hashgrid_forward_backward."""
    rng = np.random.default_rng(N)
    enc = HashGridEncoder(**CONFIGS["l16_t2e19"], generator=torch.Generator().manual_seed(1)).to(dev)
    if kind == "random":
        pos = rng.uniform(-1, 1, (N, 3))
    elif kind == "ray":
        d = np.array([0.48, -0.6, 0.64])
        pos = (np.arange(N)[:, None] - N / 2) * (2 * 3 ** 0.5 / 1024) * d
    else:
        pos = 0.3 + rng.uniform(0, 2e-4, (N, 3))
    pos = pos.astype(np.float32)
    g = rng.normal(size=(N, 32)).astype(np.float32)
    got = _backward_raw(enc, torch.from_numpy(pos).to(dev), torch.from_numpy(g).to(dev)).cpu().numpy().astype(np.float64)
    want, absw = _c_backward(enc, pos, g), _c_backward(enc, pos, np.abs(g))
    assert (got[absw == 0] == 0).all()
    assert (np.abs(got - want) <= 1e-5 * absw + 1e-30).all()


def test_backward_scale_free(dev):
    """The table gradient's sums keep relative precision at any magnitude:
    cotangents scaled by 2^-60 or 2^+60 give the gradient scaled by the same power
    of two, within the f32 tolerance (contributions stay in the f32 normal range)."""
    rng = np.random.default_rng(21)
    enc = HashGridEncoder(**CONFIGS["l16_t2e19"], generator=torch.Generator().manual_seed(1)).to(dev)
    N = 50000
    pos = rng.uniform(-1, 1, (N, 3)).astype(np.float32)
    g = rng.normal(size=(N, 32)).astype(np.float32)
    pos_t = torch.from_numpy(pos).to(dev)
    want = _c_backward(enc, pos, g)
    absw = _c_backward(enc, pos, np.abs(g))
    for k in (-60, 60):
        gs = np.ldexp(g, k).astype(np.float32)
        d = _backward_raw(enc, pos_t, torch.from_numpy(gs).to(dev)).cpu().numpy().astype(np.float64)
        d = np.ldexp(d, -k)
        assert (d[absw == 0] == 0).all()
        assert (np.abs(d - want) <= 1e-5 * absw + 1e-30).all()


def test_backward_non_finite_reaches_its_rows(dev):
    """An inf or NaN cotangent (a loss-scaling overflow) makes exactly the rows its
    point touches non-finite, as a float sum does; the other rows stay exact."""
    rng = np.random.default_rng(22)
    cfg = CONFIGS["proposal"]
    enc = HashGridEncoder(**cfg, generator=torch.Generator().manual_seed(2)).to(dev)
    N = 20000
    pos = rng.uniform(-1, 1, (N, 3)).astype(np.float32)
    g = rng.normal(size=(N, cfg["L"] * cfg["F"])).astype(np.float32)
    g[7, 3] = np.inf
    g[11, 0] = np.nan
    d = _backward_raw(enc, torch.from_numpy(pos).to(dev), torch.from_numpy(g).to(dev)).cpu().numpy()
    want = _c_backward(enc, pos, g)
    bad = ~np.isfinite(want)
    assert bad.any()
    np.testing.assert_array_equal(~np.isfinite(d), bad)
    gf = np.where(np.isfinite(g), g, 0).astype(np.float32)
    absw = _c_backward(enc, pos, np.abs(gf))
    ok = ~bad
    assert (np.abs(d[ok].astype(np.float64) - want[ok]) <= 1e-5 * absw[ok] + 1e-30).all()


def test_fp16_table_backward(dev):
    """f16 tables (the precision path) sort f16-rounded contributions: the gradient
    is within 1e-3 of the float64 scatter relative to each row's absolute
    contributions (f16 keeps 11 bits) plus 1e-6 absolute (contributions below f16's
    smallest subnormal, 6e-8, round to zero; the loss scale keeps training's far
    above it), untouched rows stay 0, and a contribution past the f16 range reaches
    its rows as inf (what the loss-scale check looks for)."""
    from jaxngp_amd import _lib
    rng = np.random.default_rng(31)
    enc = HashGridEncoder(**CONFIGS["l16_t2e19"], param_dtype=torch.float16, generator=torch.Generator().manual_seed(4)).to(dev)
    N = 30000
    pos = rng.uniform(-1, 1, (N, 3)).astype(np.float32)
    g = rng.normal(size=(N, 32)).astype(np.float32)
    pos_t = torch.from_numpy(pos).to(dev)
    desc = enc.descriptor(N, 1.0)
    ws = torch.empty(_lib.hashgrid_backward_workspace_bytes(desc), dtype=torch.uint8, device=dev)
    d = torch.full(tuple(enc.table.shape), 5.0, dtype=torch.float32, device=dev)
    _lib.call("hashgrid_encode_backward", [pos_t, torch.from_numpy(g).to(dev), d, ws], desc)
    dt = d.cpu().numpy().astype(np.float64)
    want = _c_backward(enc, pos, g)
    absw = _c_backward(enc, pos, np.abs(g))
    assert (dt[absw == 0] == 0).all()
    assert (np.abs(dt - want) <= 1e-3 * absw + 1e-6).all()
    assert np.abs(dt - want).max() > 0  # the f16 rounding is visible: this is not the f32 path
    g[5, 7] = 1e6  # past 65504 once weighted by anything above 0.066
    _lib.call("hashgrid_encode_backward", [pos_t, torch.from_numpy(g).to(dev), d, ws], desc)
    assert torch.isinf(d).any() and torch.isfinite(d).float().mean() > 0.999


def test_fp16_table_2pow22(dev):
    """The precision workload's larger table: T = 2^22 entries per level (39,474,024
    rows, levels 0-7 dense), f16.  Forward bit-exact against the oracle's f32
    restatement on the f16 values; the table gradient within the f16 bound of the
    float64 scatter (as test_fp16_table_backward), untouched rows 0."""
    from jaxngp_amd import _lib
    rng = np.random.default_rng(41)
    cfg = dict(L=16, T=2 ** 22, F=2, N_min=16, N_max=2048)
    enc = HashGridEncoder(**cfg, param_dtype=torch.float16, generator=torch.Generator().manual_seed(5)).to(dev)
    assert enc.levels.n_rows == 39474024 and enc.levels.first_hash_level == 8
    with torch.no_grad():
        enc.table.copy_(torch.from_numpy(rng.uniform(-1e-2, 1e-2, tuple(enc.table.shape)).astype(np.float16)))
    N = 2 ** 17
    pos = rng.uniform(-1, 1, (N, 3)).astype(np.float32)
    pos_t = torch.from_numpy(pos).to(dev)
    print(f"hashgrid f16 T=2^22: N={N}", flush=True)
    out, _ = enc(pos_t, 1.0)
    table32 = enc.table.detach().float().cpu().numpy()
    np.testing.assert_array_equal(out.detach().cpu().numpy(), _c_forward(enc, pos, table32))
    del table32
    g = rng.normal(size=(N, 32)).astype(np.float32)
    desc = enc.descriptor(N, 1.0)
    ws = torch.empty(_lib.hashgrid_backward_workspace_bytes(desc), dtype=torch.uint8, device=dev)
    d = torch.full(tuple(enc.table.shape), 5.0, dtype=torch.float32, device=dev)
    _lib.call("hashgrid_encode_backward", [pos_t, torch.from_numpy(g).to(dev), d, ws], desc)
    dt = d.cpu().numpy().astype(np.float64)
    want = _c_backward(enc, pos, g)
    absw = _c_backward(enc, pos, np.abs(g))
    assert (dt[absw == 0] == 0).all()
    assert (np.abs(dt - want) <= 1e-3 * absw + 1e-6).all()


def test_fused_table_update_matches_gradient_then_adam(dev):
    """hashgrid_encode_backward_adam (the optimizer step taken in the table gradient's
    last pass) against hashgrid_encode_backward followed by adam_update on the same
    state, over three steps: 2^16 points (coarse slices summed in several parts, so
    the combine pass updates them), 20,001 points, and no points (every row takes a
    zero-gradient step).  Both use one element update; the gradient's f64 sums are
    taken in LDS-atomic order, so a row's f32 gradient may differ by its last bit
    between two runs, hence the tolerance; with no points the results are equal."""
    from jaxngp_amd import _lib
    rng = np.random.default_rng(31)
    enc = HashGridEncoder(**CONFIGS["l16_t2e19"], generator=torch.Generator().manual_seed(5)).to(dev)
    L, F = 16, 2
    with torch.no_grad():
        enc.table.uniform_(-1e-2, 1e-2)
    p1 = enc.table.detach().clone()
    m1 = torch.from_numpy(rng.normal(0, 1e-3, tuple(p1.shape)).astype(np.float32)).to(dev)
    v1 = torch.from_numpy(rng.uniform(0, 1e-5, tuple(p1.shape)).astype(np.float32)).to(dev)
    p2, m2, v2 = p1.clone(), m1.clone(), v1.clone()
    n = p1.numel()
    for t, N in ((1, 1 << 16), (2, 20001), (3, 0)):
        print(f"fused table update: step {t}, {N} points", flush=True)
        pos = torch.from_numpy(rng.uniform(-1, 1, (max(N, 1), 3)).astype(np.float32)).to(dev)[:N]
        g = torch.from_numpy(rng.normal(0, 1e-3, (L, max(N, 1), F)).astype(np.float32)).to(dev)[:, :N].contiguous()
        desc = enc.descriptor(N, 1.0, _lib.ENC_LEVEL_MAJOR)
        assert _lib.hashgrid_backward_adam_supported(desc)
        ws = torch.empty(_lib.hashgrid_backward_workspace_bytes(desc) if N else 256, dtype=torch.uint8, device=dev)
        adam = _lib.adam_descriptor(n, 1e-2, 0.9, 0.99, 1e-15, 1e-15, 0.9 ** t, 0.99 ** t, 0.0)
        d = torch.empty_like(p1)
        _lib.call("hashgrid_encode_backward", [pos, g, d, ws], desc)
        _lib.call("adam_update", [p1, d, m1, v1, torch.empty(0, device=dev)], adam)
        _lib.call("hashgrid_encode_backward_adam", [pos, g, p2, m2, v2, ws], _lib.hashgrid_adam_descriptor(desc, adam))
        torch.cuda.synchronize()
        for a, b, name in ((p2, p1, "params"), (m2, m1, "m"), (v2, v1, "v")):
            if N == 0:
                assert torch.equal(a, b), name
            else:
                torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-9, msg=name)
        same = (p2 == p1).float().mean().item()
        print(f"  params equal bit for bit: {same:.6f}", flush=True)
        assert same > 0.999


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("n, L", [((3 << 15) - 1, 16), (3 << 15, 16), ((3 << 15) + 65, 5), (1 << 18, 16)])
def test_point_major_gradient_on_both_sides_of_the_transpose(dev, n, L, half):
    """The table gradient of a point-major gradient, copied level-major first from 98,304 points
    on, against the same gradient given level-major: the same f64 sums up to the order of
    entries, rounded to f32 at most a few times (1e-6 of the largest row)."""
    from jaxngp_amd import _lib
    enc = HashGridEncoder(L=L, T=1 << 15, F=2, N_min=16, N_max=512, generator=torch.Generator().manual_seed(3))
    if half:
        enc.table.data = enc.table.data.half()
    enc = enc.to(dev)
    g = torch.Generator(device=dev).manual_seed(n)
    pos = torch.rand(n, 3, generator=g, device=dev) * 2 - 1
    lm = torch.randn(L, n, 2, generator=g, device=dev)
    got = []
    for layout, grad in ((0, lm.permute(1, 0, 2).reshape(n, 2 * L).contiguous()), (1, lm)):
        d = enc.descriptor(n, 1.0, layout)
        ws = torch.empty(_lib.hashgrid_backward_workspace_bytes(d), dtype=torch.uint8, device=dev)
        out = torch.empty(enc.table.shape, device=dev)
        _lib.call("hashgrid_encode_backward", [pos, grad, out, ws], d)
        got.append(out)
    assert (got[0] - got[1]).abs().max() <= 1e-6 * got[1].abs().max()


@pytest.mark.parametrize("n, T", [(0, 1 << 15), (1, 1 << 15), (1000, 1 << 19), (77_777, 1 << 15), (130_000, 1 << 19)])
def test_f16_rows_equal_the_cast_of_f32_rows(dev, n, T):
    """hashgrid_encode_backward_f16 against a cast of hashgrid_encode_backward's rows: no points,
    slices in one part, cut slices and both kinds of launches.  The f32 sums may differ in
    their last bits (the order of an f64 sum), so at most one f16 step, in few rows."""
    from jaxngp_amd import _lib
    enc = HashGridEncoder(L=16, T=T, F=2, N_min=16, N_max=2048, generator=torch.Generator().manual_seed(3))
    enc.table.data = enc.table.data.half()
    enc = enc.to(dev)
    g = torch.Generator(device=dev).manual_seed(n)
    pos = torch.rand(n, 3, generator=g, device=dev) * 2 - 1
    grad = torch.randn(n, 32, generator=g, device=dev)
    if n > 1:
        grad[0] = 1e6  # past f16: inf in both
    d = enc.descriptor(n, 1.0)
    assert _lib.hashgrid_backward_f16_supported(d)
    ws = torch.empty(_lib.hashgrid_backward_workspace_bytes(d), dtype=torch.uint8, device=dev)
    out = [torch.full(enc.table.shape, 3.0, dtype=dt, device=dev) for dt in (torch.float32, torch.float16)]
    _lib.call("hashgrid_encode_backward", [pos, grad, out[0], ws], d)
    _lib.call("hashgrid_encode_backward_f16", [pos, grad, out[1], ws], d)
    want, got = out[0].half(), out[1]
    apart = (want.view(torch.int16).int() - got.view(torch.int16).int()).abs()
    assert int(apart.max()) <= 1 and float((apart > 0).float().mean()) < 1e-3
    assert n < 2 or bool(torch.isinf(got).any())
