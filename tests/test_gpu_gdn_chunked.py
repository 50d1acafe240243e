"""GPU checks of the chunked prefill form of the delta rule (q27h_gdn_step_chunked through the C ABI): o and the
final state against the sequential CPU oracle (itself pinned bit for bit against the sequential GPU kernel and by a
float64 recurrence) and against a float64 recurrence; plane semantics bit for bit (only the other of planes 0 / 1 is
written).

Tolerance, per 128-value vector (one (token, head) row of o, one state column of a head), so that a wrong block fails
on its own whatever the other heads hold: |got - want| <= RTOL * A for every value, A the vector's largest magnitude.
RTOL is 1e-5 (the north_star's fp32 bar) against a float64 recurrence, and 2e-5 against the sequential float32 oracle
(both float32 forms are within 1e-5 of the exact values). Relative 1e-5 per value is not a bar that float32 can meet
here: o's small values are differences of larger terms, and the sequential float32 order of the reference itself is
off the float64 result by up to 6.6e-5 relative on values above 1/64 of their vector's maximum (M = 2048). The
per-value figures of both forms are printed beside each check."""
import sys

import numpy as np
import pytest

import cfgdata as cd

pytestmark = pytest.mark.gpu

SCALE = np.float32(1.0 / np.sqrt(128.0))
RTOL_F64 = 1e-5   # against the float64 recurrence
RTOL_SEQ = 2e-5   # against the sequential float32 oracle
FLOOR = 2.0 ** -6  # values reported per value: those above FLOOR of their vector's maximum


def say(msg):
    print(f"[gpu-gdn-chunked] {msg}", flush=True)
    sys.stdout.flush()


def _run(q27, dev, x, stride, g, beta, planes, in_plane, H, HK, T):
    import torch

    dx = torch.from_numpy(x).to(dev)
    dp = torch.from_numpy(planes).to(dev)
    pin = torch.tensor([in_plane], dtype=torch.int32, device=dev)
    o = torch.full((max(T, 1) * H * 128,), float("nan"), device=dev)
    q27.ops.gdn_step_chunked(dx, dx[HK * 128:], dx[2 * HK * 128:], stride, torch.from_numpy(g).to(dev),
                             torch.from_numpy(beta).to(dev), dp, pin, o, H, HK, T, float(SCALE))
    torch.cuda.synchronize()
    return o.cpu().numpy()[: T * H * 128], dp.cpu().numpy()


def _close(got, want, what, rtol=RTOL_SEQ):
    """Per 128-value vector: |got - want| <= rtol * (the vector's largest |want|). Returns the largest error relative
    to its vector's maximum; prints it with the largest per-value relative error of values above FLOOR of it."""
    assert np.all(np.isfinite(got)), f"{what}: non-finite values"
    g = got.astype(np.float64).reshape(-1, 128)
    w = want.astype(np.float64).reshape(-1, 128)
    err = np.abs(g - w)
    vmax = np.abs(w).max(1, keepdims=True)
    bad = np.argwhere(err > rtol * vmax)
    rel_blk = (err / np.where(vmax > 0, vmax, 1)).max()
    big = np.abs(w) >= FLOOR * vmax
    rel_el = (err[big] / np.abs(w[big])).max() if big.any() else 0.0
    say(f"{what}: max error / vector max {rel_blk:.2e} (bound {rtol:g}); max relative error of values >= "
        f"{FLOOR} x max {rel_el:.2e}")
    assert bad.size == 0, (f"{what}: {len(bad)} values outside the bound; first vector {bad[0][0]} index {bad[0][1]}: "
                           f"{g[tuple(bad[0])]!r} vs {w[tuple(bad[0])]!r} (vector max {vmax[bad[0][0], 0]:.3e})")
    return rel_blk

def _f64_recurrence(x, stride, g, beta, planes, in_plane, H, HK, T):
    """The delta rule in float64 (delta = (v - e^g S^T k) beta, S <- e^g S + k delta^T, o = scale S^T q)."""
    S = planes.reshape(4, H, 128, 128)[in_plane].astype(np.float64).transpose(0, 2, 1).copy()  # [h][i][col]
    X = x.reshape(T, stride).astype(np.float64)
    kh = np.arange(H) % HK
    o = np.empty((T, H, 128))
    for t in range(T):
        q = X[t, : HK * 128].reshape(HK, 128)[kh]
        k = X[t, HK * 128: 2 * HK * 128].reshape(HK, 128)[kh]
        v = X[t, 2 * HK * 128:].reshape(H, 128)
        e = np.exp(g[t * H: (t + 1) * H].astype(np.float64))[:, None]
        kv = np.einsum("hi,hic->hc", k, S)
        d = (v - e * kv) * beta[t * H: (t + 1) * H].astype(np.float64)[:, None]
        S = e[:, :, None] * S + k[:, :, None] * d[:, None, :]
        o[t] = np.einsum("hi,hic->hc", q, S) * float(SCALE)
    return o.reshape(-1), S.transpose(0, 2, 1).reshape(-1)


@pytest.mark.parametrize("M,in_plane", [(2048, 0), (333, 1), (64, 0), (63, 3), (40, 2), (32, 1), (17, 3), (16, 1), (5, 0),
                                        (1, 1)])
def test_gdn_chunked_vs_sequential_oracle(q27, oracle, dev, M, in_plane):
    H, HK = cd.HV, cd.KH
    say(f"gdn chunked M={M} in_plane={in_plane}")
    x, stride, g, beta, planes = cd.gdn_inputs(cd.rng(200 + M), M)
    got_o, got_p = _run(q27, dev, x, stride, g, beta, planes, in_plane, H, HK, M)
    want_o, want_p = oracle.gdn_step(x, x[HK * 128:], x[2 * HK * 128:], stride, g, beta, planes, in_plane, H, HK, M,
                                     SCALE, False, True)
    out = 1 if in_plane == 0 else 0
    n = H * 128 * 128
    _close(got_o, want_o, f"o M={M}")
    _close(got_p[out * n:(out + 1) * n], want_p[out * n:(out + 1) * n], f"final state M={M}")
    for p in range(4):  # every other plane untouched, bit for bit
        if p != out:
            assert np.array_equal(got_p[p * n:(p + 1) * n].view(np.uint32), planes[p * n:(p + 1) * n].view(np.uint32)), p


@pytest.mark.parametrize("M", [8192, 333, 40])
def test_gdn_chunked_vs_float64(q27, dev, M):
    """M = 8192: 256 chunks, so the state carries the chunked form's rounding through a long sequence."""
    H, HK = cd.HV, cd.KH
    say(f"gdn chunked vs float64 M={M}")
    x, stride, g, beta, planes = cd.gdn_inputs(cd.rng(400 + M), M)
    got_o, got_p = _run(q27, dev, x, stride, g, beta, planes, 0, H, HK, M)
    want_o, want_s = _f64_recurrence(x, stride, g, beta, planes, 0, H, HK, M)
    n = H * 128 * 128
    _close(got_o, want_o, f"o vs float64 M={M}", RTOL_F64)
    _close(got_p[n:2 * n], want_s, f"state vs float64 M={M}", RTOL_F64)


def test_gdn_chunked_edge_values(q27, oracle, dev):
    """HK = H = 5, beta 0 / 1, g = 0 and -60 (decays that underflow inside a chunk), larger state values."""
    H, HK, M = 5, 5, 70
    say(f"gdn chunked edge H={H} HK={HK} M={M}")
    x, stride, g, beta, planes = cd.gdn_inputs(cd.rng(300), M, H, HK, planes_std=3.0)
    beta[::7] = 0
    beta[1::7] = 1
    g[::5] = 0
    g[2::5] = -60
    got_o, got_p = _run(q27, dev, x, stride, g, beta, planes, 0, H, HK, M)
    want_o, want_p = oracle.gdn_step(x, x[HK * 128:], x[2 * HK * 128:], stride, g, beta, planes, 0, H, HK, M, SCALE,
                                     False, True)
    n = H * 128 * 128
    _close(got_o, want_o, "edge o")
    _close(got_p[n:2 * n], want_p[n:2 * n], "edge state")
    f_o, f_s = _f64_recurrence(x, stride, g, beta, planes, 0, H, HK, M)
    _close(got_o, f_o, "edge o vs float64", RTOL_F64)
    _close(got_p[n:2 * n], f_s, "edge state vs float64", RTOL_F64)


def _run_step(q27, dev, x, stride, g, beta, planes, in_plane, H, HK, T):
    import torch

    dx = torch.from_numpy(x).to(dev)
    dp = torch.from_numpy(planes).to(dev)
    pin = torch.tensor([in_plane], dtype=torch.int32, device=dev)
    o = torch.full((max(T, 1) * H * 128,), float("nan"), device=dev)
    q27.ops.gdn_step(dx, dx[HK * 128:], dx[2 * HK * 128:], stride, torch.from_numpy(g).to(dev),
                     torch.from_numpy(beta).to(dev), dp, pin, o, H, HK, T, float(SCALE), False, flip=True)
    torch.cuda.synchronize()
    return o.cpu().numpy()[: T * H * 128], dp.cpu().numpy()


def test_gdn_step_prefill_dispatch(q27, oracle, dev):
    """gdn_step with flip: from 128 tokens on the chunked form (same bits as q27h_gdn_step_chunked), below it and in
    exact mode the sequential kernel (the checker's bits)."""
    H, HK = cd.HV, cd.KH
    prev = q27.ops.gdn_prefill_exact(False)
    try:
        for M in (2048, 128):
            say(f"gdn_step prefill dispatch M={M}")
            x, stride, g, beta, planes = cd.gdn_inputs(cd.rng(500 + M), M)
            got_o, got_p = _run_step(q27, dev, x, stride, g, beta, planes, 0, H, HK, M)
            ch_o, ch_p = _run(q27, dev, x, stride, g, beta, planes, 0, H, HK, M)
            assert np.array_equal(got_o.view(np.uint32), ch_o.view(np.uint32)), M
            assert np.array_equal(got_p.view(np.uint32), ch_p.view(np.uint32)), M
        for M, exact in ((127, False), (300, True)):
            say(f"gdn_step prefill sequential M={M} exact={exact}")
            q27.ops.gdn_prefill_exact(exact)
            x, stride, g, beta, planes = cd.gdn_inputs(cd.rng(600 + M), M)
            got_o, got_p = _run_step(q27, dev, x, stride, g, beta, planes, 1, H, HK, M)
            want_o, want_p = oracle.gdn_step(x, x[HK * 128:], x[2 * HK * 128:], stride, g, beta, planes, 1, H, HK, M,
                                             SCALE, False, True)
            assert np.array_equal(got_o.view(np.uint32), want_o.view(np.uint32)), M
            assert np.array_equal(got_p.view(np.uint32), want_p.view(np.uint32)), M
    finally:
        q27.ops.gdn_prefill_exact(prev)


@pytest.mark.parametrize("M,H,HK", [(672, 48, 16), (673, 48, 16), (70, 5, 2), (70, 3, 5)])
def test_gdn_chunked_prep_split(q27, dev, M, H, HK):
    """One preparing workgroup per value head up to 1024 of them (672 tokens of 48 heads: 1008), per key head beyond
    (673 tokens: 1056); a last set of value heads that covers only some key heads; more key heads than value heads."""
    say(f"gdn chunked prep split M={M} H={H} HK={HK}")
    x, stride, g, beta, planes = cd.gdn_inputs(cd.rng(900 + M + H), M, H, HK)
    got_o, got_p = _run(q27, dev, x, stride, g, beta, planes, 0, H, HK, M)
    want_o, want_s = _f64_recurrence(x, stride, g, beta, planes, 0, H, HK, M)
    n = H * 128 * 128
    _close(got_o, want_o, f"o vs float64 M={M} H={H} HK={HK}", RTOL_F64)
    _close(got_p[n:2 * n], want_s, f"state vs float64 M={M} H={H} HK={HK}", RTOL_F64)


@pytest.mark.parametrize("short,full,M,H,HK", [(672, 672, 673, 48, 16), (70, 64, 5472, 5, 2)])
def test_gdn_chunked_prep_split_same_bits(q27, dev, short, full, M, H, HK):
    """The preparing launch with one workgroup per value head (the first `short` tokens) and per key head (all M): the same
    bits of o in the full chunks that both batches share."""
    say(f"gdn chunked prep split {short} of {M} tokens H={H} HK={HK}")
    x, stride, g, beta, planes = cd.gdn_inputs(cd.rng(930 + M), M, H, HK)
    want, _ = _run(q27, dev, x, stride, g, beta, planes, 0, H, HK, M)
    got, _ = _run(q27, dev, x[: short * stride].copy(), stride, g[: short * H].copy(), beta[: short * H].copy(), planes, 0,
                  H, HK, short)
    n = full * H * 128
    assert np.array_equal(got[:n].view(np.uint32), want[:n].view(np.uint32))


@pytest.mark.parametrize("n", [1, 15, 16, 17, 31])
def test_gdn_chunked_ragged_rows_inside_a_larger_batch(q27, dev, n):
    """Every row behind the last token is NaN (x, g, beta): a last chunk of n tokens gives the bits of the compact batch,
    and the rows of o behind it are not written."""
    import torch

    H, HK, M, pad = 6, 2, 32 + n, 32
    say(f"gdn chunked ragged n={n}")
    x, W, g, beta, planes = cd.gdn_inputs(cd.rng(950 + n), M, H, HK)
    want_o, want_p = _run(q27, dev, x, W, g, beta, planes, 0, H, HK, M)
    dx, dg, db = (torch.cat([torch.from_numpy(a).to(dev), torch.full((pad * w,), float("nan"), device=dev)])
                  for a, w in ((x, W), (g, H), (beta, H)))
    dp = torch.from_numpy(planes).to(dev)
    pin = torch.zeros(1, dtype=torch.int32, device=dev)
    o = torch.full(((M + pad) * H * 128,), -7.0, device=dev)
    q27.ops.gdn_step_chunked(dx, dx[HK * 128:], dx[2 * HK * 128:], W, dg, db, dp, pin, o, H, HK, M, float(SCALE))
    torch.cuda.synchronize()
    got = o.cpu().numpy()
    assert np.array_equal(got[: M * H * 128].view(np.uint32), want_o.view(np.uint32))
    assert np.array_equal(dp.cpu().numpy().view(np.uint32), want_p.view(np.uint32))
    assert np.all(got[M * H * 128:] == -7.0)


@pytest.mark.parametrize("stride", [1 << 24, (1 << 24) + 4])
def test_gdn_chunked_wide_rows(q27, dev, stride):
    """Rows 2^24 floats apart (the last stride whose chunk 32-bit offsets reach) and farther (64-bit offsets): the bits of
    compact rows. 65 rows: a full chunk, a second one and a ragged one."""
    import torch

    H, HK, M = 2, 1, 65
    say(f"gdn chunked stride={stride}")
    x, W, g, beta, planes = cd.gdn_inputs(cd.rng(800), M, H, HK)
    want_o, want_p = _run(q27, dev, x, W, g, beta, planes, 0, H, HK, M)
    dx = torch.empty((M - 1) * stride + W, device=dev)
    dx.as_strided((M, W), (stride, 1)).copy_(torch.from_numpy(x).to(dev).view(M, W))
    dp = torch.from_numpy(planes).to(dev)
    pin = torch.zeros(1, dtype=torch.int32, device=dev)
    o = torch.full((M * H * 128,), float("nan"), device=dev)
    q27.ops.gdn_step_chunked(dx, dx[HK * 128:], dx[2 * HK * 128:], stride, torch.from_numpy(g).to(dev),
                             torch.from_numpy(beta).to(dev), dp, pin, o, H, HK, M, float(SCALE))
    torch.cuda.synchronize()
    assert np.array_equal(o.cpu().numpy().view(np.uint32), want_o.view(np.uint32))
    assert np.array_equal(dp.cpu().numpy().view(np.uint32), want_p.view(np.uint32))


def test_gdn_chunked_replays_in_hip_graph(q27, dev):
    """The chunked prefill (two launches, Tinv / M staged in o) captured in a HIP graph: every replay gives the eager
    launch's bits (no allocation, no host synchronisation, nothing left over from the previous replay)."""
    import torch

    H, HK, M = cd.HV, cd.KH, 300
    say(f"gdn chunked graph replay M={M}")
    x, stride, g, beta, planes = cd.gdn_inputs(cd.rng(700), M)
    want_o, want_p = _run(q27, dev, x, stride, g, beta, planes, 1, H, HK, M)
    dx, dg, db = (torch.from_numpy(a).to(dev) for a in (x, g, beta))
    p0 = torch.from_numpy(planes).to(dev)
    dp = p0.clone()
    pin = torch.ones(1, dtype=torch.int32, device=dev)
    o = torch.zeros(M * H * 128, device=dev)
    s = torch.cuda.Stream()
    gr = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        q27.ops.gdn_step_chunked(dx, dx[HK * 128:], dx[2 * HK * 128:], stride, dg, db, dp, pin, o, H, HK, M,
                                 float(SCALE))
        torch.cuda.synchronize()
        with torch.cuda.graph(gr, stream=s):
            q27.ops.gdn_step_chunked(dx, dx[HK * 128:], dx[2 * HK * 128:], stride, dg, db, dp, pin, o, H, HK, M,
                                     float(SCALE))
    for _ in range(3):
        dp.copy_(p0)
        o.fill_(float("nan"))
        torch.cuda.synchronize()
        gr.replay()
        torch.cuda.synchronize()
        assert np.array_equal(o.cpu().numpy().view(np.uint32), want_o.view(np.uint32)), "graph replay o"
        assert np.array_equal(dp.cpu().numpy().view(np.uint32), want_p.view(np.uint32)), "graph replay planes"


def test_gdn_chunked_downstream_int8(q27, oracle, dev):
    """How many int8 values of the next op (gated_rmsnorm_q8 of o, src/model.cu's order) differ between the chunked
    and the sequential prefill at M = 2048: a value differs only where o's rounding moves y / d across a half-integer,
    so a small share is expected; the count is reported and bounded, the scales of the blocks checked."""
    import torch

    H, HK, M = cd.HV, cd.KH, 2048
    say(f"gdn chunked vs sequential, downstream gated_rmsnorm_q8 int8 M={M}")
    x, stride, g, beta, planes = cd.gdn_inputs(cd.rng(800), M)
    ch_o, _ = _run(q27, dev, x, stride, g, beta, planes, 0, H, HK, M)
    prev = q27.ops.gdn_prefill_exact(True)
    try:
        sq_o, _ = _run_step(q27, dev, x, stride, g, beta, planes, 0, H, HK, M)
    finally:
        q27.ops.gdn_prefill_exact(prev)
    r = cd.rng(801)
    w = torch.from_numpy((1 + 0.1 * r.standard_normal(128)).astype(np.float32)).to(dev)
    z = torch.from_numpy(r.standard_normal(M * H * 128).astype(np.float32)).to(dev)
    out = []
    for o in (ch_o, sq_o):
        xq = torch.zeros(M * H * 128, dtype=torch.int8, device=dev)
        xd = torch.zeros(M * H * 4, device=dev)
        q27.ops.gated_rmsnorm_q8(torch.from_numpy(o).to(dev), w, z, xq, xd, M * H, cd.EPS)
        torch.cuda.synchronize()
        out.append((xq.cpu().numpy().astype(np.int32), xd.cpu().numpy()))
    dq = np.abs(out[0][0] - out[1][0])
    frac = np.count_nonzero(dq) / dq.size
    dscale = np.count_nonzero(out[0][1] != out[1][1]) / out[0][1].size
    say(f"int8 values differing: {np.count_nonzero(dq)} of {dq.size} ({frac:.2e}), max |diff| {dq.max()}; "
        f"fp16 block scales differing: {dscale:.2e}")
    assert dq.max() <= 1
    assert frac < 1e-3
