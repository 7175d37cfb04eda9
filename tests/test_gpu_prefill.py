"""GPU parity of the mxfp4 prefill GEMM (block-scaled MFMA over a direct-to-LDS ring) and
of the bf16-in gemm_nt_q_mxfp4a16 row, through the C ABI on guarded operands.

gemm_nt_q_mxfp4 (e4m3 + f32 a_scale per 128) is held to the per-element bound of
tests/test_gpu_gemm.py against oracle.quant_dot_mxfp4a8 at shapes that walk every tile
edge: ragged M and N, one K step, odd and even step counts, every tile width the planner
picks.

gemm_nt_q_mxfp4a16 has no reference counterpart.  Its two stages are checked apart:
  * the mxfp8 quantiser (bf16 -> e4m3 + E8M0 per 32) must leave in the launch scratch
    exactly the bytes of oracle.quant_act_mxfp8, edge values included (zeros, NaN,
    +-inf, bf16 subnormals, the largest finite bf16, rounding ties);
  * the GEMM must match oracle.dot_mx8_mxfp4 on those codes within
    |y - y_oracle| <= ulp_bf16 + 2*K*2^-24*S + 2^-10*S8 (S8 with the per-32 scales).
"""
import numpy as np
import pytest
import torch

import libr3d_amd as R
from libr3d_amd import synth
import oracle as O

pytestmark = pytest.mark.gpu

MX_TILE, A16 = "gemm_nt_q_mxfp4", "gemm_nt_q_mxfp4a16"


def _gu():
    from tests import gpu_util
    return gpu_util


def _mx_case(M, N, K, seed):
    rng = np.random.default_rng(seed)
    A = synth.random_e4m3_codes((M, K), rng)
    AS = (0.001 + 0.01 * rng.random((M, K // 128))).astype(np.float32)
    B = rng.integers(0, 256, size=(N, K // 2), dtype=np.uint8)
    BS = rng.integers(115, 140, size=(N, K // 32)).astype(np.uint8)
    return A, AS, B, BS


# every tile width the planner picks (bn 256/224/192/128) shows up across these N
@pytest.mark.parametrize("M,N,K", [(17, 300, 128), (128, 256, 256), (129, 448, 384),
                                   (300, 700, 640), (512, 1000, 1152), (260, 64, 512),
                                   (1000, 2176, 256)])
def test_mxfp4a8_prefill_shapes(gpu, M, N, K):
    gu = _gu()
    A, AS, B, BS = _mx_case(M, N, K, M * 7 + N + K)
    rc, Y, guards = gu.run_row(MX_TILE, "mxfp4a8", A, AS, B, BS, M, N, K, gpu)
    assert rc == R.RAD_OK and guards
    Yr, Yf, S = O.quant_dot_mxfp4a8(A, AS, B, BS, nthreads=16)
    S8 = O.group8_mag("mxfp4a8", A, AS, B, BS, nthreads=16)
    c = gu.compare(Y, Yr, Yf, S, K, S8)
    assert c["sentinel_left"] == 0, c
    assert c["nan_mismatch"] == 0 and c["inf_mismatch"] == 0, c
    assert c["max_viol"] <= 1.0, c
    assert c["rel_l2"] <= 3e-2, c


def run_a16(X, B, BS, M, N, K, dev, scratch_bytes=None):
    """Launch gemm_nt_q_mxfp4a16 on guarded operands; returns (rc, Y, Q, SX, guards_ok)."""
    gu = _gu()
    gX, gB, gBS = gu.Guarded(X, dev), gu.Guarded(B, dev), gu.Guarded(BS, dev)
    gY = gu.y_buffer(M, N, dev)
    ops = R.GemmOperands(gX.t, None, gB.t, gBS.t, gY.t, dtype="mxfp4a16", N=N, K=K,
                         group=32, M=M)
    need = R.row_scratch_bytes(A16, ops)
    assert need == ((M * K + 255) // 256) * 256 + M * (K // 32)
    nbytes = need if scratch_bytes is None else scratch_bytes
    gS = gu.Guarded(np.zeros(max(nbytes, 1), np.uint8), dev, fill=0x5A)
    ops.set_scratch(gS.t, nbytes)
    rc = R.launch_row(A16, ops, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    Y = gY.t.cpu().numpy().view(np.uint16).reshape(M, N)
    raw = gS.t.cpu().numpy()
    qb = ((M * K + 255) // 256) * 256
    Q = raw[:M * K].reshape(M, K) if nbytes >= need else None
    SX = raw[qb:qb + M * (K // 32)].reshape(M, K // 32) if nbytes >= need else None
    ok = all(g.guards_intact() for g in (gX, gB, gBS, gY, gS))
    return rc, Y, Q, SX, ok


def _bf16_acts(M, K, seed, edges=False):
    rng = np.random.default_rng(seed)
    X = synth.bf16_bits(rng.standard_normal((M, K)).astype(np.float32))
    if edges:
        X = X.copy()
        X[0, :32] = 0                                          # all-zero block -> e = 0
        X[0, 32:64] = 0x8000                                   # -0 block
        X[1, 5] = 0x7FC0                                       # NaN (never the max)
        X[1, 40] = 0x7F80                                      # +inf block -> e = 0, clamps
        X[1, 70] = 0xFF80                                      # -inf
        X[2, :32] = np.arange(1, 33, dtype=np.uint16)          # bf16 subnormals only
        X[2, 32:64] = 0x7F7F                                   # largest finite bf16
        X[3, :32] = synth.bf16_bits(np.float32(448.0) * np.ones(32, np.float32))
        X[3, 0] = synth.bf16_bits(np.array([464.0], np.float32))[0]   # above the range
        X[4, :32] = synth.bf16_bits((np.arange(32) - 16).astype(np.float32) * 2.0 ** -10)
        X[5, :32] = synth.bf16_bits(np.float32(2.0 ** -133) * np.ones(32, np.float32))
    return X


@pytest.mark.parametrize("edges", [False, True])
def test_mxfp4a16_quantiser_bit_exact(gpu, edges):
    M, N, K = 37, 64, 384
    X = _bf16_acts(M, K, 5 + edges, edges)
    B, BS = synth.mxfp4_weights(N, K, 6)
    rc, Y, Q, SX, ok = run_a16(X, B, BS, M, N, K, gpu)
    assert rc == R.RAD_OK and ok
    Qr, SXr = O.quant_act_mxfp8(X)
    assert np.array_equal(SX, SXr), np.argwhere(SX != SXr)[:8]
    assert np.array_equal(Q, Qr), np.argwhere(Q != Qr)[:8]


@pytest.mark.parametrize("M,N,K", [(1, 128, 128), (17, 200, 256), (256, 512, 1024),
                                   (300, 700, 640), (513, 1000, 1152), (64, 2176, 384)])
def test_mxfp4a16_gemm(gpu, M, N, K):
    gu = _gu()
    X = _bf16_acts(M, K, M + N + K)
    B, BS = synth.mxfp4_weights(N, K, M + 3)
    rc, Y, Q, SX, ok = run_a16(X, B, BS, M, N, K, gpu)
    assert rc == R.RAD_OK and ok
    Qr, SXr = O.quant_act_mxfp8(X)
    assert np.array_equal(Q, Qr) and np.array_equal(SX, SXr)
    Yr, Yf, S = O.dot_mx8_mxfp4(Qr, SXr, B, BS, nthreads=16)
    S8 = O.group8_mag("mxfp4a16", Qr, SXr, B, BS, nthreads=16)
    c = gu.compare(Y, Yr, Yf, S, K, S8)
    assert c["sentinel_left"] == 0, c
    assert c["nan_mismatch"] == 0 and c["inf_mismatch"] == 0, c
    assert c["max_viol"] <= 1.0, c
    assert c["row_rel_l2_max"] <= 2.0 ** -8, c


def test_mxfp4a16_short_scratch_refused(gpu):
    M, N, K = 40, 64, 256
    X = _bf16_acts(M, K, 9)
    B, BS = synth.mxfp4_weights(N, K, 10)
    rc, Y, _, _, ok = run_a16(X, B, BS, M, N, K, gpu, scratch_bytes=M * K)
    assert rc == R.RAD_E_UNSUPPORTED and ok
    assert np.all(Y == _gu().Y_SENTINEL)                    # nothing launched


F8_WIDE = [  # M, N, K, scratch, the tile's tokens, chunks: the fp8a8 wide tile, whole K and split
    (1030, 8200, 128, None, 256, 1),      # one step, six live tokens in the last tile, ragged N
    (1030, 8448, 256, None, 256, 1),      # two steps
    (300, 21700, 384, None, 128, 1),      # an odd step count, ragged M and N
    (144, 300, 21504, "hook", 128, 28),   # split: the least M, a ragged N past one tile
    (260, 514, 5376, "hook", 128, 14),    # split, N off a multiple of 4
    (513, 300, 8192, "hook", 128, 16),    # split, one live token in the last tile
    (513, 3073, 13568, "hook", 256, 6),   # split of the larger tile: one live token and one live
]                                         # row in the last ones, a shorter last chunk


@pytest.mark.parametrize("scales", ["block", "channel", "vary", "late"])
@pytest.mark.parametrize("M,N,K,scratch,bm,kc", F8_WIDE)
def test_fp8_wide_tile(gpu, M, N, K, scratch, bm, kc, scales):
    """The wide tile at its edges, on both scale grids; on the per-row grid with one scale a row
    (applied once after the walk), with scales that vary everywhere, and with one row's scale
    that differs in its last group alone (that row's tile must take the per-group walk)."""
    from tests.test_gpu_gemm import F8_TILE, _check, _f8_case
    rblk = 128 if scales == "block" else 1
    A, AS, B, BS = _f8_case(M, N, K, M + N + K, rblk)
    if scales in ("channel", "late"):
        BS = np.repeat(BS[:, :1], K // 128, axis=1).copy()
    if scales == "late":
        BS[N - 1, -1] += 0x80                              # twice as large
    A, AS, B, BS = (np.ascontiguousarray(t) for t in (A, AS, B, BS))
    g = _f8_geom(M, N, K, rblk, scratch)
    assert (g["bm"], g.get("kc", "1")) == (str(bm), str(kc)), g
    if M * N * K < 1 << 33:
        _check(F8_TILE, "fp8a8", A, AS, B, BS, M, N, K, gpu, rblk=rblk, scratch=scratch)
        return
    gu = _gu()
    rc, Y, ok = gu.run_row(F8_TILE, "fp8a8", A, AS, B, BS, M, N, K, gpu, scratch=scratch)
    assert rc == R.RAD_OK and ok and (Y != gu.Y_SENTINEL).any(axis=0).all()
    for lo, hi in _ends(N):                                # the first and last rows' columns
        b = BS[lo // rblk:-(-hi // rblk)]
        Yr, Yf, S = O.quant_dot_fp8a8(A, AS, B[lo:hi], b, rblk, nthreads=16)
        S8 = O.group8_mag("fp8a8", A, AS, B[lo:hi], b, rblk, nthreads=16)
        _within(gu.compare(np.ascontiguousarray(Y[:, lo:hi]), Yr, Yf, S, K, S8))


def _ends(N):
    return (0, 256), ((N - 200) // 128 * 128, N)


def _within(c):
    assert c["sentinel_left"] == 0 and c["nan_mismatch"] == 0 and c["inf_mismatch"] == 0, c
    assert c["max_viol"] <= 1.0, c


def _f8_geom(M, N, K, rblk, scratch):
    """describe's fields of a launch that the wide tile must take."""
    rows = N if rblk == 1 else (N + 127) // 128
    z = lambda *s, dt=torch.uint8: torch.zeros(s, dtype=dt)
    ops = R.GemmOperands(z(M, K), z(M, K // 128, dt=torch.float32), z(N, K),
                         z(rows, K // 128, dt=torch.int16), z(M, N, dt=torch.int16),
                         dtype="fp8a8", N=N, K=K)
    if scratch:
        ops.set_scratch(z(64), R.row_scratch_bytes("gemm_nt_q_fp8a8", ops))
    d = R.describe("gemm_nt_q_fp8a8", ops)[1]
    assert ("kernel=f8wide" if scratch else "wide=") in d, d
    return dict(f.split("=", 1) for f in d.split() if "=" in f)


@pytest.mark.parametrize("bad", [0x7F80, 0x7FC0])
def test_fp8_wide_tile_non_finite_row_scale(gpu, bad):
    """A row whose scale is Inf or NaN in every group is one scale a row, but its sum is not
    sum(D * sa) * sb: it takes the per-group walk, NaN and Inf classes as the oracle's."""
    from tests.test_gpu_gemm import F8_TILE, _f8_case
    from tests import gpu_util as gu
    M, N, K = 500, 2050, 5376
    A, AS, B, BS = _f8_case(M, N, K, 5, 1)
    BS = np.repeat(BS[:, :1], K // 128, axis=1).copy()
    BS[700, :] = bad
    rc, Y, ok = gu.run_row(F8_TILE, "fp8a8", A, AS, B, BS, M, N, K, gpu, scratch="hook")
    assert rc == R.RAD_OK and ok
    rows = slice(640, 768)                                 # the row's neighbours too
    Yr, Yf, S = O.quant_dot_fp8a8(A, AS, B[rows], BS[rows], 1, nthreads=16)
    S8 = O.group8_mag("fp8a8", A, AS, B[rows], BS[rows], 1, nthreads=16)
    c = gu.compare(np.ascontiguousarray(Y[:, rows]), Yr, Yf, S, K, S8)
    assert c["nan_mismatch"] == 0 and c["inf_mismatch"] == 0 and c["max_viol"] <= 1.0, c


@pytest.mark.parametrize("M,N,K,scratch", [(300, 21700, 384, None), (1030, 8448, 256, None),
                                           (260, 514, 5376, "hook")])
def test_fp8_wide_tile_large_token_scale(gpu, M, N, K, scratch):
    """One scale a row, a token scale of 1e31 on codes of 448: every group's D * sa is finite
    (2.6e38) and any two overflow, but the rows' 1e-10 scales bring the per-group products to
    2.6e28.  The result is the per-group order's: finite, within the bound."""
    from tests.test_gpu_gemm import F8_TILE, _check, _f8_case
    A, AS, B, BS = _f8_case(M, N, K, M + K, 1)
    BS = np.repeat(BS[:, :1], K // 128, axis=1).copy()
    for m in (7, M - 1):
        A[m], AS[m] = 0x7E, 1e31
    for n in (3, 300, N - 1):
        B[n], BS[n] = 0x7E, synth.bf16_bits(np.array([1e-10], np.float32))[0]
    _f8_geom(M, N, K, 1, scratch)
    _, Y = _check(F8_TILE, "fp8a8", A, AS, B, BS, M, N, K, gpu, scratch=scratch)
    assert np.isfinite(O.bf16_to_f32(Y)[:, [3, 300, N - 1]]).all()


MX_SPLIT = [  # M, N, K, the tile's tokens, chunks
    (144, 300, 8192, 128, 16), (260, 514, 5376, 128, 14), (513, 130, 6144, 128, 16),
    (385, 3001, 8192, 256, 5)]            # 128 x 256: one live token, a shorter last chunk


def _mx_geom(row, ops, M, N, bm, kc):
    g = dict(f.split("=", 1) for f in R.describe(row, ops)[1].split() if "=" in f)
    assert (g["arm"], g["bn"], g["bm"], g["kc"]) == ("splitk", "128", str(bm), str(kc)), g
    assert g["partials"] == str(4 * kc * M * N)


@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("M,N,K,bm,kc", MX_SPLIT)
def test_mxfp4a8_prefill_splitk(gpu, M, N, K, bm, kc, special):
    """K split past 128 tokens on the e2m1 tiles (ragged M and N, N off a multiple of 4, one
    live token in the last tile), against the bar of the unsplit tiles; a scratch one byte
    short runs those.  special: NaN codes, token scales and weight scales in the first and the
    last chunk.  (Not Inf token scales: the oracle applies them to each 32-wide block, the MFMA
    to a group's sum, and Inf - Inf is NaN in the former alone, split or not.)"""
    gu = _gu()
    A, AS, B, BS = _mx_case(M, N, K, M + N + K)
    if special:
        A[3, 5], A[M - 1, K - 1] = 0x7F, 0xFF
        AS[7, 2], AS[11, -1] = np.nan, np.nan
        BS[2, 1], BS[N - 1, -1] = 0xFF, 0xFF
    z = lambda *s, dt=torch.uint8: torch.zeros(s, dtype=dt)
    ops = R.GemmOperands(z(M, K), z(M, K // 128, dt=torch.float32), z(N, K // 2), z(N, K // 32),
                         z(M, N, dt=torch.int16), dtype="mxfp4a8", N=N, K=K)
    need = R.row_scratch_bytes(MX_TILE, ops)
    assert need == 4 * kc * M * N
    ops.set_scratch(z(64), need)
    _mx_geom(MX_TILE, ops, M, N, bm, kc)
    for scratch in ("hook", None):
        rc, Y, guards = gu.run_row(MX_TILE, "mxfp4a8", A, AS, B, BS, M, N, K, gpu, scratch=scratch)
        assert rc == R.RAD_OK and guards
        for lo, hi in _ends(N) if N > 1024 else ((0, N),):
            Yr, Yf, S = O.quant_dot_mxfp4a8(A, AS, B[lo:hi], BS[lo:hi], nthreads=16)
            S8 = O.group8_mag("mxfp4a8", A, AS, B[lo:hi], BS[lo:hi], nthreads=16)
            c = gu.compare(np.ascontiguousarray(Y[:, lo:hi]), Yr, Yf, S, K, S8)
            _within(c)
            assert c["rel_l2"] <= 3e-2, c


@pytest.mark.parametrize("M,N,K,bm,kc", MX_SPLIT)
def test_mxfp4a16_prefill_splitk(gpu, M, N, K, bm, kc):
    """The same on the bf16-in row, whose hook asks for the planes past the quantised
    activations; with the activations' bytes alone, or one byte short of both, it runs
    unsplit."""
    gu = _gu()
    X = _bf16_acts(M, K, M + N + K)
    B, BS = synth.mxfp4_weights(N, K, M + 3)
    Qr, SXr = O.quant_act_mxfp8(X)
    base = ((M * K + 255) // 256) * 256 + M * (K // 32)
    gX, gB, gBS = gu.Guarded(X, gpu), gu.Guarded(B, gpu), gu.Guarded(BS, gpu)
    for short in (None, 1, 0):                             # whole, one byte short, no planes
        gY = gu.y_buffer(M, N, gpu)
        ops = R.GemmOperands(gX.t, None, gB.t, gBS.t, gY.t, dtype="mxfp4a16", N=N, K=K, group=32,
                             M=M)
        need = R.row_scratch_bytes(A16, ops)
        assert need - (base + 255) // 256 * 256 == 4 * kc * M * N
        nbytes = need if short is None else need - 1 if short else base
        gS = gu.Guarded(np.zeros(nbytes, np.uint8), gpu, fill=0x5A)
        ops.set_scratch(gS.t, nbytes)
        if short is None:
            _mx_geom(A16, ops, M, N, bm, kc)
        else:
            assert "arm=prefill" in R.describe(A16, ops)[1]
        rc = R.launch_row(A16, ops, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert rc == R.RAD_OK and all(g.guards_intact() for g in (gX, gB, gBS, gY, gS))
        raw = gS.t.cpu().numpy()
        assert np.array_equal(raw[:M * K].reshape(M, K), Qr)
        Y = gY.t.cpu().numpy().view(np.uint16).reshape(M, N)
        for lo, hi in _ends(N) if N > 1024 else ((0, N),):
            Yr, Yf, S = O.dot_mx8_mxfp4(Qr, SXr, B[lo:hi], BS[lo:hi], nthreads=16)
            S8 = O.group8_mag("mxfp4a16", Qr, SXr, B[lo:hi], BS[lo:hi], nthreads=16)
            c = gu.compare(np.ascontiguousarray(Y[:, lo:hi]), Yr, Yf, S, K, S8)
            _within(c)
            assert c["row_rel_l2_max"] <= 2.0 ** -8, c
