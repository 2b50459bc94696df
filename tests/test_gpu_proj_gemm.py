"""GPU parity of the hand-written grouped projection GEMM (kvp_proj_gemm)
against the oracle's nn.Linear (oracle/backbone.py: float64 of the same
bf16-rounded operands).

bf16 outputs: within one bf16 ulp of the wide result; fp32 outputs (plain or
accumulated into the existing values, the residual add of out_proj):
max-abs <= 1e-4. Rows past `rows` are never written.
"""

import numpy as np
import pytest
import torch

from kvpersist import _lib
from kvpersist import backbone as kb
from oracle import backbone as ob

DEV = "cuda"


def _bf16_close(got, want):
    got = np.asarray(got, np.float64)
    want = np.asarray(want, np.float64)
    bad = np.abs(got - want) > np.abs(want) * 2.0 ** -7 + 1e-5
    assert not bad.any(), (int(bad.sum()), got[bad][:4], want[bad][:4])


CASES = [
    # rows, K, N, groups, tile_n, out_dtype, accumulate, bias
    (1, 64, 256, 1, 256, 1, False, True),
    (300, 256, 256, 3, 128, 1, False, True),
    (1560, 1536, 1536, 3, 256, 1, False, True),
    (1560, 1536, 1536, 3, 128, 1, False, False),
    (257, 128, 384, 2, 128, 0, False, True),
    (1000, 1536, 1536, 1, 256, 0, True, True),
    # accumulate form, K of one chunk (residual loaded in the epilogue) and of
    # two (loaded during the first), ragged last row tile
    (130, 64, 128, 1, 128, 0, True, True),
    (257, 128, 256, 1, 128, 0, True, False),
    (1560, 1536, 1536, 1, 128, 0, True, True),
    (12480, 1536, 1536, 3, 256, 1, False, True),
    (12480, 1536, 1536, 3, 128, 1, False, True),
    (12480, 1536, 1536, 1, 128, 0, True, True),
]


@pytest.mark.gpu
@pytest.mark.parametrize("rows,K,N,groups,tile_n,out_dt,acc,bias", CASES)
def test_proj_gemm_matches_oracle(rows, K, N, groups, tile_n, out_dt, acc, bias):
    print(f"proj_gemm rows={rows} K={K} N={N} groups={groups} tile={tile_n} out={out_dt} "
          f"acc={acc}", flush=True)
    rng = np.random.default_rng(rows + K + N + groups)
    x = ob.round_bf16(rng.standard_normal((rows, K)).astype(np.float32))
    w = ob.round_bf16((0.02 * rng.standard_normal((groups * N, K))).astype(np.float32))
    b = (0.1 * rng.standard_normal(groups * N)).astype(np.float32) if bias else None
    odt = torch.bfloat16 if out_dt == 1 else torch.float32
    guard = 3
    y0 = rng.standard_normal((groups, rows + guard, N)).astype(np.float32)
    if out_dt == 1:
        y0 = ob.round_bf16(y0)
    ys = [torch.from_numpy(y0[g]).to(DEV).to(odt) for g in range(groups)]
    xd = torch.from_numpy(x).to(DEV).to(torch.bfloat16)
    wd = torch.from_numpy(w).to(DEV).to(torch.bfloat16)
    bd = None if b is None else torch.from_numpy(b).to(DEV)
    kb.proj_gemm(xd, wd, bd, [y[:rows] for y in ys], accumulate=acc, tile_n=tile_n)
    torch.cuda.synchronize()
    # the oracle on a bounded sample of rows for the largest case
    sample = np.arange(rows) if rows <= 2000 else np.unique(
        np.concatenate([np.arange(300), rng.choice(rows, 700, replace=False), [rows - 1]]))
    for g in range(groups):
        got = ys[g].float().cpu().numpy()
        assert np.array_equal(got[rows:], y0[g][rows:]), "rows past the end were written"
        want = ob.linear(x[sample], w[g * N:(g + 1) * N], None if b is None else
                         b[g * N:(g + 1) * N])
        if acc:
            want = want + y0[g][sample]
        if out_dt == 1:
            _bf16_close(got[sample], want)
        else:
            assert np.abs(got[sample] - want).max() <= 1e-4, g


def test_proj_gemm_rejects_unsupported_shapes(lib):
    """Shape errors are reported before any device work (runs without a GPU)."""
    assert lib.kvp_proj_gemm(16, 16, None, 16, None, None, 1, 4, 96, 256, 1, 0, 256, None) != 0
    assert "not supported" in _lib.last_error()
    assert lib.kvp_proj_gemm(16, 16, None, 16, None, None, 1, 4, 64, 192, 1, 0, 256, None) != 0
    assert lib.kvp_proj_gemm(16, 16, None, 16, None, None, 1, 4, 64, 256, 1, 1, 256, None) != 0
    assert "fp32" in _lib.last_error()
    assert lib.kvp_proj_gemm(16, 16, None, 16, None, None, 4, 4, 64, 256, 1, 0, 256, None) != 0
    assert lib.kvp_proj_gemm(16, 16, None, 16, None, None, 2, 4, 64, 256, 1, 0, 256, None) != 0
    assert lib.kvp_proj_gemm(16, 16, None, 16, None, None, 1, 4, 64, 256, 1, 0, 64, None) != 0


# fp32 operands on the tiled kernel: one and many K chunks of 32, one row, the
# edges of a 128-row tile, several feature tiles, both forms
@pytest.mark.gpu
@pytest.mark.parametrize("rows,K,N,acc,bias", [
    (1, 32, 128, False, True), (127, 64, 128, True, True), (128, 96, 256, False, False),
    (129, 32, 128, True, False), (1560, 1536, 1536, False, True), (300, 1536, 384, True, True),
])
def test_fp32_linear_tiled(rows, K, N, acc, bias):
    _check_fp32_linear(rows, K, N, acc, bias)


# short inner dimension: every K of the register kernel and its neighbours on
# the general one, rows around a wave's 16 and a block's 64, features around
# the block's 256 and a multiple of 4 or not
@pytest.mark.gpu
@pytest.mark.parametrize("rows,K,N,acc,bias", [
    (1, 4, 4, False, True), (15, 8, 252, False, False), (17, 12, 256, True, True),
    (65, 16, 260, False, True), (1560, 16, 1536, False, True), (63, 16, 258, True, True),
    (129, 20, 256, False, True), (64, 15, 256, False, True), (64, 16, 1024, True, False),
])
def test_fp32_linear_short_inner(rows, K, N, acc, bias):
    _check_fp32_linear(rows, K, N, acc, bias)


# the same where the register kernel is the one that runs: rows around a wave's
# 16 and a block's 64, column blocks that end after 64, 128, 252 and 44 features
@pytest.mark.gpu
@pytest.mark.parametrize("rows,K,N,acc,bias", [
    (64, 4, 4, False, True), (65, 8, 64, True, True), (79, 12, 252, False, False),
    (130, 16, 128, True, False), (81, 16, 512, False, True), (16385, 8, 300, True, True),
])
def test_fp32_linear_short_inner_kernel(lib, rows, K, N, acc, bias):
    assert lib.kvp_linear_kernel(0, 0, rows, K, N, 1, int(acc)) == 1
    _check_fp32_linear(rows, K, N, acc, bias)


def _check_fp32_linear(rows, K, N, acc, bias):
    print(f"fp32 linear rows={rows} K={K} N={N} acc={acc}", flush=True)
    rng = np.random.default_rng(rows + K + N)
    x = rng.standard_normal((rows, K)).astype(np.float32)
    w = (0.02 * rng.standard_normal((N, K))).astype(np.float32)
    b = (0.1 * rng.standard_normal(N)).astype(np.float32) if bias else None
    y0 = rng.standard_normal((rows + 3, N)).astype(np.float32)
    y = torch.from_numpy(y0).to(DEV)
    kb.linear(torch.from_numpy(x).to(DEV), torch.from_numpy(w).to(DEV),
              None if b is None else torch.from_numpy(b).to(DEV), y[:rows], accumulate=acc)
    torch.cuda.synchronize()
    got = y.cpu().numpy()
    assert np.array_equal(got[rows:], y0[rows:]), "rows past the end were written"
    want = ob.linear(x, w, b) + (y0[:rows] if acc else 0)
    # each value is a chain of at most K + 2 rounded fp32 additions of terms
    # whose magnitudes sum to |x| |w|^T + |b| + |y0|
    mag = np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T
    mag += (0 if b is None else np.abs(b)) + (np.abs(y0[:rows]) if acc else 0)
    assert (np.abs(got[:rows] - want) <= (K + 2) * 2.0 ** -24 * mag).all()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,heads", [(1, 1), (131, 3)])
def test_fp32_qkv_project_is_three_linears(rows, heads):
    """The grouped fp32 launch equals three single launches of its weight blocks, bit for bit."""
    D = 128 * heads
    print(f"fp32 qkv rows={rows} D={D}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(rows)
    x = torch.randn(rows, D, generator=g, device=DEV)
    w = 0.02 * torch.randn(3 * D, D, generator=g, device=DEV)
    b = torch.randn(3 * D, generator=g, device=DEV)
    ln_w, ln_b = torch.ones(D, device=DEV), torch.zeros(D, device=DEV)
    xn, q, k, v = (torch.empty(rows, D, device=DEV) for _ in range(4))
    kb.qkv_project(x, ln_w, ln_b, w, b, xn, q, k, v)
    for i, got in enumerate((q, k, v)):
        want = torch.empty(rows, D, device=DEV)
        kb.linear(xn, w[i * D:(i + 1) * D], b[i * D:(i + 1) * D], want)
        assert torch.equal(got, want), i


# tokens that end inside a tile of 320, 256 or 128, feature tiles that hold two
# groups and reach past the last one, one and several K chunks: the wide tiles for
# tile_n 256; so few chunks run 128 x 128 tiles for tile_n 128 (where it picks the
# wide ones: test_chosen_wide_tiles_match_oracle)
@pytest.mark.gpu
@pytest.mark.parametrize("rows,K,N,groups,tile_n,out_dt,acc,bias", [
    (12473, 64, 1408, 3, 128, 1, False, True),
    (12473, 192, 1536, 1, 128, 0, True, True),
    (12473, 128, 384, 3, 128, 0, False, False),
    (255, 128, 256, 3, 256, 1, False, True),
    (513, 64, 512, 1, 256, 0, True, True),
])
def test_wide_tiles_match_oracle(rows, K, N, groups, tile_n, out_dt, acc, bias):
    test_proj_gemm_matches_oracle(rows, K, N, groups, tile_n, out_dt, acc, bias)


# the same where a launch picks the wide tiles itself (K from 256, from 768 when it
# accumulates), with features past the last group and a wave's accumulators there
@pytest.mark.gpu
@pytest.mark.parametrize("rows,K,N,groups,out_dt,acc,kernel", [
    (12473, 256, 1408, 3, 1, False, 4), (12473, 256, 384, 3, 0, False, 3),
    (12473, 768, 1408, 1, 0, True, 4), (3117, 256, 1408, 3, 1, False, 3),
    (3117, 768, 4480, 1, 0, True, 3),
])
def test_chosen_wide_tiles_match_oracle(lib, rows, K, N, groups, out_dt, acc, kernel):
    assert lib.kvp_linear_kernel(1, out_dt, rows, K, N, groups, int(acc)) == kernel
    test_proj_gemm_matches_oracle(rows, K, N, groups, 128, out_dt, acc, True)


@pytest.mark.gpu
@pytest.mark.parametrize("out_dt,acc", [(1, False), (0, False), (0, True)])
def test_all_tiles_give_the_same_bits(lib, out_dt, acc):
    """The same rows through 256 x 320, 256 x 256 and 128 x 128 tiles."""
    rows, K, N, few = 12473, 768, 1536, 1500
    print(f"tiles bitwise out={out_dt} acc={acc}", flush=True)
    kernels = [lib.kvp_linear_kernel(1, out_dt, r, K, N, 1, int(acc)) for r in (rows, few)]
    assert kernels == [4, 2]
    g = torch.Generator(device=DEV).manual_seed(out_dt + 2 * acc)
    x = torch.randn(rows, K, generator=g, device=DEV).to(torch.bfloat16)
    w = (0.02 * torch.randn(N, K, generator=g, device=DEV)).to(torch.bfloat16)
    b = torch.randn(N, generator=g, device=DEV)
    odt = torch.bfloat16 if out_dt else torch.float32
    y0 = torch.randn(rows, N, generator=g, device=DEV).to(odt)
    outs = []
    for n, tile_n in ((rows, 128), (rows, 256), (few, 128)):
        y = y0.clone()
        kb.proj_gemm(x[:n], w, b, [y[:n]], accumulate=acc, tile_n=tile_n)
        outs.append(y)
    assert torch.equal(outs[0], outs[1])
    assert torch.equal(outs[0][:few], outs[2][:few]) and torch.equal(outs[2][few:], y0[few:])
