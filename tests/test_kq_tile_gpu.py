"""The k-quant tile GEMMs (M > 16) over the ways a call is cut: 32, 64 and 128-row tiles, whole,
split over K (scratch), cut in row quarters in the last round (no scratch), and whole and split
tiles of one call, row-major and in XCD order. Against the oracle's exact integer sums (reference
tests/test_gemm_q4k.py:430-528)."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import kquant as okq
from oracle import q4k as oq
from superl8_amd import _C, _lib

RANDOM = {4: oq.random_weights, 5: okq.q5k_random, 6: okq.q6k_random}
GEMV = {4: oq.gemv, 5: okq.q5k_gemv, 6: okq.q6k_gemv}
GEMM = {4: _C.gemm_q4k, 5: _C.gemm_q5k, 6: _C.gemm_q6k}


def _plan(fmt, M, N, K, scratch):
    """(rows of a tile, whole tiles, tiles split over K, their parts, tiles cut in quarters)"""
    p = (ctypes.c_int64 * 5)()
    _lib.call("sl8_gemm_kq_plan", fmt, M, N, K, int(scratch), p)
    return tuple(p)


def _kind(plan):
    rows, whole, split, _, cut = plan
    return rows, "cut" if cut else "mixed" if whole and split else "split" if split else "whole"


def _gemm(fmt, x_i8, xs, wd, scratch):
    if scratch:
        return GEMM[fmt](x_i8, xs, wd, torch.float32)
    M, K = x_i8.shape
    out = torch.full((M, wd.shape[0]), float("nan"), device=wd.device)
    _lib.call(f"sl8_gemm_q{fmt}k", x_i8.data_ptr(), xs.data_ptr(), wd.data_ptr(), out.data_ptr(),
              _lib.F32, M, wd.shape[0], K, _lib.stream_of(wd))
    return out


def _case(device, fmt, M, N, K):
    w = RANDOM[fmt](N, K, seed=M + N)
    g = torch.Generator(device="cpu").manual_seed(M)
    x_i8, xs = _C.quantize_i8_rowwise(torch.randn(M, K, generator=g).half().to(device))
    return w, torch.from_numpy(w).to(device), x_i8, xs


# (format, scratch, M, N, K) -> rows of a tile and how the tiles are cut on 256 CUs; ragged rows and
# columns, odd counts of super-blocks (uneven K parts). 17408 columns: 136 column tiles, XCD order;
# 16770: 132, row-major
CASES = [
    (4, True, 17, 40, 2304, (32, "split")), (4, True, 33, 130, 768, (32, "whole")),
    (4, True, 33, 4100, 3328, (64, "split")), (4, True, 100, 8250, 768, (64, "whole")),
    (4, True, 500, 8250, 1280, (64, "mixed")), (4, True, 500, 4100, 5120, (128, "split")),
    (4, True, 500, 12300, 768, (128, "whole")), (4, True, 500, 16770, 2304, (128, "mixed")),
    (4, True, 512, 17408, 5120, (128, "mixed")),
    (4, False, 17, 40, 2304, (64, "whole")), (4, False, 500, 4100, 5120, (128, "whole")),
    (4, False, 500, 16770, 2304, (128, "cut")), (4, False, 512, 17408, 2304, (128, "cut")),
    (5, True, 17, 40, 2304, (32, "split")), (5, True, 33, 130, 768, (32, "whole")),
    (5, True, 512, 4100, 2304, (32, "mixed")), (5, True, 33, 8250, 2304, (64, "split")),
    (5, True, 100, 8250, 768, (64, "whole")), (5, True, 700, 6100, 1280, (64, "mixed")),
    (5, True, 1500, 1000, 5120, (128, "split")), (5, True, 1000, 4100, 768, (128, "whole")),
    (5, True, 500, 16770, 2304, (128, "mixed")), (5, True, 512, 17408, 2304, (128, "mixed")),
    (5, False, 17, 40, 2304, (64, "whole")), (5, False, 500, 4100, 5120, (128, "whole")),
    (5, False, 500, 16770, 2304, (128, "cut")), (5, False, 512, 17408, 2304, (128, "cut")),
    (6, True, 17, 40, 2304, (32, "split")), (6, True, 33, 130, 768, (32, "whole")),
    (6, True, 129, 16770, 2304, (32, "mixed")), (6, True, 500, 130, 5120, (64, "split")),
    (6, True, 100, 8250, 768, (64, "whole")), (6, True, 512, 4100, 5120, (64, "mixed")),
    (6, True, 100, 4100, 3328, (128, "split")), (6, True, 1000, 4100, 768, (128, "cut")),
    (6, True, 500, 16770, 2304, (128, "mixed")), (6, True, 512, 17408, 2304, (128, "mixed")),
    (6, False, 500, 16770, 2304, (128, "cut")), (6, False, 512, 17408, 2304, (128, "cut")),
]


@pytest.mark.parametrize("fmt,scratch,M,N,K,kind", CASES)
def test_plan(fmt, scratch, M, N, K, kind):
    """The cases below run what they are there for (the plan needs no GPU; 256 CUs are assumed
    where there is none)."""
    assert _kind(_plan(fmt, M, N, K, scratch)) == kind


@pytest.mark.parametrize("fmt", [4, 5, 6])
def test_plan_covers_every_tile(fmt):
    for M in (17, 64, 65, 300, 512, 777, 2000):
        for N in (1, 130, 4096, 16770, 17408):
            for K in (256, 1280, 5120):
                for scratch in (True, False):
                    rows, whole, split, parts, cut = _plan(fmt, M, N, K, scratch)
                    assert whole + split + cut == -(-M // rows) * -(-N // 128)
                    assert 1 <= parts <= max(1, K // 512) and (parts > 1) == (split > 0)
                    assert not (split and not scratch) and not (cut and rows != 128)


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,scratch,M,N,K,kind", CASES)
def test_tiles(device, fmt, scratch, M, N, K, kind):
    """fp32 accumulation over K / 256 super-blocks and parts (2^-24 relative to the partial sums per
    step): the first and the last columns, which hold the split or cut tiles, against the exact sums,
    and every element against the other route."""
    assert _kind(_plan(fmt, M, N, K, scratch)) == kind
    w, wd, x_i8, xs = _case(device, fmt, M, N, K)
    y = _gemm(fmt, x_i8, xs, wd, scratch)
    for c in (slice(0, 130), slice(max(0, N - 300), N)):
        ref = GEMV[fmt](x_i8.cpu().numpy(), xs.cpu().numpy(), w[c], K)
        err = np.abs(y[:, c].cpu().numpy().astype(np.float64) - ref)
        assert (err <= 1e-5 * np.abs(ref) + 1e-5 * np.abs(ref).max()).all(), f"max err {err.max():.3e}"
    z = _gemm(fmt, x_i8, xs, wd, not scratch)
    assert ((y - z).abs() <= 1e-5 * z.abs() + 1e-5 * z.abs().max()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [4, 5, 6])
def test_quarters_bit_match_whole_tiles(device, fmt):
    """The quarter launch applies the whole tiles' operations in the same order: without the first
    1024 columns the 512 tiles are one even round, and the columns whose tiles were cut (16384 on)
    match bit for bit."""
    M, N, K = 512, 17408, 2304
    assert _kind(_plan(fmt, M, N, K, False)) == (128, "cut")
    assert _kind(_plan(fmt, M, N - 1024, K, False)) == (128, "whole")
    _, wd, x_i8, xs = _case(device, fmt, M, N, K)
    y = _gemm(fmt, x_i8, xs, wd, False)
    assert torch.equal(y[:, 1024:], _gemm(fmt, x_i8, xs, wd[1024:].contiguous(), False))


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [4, 5, 6])
def test_whole_tiles_beside_split_ones(device, fmt):
    """Where whole and split tiles share a call, the whole ones (the first 16384 of 17408 columns)
    hold the bits of a call in which nothing is split."""
    M, N, K, n = 512, 17408, 2304, 16384
    assert _kind(_plan(fmt, M, N, K, True)) == (128, "mixed")
    assert _kind(_plan(fmt, M, n, K, True)) == (128, "whole")
    _, wd, x_i8, xs = _case(device, fmt, M, N, K)
    y = _gemm(fmt, x_i8, xs, wd, True)
    assert torch.equal(y[:, :n], _gemm(fmt, x_i8, xs, wd[:n].contiguous(), True))


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,q_max", [(4, 15), (5, 31)])
@pytest.mark.parametrize("scratch", [True, False])
@pytest.mark.parametrize("M", [40, 512])
def test_largest_sums(device, fmt, q_max, scratch, M):
    """Every code, scale and min at its largest and x rows of all +127, all -127 and halves that
    cancel: the running sums of a super-block reach 256 * 127 * 63 * q_max (6.3e7, above 2^24). The
    int8 kernel (M = 512 without scratch) holds them exactly, the fp16 one rounds 16 times per
    super-block at 2^-23 of the largest; then fp32 sums over the super-blocks."""
    N, K = 4864, 1024
    nsb = K // 256
    one = np.ones((N, nsb), np.float16)
    sc = np.full((N, nsb, 8), 63, np.uint8)
    q = np.full((N, nsb, 8, 32), q_max, np.uint8)
    q[1::2, :, :, ::3] = 0
    make = oq.make_blocks if fmt == 4 else okq.q5k_make
    w = make(one, one, sc, sc.copy(), q).reshape(N, -1)
    x = np.full((M, K), 127, np.int8)
    x[1::3] = -127
    x[2::3] = np.where(np.arange(K) % 256 < 128, 127, -127)
    xt, wd = torch.from_numpy(x).to(device), torch.from_numpy(w).to(device)
    y = _gemm(fmt, xt, torch.ones(M, device=device), wd, scratch)
    ref = GEMV[fmt](x[:3], np.ones(3, np.float32), w[:2], K)  # rows and columns repeat
    ref = np.tile(ref, (-(-M // 3), N // 2))[:M]
    top = 256 * 127 * 63.0 * q_max
    tol = nsb * 16 * 2.0 ** -23 * top + nsb * 2.0 ** -23 * nsb * top
    assert np.abs(y.cpu().numpy().astype(np.float64) - ref).max() <= tol
