"""The decode's merges (a wave's row groups, a workgroup's waves, a cut row's
records) at every remainder of the four states and records they take at a time."""
import math

import numpy as np
import pytest
import torch

from oracle import oracle as orc
from tests.gpu_util import approx, assert_close, new_context, new_pool, to_dev, to_host

pytestmark = pytest.mark.gpu

LENGTHS = [1, 16, 17, 33, 100, 161, 300, 520]


@pytest.fixture(scope="module")
def ctx():
    c = new_context()
    yield c
    c.sync()
    c.close()


@pytest.mark.parametrize("code,dim,group", [(orc.BF16, 128, 2), (orc.F32, 128, 1), (orc.F16, 256, 4)])
def test_merges_at_every_remainder(ctx, code, dim, group, monkeypatch):
    """1 to 10 waves per workgroup, rows cut into 1 to 33 records."""
    H, Hq, rows = 2, 2 * group, len(LENGTHS)
    rng = orc.Mt64(300 + dim + code)
    pages = [-(-n // 16) for n in LENGTHS]
    blocks = sum(pages)
    flat, offsets = rng.permutation(blocks), np.cumsum([0] + pages[:-1])
    positions = [n - 1 for n in LENGTHS]
    geom, n = (1, blocks, 16, H, dim), blocks * 16 * H * dim
    kc, vc = rng.normal(n, code), rng.normal(n, code)
    q = rng.normal(rows * Hq * dim, code).reshape(rows, -1)
    scale = float(np.float32(1 / math.sqrt(dim)))
    expected = orc.Attention(geom, kc, vc, code, q, code, positions, flat, offsets, pages, Hq, 0,
                             scale).reference()
    pool, kd, vd = new_pool(ctx, geom, code)
    kd.copy_(to_dev(kc, code))
    vd.copy_(to_dev(vc, code))
    qd = to_dev(q, code)
    for waves in (1, 2, 3, 4, 5, 6, 7, 8, 10):
        for split in (1, 2, 3, 4, 7, 0):
            monkeypatch.setenv("CKV_DECODE_WAVES", str(waves))
            monkeypatch.setenv("CKV_DECODE_SPLIT", str(split))
            pool.upload(flat, offsets, pages, positions)
            out = torch.full_like(qd, float("nan"))
            pool.decode(0, qd, Hq, scale, out)
            ctx.sync()
            got = to_host(out, code)
            if code == orc.F32:  # sums of up to 520 terms in another order
                assert approx(got, expected, 3e-5, 1.0), (waves, split)
            else:
                assert_close(orc.to_f32(got, code), expected, what=f"{waves} waves, split {split}")
    pool.close()


@pytest.mark.parametrize("code,dim,group", [(orc.BF16, 128, 2), (orc.F32, 128, 1), (orc.F16, 256, 4)])
def test_merges_keep_infinities(ctx, code, dim, group, monkeypatch):
    """An infinite value stays an infinity, whichever wave's or slice's state
    holds it: every third token but a row's last has one, at a feature of its own
    (positive at even ones), so each state and record has some."""
    H, Hq, rows = 2, 2 * group, len(LENGTHS)
    rng = orc.Mt64(340 + dim + code)
    pages = [-(-n // 16) for n in LENGTHS]
    blocks = sum(pages)
    flat, offsets = rng.permutation(blocks), np.cumsum([0] + pages[:-1])
    tables = np.split(flat, offsets[1:])
    geom = (1, blocks, 16, H, dim)
    kc = rng.normal(blocks * 16 * H * dim, code)
    v = rng.normal(blocks * 16 * H * dim, orc.F32).reshape(-1, H, dim)
    infinite = np.zeros((rows, dim))
    for r, n in enumerate(LENGTHS):
        for t in range(0, n - 1, 3):
            f = t % dim
            infinite[r, f] = -np.inf if f % 2 else np.inf
            v[orc.slot(tables[r], t, 16), :, f] = infinite[r, f]
    pool, kd, vd = new_pool(ctx, geom, code)
    kd.copy_(to_dev(kc, code))
    vd.copy_(torch.from_numpy(v.reshape(-1)).to(vd.dtype))
    qd = to_dev(rng.normal(rows * Hq * dim, code).reshape(rows, -1), code)
    where = np.broadcast_to(infinite[:, None], (rows, Hq, dim))
    for waves in (1, 2, 3, 5, 6, 7, 8, 10):
        for split in (1, 2, 3, 4, 7, 0):
            monkeypatch.setenv("CKV_DECODE_WAVES", str(waves))
            monkeypatch.setenv("CKV_DECODE_SPLIT", str(split))
            pool.upload(flat, offsets, pages, [n - 1 for n in LENGTHS])
            out = torch.zeros_like(qd)
            pool.decode(0, qd, Hq, 1 / math.sqrt(dim), out)
            ctx.sync()
            got = out.double().cpu().numpy().reshape(rows, Hq, dim)
            assert not np.isnan(got).any(), (waves, split)
            assert np.array_equal(np.where(np.isinf(got), got, 0.0), where), (waves, split)
    pool.close()


@pytest.mark.parametrize("code,dim,group", [(orc.BF16, 128, 2), (orc.F32, 128, 1), (orc.F16, 256, 4),
                                            (orc.F32, 256, 2)])
def test_keys_with_scores_of_minus_infinity_weigh_nothing(ctx, code, dim, group, monkeypatch):
    """Keys whose product with every query is -inf: the first of a row, single ones,
    whole pages and a row's last, so that lanes, waves and chunks see no other
    score (the double reference gives such keys weight 0)."""
    H, Hq, rows = 2, 2 * group, len(LENGTHS)
    rng = orc.Mt64(420 + dim + code)
    pages = [-(-n // 16) for n in LENGTHS]
    blocks = sum(pages)
    flat, offsets = rng.permutation(blocks), np.cumsum([0] + pages[:-1])
    tables = np.split(flat, offsets[1:])
    positions = [n - 1 for n in LENGTHS]
    geom, n = (1, blocks, 16, H, dim), blocks * 16 * H * dim
    kc, vc = rng.normal(n, code), rng.normal(n, code)
    keys = kc.reshape(-1, H, dim)
    for r, length in enumerate(LENGTHS[1:], 1):
        for t in range(length):
            if t == 0 or t == length - 1 or t % 5 == 3 or 32 <= t < 80:
                keys[orc.slot(tables[r], t, 16), :, 7] = {orc.F32: -np.inf, orc.BF16: 0xFF80,
                                                          orc.F16: 0xFC00}[code]
    q = rng.normal(rows * Hq * dim, code).reshape(rows, Hq, dim)
    q[:, :, 7] = {orc.F32: 1, orc.BF16: 0x3F80, orc.F16: 0x3C00}[code]
    q = q.reshape(rows, -1)
    scale = float(np.float32(1 / math.sqrt(dim)))
    expected = orc.Attention(geom, kc, vc, code, q, code, positions, flat, offsets, pages, Hq, 0,
                             scale).reference()
    assert np.isfinite(expected).all()
    pool, kd, vd = new_pool(ctx, geom, code)
    kd.copy_(to_dev(kc, code))
    vd.copy_(to_dev(vc, code))
    qd = to_dev(q, code)
    for waves in (1, 3, 8):
        for split in (1, 2, 4, 0):
            monkeypatch.setenv("CKV_DECODE_WAVES", str(waves))
            monkeypatch.setenv("CKV_DECODE_SPLIT", str(split))
            pool.upload(flat, offsets, pages, positions)
            out = torch.zeros_like(qd)
            pool.decode(0, qd, Hq, scale, out)
            ctx.sync()
            got = to_host(out, code)
            if code == orc.F32:  # sums of up to 520 terms in another order
                assert approx(got, expected, 3e-5, 1.0), (waves, split)
            else:
                assert_close(orc.to_f32(got, code), expected, what=f"{waves} waves, split {split}")
    pool.close()


@pytest.mark.parametrize("code,dim,group,rotary", [
    (orc.BF16, 256, 4, 64), (orc.F16, 256, 1, None), (orc.F32, 256, 2, None), (orc.BF16, 128, 2, 128),
    (orc.F16, 128, 8, None), (orc.F32, 128, 4, None)])
def test_newest_value_row_keeps_infinities(ctx, code, dim, group, rotary):
    """The newest token's infinities at every position of a page: the lanes past it,
    which re-read it, make no NaN of them, in the appending call and in a decode
    of the same pages (there with the queries as they are)."""
    lengths = list(range(1, 18)) + [47, 48, 200]
    H, Hq, rows = 2, 2 * group, len(lengths)
    rng = orc.Mt64(380 + dim + code)
    pages = [-(-n // 16) for n in lengths]
    blocks = sum(pages)
    flat, offsets = rng.permutation(blocks), np.cumsum([0] + pages[:-1])
    positions = [n - 1 for n in lengths]
    slots = [orc.slot(t, p, 16) for t, p in zip(np.split(flat, offsets[1:]), positions)]
    geom, n = (1, blocks, 16, H, dim), blocks * 16 * H * dim
    pool, kd, vd = new_pool(ctx, geom, code)
    kd.copy_(to_dev(rng.normal(n, code), code))
    vd.copy_(to_dev(rng.normal(n, code), code))
    qd = to_dev(rng.normal(rows * Hq * dim, code).reshape(rows, -1), code)
    kn = to_dev(rng.normal(rows * H * dim, code).reshape(rows, -1), code)
    vn = to_dev(rng.normal(rows * H * dim, code).reshape(rows, H, dim), code)
    where = np.zeros((rows, Hq, dim))
    for f, sign in ((0, 1), (5, -1), (dim - 3, 1)):
        vn[:, :, f] = sign * math.inf
        where[:, :, f] = sign * np.inf
    vn, scale = vn.reshape(rows, -1), 1 / math.sqrt(dim)
    pool.upload(flat, offsets, pages, positions, slots)
    for again in (False, True):
        out = torch.zeros_like(qd)
        if again:
            pool.decode(0, qd, Hq, scale, out)
        elif rotary:
            pool.rope_append_decode(0, kn, vn, qd, Hq, scale, 1e6, out, rotary)
        else:
            pool.append_decode(0, kn, vn, qd, Hq, scale, out)
        ctx.sync()
        got = out.double().cpu().numpy().reshape(rows, Hq, dim)
        assert not np.isnan(got).any(), again
        assert np.array_equal(np.where(np.isinf(got), got, 0.0), where), again
    pool.close()
