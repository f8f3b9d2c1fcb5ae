"""Attention over 256-wide heads against the oracle (rope_f32, store_kv, paged
attention, gate) and against the general path, which misaligned queries take.

Pages hold NaN wherever no token was written, so a read past a row's tokens
shows in the output. Rows end at and around the edges of a page and of the
half page a wave reads at a time."""
import math

import numpy as np
import pytest
import torch

from oracle import oracle as orc
from tests.gpu_util import (approx, assert_close, force_plan, new_context, new_pool, to_dev,
                            to_host)

pytestmark = pytest.mark.gpu

D = 256
LENGTHS = [1, 2, 7, 8, 9, 15, 16, 17, 24, 25, 160, 161, 401, 700]


@pytest.fixture(scope="module")
def ctx():
    c = new_context()
    yield c
    c.sync()
    c.close()


def nan_pages(code, n):
    if code == orc.F32:
        return np.full(n, np.nan, np.float32)
    return np.full(n, 0x7FC0 if code == orc.BF16 else 0x7E00, np.uint16)


def misaligned(t):
    """A copy one element past a 16-byte boundary."""
    base = torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)
    view = base[1:1 + t.numel()].view(t.shape)
    view.copy_(t)
    return view


@pytest.mark.parametrize("code,group,rotary,gated,split", [
    (orc.BF16, 4, 64, True, None), (orc.BF16, 4, 256, False, "0"), (orc.F16, 4, 128, True, "3"),
    (orc.BF16, 2, 64, True, "b6"), (orc.F16, 1, 16, False, "1"), (orc.BF16, 8, 256, True, "5"),
    (orc.BF16, 2, None, False, "2"), (orc.F32, 4, None, True, "4"), (orc.F32, 8, None, False, "2"),
    (orc.F32, 1, 64, False, None), (orc.BF16, 4, 48, False, None)])
def test_wide_decode_matches_oracle_and_general_path(ctx, code, group, rotary, gated, split,
                                                     monkeypatch):
    print(f"wide decode dtype {code} group {group} rotary {rotary} gated {gated} split {split}",
          flush=True)
    force_plan(monkeypatch, split)
    rng = orc.Mt64(900 + 10 * group + code)
    H = 2
    Hq, rows, theta = H * group, len(LENGTHS), 1e7
    pages = [-(-n // 16) for n in LENGTHS]
    blocks = sum(pages) + 3
    order = rng.permutation(blocks)
    tables = np.split(order[:sum(pages)], np.cumsum(pages)[:-1])
    flat, offsets = np.concatenate(tables), np.cumsum([0] + pages[:-1])
    positions = [n - 1 for n in LENGTHS]
    slots = [orc.slot(t, p, 16) for t, p in zip(tables, positions)]
    geom, F = (1, blocks, 16, H, D), H * D
    kc, vc = nan_pages(code, blocks * 16 * F), nan_pages(code, blocks * 16 * F)
    for t, n in zip(tables, LENGTHS):
        held = [orc.slot(t, p, 16) for p in range(n - 1)]
        if held:
            orc.store_kv(kc, vc, rng.normal(len(held) * F, code).reshape(-1, F),
                         rng.normal(len(held) * F, code).reshape(-1, F), held, 0, blocks * 16)
    q = rng.normal(rows * Hq * D, code).reshape(rows, Hq * D)
    kn, vn = (rng.normal(rows * F, code).reshape(rows, F) for _ in range(2))
    gate = rng.normal(rows * Hq * D, code).reshape(rows, Hq * D) if gated else None
    scale = float(np.float32(1 / math.sqrt(D)))

    outs, caches = [], []
    for shift in (lambda t: t, misaligned):
        pool, kd, vd = new_pool(ctx, geom, code)
        kd.copy_(to_dev(kc, code))
        vd.copy_(to_dev(vc, code))
        pool.upload(flat, offsets, pages, positions, slots)
        qd, knd, vnd = shift(to_dev(q, code)), to_dev(kn, code), to_dev(vn, code)
        gd = to_dev(gate, code) if gated else None
        out = shift(torch.full((rows, Hq * D), float("nan"), dtype=qd.dtype, device="cuda"))
        if rotary is not None:
            pool.rope_append_decode(0, knd, vnd, qd, Hq, scale, theta, out, rotary, gd)
        elif gated:
            pool.append_decode_gated(0, knd, vnd, qd, Hq, scale, gd, out)
        else:
            pool.append_decode(0, knd, vnd, qd, Hq, scale, out)
        ctx.sync()
        outs.append(to_host(out, code))
        caches.append((to_host(kd, code), to_host(vd, code)))
        if rotary is None and not gated:  # the unfused call over the same pages
            again = torch.full_like(out, float("nan"))
            pool.decode(0, qd, Hq, scale, again)
            ctx.sync()
            assert np.array_equal(to_host(again, code), outs[-1])
        pool.close()

    want_k, want_v = kc.copy(), vc.copy()
    rk = kn if rotary is None else orc.rope(kn, code, H, positions, theta, rotary)
    orc.store_kv(want_k, want_v, rk, vn, slots, 0, blocks * 16)
    for got_k, got_v in caches:
        assert np.array_equal(got_v.view(np.uint8), want_v.view(np.uint8))
        if rotary is None:
            assert np.array_equal(got_k.view(np.uint8), want_k.view(np.uint8))
        elif code == orc.F32:
            assert np.allclose(got_k, want_k, rtol=1e-5, atol=1e-5, equal_nan=True)
        else:  # a rotated element within one unit in the last place (sign and magnitude)
            a, b = (np.where(x & 0x8000, -(x & 0x7FFF).astype(np.int32), x & 0x7FFF)
                    for x in (got_k.astype(np.int32), want_k.astype(np.int32)))
            assert np.abs(a - b).max() <= 1
    rq = q if rotary is None else orc.rope(q, code, Hq, positions, theta, rotary)
    expected = orc.Attention(geom, caches[0][0], caches[0][1], code, rq, code, positions, flat,
                             offsets, pages, Hq, 0, scale).online_threads(8)
    if gated:
        g = gate if code == orc.F32 else orc.to_f32(gate, code)
        expected = expected * (1.0 / (1.0 + np.exp(-np.asarray(g, np.float64))))
    for got, what in zip(outs, ("fast", "general")):
        if code == orc.F32:
            assert approx(got, expected, 3e-5, 1.0), what
        else:
            assert_close(orc.to_f32(got, code), expected, what=what)


# (prefix, rows) of each sequence: single rows, tile and block edges, tiles of several workgroups
CHUNKS = [(0, 1), (0, 33), (5, 40), (31, 64), (100, 128), (16, 257), (700, 1), (1000, 70), (63, 2)]


@pytest.mark.parametrize("code,group,gated,split,min_blocks", [
    (orc.BF16, 4, True, None, None), (orc.F16, 4, False, "1", None), (orc.BF16, 2, False, "3", "1"),
    (orc.F16, 1, True, "8", "2"), (orc.BF16, 8, True, "2", "1"), (orc.F16, 2, True, "8", "1"),
    (orc.BF16, 1, False, None, None), (orc.F32, 4, True, None, None)])
def test_wide_prefill_matches_oracle_and_general_path(ctx, code, group, gated, split, min_blocks,
                                                      monkeypatch):
    """Tiles on the matrix cores (f32 pools: decode rows) with keys unsplit and
    split. Probabilities enter as three 16-bit terms, so the error against the
    double reference is that of the general path, which holds them in 32 bits:
    both round the same stored values once (bounded at 1.1 times here, for the
    order of sums)."""
    print(f"wide prefill dtype {code} group {group} gated {gated} split {split}", flush=True)
    if split is not None:
        monkeypatch.setenv("CKV_PREFILL_SPLIT", split)
    if min_blocks is not None:
        monkeypatch.setenv("CKV_PREFILL_SPLIT_MIN", min_blocks)
    rng = orc.Mt64(1200 + 10 * group + code)
    H = 2
    Hq, F = H * group, H * D
    spans = [p + n for p, n in CHUNKS]
    pages = [-(-n // 16) for n in spans]
    blocks = sum(pages) + 2
    order = rng.permutation(blocks)
    tables = np.split(order[:sum(pages)], np.cumsum(pages)[:-1])
    flat, starts = np.concatenate(tables), np.cumsum([0] + pages[:-1])
    seq = np.repeat(np.arange(len(CHUNKS)), [n for _, n in CHUNKS])
    positions = np.concatenate([np.arange(p, p + n) for p, n in CHUNKS]).astype(np.uint32)
    offsets, lengths = starts[seq], np.array(pages)[seq]
    rows, geom = len(positions), (1, blocks, 16, H, D)
    kc, vc = nan_pages(code, blocks * 16 * F), nan_pages(code, blocks * 16 * F)
    for t, n in zip(tables, spans):
        orc.store_kv(kc, vc, rng.normal(n * F, code).reshape(-1, F),
                     rng.normal(n * F, code).reshape(-1, F), [orc.slot(t, p, 16) for p in range(n)],
                     0, blocks * 16)
    q = rng.normal(rows * Hq * D, code).reshape(rows, -1)
    gate = rng.normal(rows * Hq * D, code).reshape(rows, -1) if gated else None
    scale = float(np.float32(1 / math.sqrt(D)))
    pool, kd, vd = new_pool(ctx, geom, code)
    kd.copy_(to_dev(kc, code))
    vd.copy_(to_dev(vc, code))
    pool.upload(flat, offsets, lengths, positions)
    gd = to_dev(gate, code) if gated else None
    outs = []
    for shift in (lambda t: t, lambda t: t, misaligned):
        qd = shift(to_dev(q, code))
        out = shift(torch.full((rows, Hq * D), float("nan"), dtype=qd.dtype, device="cuda"))
        if gated:
            pool.attention_gated(0, qd, Hq, scale, gd, out)
        else:
            pool.attention(0, qd, Hq, scale, out)
        ctx.sync()
        outs.append(to_host(out, code))
    pool.close()
    assert np.array_equal(outs[0], outs[1]), "a second call differs"
    expected = orc.Attention(geom, kc, vc, code, q, code, positions, flat, offsets, lengths, Hq, 0,
                             scale).reference()
    if gated:
        g = gate if code == orc.F32 else orc.to_f32(gate, code)
        expected = expected * (1.0 / (1.0 + np.exp(-np.asarray(g, np.float64))))
    got, general = ((x if code == orc.F32 else orc.to_f32(x, code)).astype(np.float64)
                    for x in (outs[0], outs[2]))
    if code == orc.F32:
        assert approx(got, expected, 3e-5, 1.0)
    else:
        assert_close(got, expected, what="prefill")
        off, off_general = (np.linalg.norm(x - expected) for x in (got, general))
        assert off <= 1.1 * off_general, (off, off_general)


@pytest.mark.parametrize("code,group,gated,split", [
    (orc.BF16, 4, True, "1"), (orc.F16, 2, False, "4"), (orc.BF16, 8, False, "2"), (orc.F16, 1, True, "1")])
def test_wide_prefill_keeps_values_that_are_not_finite_with_their_rows(ctx, code, group, gated, split,
                                                                       monkeypatch):
    """Infinities and a NaN among the keys and values reach exactly the rows
    that attend them, as in the general path: a query of the same tile that stands
    before such a token has none of it, and an infinite value stays an infinity."""
    print(f"wide prefill, not finite: dtype {code} group {group} gated {gated} split {split}", flush=True)
    monkeypatch.setenv("CKV_PREFILL_SPLIT", split)
    monkeypatch.setenv("CKV_PREFILL_SPLIT_MIN", "1")
    rng = orc.Mt64(1500 + 10 * group + code)
    H, prefix, rows = 2, 21, 150
    span, Hq, F = prefix + rows, H * group, H * D
    pages = -(-span // 16)
    geom, table = (1, pages + 1, 16, H, D), rng.permutation(pages + 1)[:pages]
    k, v = (rng.normal(span * F, code).reshape(span, F).copy() for _ in range(2))
    q = rng.normal(rows * Hq * D, code).reshape(rows, -1)
    gate = rng.normal(rows * Hq * D, code).reshape(rows, -1)
    inf, nan = (0x7F80, 0x7FC0) if code == orc.BF16 else (0x7C00, 0x7E00)
    v[40, 3] = v[77, 200] = inf          # kv head 0, two features
    v[60, D + 9] = v[61, D + 9] = inf | 0x8000  # kv head 1
    k[130, 5] = inf                      # scores of one sign or the other
    v[150, D + 30] = nan
    kc, vc = nan_pages(code, geom[1] * 16 * F), nan_pages(code, geom[1] * 16 * F)
    orc.store_kv(kc, vc, k, v, [orc.slot(table, p, 16) for p in range(span)], 0, geom[1] * 16)
    pool, kd, vd = new_pool(ctx, geom, code)
    kd.copy_(to_dev(kc, code))
    vd.copy_(to_dev(vc, code))
    pool.upload(table, np.zeros(rows, np.uint32), np.full(rows, pages),
                np.arange(prefix, span).astype(np.uint32))
    outs = []
    for shift in (lambda t: t, misaligned):
        qd = shift(to_dev(q, code))
        out = shift(torch.full((rows, Hq * D), float("nan"), dtype=qd.dtype, device="cuda"))
        if gated:
            pool.attention_gated(0, qd, Hq, 1 / math.sqrt(D), to_dev(gate, code), out)
        else:
            pool.attention(0, qd, Hq, 1 / math.sqrt(D), out)
        ctx.sync()
        outs.append(orc.to_f32(to_host(out, code), code).reshape(rows, Hq * D))
    pool.close()
    got, general = outs
    assert np.isfinite(general[:40 - prefix]).all() and np.isinf(general).any() and np.isnan(general).any()
    assert np.array_equal(np.isnan(got), np.isnan(general))
    assert np.array_equal(np.isinf(got), np.isinf(general))
    fin = np.isfinite(general)
    assert_close(got[fin], general[fin], what="finite values")
    assert np.array_equal(np.sign(got[~fin & ~np.isnan(got)]), np.sign(general[~fin & ~np.isnan(general)]))


@pytest.mark.parametrize("code,group", [(orc.BF16, 4), (orc.F16, 2)])
def test_wide_prefill_keeps_nan_of_keys_that_weigh_nothing(ctx, code, group):
    """0 * NaN and 0 * inf are NaN in the reference: a key whose probability rounds
    to 0 still passes its NaN on to every query that attends it, as on the general
    path, however few keys the query attends."""
    rng = orc.Mt64(1700 + code)
    H, rows = 2, 40
    Hq, F, pages = H * group, H * D, 3
    geom, table = (1, pages, 16, H, D), rng.permutation(pages)
    k, v = (rng.normal(rows * F, code).reshape(rows, F).copy() for _ in range(2))
    q = rng.normal(rows * Hq * D, code).reshape(rows, Hq, D)
    one, low, inf, nan = ((0x3F80, 0xC600, 0x7F80, 0x7FC0) if code == orc.BF16
                          else (0x3C00, 0xF000, 0x7C00, 0x7E00))
    q[:, :, 7] = one
    k[0, 7] = k[0, D + 7] = low  # -8192: a probability of 2^-700 beside any other key's
    v[0, 3], v[0, D + 9] = nan, inf
    kc, vc = nan_pages(code, pages * 16 * F), nan_pages(code, pages * 16 * F)
    orc.store_kv(kc, vc, k, v, [orc.slot(table, p, 16) for p in range(rows)], 0, pages * 16)
    pool, kd, vd = new_pool(ctx, geom, code)
    kd.copy_(to_dev(kc, code))
    vd.copy_(to_dev(vc, code))
    pool.upload(table, np.zeros(rows, np.uint32), np.full(rows, pages), np.arange(rows).astype(np.uint32))
    outs = []
    for shift in (lambda t: t, misaligned):
        qd = shift(to_dev(q.reshape(rows, -1), code))
        out = shift(torch.zeros((rows, Hq * D), dtype=qd.dtype, device="cuda"))
        pool.attention(0, qd, Hq, 1 / math.sqrt(D), out)
        ctx.sync()
        outs.append(orc.to_f32(to_host(out, code), code).reshape(rows, H, group, D))
    pool.close()
    got, general = outs
    assert np.isnan(general[:, 0, :, 3]).all() and np.isnan(general[1:, 1, :, 9]).all()
    assert np.array_equal(np.isnan(got), np.isnan(general))
    assert np.array_equal(np.isinf(got), np.isinf(general))
    fin = np.isfinite(general)
    assert_close(got[fin], general[fin], what="finite values")


@pytest.mark.parametrize("code,group", [(orc.BF16, 4), (orc.F16, 8)])
def test_wide_prefill_with_an_infinity_early_in_a_prefix(ctx, code, group):
    """Every query of the launch attends an infinite value and is attended again by
    vector arithmetic, several at a time: the counts of such queries in a wave
    run over 1 to 32, and all values but the infinite ones stay those of the
    double reference."""
    rng = orc.Mt64(1800 + code)
    H, chunks = 1, [(19, n) for n in (1, 2, 3, 4, 5, 31, 32, 33, 70)]
    Hq, F = H * group, H * D
    spans = [p + n for p, n in chunks]
    pages = [-(-n // 16) for n in spans]
    blocks = sum(pages)
    tables = np.split(rng.permutation(blocks), np.cumsum(pages)[:-1])
    seq = np.repeat(np.arange(len(chunks)), [n for _, n in chunks])
    positions = np.concatenate([np.arange(p, p + n) for p, n in chunks]).astype(np.uint32)
    flat, offsets = np.concatenate(tables), np.cumsum([0] + pages[:-1])[seq]
    lengths, rows, geom = np.array(pages)[seq], len(positions), (1, blocks, 16, H, D)
    kc, vc = nan_pages(code, blocks * 16 * F), nan_pages(code, blocks * 16 * F)
    for t, n in zip(tables, spans):
        orc.store_kv(kc, vc, rng.normal(n * F, code).reshape(-1, F), rng.normal(n * F, code).reshape(-1, F),
                     [orc.slot(t, p, 16) for p in range(n)], 0, blocks * 16)
    q = rng.normal(rows * Hq * D, code).reshape(rows, -1)
    scale = float(np.float32(1 / math.sqrt(D)))
    expected = orc.Attention(geom, kc, vc, code, q, code, positions, flat, offsets, lengths, Hq, 0,
                             scale).reference().reshape(rows, Hq, D).copy()
    expected[:, :, 17] = np.inf
    for t in tables:
        vc.reshape(-1, F)[orc.slot(t, 2, 16), 17] = 0x7F80 if code == orc.BF16 else 0x7C00
    pool, kd, vd = new_pool(ctx, geom, code)
    kd.copy_(to_dev(kc, code))
    vd.copy_(to_dev(vc, code))
    pool.upload(flat, offsets, lengths, positions)
    qd = to_dev(q, code)
    out = torch.full_like(qd, float("nan"))
    pool.attention(0, qd, Hq, scale, out)
    ctx.sync()
    got = orc.to_f32(to_host(out, code), code).reshape(rows, Hq, D)
    pool.close()
    assert np.array_equal(got[:, :, 17], expected[:, :, 17])
    others = np.arange(D) != 17
    assert_close(got[:, :, others], expected[:, :, others], what="finite values")


@pytest.mark.parametrize("code", [orc.BF16, orc.F16])
def test_wide_prefill_holds_probabilities_in_32_bits(ctx, code):
    """Values that cancel show a probability's own rounding. In each sequence of
    four tokens the first key has probability p = e^(-y / 16) beside three of 1,
    whose values are the parts of -p in the 16-bit type: the last row's output
    is what p's roundings leave, over 3 + p > 3.3. Bound: p off by 2^-22 (its
    exponent's two roundings and the exponential's last place), its parts by 2^-24,
    and six matrix products rounding sums of at most 1 twice, 12 * 2^-24: 3e-7, plus
    half of fp16's smallest value. (bf16 probabilities in two terms, 16 bits, leave
    up to 1e-6 for half of these y.)"""
    H, group, n, count = 1, 4, 4, 64
    to = torch.bfloat16 if code == orc.BF16 else torch.float16
    y = torch.arange(1, count + 1, dtype=torch.float64) / 4
    k, v = (torch.zeros(count, 16, D, dtype=torch.float64) for _ in range(2))
    k[:, 0, 0] = -y
    v[:, 0] = 1.0
    left = -torch.exp(-y / 16)
    for part in (1, 2, 3):
        v[:, part] = left.to(to).double()[:, None]
        left = left - v[:, part, 0]
    q = torch.zeros(count, n, group, D, dtype=torch.float64)
    q[..., 0] = 1.0
    order = torch.arange(count - 1, -1, -1)  # sequence i on page count - 1 - i
    pool, kd, vd = new_pool(ctx, (1, count, 16, H, D), code)
    kd.copy_(k[order].to(to).reshape(-1).cuda())
    vd.copy_(v[order].to(to).reshape(-1).cuda())
    rows = count * n
    pool.upload(order.numpy().astype(np.uint32), np.repeat(np.arange(count), n), np.ones(rows, np.uint32),
                np.tile(np.arange(n), count).astype(np.uint32))
    qd = q.reshape(rows, -1).to(to).cuda()
    out = torch.full_like(qd, float("nan"))
    pool.attention(0, qd, group, 1 / 16, out)
    ctx.sync()
    pool.close()
    last = out.double().cpu().reshape(count, n, group, D)[:, -1]
    assert last.abs().max() <= 3e-7 + 2.0 ** -25, float(last.abs().max())


@pytest.mark.parametrize("code,split", [(orc.BF16, "1"), (orc.F16, "3")])
def test_wide_heads_in_a_layer_past_4_gib(ctx, code, split, monkeypatch):
    """A layer of 140,000 pages of 32 KiB (4.3 GiB per tensor): pages above the
    4 GiB line, alone and among low ones, in prefill and decode."""
    monkeypatch.setenv("CKV_PREFILL_SPLIT", split)
    monkeypatch.setenv("CKV_PREFILL_SPLIT_MIN", "1")
    rng = orc.Mt64(2000 + code)
    H, group, n, chunk, blocks = 4, 2, 210, 70, 140_000
    Hq, F, pages = H * group, H * D, 14
    assert blocks * 16 * F * 2 > 1 << 32
    print(f"256-wide heads over {blocks} pages, dtype {code} split {split}", flush=True)
    high = np.arange(blocks - pages, blocks, dtype=np.uint32)
    mixed = np.where(np.arange(pages) % 2, blocks - 40 + np.arange(pages), 5 + np.arange(pages)).astype(np.uint32)
    tables = [high, mixed]
    k, v = (rng.normal(2 * n * F, code).reshape(2, n, F) for _ in range(2))
    q = rng.normal(2 * chunk * Hq * D, code).reshape(2 * chunk, -1)
    kc, vc = (np.zeros(2 * pages * 16 * F, np.uint16) for _ in range(2))
    pool, _, _ = new_pool(ctx, (1, blocks, 16, H, D), code)
    for i, t in enumerate(tables):
        pool.upload(t, [0] * n, [pages] * n, list(range(n)), [orc.slot(t, p, 16) for p in range(n)])
        pool.append(0, to_dev(k[i], code), to_dev(v[i], code))
        compact = np.arange(i * pages, (i + 1) * pages, dtype=np.uint32)
        orc.store_kv(kc, vc, k[i], v[i], [orc.slot(compact, p, 16) for p in range(n)], 0, 2 * pages * 16)
    positions = list(range(n - chunk, n)) * 2
    offsets, lengths = [0] * chunk + [pages] * chunk, [pages] * (2 * chunk)
    scale = float(np.float32(1 / math.sqrt(D)))
    expected = orc.Attention((1, 2 * pages, 16, H, D), kc, vc, code, q, code, positions,
                             np.arange(2 * pages, dtype=np.uint32), offsets, lengths, Hq, 0, scale).reference()
    pool.upload(np.concatenate(tables), offsets, lengths, positions)
    qd = to_dev(q, code)
    for name in ("attention", "decode"):
        out = torch.full_like(qd, float("nan"))
        getattr(pool, name)(0, qd, Hq, scale, out)
        ctx.sync()
        assert_close(orc.to_f32(to_host(out, code), code), expected, what=name)
    pool.close()
    del pool
    torch.cuda.empty_cache()
