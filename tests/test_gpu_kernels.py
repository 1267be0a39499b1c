"""Kernel-level parity on the GPU: each HIP kernel against the oracle on the same seeded inputs.

Bar: bit-exact for integer/byte work (quantisation, generators, routing ids) and for the f32
arithmetic the reference fixes (GEMV epilogue, dot orders, exp512/SwiGLU, RMSNorm).  Routing
weights use libm expf on the CPU and a double-rounded exp on the GPU: they may differ by one ulp
(tolerance written below)."""
from __future__ import annotations

import sys

import numpy as np
import pytest

import oracle as O
import trmoe

pytestmark = pytest.mark.gpu


def torch_dev():
    import torch
    assert torch.cuda.is_available(), "GPU test on a host without a GPU"
    return torch


def say(msg):
    print(f"[gpu] {msg}", flush=True)
    sys.stdout.flush()


def to_dev(a):
    torch = torch_dev()
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    return t.detach().cpu().numpy()


def ulp_diff(a, b):
    a = np.ascontiguousarray(a, np.float32).view(np.int32).astype(np.int64)
    b = np.ascontiguousarray(b, np.float32).view(np.int32).astype(np.int64)
    return np.abs(a - b)


@pytest.mark.parametrize("fmt,rows,K", [(O.FMT_Q4_K, 33, 2048), (O.FMT_Q6_K, 17, 512), (O.FMT_Q8_0, 9, 768), (O.FMT_Q5_1, 9, 768)])
def test_generator_bytes_match_oracle(fmt, rows, K):
    say(f"gen_gguf fmt={fmt} rows={rows} K={K}")
    g = host(trmoe.gen_gguf(fmt, 7, (3 << 32) | 99, rows, K))
    o = O.gen_gguf(fmt, 7, (3 << 32) | 99, rows, K)
    assert np.array_equal(g, o)
    say("gen_normal")
    gn = host(trmoe.gen_normal(7, 5, 4096, 0.02))
    on = O.gen_normal(7, 5, 4096, 0.02)
    assert np.allclose(gn, on, rtol=1e-6, atol=1e-12)


@pytest.mark.parametrize("kb", [16, 32])
@pytest.mark.parametrize("m", [1, 5])
def test_quantize_rows_bit_exact(kb, m):
    say(f"quantize rows kb={kb} m={m}")
    rng = np.random.default_rng(kb + m)
    x = (rng.standard_normal((m, 2048)) * 3).astype(np.float32)
    x[0, :kb] = 0.0                                   # all-zero block
    x[0, kb:2 * kb] = np.arange(kb) - kb / 2 + 0.5    # exact .5 ties after scaling
    q, s, su = trmoe.quantize(to_dev(x), kb)
    oq, os_, osu = O.quant_rows(x, kb)
    assert np.array_equal(host(q), oq) and np.array_equal(host(s).view(np.uint32), os_.view(np.uint32))
    assert np.array_equal(host(su), osu)


@pytest.mark.parametrize("kb", [16, 32])
def test_quantize_pair_bit_exact(kb):
    say(f"quantize pair kb={kb}")
    rng = np.random.default_rng(11)
    x = (rng.standard_normal(2048) * 2).astype(np.float32)
    q, s, su = trmoe.quantize(to_dev(x), kb, pair=True)
    oq, os_, osu = O.quant_pair(x, kb)
    assert np.array_equal(host(q), oq) and np.array_equal(host(s).view(np.uint32), os_.view(np.uint32))
    assert np.array_equal(host(su), osu)


@pytest.mark.parametrize("m", [1, 3, 16, 37])
def test_router_logits_bit_exact(m):
    say(f"router logits m={m}")
    E, H = 512, 2048
    router = O.gen_normal(1, 1, E * H, 0.02).reshape(E, H)
    shg = O.gen_normal(1, 2, H, 0.02)
    x = O.gen_normal(1, 3, m * H, 1.0).reshape(m, H)
    bias = (O.gen_normal(1, 4, E, 1.0)).astype(np.float32)
    dr, dx, ds, db = to_dev(router), to_dev(x), to_dev(shg), to_dev(bias)
    lg, sh = trmoe.router_logits(dr, dx, bias=db, shexp_gate=ds, gemm_order=False)
    want = np.array([[np.float32(O.dot(router[e], x[i]) + bias[e]) for e in range(E)] for i in range(m)], np.float32)
    assert np.array_equal(host(lg).view(np.uint32), want.view(np.uint32))
    wsh = np.array([O.dot(shg, x[i]) for i in range(m)], np.float32)
    assert np.array_equal(host(sh).view(np.uint32), wsh.view(np.uint32))
    lg2, _ = trmoe.router_logits(dr, dx, gemm_order=True)
    want2 = O.gemm_f32_nt(x, router)
    assert np.array_equal(host(lg2).view(np.uint32), want2.view(np.uint32))


@pytest.mark.parametrize("m", [70, 300])
def test_router_gemm_tiles_bit_exact(m):
    # the gemm tiles chosen for 64 <= m < 256 and m >= 256 (smallgemm.rs:8-59 order)
    say(f"router gemm m={m}")
    E, H = 512, 2048
    router = O.gen_normal(1, 1, E * H, 0.02).reshape(E, H)
    x = O.gen_normal(1, 5, m * H, 1.0).reshape(m, H)
    lg, _ = trmoe.router_logits(to_dev(router), to_dev(x), gemm_order=True)
    want = O.gemm_f32_nt(x, router)
    assert np.array_equal(host(lg).view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("m,E,H", [(512, 512, 2048), (700, 96, 768), (1024, 512, 2048), (1100, 80, 512),
                                   (1057, 96, 2560), (3072, 512, 2048)])
def test_router_mfma_bit_exact(m, E, H):
    """The matrix-core router gemm: the same bits as gemm_f32_nt's chains and halving
    tree, with ragged token and expert tiles, a bias, and the full shapes of configs 3 and 4."""
    say(f"router mfma m={m} E={E} H={H}")
    router = O.gen_normal(2, 1, E * H, 0.02).reshape(E, H)
    x = O.gen_normal(2, 5, m * H, 1.0).reshape(m, H)
    bias = O.gen_normal(2, 6, E, 1.0).astype(np.float32)
    lg, _ = trmoe.router_logits(to_dev(router), to_dev(x), bias=to_dev(bias), gemm_order=True)
    want = (O.gemm_f32_nt(x, router) + bias[None, :]).astype(np.float32)
    got = host(lg)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), np.abs(got - want).max()


@pytest.mark.parametrize("m,E,H", [(159, 96, 768), (160, 33, 768), (161, 512, 1024), (480, 512, 256), (500, 512, 384),
                                   (193, 70, 192), (290, 16, 2560), (330, 161, 192), (1025, 40, 64), (1025, 33, 768),
                                   (401, 257, 512), (400, 120, 768), (400, 121, 768), (1024, 61, 320), (401, 33, 256)])
def test_router_mfma_chunks_bit_exact(m, E, H):
    """Either side of the line to the matrix cores (160 rows, and enough experts to fill the VALU tiles'
    workgroups: 480 of them up to 400 rows), every chunk width (256 while the tiles and the shared
    gate's workgroups have CUs of their own, 128, 64; one chunk, odd counts), ragged tiles, and the shared gate's rows beside them."""
    say(f"router mfma chunks m={m} E={E} H={H}")
    router = O.gen_normal(2, 1, E * H, 0.02).reshape(E, H)
    x = O.gen_normal(2, 5, m * H, 1.0).reshape(m, H)
    shg = O.gen_normal(2, 7, H, 0.02)
    lg, sh = trmoe.router_logits(to_dev(router), to_dev(x), shexp_gate=to_dev(shg), gemm_order=True)
    assert np.array_equal(host(lg).view(np.uint32), O.gemm_f32_nt(x, router).view(np.uint32))
    want = np.array([O.dot(shg, x[i]) for i in range(m)], np.float32)
    assert np.array_equal(host(sh).view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("m,E,H", [(512, 512, 256), (200, 512, 192), (1030, 64, 384), (40, 64, 256)])
def test_router_gemm_special_values_bit_exact(m, E, H):
    """Denormal inputs, products and sums, signed zeros, overflow and infinities through the outer products (and
    the VALU tiles): the bits of the oracle's fma chains, NaN where it has NaN."""
    say(f"router special values m={m} E={E} H={H}")
    rng = np.random.default_rng(m)
    scale = np.float32(2.0) ** rng.integers(-40, 30, (m, 1)).astype(np.float32)
    x = (rng.standard_normal((m, H)).astype(np.float32) * scale)
    router = rng.standard_normal((E, H)).astype(np.float32)
    x[0::8] *= np.float32(2.0 ** -60)   # products in the denormal range
    router[0::4] *= np.float32(2.0 ** -60)
    x[1::8] = (rng.integers(0, 1 << 23, x[1::8].shape).astype(np.uint32) | (rng.integers(0, 2, x[1::8].shape).astype(np.uint32) << 31)).view(np.float32)
    x[2::8] = np.where(rng.random(x[2::8].shape) < 0.5, np.float32(-0.0), x[2::8])
    x[3::8, 5] = np.float32(3e38)       # overflow inside a chain
    router[1::4, 5] = np.float32(3e38)
    x[4::8, 7] = np.inf
    x[5::8, 9], x[5::8, 25] = np.inf, -np.inf  # one chain, or two that meet in the tree
    router[2::4, 9] = 0.0               # inf * 0
    with np.errstate(all="ignore"):
        want = O.gemm_f32_nt(x, router)
    got = host(trmoe.router_logits(to_dev(router), to_dev(x), gemm_order=True)[0])
    nan = np.isnan(want)
    assert nan.any() and np.isinf(want).any() and ((np.abs(want) < 1e-38) & (want != 0)).any()
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got.view(np.uint32)[~nan], want.view(np.uint32)[~nan])


@pytest.mark.parametrize("n,H", [(32 * 2897, 64), (23200, 16)])
def test_router_more_tiles_than_one_grid_row(n, H):
    """n x n logits whose tiles pass 2^32 threads (32 x 32 of 512 threads, 34 GB; 16 x 2 of 256): every sampled
    row, the last ones too, as a call of its own gives it."""
    torch = torch_dev()
    say(f"router {n} x {n} logits, H={H}")
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)
    x, router = (torch.randn((n, H), device="cuda", generator=gen) for _ in range(2))
    lg, _ = trmoe.router_logits(router, x, gemm_order=True)
    for r in (0, 31, n // 2, n - 40, n - 1):
        one, _ = trmoe.router_logits(router, x[r:r + 1].contiguous(), gemm_order=True)
        assert torch.equal(lg[r].view(torch.int32), one[0].view(torch.int32)), r
    del lg
    torch.cuda.empty_cache()


def routing_cases(E=512):
    rng = np.random.default_rng(5)
    lg = [rng.standard_normal((8, E)).astype(np.float32),
          (rng.integers(0, 40, (8, E)) * 0.25).astype(np.float32),   # many exact ties (router.rs:277-312)
          np.tile(np.array([((i * 37) % 101) * 0.1 for i in range(E)], np.float32), (2, 1))]
    peaked = np.full((1, E), -12.0, np.float32)
    for i, p in enumerate([0.61, 0.19, 0.09, 0.05, 0.025, 0.015]):
        peaked[0, i * 7] = np.float32(np.log(np.float32(p)))
    lg.append(peaked)
    nanrow = rng.standard_normal((1, E)).astype(np.float32)
    nanrow[0, ::3] = np.nan
    nanrow[0, 1::7] = -np.inf
    lg.append(nanrow)
    # more than 64 keys at or above the selection threshold: every logit equal, and 100 copies
    # of the maximum (with -0.0 / +0.0 mixed, which compare equal)
    lg.append(np.zeros((1, E), np.float32))
    signed_zero = np.zeros((1, E), np.float32)
    signed_zero[0, 1::2] = -0.0
    lg.append(signed_zero)
    hundred = np.clip(rng.standard_normal((1, E)), -4, 2.9).astype(np.float32)
    hundred[0, rng.permutation(E)[:100]] = 3.0
    lg.append(hundred)
    return np.concatenate(lg)


@pytest.mark.parametrize("E", [512, 1000])
@pytest.mark.parametrize("policy", [None, (1, 10, 0.9, O.BASIS_TOP), (1, 10, 0.95, O.BASIS_ALL), (4, 4, 0.5, O.BASIS_TOP),
                                    (1, 32, 1.0, O.BASIS_ALL), (8, 10, 0.5, O.BASIS_ALL)])
def test_route_matches_oracle(policy, E):
    say(f"route policy={policy} E={E}")
    lg = routing_cases(E)
    ids, w, n = trmoe.route(to_dev(lg), 10, policy)
    ids, w, n = host(ids).view(np.uint32), host(w), host(n)
    worst = 0
    for r in range(lg.shape[0]):
        oi, ow = O.route_mass(lg[r], *policy) if policy else O.route_topk(lg[r], 10)
        assert n[r] == len(oi), r
        assert np.array_equal(ids[r, :n[r]], oi), r
        worst = max(worst, int(ulp_diff(w[r, :n[r]], ow).max()))
    assert worst <= 1  # libm expf vs correctly rounded exp


def act_rows(x, kb, pair):
    """int8 activation rows as the reference quantises them: one row each, or (coarse, residual)
    pairs (quant.rs:36-53)."""
    if not pair:
        return O.quant_rows(x, kb)
    qs = [O.quant_pair(x[i], kb) for i in range(x.shape[0])]
    return tuple(np.concatenate([a[c] for a in qs]) for c in range(3))


def gemv_check(w_dev, w_tq, rows, K, fmt, bits, kb, x, pair, strips):
    """trk_gemv against the oracle's gemm_tq_rows on the same TQ bytes: identity rows, then a row
    map with repeats (accumulate and overwrite) into a wider y (ldy > rows)."""
    q, s, su = act_rows(x, kb, pair)
    m = x.shape[0]
    nstrips = (rows + 15) // 16
    s0, s1 = strips if strips else (0, nstrips)
    width = 16 * nstrips  # the oracle stores whole strips
    cut = width if fmt in trmoe.TQ_FMTS else rows  # GGUF rows past `rows` are never written
    want = O.gemv_tq(w_tq, K, bits, kb, width, q, s, su, pair=pair, s0=s0, s1=s1)
    y = trmoe.gemv(w_dev, rows, K, fmt, 0, 1, kb, to_dev(q), to_dev(s), to_dev(su), pair=pair, s0=s0, s1=s1,
                   y=to_dev(np.zeros((m, width), np.float32)), ldy=width)
    got = host(y)
    assert np.array_equal(got[:, :cut].view(np.uint32), want[:, :cut].view(np.uint32))
    assert not got[:, cut:].any()
    # a row map with repeats: logical rows in order onto 3 y rows of pitch width + 5
    rmap = np.array([(2 * i + 1) % 3 for i in range(m)], np.uint32)
    ldy = width + 5
    for acc in (True, False):
        base = np.arange(3 * ldy, dtype=np.float32).reshape(3, ldy) * 0.25
        want2 = O.gemv_tq(w_tq, K, bits, kb, width, q, s, su, pair=pair, y=base.copy(), rows=rmap,
                          accumulate=acc, s0=s0, s1=s1, ldy=ldy)
        y2 = trmoe.gemv(w_dev, rows, K, fmt, 0, 1, kb, to_dev(q), to_dev(s), to_dev(su), pair=pair,
                        y=to_dev(base.copy()), ldy=ldy, rowmap=to_dev(rmap.view(np.int32)), accumulate=acc,
                        s0=s0, s1=s1)
        got2 = host(y2)
        c0, c1 = 16 * s0, min(16 * s1, cut)
        assert np.array_equal(got2[:, c0:c1].view(np.uint32), want2[:, c0:c1].view(np.uint32)), acc
        keep = np.ones(ldy, bool)
        keep[c0:c1] = False
        assert np.array_equal(got2[:, keep], base[:, keep]), acc


# GGUF matrices read as their TQ conversion: every format and kb, sub-ranges of strips, rows not
# a multiple of 16, one to nine activation rows (passes of four), pairs
GEMV_GGUF_CASES = [(O.FMT_Q4_K, 32, 64, 2048, False, 3, None), (O.FMT_Q4_K, 32, 48, 512, True, 4, (1, 3)),
                   (O.FMT_Q4_K, 16, 96, 512, True, 6, (1, 5)), (O.FMT_Q4_K, 16, 40, 256, False, 5, None),
                   (O.FMT_Q6_K, 16, 64, 512, False, 3, (2, 4)), (O.FMT_Q6_K, 16, 40, 2048, True, 2, None),
                   (O.FMT_Q8_0, 32, 64, 512, False, 9, None), (O.FMT_Q8_0, 16, 48, 768, True, 4, (1, 3)),
                   (O.FMT_Q5_1, 32, 64, 1024, False, 1, None), (O.FMT_Q5_1, 16, 80, 512, False, 7, (2, 5))]


@pytest.mark.parametrize("fmt,kb,rows,K,pair,m,strips", GEMV_GGUF_CASES)
def test_gemv_gguf_bit_exact(fmt, kb, rows, K, pair, m, strips):
    say(f"gemv gguf fmt={fmt} kb={kb} rows={rows} K={K} pair={pair} m={m} strips={strips}")
    raw = O.gen_gguf(fmt, 3, 40 + fmt + kb, rows, K)
    tq, bits = O.gguf_to_tq(fmt, raw, rows, K, kb)
    x = O.gen_normal(3, 41 + m, m * K, 1.0).reshape(m, K)
    gemv_check(to_dev(raw), tq, rows, K, fmt, bits, kb, x, pair, strips)


def random_tq(seed, rows, K, bits, kb):
    """A packed TQ matrix (codec.rs:1-46) of uniform q and f16 scales / mins of real magnitudes."""
    rng = np.random.default_rng(seed)
    q = rng.integers(0, 1 << bits, (rows, K), dtype=np.uint8)
    nb = K // kb
    d = (rng.uniform(1e-4, 3e-3, (rows, nb)) * rng.choice([-1, 1], (rows, nb))).astype(np.float16)
    m = (-d.astype(np.float32) * rng.uniform(0, 1 << (bits - 1), (rows, nb))).astype(np.float16)
    return O.pack_tq(q, d, m, bits, kb)


# The reference's own packed codecs: its real expert shapes (gate TQ4_32 [640][2560], down
# TQ5_16 [2560][640], python/tests/test_blocks_real.py:23-26), k not a multiple of 256, ragged
# slices (33 blocks), padded strips, sub-ranges, pairs and row maps
GEMV_TQ_CASES = [(4, 32, 640, 2560, False, 1, None), (5, 16, 2560, 640, False, 1, None),
                 (5, 16, 2560, 640, True, 2, (40, 100)), (4, 16, 40, 80, False, 5, None),
                 (8, 16, 64, 96, False, 9, (1, 3)), (8, 32, 48, 2048, True, 6, None),
                 (5, 32, 100, 320, False, 3, None), (4, 32, 64, 1056, False, 4, (0, 2)),
                 (8, 16, 2560, 640, False, 2, (3, 160))]


@pytest.mark.parametrize("bits,kb,rows,K,pair,m,strips", GEMV_TQ_CASES)
def test_gemv_tq_bit_exact(bits, kb, rows, K, pair, m, strips):
    say(f"gemv tq bits={bits} kb={kb} rows={rows} K={K} pair={pair} m={m} strips={strips}")
    fmt = (bits << 8) | kb
    tq = random_tq(7 + bits + kb + m, rows, K, bits, kb)
    assert tq.size == trmoe.matrix_bytes(fmt, rows, K)
    x = O.gen_normal(4, 50 + m, m * K, 1.0).reshape(m, K)
    gemv_check(to_dev(tq), tq, rows, K, fmt, bits, kb, x, pair, strips)


# Few TQ rows of enough blocks take four rows per workgroup (rows x passes of four up to 2048; from 20 to 96 blocks
# by those, the activation rows and the bits), others a strip per workgroup: both sides of the lines, slices of 256
# blocks (128 from three activation rows) and one block past them
GEMV_QUAD_CASES = [(4, 32, 2048, 320, False, 1, None), (4, 32, 2064, 320, False, 3, None),
                   (5, 32, 2064, 352, True, 1, None), (8, 32, 2064, 96, False, 2, None),
                   (4, 16, 2080, 80, False, 4, (1, 130)), (5, 16, 512, 4112, True, 1, (3, 32)),
                   (8, 32, 320, 10240, True, 1, None), (8, 32, 64, 4128, False, 4, None),
                   (8, 16, 48, 2064, False, 3, (0, 2)), (4, 16, 1024, 4096, False, 8, None),
                   (4, 32, 256, 608, False, 1, None), (4, 32, 256, 640, False, 1, None),
                   (8, 32, 96, 1248, True, 1, None), (8, 32, 96, 1280, True, 1, None), (8, 32, 96, 640, False, 3, None),
                   (5, 16, 1040, 1008, False, 1, None), (5, 16, 1040, 1024, False, 2, None),
                   (8, 16, 2048, 1520, False, 1, (0, 128)), (8, 16, 2048, 1536, False, 1, (0, 128)),
                   (4, 16, 2048, 624, False, 4, None), (4, 16, 2048, 640, False, 4, None)]


@pytest.mark.parametrize("bits,kb,rows,K,pair,m,strips", GEMV_QUAD_CASES)
def test_gemv_few_rows_bit_exact(bits, kb, rows, K, pair, m, strips):
    say(f"gemv quads bits={bits} kb={kb} rows={rows} K={K} pair={pair} m={m} strips={strips}")
    tq = random_tq(9 + bits + kb + m, rows, K, bits, kb)
    x = O.gen_normal(4, 80 + m, m * K, 1.0).reshape(m, K)
    gemv_check(to_dev(tq), tq, rows, K, (bits << 8) | kb, bits, kb, x, pair, strips)


# TQ strips that stay a workgroup per strip (64 rows a workgroup from 65,536), also with a row map: more rows than
# the quads take, several passes of four activation rows (the last one partial), several slices of blocks
GEMV_STRIP_CASES = [(5, 32, 2064, 2592, False, 7, None), (8, 32, 2064, 2080, True, 3, None), (8, 16, 2080, 1104, False, 9, None),
                    (4, 16, 2064, 2064, False, 4, None), (5, 16, 2096, 1040, True, 2, None), (4, 32, 2064, 4128, False, 1, None),
                    (4, 32, 65552, 1056, False, 3, None), (8, 32, 65536, 1056, False, 1, None),
                    (5, 16, 65552, 560, True, 1, (0, 4097))]


@pytest.mark.parametrize("bits,kb,rows,K,pair,m,strips", GEMV_STRIP_CASES)
def test_gemv_strips_bit_exact(bits, kb, rows, K, pair, m, strips):
    say(f"gemv strips bits={bits} kb={kb} rows={rows} K={K} pair={pair} m={m} strips={strips}")
    assert rows > 2048 and (rows // 16) * ((m * (2 if pair else 1) + 3) // 4) < (1792 if m > 4 else 1 << 32)
    tq = random_tq(13 + bits + kb + m, rows, K, bits, kb)
    x = O.gen_normal(4, 90 + m, m * K, 1.0).reshape(m, K)
    gemv_check(to_dev(tq), tq, rows, K, (bits << 8) | kb, bits, kb, x, pair, strips)


@pytest.mark.parametrize("kind,kb", [(4, 32), (4, 16), (5, 32), (5, 16), (6, 32), (6, 16)])
@pytest.mark.parametrize("na", [1, 2, 4])
def test_gemv_quads_two_workgroups_per_cu(kind, kb, na):
    """The row quads' rule counts two of their workgroups per CU: registers and LDS leave room for them."""
    import ctypes as C
    torch_dev().zeros(1, device="cuda")
    hip = C.CDLL("libamdhip64.so")
    kernel = getattr(trmoe.lib(), f"_ZN3trk16gemv_quad_kernelILi{kind}ELi{kb}ELi{na}EEEvNS_8GemvArgsE")
    n = C.c_int()
    assert hip.hipOccupancyMaxActiveBlocksPerMultiprocessor(C.byref(n), C.cast(kernel, C.c_void_p), 512, C.c_size_t(0)) == 0
    assert n.value >= 2


# Enough (strip, pass) workgroups for the MFMA tiles: every codec, ragged row and activation tiles (the
# last workgroup nearly empty), k short of a slice and past one, strip sub-ranges, pairs, accumulate;
# 64-row workgroups past three of 32 rows per CU (m = 520 at 48 row blocks)
GEMM_CASES = [(O.FMT_Q4_K, 32, 1000, 512, False, 129, None), (O.FMT_Q4_K, 16, 440, 256, True, 145, (1, 27)),
              (O.FMT_Q6_K, 16, 520, 768, False, 241, (3, 33)), (O.FMT_Q8_0, 32, 1160, 256, False, 100, None),
              (O.FMT_Q8_0, 16, 240, 512, True, 260, None), (O.FMT_Q5_1, 32, 480, 256, False, 241, None),
              (O.FMT_Q5_1, 16, 1040, 256, False, 111, None), ((4, 32), 32, 900, 1056, False, 127, None),
              ((4, 16), 16, 1800, 80, False, 65, None), ((5, 32), 32, 700, 320, True, 91, (2, 44)),
              ((5, 16), 16, 2560, 176, False, 45, (0, 157)), ((8, 32), 32, 28700, 32, False, 5, None),
              ((8, 16), 16, 400, 640, False, 289, None), ((8, 32), 32, 6100, 160, False, 520, None),
              ((5, 16), 16, 6100, 272, True, 260, None), (O.FMT_Q6_K, 16, 6100, 256, False, 520, None),
              # past three workgroups per CU: one block of activation rows, a half-empty one, three blocks
              ((4, 32), 32, 98400, 32, False, 5, None), ((8, 32), 32, 98400, 32, False, 33, None),
              ((5, 32), 32, 33000, 64, False, 90, None),
              # longer TQ columns take the GEMV's passes for two rounds ([900][1056], [400][640] above), then the tiles
              ((4, 32), 32, 1000, 1056, False, 127, None), ((8, 16), 16, 480, 640, False, 289, None),
              ((5, 32), 32, 256, 1024, False, 512, None), ((5, 32), 32, 256, 1024, False, 513, None)]


@pytest.mark.parametrize("fmt,kb,rows,K,pair,m,strips", GEMM_CASES)
def test_gemv_many_rows_bit_exact(fmt, kb, rows, K, pair, m, strips):
    """trk_gemv of many activation rows against the oracle's gemm_tq_rows, written and accumulated,
    into a y wider than the matrix: the bits of the chain, nothing outside the strip range."""
    say(f"gemm fmt={fmt} kb={kb} rows={rows} K={K} pair={pair} m={m} strips={strips}")
    if isinstance(fmt, tuple):
        bits, code = fmt[0], (fmt[0] << 8) | fmt[1]
        raw = tq = random_tq(11 + bits + m, rows, K, bits, kb)
    else:
        code, raw = fmt, O.gen_gguf(fmt, 3, 60 + fmt + kb, rows, K)
        tq, bits = O.gguf_to_tq(fmt, raw, rows, K, kb)
    q, s, su = act_rows(O.gen_normal(5, 70 + m, m * K, 1.0).reshape(m, K), kb, pair)
    nstrips = (rows + 15) // 16
    s0, s1 = strips or (0, nstrips)
    assert (s1 - s0) * ((q.shape[0] + 3) // 4) >= 7 * 256  # the tiles' range (TQ of long columns: from 1920 or 2049)
    c0, c1 = 16 * s0, 16 * s1 if isinstance(fmt, tuple) else min(16 * s1, rows)
    ldy = 16 * nstrips + 3
    base = (np.arange(m * ldy, dtype=np.float32).reshape(m, ldy) % 97) * 0.25
    for acc in (False, True):
        want = O.gemv_tq(tq, K, bits, kb, 16 * nstrips, q, s, su, pair=pair, y=base.copy(),
                         rows=np.arange(m, dtype=np.uint32), accumulate=acc, s0=s0, s1=s1, ldy=ldy)
        got = host(trmoe.gemv(to_dev(raw), rows, K, code, 0, 1, kb, to_dev(q), to_dev(s), to_dev(su), pair=pair,
                              y=to_dev(base.copy()), ldy=ldy, accumulate=acc, s0=s0, s1=s1))
        assert np.array_equal(got[:, c0:c1].view(np.uint32), want[:, c0:c1].view(np.uint32)), acc
        assert np.array_equal(got[:, :c0], base[:, :c0]) and np.array_equal(got[:, c1:], base[:, c1:]), acc


def test_gemv_more_tiles_than_one_grid_row():
    """A strip against so many activation rows that its tiles of 256 threads pass 2^32 threads: every sampled
    row, the last ones too, as a call of its own gives it."""
    torch = torch_dev()
    m, kb = (1 << 30) + 200, 16
    if torch.cuda.mem_get_info()[0] < 120 << 30:
        pytest.skip("needs 100 GB of free memory")
    say(f"gemv of {m} activation rows")
    tq = to_dev(random_tq(3, 16, kb, 4, kb))
    q = torch.arange(m, dtype=torch.int32, device="cuda").view(m, 1).expand(m, kb // 4).contiguous().view(torch.int8)
    s = torch.full((m, 1), 0.5, device="cuda")
    su = torch.full((m, 1), 3, dtype=torch.int32, device="cuda")
    y = trmoe.gemv(tq, 16, kb, trmoe.FMT_TQ4_16, 0, 1, kb, q, s, su)
    for r in (0, 63, m // 2, m - 300, m - 1):
        one = trmoe.gemv(tq, 16, kb, trmoe.FMT_TQ4_16, 0, 1, kb, q[r:r + 1].clone(), s[:1], su[:1])
        assert torch.equal(y[r].view(torch.int32), one[0].view(torch.int32)), r
    del y, q, s, su
    torch.cuda.empty_cache()


@pytest.mark.parametrize("m", [1, 70, 300, 512])
def test_designed_rounding_orders(m):
    """The designed cases that pin the oracle's f32 orders (test_oracle.py: test_gemv_epilogue_order,
    test_gemm_f32_nt_lane_map, test_rmsnorm_product_order) through the GPU kernels: the GEMV's
    two-FMA epilogue (gemv.rs:141-148), the router GEMM's lane / chain map on each of its tile paths
    (smallgemm.rs:8-59; m = 1 and 70 VALU tiles of two sizes, 300 the 16 x 16 tiles, 512 the matrix
    cores) and RMSNorm's (x r) w (elem.rs:255-262), each against the literal the case was built
    for."""
    from test_oracle import epilogue_order_case, rmsnorm_order_case
    say(f"designed rounding orders m={m}")
    w, k, bits, kb, xq, s, su = epilogue_order_case()
    y = host(trmoe.gemv(to_dev(w), 16, k, (bits << 8) | kb, 0, 1, kb, to_dev(xq), to_dev(s), to_dev(su)))
    assert y[0, 0] == np.float32(2.0 ** -10) and np.all(y[0, 1:] == 0)
    a = np.float32(1 + 2.0 ** -12)
    H, E = 256, 8
    router = np.zeros((E, H), np.float32)
    router[0, 0], router[0, 16] = a, a
    router[1, 0], router[1, 16], router[1, 1] = 1e8, -1e8, 1.0
    router[2, 0], router[2, 8], router[2, 1] = 1e8, 1.0, -1e8
    x = np.ones((m, H), np.float32)
    x[:, 0], x[:, 16] = a, -a
    # row 0: the fused chain of lane 0 leaves -2^-24; rows 1 and 2 see x = a at k = 0 and -a at
    # k = 16, so their designed sums are taken on rows of ones
    lg, _ = trmoe.router_logits(to_dev(router), to_dev(x), gemm_order=True)
    assert np.all(host(lg)[:, 0] == np.float32(-(2.0 ** -24)))
    lg, _ = trmoe.router_logits(to_dev(router), to_dev(np.ones((m, H), np.float32)), gemm_order=True)
    got = host(lg)
    assert np.all(got[:, 1] == 1.0) and np.all(got[:, 2] == 0.0)
    xr, wr, want = rmsnorm_order_case()
    yr = host(trmoe.rmsnorm(to_dev(np.tile(xr, (2, 1))), to_dev(wr), 0.0))
    assert np.array_equal(yr.view(np.uint32), np.tile(want, (2, 1)).view(np.uint32))


def test_swiglu_and_rmsnorm_bit_exact():
    say("swiglu / rmsnorm")
    rng = np.random.default_rng(2)
    g = (rng.standard_normal(4096 + 7) * 4).astype(np.float32)
    u = rng.standard_normal(4096 + 7).astype(np.float32)
    y = host(trmoe.swiglu(to_dev(g), to_dev(u)))
    want = O.swiglu(g, u)
    body = g.size // 16 * 16  # exp512 body: bit-exact; scalar tail uses libm expf (<= 1 ulp apart)
    assert np.array_equal(y[:body].view(np.uint32), want[:body].view(np.uint32))
    assert np.allclose(y[body:], want[body:], rtol=1e-6, atol=0)
    x = rng.standard_normal((3, 2048)).astype(np.float32)
    w = rng.uniform(0.9, 1.1, 2048).astype(np.float32)
    yn = host(trmoe.rmsnorm(to_dev(x), to_dev(w), 1e-6))
    want = np.stack([O.rmsnorm(x[i], w, 1e-6) for i in range(3)])
    assert np.array_equal(yn.view(np.uint32), want.view(np.uint32))
    # ragged width: one 1024-wide batch, a 64-wide step, a 16-wide tail and a scalar tail
    n = 1024 + 64 + 16 + 5
    x = rng.standard_normal((2, n)).astype(np.float32)
    w = rng.uniform(0.9, 1.1, n).astype(np.float32)
    yn = host(trmoe.rmsnorm(to_dev(x), to_dev(w), 1e-6))
    want = np.stack([O.rmsnorm(x[i], w, 1e-6) for i in range(2)])
    assert np.array_equal(yn.view(np.uint32), want.view(np.uint32))


def test_row_and_element_kernels_past_one_grid_row():
    """swiglu, add, rmsnorm, route and the normal generator past 2^32 threads: the last elements and rows as a call
    of their own gives them (swiglu's scalar tail is the whole array's)."""
    torch = torch_dev()
    if torch.cuda.mem_get_info()[0] < 80 << 30:
        pytest.skip("needs 60 GB of free memory")
    n = (1 << 32) + 16 * 1000
    cuts = [slice(0, 4096), slice(n // 2, n // 2 + 4096), slice(n - 4096, n)]
    say("swiglu, add of 2^32 elements")
    part = torch.randn(1 << 20, device="cuda")
    g = part.repeat(n // (1 << 20) + 1)[:n]
    y = torch.empty(n, device="cuda")
    trmoe.check(trmoe.lib().trk_swiglu(g.data_ptr(), g.data_ptr(), y.data_ptr(), n, None))
    for c in cuts:
        one = trmoe.swiglu(g[c].clone(), g[c].clone())
        assert torch.equal(y[c].view(torch.int32), one.view(torch.int32)), c
    trmoe.check(trmoe.lib().trk_add_inplace(y.data_ptr(), g.data_ptr(), n, None))
    for c in cuts:
        one = trmoe.swiglu(g[c].clone(), g[c].clone()) + g[c]
        assert torch.equal(y[c].view(torch.int32), one.view(torch.int32)), c
    say("rmsnorm, route of 2^26 rows")
    m = (1 << 26) + 50
    x = g[:4 * m].view(m, 4)
    out = trmoe.rmsnorm(x, None, 1e-6)
    ids, w, k = trmoe.route(x, 2)
    for r in (0, m // 2, m - 10, m - 1):
        assert torch.equal(out[r], trmoe.rmsnorm(x[r:r + 1].clone(), None, 1e-6)[0]), r
        i1, w1, k1 = trmoe.route(x[r:r + 1].clone(), 2)
        assert int(k[r]) == 2 and torch.equal(ids[r], i1[0]) and torch.equal(w[r], w1[0]), r
    del g, y, out, ids, w, k, x
    say("2^32 normals")
    z = trmoe.gen_normal(7, 3, n)
    assert torch.isfinite(z[n - 4096:]).all() and (z[n - 4096:] != z[n - (1 << 32) - 4096:n - (1 << 32)]).any()
    assert 0.9 < float(z[n - 4096:].std()) < 1.1 and 0.9 < float(z[n // 2:n // 2 + 4096].std()) < 1.1
    del z
    torch.cuda.empty_cache()
