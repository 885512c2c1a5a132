"""GPU parity of the register-held weight units (decode, window and GEMV
kernels) at the shapes where their lane layouts change or leave remainders
(4 to 128 units per gate/up row, 4 to 16 per down row, output rows that do
not fill the last block, lists of one entry and of nearly 64), and of the
8-values-per-lane q8 quantizer's general path (groups of zeros, of products
below the normal range, with a NaN), against the C oracle; the GEMV's tile
kernel, which takes weights that are not whole dwords, and its bits against
the register kernel's."""
import ctypes

import numpy as np
import pytest

from test_gpu_decode import dev, host
from test_gpu_formats import check_tokens, packed_experts

import q4mi
from q4mi.synth import (T_IQ2_S, T_IQ2_XS, T_IQ2_XXS, T_IQ3_S, T_IQ3_XXS, T_IQ4_NL, T_IQ4_XS,
                        T_Q2_0, T_Q6_K, T_Q8_0)

pytestmark = pytest.mark.gpu

SHAPES = [(T_Q8_0, T_Q8_0, 256, 256), (T_Q8_0, T_Q2_0, 640, 640), (T_IQ3_S, T_IQ3_S, 512, 1024),
          (T_IQ2_XS, T_IQ4_NL, 1024, 256), (T_IQ4_XS, T_Q8_0, 2560, 1024),
          (T_IQ2_XXS, T_Q2_0, 4096, 640), (T_IQ3_XXS, T_IQ2_S, 8192, 512)]


@pytest.mark.parametrize("tg,td,H,F", SHAPES)
@pytest.mark.parametrize("n_tok,k", [(1, 1), (1, 40), (3, 5), (8, 7)])
def test_units_layer(gpu, oracle, tg, td, H, F, n_tok, k):
    E = 48
    if H * F > 1 << 20:
        E, k = 12, min(k, 12)
    rng = np.random.default_rng(tg * 1000 + H + 10 * n_tok + k)
    arena, stride, og, ou, od = packed_experts(rng, E, H, F, tg, td)
    d_arena = dev(arena)
    x = rng.standard_normal((n_tok, H)).astype(np.float32)
    if n_tok == 3:            # groups the short quantizer forms do not take
        x[0, :32] = 0.0
        x[1, 32:64] *= np.float32(1e-36)
        x[2, 70] = np.nan
    ids = np.stack([rng.choice(E, k, replace=False) for _ in range(n_tok)]).astype(np.int32)
    w = rng.random((n_tok, k)).astype(np.float32)
    yo, h = oracle.moe_tokens(H, F, tg, td, arena, stride, x, ids, w, want_h=True)
    P = q4mi.ptr
    if n_tok == 1:
        y = dev(np.zeros(H, np.float32))
        i0, w0 = np.ascontiguousarray(ids[0]), np.ascontiguousarray(w[0])
        q4mi.check(gpu.q4_hip_moe_exec(P(d_arena), stride, i0.ctypes.data_as(ctypes.c_void_p),
                                       w0.ctypes.data_as(ctypes.c_void_p), k, tg, og, tg, ou, td,
                                       od, P(dev(x[0])), None, None, None, P(y), F, H, H),
                   "q4_hip_moe_exec")
        got = host(y)[None]
    else:
        es = np.full((n_tok, 64), -1, np.int32)
        ew = np.zeros((n_tok, 64), np.float32)
        es[:, :k], ew[:, :k] = ids, w
        y = dev(np.zeros((n_tok, H), np.float32))
        q4mi.check(gpu.q4_hip_moe_exec_win(P(d_arena), stride, P(dev(es)), P(dev(ew)),
                                           P(dev(np.full(n_tok, k, np.int32))), n_tok, tg, og, tg,
                                           ou, td, od, P(dev(x)), None, P(y), F, H, H), "exec_win")
        got = host(y)
    ties = check_tokens(oracle, got, yo, h, ids, w, arena, stride, od, td, H, F)
    assert ties <= max(1, n_tok // 2)


@pytest.mark.parametrize("K", [1024, 2048, 2560, 4096])
def test_tall_q80_same_bits_for_every_token_count(gpu, K):
    """A tall Q8_0 matrix: one and two tokens may take the tile kernel, more
    the register kernel; a row's bits do not depend on it."""
    import torch
    from q4mi import synth
    rows = (170 << 20) // (K // 32 * 34) + 3
    w = synth.device_q80(rows * (K // 32 * 34), seed=K)
    x = torch.randn((3, K), device="cuda", generator=torch.Generator("cuda").manual_seed(K))
    ys = []
    for n in (1, 2, 3):
        y = torch.empty((n, rows), device="cuda")
        gpu.q4_mmvq_warm()
        q4mi.check(gpu.q4_mmvq_n(T_Q8_0, q4mi.ptr(w), rows, K, q4mi.ptr(x), q4mi.ptr(y), 0.5, n),
                   "q4_mmvq_n")
        ys.append(y)
    assert torch.equal(ys[0][0], ys[2][0])
    assert torch.equal(ys[1][1], ys[2][1])


@pytest.mark.parametrize("ty", [T_IQ3_S, T_Q8_0, T_IQ4_NL, T_Q2_0, T_IQ2_S, T_Q6_K])
@pytest.mark.parametrize("rows,K", [(1, 512), (3, 8192), (515, 1024), (517, 2560), (66, 4096)])
def test_units_gemv(gpu, oracle, ty, rows, K):
    """Row counts around a wave's task and lane layouts of 8 to 128 units:
    group sums bit-exact, y to 1e-3, the fp32-x entry the same bits as the
    pre-quantized one, a row the same for 1 and 5 tokens."""
    import torch
    from test_gpu_decode import empty
    from conftest import rel_err
    from q4mi import synth
    rng = np.random.default_rng(ty + rows + K)
    w = synth.matrix(rng, ty, rows, K)
    x = rng.standard_normal((5, K)).astype(np.float32)
    q, d = (np.stack([oracle.quant8(x[t])[i] for t in range(5)]) for i in (0, 1))
    dw, P, bits = dev(w), q4mi.ptr, []
    gpu.q4_mmvq_warm()
    for n in (5, 1):
        y, s = empty((n, rows), torch.float32), empty((n, rows, K // 32), torch.int32)
        q4mi.check(gpu.q4mi_mmvq(ty, P(dw), rows, K, P(dev(q)), P(dev(d)), n, P(y), 1.0, P(s)),
                   "q4mi_mmvq")
        y2 = empty((n, rows), torch.float32)
        q4mi.check(gpu.q4_mmvq_n(ty, P(dw), rows, K, P(dev(x)), P(y2), 1.0, n), "q4_mmvq_n")
        assert np.array_equal(host(y).view(np.uint32), host(y2).view(np.uint32))
        bits.append(host(y)[0].view(np.uint32))
        if n == 5:
            sums = host(s)
            rb = w.size // rows
            for t in (0, 4):
                for r in {0, rows // 2, rows - 1}:
                    want = oracle.group_sums(ty, w[r * rb:(r + 1) * rb], K, q[t])
                    assert np.array_equal(sums[t, r], want), (t, r)
            assert rel_err(host(y), oracle.dot8_rows(ty, w, rows, K, x)) <= 1e-3
    assert np.array_equal(bits[0], bits[1])


GEMV_TYPES = [T_IQ3_S, T_Q8_0, T_IQ4_NL, T_Q2_0, T_IQ2_S, T_Q6_K]


def offset_dev(w, by):
    """A device copy of w that starts `by` bytes into an allocation."""
    import torch
    b = torch.zeros(w.size + by, dtype=torch.uint8, device="cuda")
    b[by:] = torch.from_numpy(w).cuda()
    return b[by:]


@pytest.mark.parametrize("ty", GEMV_TYPES)
@pytest.mark.parametrize("rows,K", [(33, 256), (9, 640), (70, 512), (4100, 2048), (37, 2560),
                                    (130, 4096), (35, 8192)])
def test_gemv_weights_two_bytes_into_a_dword(gpu, oracle, ty, rows, K):
    """Weights that start 2 bytes into a dword, and rows that are not whole
    dwords (256 columns of the 256-value superblock types), take the tile
    kernel: group sums bit-exact and y to 1e-3 against the oracle, fp32 x the
    same bits as pre-quantized codes, and the same bits as the register kernel
    gives the same rows where their start is a whole dword."""
    import torch
    from test_gpu_decode import empty
    from conftest import rel_err
    from q4mi import synth
    if K == 640 and ty in (T_IQ3_S, T_IQ2_S, T_Q6_K):
        pytest.skip("not a whole number of superblocks")
    rng = np.random.default_rng(ty + rows + K)
    w = synth.matrix(rng, ty, rows, K)
    x = rng.standard_normal((8, K)).astype(np.float32)
    q, d = (np.stack([oracle.quant8(x[t])[i] for t in range(8)]) for i in (0, 1))
    P, bases = q4mi.ptr, [offset_dev(w, 2), offset_dev(w, 0)]
    dx, dq, dd = dev(x), dev(q), dev(d)
    rb = w.size // rows
    gpu.q4_mmvq_warm()
    for n in (1, 2, 4, 8):
        bits = []
        for dw in bases:
            y, s = empty((n, rows), torch.float32), empty((n, rows, K // 32), torch.int32)
            q4mi.check(gpu.q4mi_mmvq(ty, P(dw), rows, K, P(dq), P(dd), n, P(y), 1.0, P(s)),
                       "q4mi_mmvq")
            y2 = empty((n, rows), torch.float32)
            q4mi.check(gpu.q4_mmvq_n(ty, P(dw), rows, K, P(dx), P(y2), 1.0, n), "q4_mmvq_n")
            assert np.array_equal(host(y).view(np.uint32), host(y2).view(np.uint32))
            bits.append(host(y).view(np.uint32))
            sums = host(s)
            for t in {0, n - 1}:
                for r in {0, rows // 2, rows - 1}:
                    want = oracle.group_sums(ty, w[r * rb:(r + 1) * rb], K, q[t])
                    assert np.array_equal(sums[t, r], want), (t, r)
        assert np.array_equal(bits[0], bits[1]), n
        if n in (1, 8):
            m = min(rows, 200)
            assert rel_err(host(y)[:, :m], oracle.dot8_rows(ty, w[:m * rb], m, K, x[:n])) <= 1e-3


@pytest.mark.parametrize("ty", GEMV_TYPES)
@pytest.mark.parametrize("K", [4096, 8192])
def test_gemv_lane_layouts_same_bits(gpu, ty, K):
    """Rows of 128 and 256 groups: the 64-lane layout (one token, or few rows)
    and the 32-lane one (many rows, three tokens and more) give the same bits."""
    import torch
    rows = 32768 + 5
    bv, bs, at = {T_IQ3_S: (256, 110, 0), T_Q8_0: (32, 34, 0), T_IQ4_NL: (32, 18, 0),
                  T_Q2_0: (64, 18, 0), T_IQ2_S: (256, 82, 0), T_Q6_K: (256, 210, 208)}[ty]
    gen = torch.Generator("cuda").manual_seed(ty + K)
    w = torch.randint(0, 256, (rows * K // bv, bs), dtype=torch.uint8, device="cuda", generator=gen)
    w[:, at + 1] = w[:, at + 1] % 8 + 0x10          # block scales 2^-11 .. 2^-9
    x = torch.randn((5, K), device="cuda", generator=gen)
    few = 300 * (K // bv) * bs
    ys = []
    for n, r in ((1, rows), (3, rows), (5, rows), (5, 300)):
        y = torch.empty((n, r), device="cuda")
        ww = w if r == rows else w.view(-1)[:few]
        q4mi.check(gpu.q4_mmvq_n(ty, q4mi.ptr(ww), r, K, q4mi.ptr(x), q4mi.ptr(y), 1.0, n),
                   "q4_mmvq_n")
        ys.append(y)
    one, three, five, short = ys
    assert bool(torch.isfinite(five).all())
    assert torch.equal(one[0], three[0]) and torch.equal(three, five[:3])
    assert torch.equal(five[:, :300], short)


# exponents of a group's largest magnitude: the short divisions' range is 2^-100 .. 2^100
# (both ends inside); the rest of the float range takes the full divides
@pytest.mark.parametrize("exps,calls", [((0,), 4096), ((-100,), 32), ((-101,), 32), ((-126,), 32),
                                        ((99,), 32), ((100,), 32), ((126,), 32),
                                        ((-126, -101, -100, -30, 0, 40, 99, 100, 126), 64)])
def test_in_block_quantizer_every_mantissa(gpu, exps, calls):
    """The quantizer inside the decode, window and GEMV kernels (eight values a
    lane, short exact divisions) gives the scales and codes of q4mi_quant8's
    IEEE divides bit for bit: all 2^23 mantissas of a group's largest magnitude
    at exponent 0, 65536 evenly spread ones (first and last among them) at the
    ends of the short range and beyond, and exponents mixed within a wave.  The
    other values are the 126.5 .. 0.5 steps, where the code rounds to even, and
    their neighbours.  An identity matrix (Q8_0, block scales 1) shows every
    value's code times its group's scale, one rounding of the two."""
    import torch
    K, n = 8192, 8
    dv = dict(device="cuda")
    w = torch.zeros((K, K // 32, 34), dtype=torch.uint8, **dv)
    w[:, :, 1] = 0x3c                                        # fp16 1.0
    r = torch.arange(K, **dv)
    w[r, r // 32, 2 + r % 32] = 1
    gen = torch.Generator("cuda").manual_seed(calls)
    groups = n * K // 32
    last = (1 << 23) - 1
    bad = torch.zeros((), dtype=torch.int64, **dv)
    P = q4mi.ptr
    for c in range(calls):
        at = torch.arange(c * groups, (c + 1) * groups, **dv)
        man = (at * last).div(calls * groups - 1, rounding_mode="floor")
        e = torch.tensor(exps, **dv)[torch.randint(0, len(exps), (groups,), generator=gen, **dv)]
        a = (((e + 127) << 23) | man).to(torch.int32).view(torch.float32)[:, None]
        step = torch.randint(-127, 127, (groups, 32), generator=gen, **dv) + 0.5
        x = (step / 127 * a)
        near = torch.randint(-1, 2, (groups, 32), generator=gen, dtype=torch.int32, **dv)
        x = (x.view(torch.int32) + near).view(torch.float32)
        pos = torch.randint(0, 32, (groups, 1), generator=gen, **dv)
        x.scatter_(1, pos, torch.where(pos % 2 == 0, a, -a))
        x = x.reshape(n, K).contiguous()
        q = torch.empty((n, K), dtype=torch.int8, **dv)
        d = torch.empty((n, K // 32), **dv)
        bs = torch.empty((n, K // 32), dtype=torch.int32, **dv)
        y = torch.empty((n, K), **dv)
        q4mi.check(gpu.q4mi_quant8(P(x), None, n, K, P(q), P(d), P(bs)), "q4mi_quant8")
        q4mi.check(gpu.q4_mmvq_n(T_Q8_0, P(w), K, K, P(x), P(y), 1.0, n), "q4_mmvq_n")
        want = q.float() * d.repeat_interleave(32, dim=1)
        bad += (y != want).sum()
        if c == 0:
            # (-128: every code of a group at -126, whose 127 / a is infinite)
            assert int(q.int().abs().max()) >= 127 and bool(torch.isfinite(want).all())
    assert int(bad) == 0
