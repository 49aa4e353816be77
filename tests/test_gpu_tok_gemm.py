"""The few-token projection kernel (grout_amd/csrc/tok_gemm.hip) against fp64
products of the f16 weights that grout_qweight_dequant gives (themselves
checked bit for bit in test_gpu_quant.py), at the edges of its tiles.

The kernel is internal to the engine, so it is called by its C++ symbol.  Its
products are exact in fp32 and K of them are added in fp32, in MFMA blocks,
then over the ranges of K: within K * 2^-24 * sum|w x| of the exact sum (each
of fewer than K additions rounds a partial sum no larger than sum|w x|), plus
half an f16 ulp for the rows it rounds itself."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle as O
from test_gpu_quant import call, ptr, random_blocks, upload

pytestmark = pytest.mark.gpu

SYM = "_ZN5grout15launch_tok_gemmEiPKvS1_PvPfliiiiP12ihipStream_t"
OK = "_ZN5grout11tok_gemm_okEiiii"


def tok_gemm(L):
    f = getattr(L, SYM)
    f.restype = C.c_int
    f.argtypes = [C.c_int] + [C.c_void_p] * 4 + [C.c_long] + [C.c_int] * 4 + [C.c_void_p]
    return f


def matrix(fmt, n, k, seed, L):
    if fmt == 0:
        w = torch.from_numpy(np.random.default_rng(seed).standard_normal((n, k)).astype(
            np.float16)).cuda()
        return w, w
    wq = upload(fmt, random_blocks(fmt, n, k, seed), n, k, L)
    w = torch.empty((n, k), dtype=torch.float16, device="cuda")
    call(L, "grout_qweight_dequant", fmt, ptr(wq), n, k, ptr(w), None)
    return wq, w


# one token tile and its edges, every instantiated tile count, two token blocks
TOKENS = [2, 15, 16, 17, 33, 49, 64, 65, 96, 97, 113, 128, 129, 160, 161, 320, 321, 480]
# rows: fewer than a workgroup's 64, a ragged last workgroup, whole ones;
# K: one sub-step (Q8_0, f16), an odd number of them, one superblock, the
# ranges' ragged end
SHAPES = {0: [(4, 128), (100, 384), (192, 1152)], 8: [(20, 128), (100, 384), (192, 1152)],
          12: [(4, 256), (100, 768), (192, 2304)], 13: [(4, 256), (100, 768), (192, 2304)],
          14: [(4, 256), (100, 768), (192, 2304)]}


@pytest.mark.parametrize("fmt", [0, O.Q8_0, O.Q4_K, O.Q5_K, O.Q6_K])
@pytest.mark.parametrize("m", TOKENS)
def test_tok_gemm_rows_and_partial_sums(gpu, fmt, m):
    from grout_amd import lib

    L = lib()
    f = tok_gemm(L)
    ok = getattr(L, OK)
    for n, k in SHAPES[fmt]:
        if not ok(fmt, m, n, k):
            assert (fmt == 0 and m > 96) or (fmt == O.Q8_0 and m > 320)
            y = torch.zeros((m, n), dtype=torch.float16, device="cuda")
            assert f(0, ptr(y), ptr(y), ptr(y), None, n, m, n, k, 1, None) != 0
            continue
        print(f"[case] tok_gemm fmt={fmt} m={m} n={n} k={k}", flush=True)
        wq, w = matrix(fmt, n, k, 3 + m, L)
        g = torch.Generator(device="cuda")
        g.manual_seed(m)
        x = torch.empty((m, k), dtype=torch.float16, device="cuda").normal_(generator=g)
        ref = x.double() @ w.double().T
        mag = x.double().abs() @ w.double().abs().T
        bound = k * 2.0 ** -24 * mag
        # f16 rows, written into columns 8 .. of wider rows whose rest stays
        ld = n + 12
        y = torch.full((m, ld), 7.0, dtype=torch.float16, device="cuda")
        assert f(fmt, ptr(wq), ptr(x), C.c_void_p(y.data_ptr() + 16), None, ld, m, n, k, 1,
                 None) == 0
        half_ulp = 2.0 ** (torch.floor(torch.log2(ref.abs().clamp(min=2.0 ** -14))) - 11)
        assert ((y[:, 8:8 + n].double() - ref).abs() <= bound + 1.01 * half_ulp).all()
        assert (y[:, :8] == 7).all() and (y[:, 8 + n:] == 7).all()
        # partial sums over the ranges of K
        units = (k // 128 + 1) // 2
        for splits in {units, (units + 1) // 2} - {0, 1}:
            per = (units + splits - 1) // splits
            splits = (units + per - 1) // per
            if splits == 1:
                continue
            part = torch.full((splits, m, ld), 5.0, dtype=torch.float32, device="cuda")
            assert f(fmt, ptr(wq), ptr(x), None, C.c_void_p(part.data_ptr() + 32), ld, m, n, k,
                     splits, None) == 0
            got = part[:, :, 8:8 + n].double().sum(0)
            assert ((got - ref).abs() <= bound).all()
            assert (part[:, :, :8] == 5).all() and (part[:, :, 8 + n:] == 5).all()


PAIR = "_ZN5grout20launch_tok_gemm_pairEiPKviiS1_iS1_PvPfliiiP12ihipStream_t"


@pytest.mark.parametrize("fmt", [O.Q4_K, O.Q5_K])
@pytest.mark.parametrize("m", [2, 17, 33, 131, 161])
@pytest.mark.parametrize("na,nb", [(192, 64), (100, 20), (4, 128)])
def test_tok_gemm_pair_equals_two_launches(gpu, fmt, m, na, nb):
    """A pair launch writes the same bits as one launch per matrix."""
    from grout_amd import lib

    L, k = lib(), 768
    f, g = tok_gemm(L), getattr(L, PAIR)
    g.restype = C.c_int
    g.argtypes = [C.c_int, C.c_void_p, C.c_int, C.c_int, C.c_void_p, C.c_int] + [C.c_void_p] * 3 \
        + [C.c_long] + [C.c_int] * 3 + [C.c_void_p]
    (wa, _), (wb, _) = matrix(fmt, na, k, 1, L), matrix(O.Q6_K, nb, k, 2, L)
    x = torch.randn((m, k), dtype=torch.float16, device="cuda")
    ld = na + nb
    off = lambda t, n: C.c_void_p(t.data_ptr() + n * t.element_size())
    for splits in (1, 3):
        y, z = (torch.full((m, ld), 7.0, dtype=torch.float16, device="cuda") for _ in range(2))
        p, q = (torch.full((splits, m, ld), 5.0, device="cuda") for _ in range(2))
        assert f(fmt, ptr(wa), ptr(x), ptr(y), ptr(p), ld, m, na, k, splits, None) == 0
        assert f(O.Q6_K, ptr(wb), ptr(x), off(y, na), off(p, na), ld, m, nb, k, splits, None) == 0
        assert g(fmt, ptr(wa), na, O.Q6_K, ptr(wb), nb, ptr(x), ptr(z), ptr(q), ld, m, k, splits,
                 None) == 0
        assert torch.equal(y, z) and torch.equal(p, q)
    assert g(O.Q6_K, ptr(wb), nb, O.Q6_K, ptr(wb), nb, ptr(x), ptr(z), ptr(q), ld, m, k, 1,
             None) != 0


def test_tok_gemm_refuses_what_it_does_not_cover(gpu):
    from grout_amd import lib

    ok = getattr(lib(), OK)
    assert ok(0, 2, 4, 128) and ok(0, 96, 4, 128) and not ok(0, 97, 4, 128)
    assert not ok(0, 1, 4, 128)          # one token: the decode GEMVs
    assert not ok(0, 2, 6, 128)          # rows in fours
    assert not ok(0, 2, 4, 120)          # K in whole sub-steps
    assert not ok(O.Q4_K, 2, 4, 128) and ok(O.Q8_0, 2, 4, 128)
    assert ok(O.Q6_K, 480, 4, 256) and not ok(O.Q6_K, 481, 4, 256)
    assert ok(O.Q8_0, 320, 4, 128) and not ok(O.Q8_0, 321, 4, 128)
    assert not ok(2, 2, 4, 256)          # an unknown format
