"""The longer-prompt projection kernel (grout_amd/csrc/tile_gemm.hip) against
fp64 products, at the edges of its tiles and ranges.

The kernel is internal to the engine, so it is called by its C++ symbol.  Its
products are exact in fp32 and K of them are added in fp32, in MFMA blocks,
then over the ranges of K: within K * 2^-24 * sum|w x| of the exact sum, plus
half an f16 ulp for the rows it rounds itself."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu

SYM = "_ZN5grout16launch_tile_gemmEPKvS1_PvPfliiiiP12ihipStream_t"
SPLITS = "_ZN5grout16tile_gemm_splitsEiii"
PAYS = "_ZN5grout14tile_gemm_paysEii"


def tile_gemm():
    from grout_amd import lib

    f = getattr(lib(), SYM)
    f.restype = C.c_int
    f.argtypes = [C.c_void_p] * 4 + [C.c_long] + [C.c_int] * 4 + [C.c_void_p]
    return f


def at(t, n=0):
    return C.c_void_p(t.data_ptr() + n * t.element_size())


# every block count of a wave and its edges, two and three token tiles
@pytest.mark.parametrize("m", [1, 32, 33, 64, 65, 96, 97, 128, 129, 193, 257, 300])
# rows: fewer than a tile, a ragged last tile, more tiles than XCDs; K: the
# fewest steps, an odd number of them, many
@pytest.mark.parametrize("n,k", [(4, 128), (132, 192), (260, 1152), (1284, 832)])
def test_tile_gemm_rows_and_partial_sums(gpu, m, n, k):
    f = tile_gemm()
    print(f"[case] tile_gemm m={m} n={n} k={k}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(m + n)
    w = torch.empty((n, k), dtype=torch.float16, device="cuda").normal_(generator=g)
    x = torch.empty((m, k), dtype=torch.float16, device="cuda").normal_(generator=g)
    ref = x.double() @ w.double().T
    bound = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    # f16 rows, written into columns 8 .. of wider rows whose rest stays
    ld = n + 12
    y = torch.full((m, ld), 7.0, dtype=torch.float16, device="cuda")
    assert f(at(w), at(x), at(y, 8), None, ld, m, n, k, 1, None) == 0
    half_ulp = 2.0 ** (torch.floor(torch.log2(ref.abs().clamp(min=2.0 ** -14))) - 11)
    assert ((y[:, 8:8 + n].double() - ref).abs() <= bound + 1.01 * half_ulp).all()
    assert (y[:, :8] == 7).all() and (y[:, 8 + n:] == 7).all()
    # partial sums: two ranges, ragged ones, one step each
    steps = k // 64
    for splits in sorted({2, 3, steps} & set(range(2, 19))):
        if -(-steps // splits) * (splits - 1) >= steps:
            assert f(at(w), at(x), None, at(y), ld, m, n, k, splits, None) != 0
            continue
        part = torch.full((splits, m, ld), 5.0, dtype=torch.float32, device="cuda")
        assert f(at(w), at(x), None, at(part, 8), ld, m, n, k, splits, None) == 0
        assert ((part[:, :, 8:8 + n].double().sum(0) - ref).abs() <= bound).all()
        assert (part[:, :, :8] == 5).all() and (part[:, :, 8 + n:] == 5).all()


def test_tile_gemm_rule_and_refusals(gpu):
    from grout_amd import lib

    L, f = lib(), tile_gemm()
    pays, splits = getattr(L, PAYS), getattr(L, SPLITS)
    pays.restype = C.c_bool
    assert pays(512, 2560) and pays(131, 6144) and not pays(512, 6144) and not pays(64, 2560)
    assert not pays(4097, 128) and pays(4096, 128)
    for m, n, k in ((65, 4, 128), (131, 2560, 4096), (512, 2560, 9728), (4096, 128, 32768)):
        s, steps = splits(m, n, k), k // 64
        assert 1 <= s <= 12 and -(-steps // s) * (s - 1) < steps
    t = torch.zeros((256, 256), dtype=torch.float16, device="cuda")
    p = at(t)
    assert f(p, p, p, None, 128, 4, 6, 128, 1, None) != 0      # rows in fours
    assert f(p, p, p, None, 128, 4, 128, 96, 1, None) != 0     # K in whole steps
    assert f(p, p, p, None, 130, 4, 128, 128, 1, None) != 0    # row stride
    assert f(p, p, p, None, 128, 4, 128, 128, 2, None) != 0    # ranges without their buffer
