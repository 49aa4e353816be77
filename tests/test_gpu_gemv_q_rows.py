"""Low-bit GEMV forms at the lines of their dispatch: two rows per 16-lane team
(tall Q4_K / Q5_K, the norm-folded 8-row workgroups from 4096 rows), one row
below those lines, and the short K that used to take the looped kernel.  Bars as
test_gpu_quant.py: one f16 ulp plus 1e-5 * sum(|w x| + m |x|) of the fp64
oracle, inputs of the norm form rounded as the norm kernel rounds them."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle as O
from test_gpu_quant import call, min_term, ptr, random_blocks, ulp, upload

pytestmark = pytest.mark.gpu

FMTS = [O.Q8_0, O.Q4_K, O.Q5_K, O.Q6_K]


def bound(fmt, blocks, n, k, x):
    w = O.dequant(fmt, blocks, n * k, decode=True).reshape(n, k).astype(np.float64)
    xs = x.astype(np.float64)
    y = w @ xs
    return y, ulp(y) + 1e-5 * (np.abs(w) @ np.abs(xs) + min_term(fmt, blocks, n, k) @ np.abs(xs))


@pytest.mark.parametrize("fmt", FMTS)
# 16384 rows are tall; 16417 leaves a ragged last workgroup of one row (32 rows
# each); K of 2 and 4 pieces per lane with no slice count that fits upwards
@pytest.mark.parametrize("n,k", [(16383, 512), (16384, 512), (16417, 2560), (4096, 1024),
                                 (1024, 2048), (37, 1024)])
def test_plain_rows(gpu, fmt, n, k):
    from grout_amd import lib

    print(f"[case] gemv_q rows fmt={fmt} n={n} k={k}", flush=True)
    L = lib()
    blocks = random_blocks(fmt, n, k, n + k)
    x = np.random.default_rng(k).standard_normal(k).astype(np.float16)
    wq, y = upload(fmt, blocks, n, k, L), torch.zeros(n + 8, dtype=torch.float16, device="cuda")
    xd = torch.from_numpy(x).cuda()
    call(L, "grout_gemv_q", fmt, ptr(wq), ptr(xd), ptr(y), n, k, None)
    ref, tol = bound(fmt, blocks, n, k, x)
    got = y.cpu().numpy().astype(np.float64)
    assert (np.abs(got[:n] - ref) <= tol).all() and (got[n:] == 0).all()


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("residual", [True, False])
# rows at the two-row lines (4095 / 4096, Q8_0 8191 / 8192) and a ragged last
# workgroup of 8; K with 2 (2560: three slices of 2, one clipped) pieces per slice
@pytest.mark.parametrize("n,k", [(4095, 1024), (4096, 2560), (4099, 4096), (8191, 1024),
                                 (8196, 2560), (16400, 2560)])
def test_norm_rows(gpu, fmt, residual, n, k):
    from grout_amd import lib

    print(f"[case] gemv_q norm rows fmt={fmt} n={n} k={k} residual={residual}", flush=True)
    L, eps = lib(), 1e-6
    blocks = random_blocks(fmt, n, k, n)
    rng = np.random.default_rng(n + k)
    x, res = (rng.standard_normal(k).astype(np.float16) for _ in range(2))
    gam = rng.uniform(0.8, 1.2, k).astype(np.float16)
    c = x.astype(np.float32) + (res.astype(np.float32) if residual else np.float32(0))
    inv = 1.0 / np.sqrt((c.astype(np.float64) ** 2).mean() + eps)
    xp = (c.astype(np.float64) * inv * gam.astype(np.float64)).astype(np.float16)
    dev = lambda a: torch.from_numpy(a).cuda()
    wq = upload(fmt, blocks, n, k, L)
    y, ro = (torch.zeros(m, dtype=torch.float16, device="cuda") for m in (n + 8, k))
    xd, gd, rd = dev(x), dev(gam), dev(res)
    call(L, "grout_gemv_q_rms_norm", fmt, ptr(wq), ptr(rd) if residual else None, ptr(xd), ptr(gd),
         ptr(ro), ptr(y), n, k, eps, None)
    ref, tol = bound(fmt, blocks, n, k, xp)
    # x' may round the other way in single elements (1/rms in another order): one
    # ulp of x', 2^-10 relative, on each weight's term
    w = O.dequant(fmt, blocks, n * k, decode=True).reshape(n, k).astype(np.float64)
    tol = tol + 2.0 ** -10 * (np.abs(w) @ np.abs(xp.astype(np.float64)))
    got = y.cpu().numpy().astype(np.float64)
    assert (np.abs(got[:n] - ref) <= tol).all() and (got[n:] == 0).all()
    assert np.array_equal(ro.cpu().numpy(), c.astype(np.float16))


PAIR = "_ZN5grout23launch_gemv_q_norm_pairEiPKviiS1_iS1_S1_S1_PvfS2_iP12ihipStream_t"


@pytest.mark.parametrize("fmt", [O.Q4_K, O.Q5_K])
@pytest.mark.parametrize("residual", [True, False])
@pytest.mark.parametrize("na,nb,k", [(4096, 1024, 2560), (5120, 1, 4096), (4099, 1021, 5120),
                                     (8192, 9, 6144)])
def test_norm_pair_equals_two_launches(gpu, fmt, residual, na, nb, k):
    """The pair launch (internal: by its C++ symbol) against one launch per
    matrix: the first matrix and residual_out bit for bit (the same kernel
    form), the second within the forms' different summation order."""
    from grout_amd import lib

    print(f"[case] gemv_q pair fmt={fmt} na={na} nb={nb} k={k} residual={residual}", flush=True)
    L, eps = lib(), 1e-6
    f = getattr(L, PAIR)
    f.restype = C.c_int
    f.argtypes = [C.c_int, C.c_void_p, C.c_int, C.c_int, C.c_void_p, C.c_int] + [C.c_void_p] * 4 \
        + [C.c_float, C.c_void_p, C.c_int, C.c_void_p]
    ba, bb = random_blocks(fmt, na, k, 1), random_blocks(O.Q6_K, nb, k, 2)
    wa, wb = upload(fmt, ba, na, k, L), upload(O.Q6_K, bb, nb, k, L)
    g = torch.Generator(device="cuda")
    g.manual_seed(k)
    x, res = (torch.empty(k, dtype=torch.float16, device="cuda").normal_(generator=g)
              for _ in range(2))
    gam = torch.empty(k, dtype=torch.float16, device="cuda").uniform_(0.8, 1.2, generator=g)
    y, z = (torch.full((na + nb + 4,), 7.0, dtype=torch.float16, device="cuda") for _ in range(2))
    ro, rp = (torch.zeros(k, dtype=torch.float16, device="cuda") for _ in range(2))
    r = ptr(res) if residual else None
    call(L, "grout_gemv_q_rms_norm", fmt, ptr(wa), r, ptr(x), ptr(gam), ptr(ro), ptr(y), na, k,
         eps, None)
    call(L, "grout_gemv_q_rms_norm", O.Q6_K, ptr(wb), r, ptr(x), ptr(gam), None,
         C.c_void_p(y.data_ptr() + 2 * na), nb, k, eps, None)
    assert f(fmt, ptr(wa), na, O.Q6_K, ptr(wb), nb, r, ptr(x), ptr(gam), ptr(rp), eps, ptr(z), k,
             None) == 0
    torch.cuda.synchronize()
    assert torch.equal(y[:na], z[:na]) and torch.equal(ro, rp) and (z[na + nb:] == 7).all()
    c = x.float() + (res.float() if residual else 0)
    xp = (c * torch.rsqrt((c * c).mean() + eps) * gam.float()).cpu().numpy()
    w = O.dequant(O.Q6_K, bb, nb * k, decode=True).reshape(nb, k).astype(np.float64)
    a, b = (t[na:na + nb].cpu().numpy().astype(np.float64) for t in (y, z))
    # x' is the same; fp32 sums of k terms in another order, then one f16 rounding
    assert (np.abs(a - b) <= ulp(a) + 1e-5 * (np.abs(w) @ np.abs(xp))).all()


def test_norm_pair_refuses_other_forms(gpu):
    from grout_amd import lib

    ok = getattr(lib(), "_ZN5grout19gemv_q_norm_pair_okEiiii")
    assert ok(O.Q4_K, O.Q6_K, 4096, 2560) and ok(O.Q5_K, O.Q6_K, 4096, 6144)
    assert not ok(O.Q4_K, O.Q6_K, 4095, 2560) and not ok(O.Q4_K, O.Q6_K, 4096, 2048)
    assert not ok(O.Q4_K, O.Q6_K, 4096, 6656) and not ok(O.Q4_K, O.Q6_K, 4096, 2816)
    assert not ok(O.Q6_K, O.Q4_K, 4096, 2560) and not ok(O.Q8_0, O.Q6_K, 8192, 2560)
