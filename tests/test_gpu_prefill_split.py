"""Prefill attention over a split kv range (grout_fmha_prefill_ws): forced range
counts against the oracle and against the unsplit kernel, at the edges of the
ranges (one tile each, ranges past a block's last tile, a last range whose rows
are partly or wholly masked), and the rule that picks them."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle as O
from test_gpu_kernels import D, assert_close, dev, host_f32, normal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,Hq,Hkv,pos0,splits", [
    (1, 32, 8, 1600, [2, 3, 16]), (61, 32, 8, 1535, [2, 5, 13]),
    (17, 16, 8, 1647, [7, 16]),    # 26 tiles, row 0 sees only 25 full ones and 48 of the last
    (65, 10, 2, 1599, [4, 16]),    # G = 5: 12 positions per block, ragged last block
    (40, 7, 1, 1580, [3]), (16, 3, 3, 1700, [16]), (100, 64, 8, 2000, [2, 16])])
def test_split_ranges_vs_oracle(gpu, monkeypatch, S, Hq, Hkv, pos0, splits):
    print(f"[case] split prefill S={S} Hq={Hq} Hkv={Hkv} pos0={pos0}", flush=True)
    max_ctx = pos0 + S + 70
    q = normal(f"sq{S}", (S, Hq, D))
    kc, vc = normal(f"sk{S}", (Hkv, max_ctx, D)), normal(f"sv{S}", (Hkv, max_ctx, D))
    ref = O.attention_prefill_rows(q, kc, vc, pos0, nthreads=8)
    kd, vd = dev(kc), dev(vc)
    kd[:, pos0 + S:] = float("nan")  # rows past the chunk are never read
    vd[:, pos0 + S:] = float("nan")
    monkeypatch.setenv("GROUT_FMHA_PREFILL_SPLITS", "1")
    one = gpu.ops.fmha_prefill(dev(q), kd, vd, pos0)
    for n in splits:
        monkeypatch.setenv("GROUT_FMHA_PREFILL_SPLITS", str(n))
        out = gpu.ops.fmha_prefill(dev(q), kd, vd, pos0)
        torch.cuda.synchronize()
        assert_close(host_f32(out), ref, f"{n} ranges")
        # f16 P against each range's own reference point: one ulp, as decode splits
        assert np.abs(host_f32(out) - host_f32(one)).max() <= 2e-3


def test_dominant_key_and_masked_range(gpu, monkeypatch):
    """One key far above the rest in one range, the other ranges' weight nil;
    then rows whose last range is wholly masked (they see none of its tile)."""
    S, Hq, Hkv, pos0 = 33, 4, 1, 1631  # tiles 0..25; rows 0..31 end inside tile 25
    q = normal("dq", (S, Hq, D))
    kc, vc = normal("dk", (Hkv, 1700, D)), normal("dv", (Hkv, 1700, D))
    kf = kc.view(np.float16)
    kf[0, 700] = q.view(np.float16)[0, 0] * np.float16(4)
    ref = O.attention_prefill_rows(q, kc, vc, pos0, nthreads=8)
    for n in (1, 13, 16):
        monkeypatch.setenv("GROUT_FMHA_PREFILL_SPLITS", str(n))
        out = gpu.ops.fmha_prefill(dev(q), dev(kc), dev(vc), pos0)
        torch.cuda.synchronize()
        assert_close(host_f32(out), ref, f"dominant key, {n} ranges")


def test_small_workspace_takes_fewer_ranges(gpu):
    L, S, Hq, Hkv, pos0 = gpu.lib(), 61, 32, 8, 4000
    need = L.grout_fmha_prefill_workspace_bytes(S, pos0, Hq, Hkv)
    per = S * Hq * 130 * 4
    assert need >= 2 * per and need % per == 0
    q = dev(normal("wq", (S, Hq, D)))
    kc, vc = dev(normal("wk", (Hkv, 4096, D))), dev(normal("wv", (Hkv, 4096, D)))
    ref = gpu.ops.fmha_prefill(q, kc, vc, pos0)
    p = lambda t: C.c_void_p(t.data_ptr())
    for nbytes in (need, 3 * per + 4, per, 0):
        guard = torch.full((need // 4 + 64,), 3.0, device="cuda")
        out = torch.empty_like(q)
        assert L.grout_fmha_prefill_ws(p(q), p(kc), p(vc), p(out), p(guard), nbytes, S, pos0, Hq,
                                       Hkv, D, 4096 * D, 1 / np.sqrt(D), None) == 0
        torch.cuda.synchronize()
        assert (out.float() - ref.float()).abs().max() <= 2e-3
        assert (guard[nbytes // 4:] == 3).all()


def test_split_captures_into_a_graph(gpu):
    S, Hq, Hkv, pos0 = 19, 16, 8, 3000
    q = dev(normal("gq", (S, Hq, D)))
    kc, vc = dev(normal("gk", (Hkv, 3072, D))), dev(normal("gv", (Hkv, 3072, D)))
    ref = gpu.ops.fmha_prefill(q, kc, vc, pos0)
    out = torch.empty_like(q)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        gpu.ops.fmha_prefill(q, kc, vc, pos0, out=out)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        gpu.ops.fmha_prefill(q, kc, vc, pos0, out=out)
    for _ in range(3):
        out.fill_(9.0)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)
