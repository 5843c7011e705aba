"""GPU parity of the dense int8 / f16 GEMV and the whole MoE block
(escha_mlx/quant.py w8a16 contract, models/qwen3_5_moe.py:257-273,
ref.moe_block escha_mlx/ref.py:314-349), through the C-ABI.

One-hot inputs pin every weight bit-exactly (a single product: x = e_k makes
y[:, o] the contract weight f16(f32(w8[o, k]) * f32(scale[o]))); other inputs
are held to the reference's own w8a16 bar (max |diff| / max |want| < 2e-3,
tests/test_mlx_cpu.py:55-65 of the reference) against its golden and against
a float64 product of the contract weights.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import ref_np as R

from .conftest import has_gpu, moe_block_weights

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not has_gpu(), reason="needs a ROCm GPU")]

DEV = "cuda"


@pytest.fixture(autouse=True)
def _announce(request):
    print(f"\n[gpu case] {request.node.nodeid}", flush=True)
    yield
    torch.cuda.synchronize()


def ops():
    from escha_mlx_amd import ops as o
    return o


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _rel(got, want):
    g, w = got.astype(np.float64), want.astype(np.float64)
    return np.abs(g - w).max() / np.abs(w).max()


def test_w8a16_vs_reference_golden(w8a16_golden):
    w8, scale, x, want = w8a16_golden
    got = ops().w8a16(_dev(x), _dev(w8), _dev(scale)).cpu().numpy()
    assert _rel(got, want) < 2e-3
    wf = (w8.astype(np.float32) * scale[:, None]).astype(np.float16).astype(np.float64)
    assert _rel(got, x.astype(np.float64) @ wf.T) < 2e-3


# K = 128 / 256 / 384: 8 / 16 / 32 lanes per row (384: 24 chunks, 8 lanes
# idle); 5120 and 8192: 5 and 8 chunks per lane, at most 2 rows per launch
@pytest.mark.parametrize("K", [128, 256, 384, 512, 1024, 2048, 4096, 5120, 8192])
@pytest.mark.parametrize("m", [1, 3, 8, 11])
def test_w8a16_one_hot_bit_exact(K, m):
    rng = np.random.default_rng(K + m)
    O = (384 if K < 4096 else 96) + 1  # a partial last wave-step where rows share a wave
    w8 = rng.integers(-128, 128, size=(O, K), dtype=np.int8)
    scale = rng.uniform(1e-3, 5e-3, O).astype(np.float16).astype(np.float32)
    ks = rng.integers(0, K, size=m)
    x = np.zeros((m, K), np.float16)
    x[np.arange(m), ks] = 1.0
    got = ops().w8a16(_dev(x), _dev(w8), _dev(scale)).cpu().numpy()
    for r, k in enumerate(ks):
        want = (w8[:, k].astype(np.float32) * scale).astype(np.float16)
        assert np.array_equal(got[r].view(np.uint16), want.view(np.uint16)), r


@pytest.mark.parametrize("K,m", [(2048, 1), (512, 4), (1024, 8), (2048, 13), (256, 3), (384, 9),
                                 (5120, 5), (8192, 3)])
def test_w8a16_vs_f64_and_deterministic(K, m):
    rng = np.random.default_rng(3 * K + m)
    O = 640
    w8 = rng.integers(-128, 128, size=(O, K), dtype=np.int8)
    scale = rng.uniform(1e-3, 5e-3, O).astype(np.float32)
    x = rng.standard_normal((m, K)).astype(np.float16)
    args = (_dev(x), _dev(w8), _dev(scale))
    y = ops().w8a16(*args)
    wf = (w8.astype(np.float32) * scale[:, None]).astype(np.float16).astype(np.float64)
    assert _rel(y.cpu().numpy(), x.astype(np.float64) @ wf.T) < 2e-3
    assert torch.equal(ops().w8a16(*args), y)


@pytest.mark.parametrize("K", [64, 200, 256, 512, 1024, 2048, 4096])
@pytest.mark.parametrize("m", [1, 5, 9])
def test_gemv_f16w_one_hot_and_f64(K, m):
    rng = np.random.default_rng(7 * K + m)
    O = 256
    w = (rng.standard_normal((O, K)) * 0.05).astype(np.float16)
    ks = rng.integers(0, K, size=m)
    x = np.zeros((m, K), np.float16)
    x[np.arange(m), ks] = 1.0
    got = ops().gemv_f16w(_dev(x), _dev(w)).cpu().numpy()
    for r, k in enumerate(ks):
        assert np.array_equal(got[r].view(np.uint16), w[:, k].view(np.uint16))
    xr = rng.standard_normal((m, K)).astype(np.float16)
    got = ops().gemv_f16w(_dev(xr), _dev(w)).cpu().numpy()
    assert _rel(got, xr.astype(np.float64) @ w.astype(np.float64).T) < 2e-3


def test_shared_act_and_block_out_vs_oracle():
    rng = np.random.default_rng(9)
    g = (rng.standard_normal((5, 512)) * 3).astype(np.float16)
    u = rng.standard_normal((5, 512)).astype(np.float16)
    got = ops().moe_shared_act(_dev(g), _dev(u)).cpu().numpy()
    want = R.shared_act(g, u)
    # device expf vs numpy exp: at most one f16 ulp apart
    ulps = np.abs(got.view(np.int16).astype(np.int32) - want.view(np.int16).astype(np.int32))
    assert ulps.max() <= 1 and (ulps > 0).mean() < 0.01
    y = rng.standard_normal((5, 512)).astype(np.float16)
    sh = rng.standard_normal((5, 512)).astype(np.float16)
    shg = (rng.standard_normal((5, 1)) * 2).astype(np.float16)
    got = ops().moe_block_out(_dev(y), _dev(sh), _dev(shg)).cpu().numpy()
    sg = np.float32(1) / (np.float32(1) + np.exp(-shg.astype(np.float32)))
    want = (y.astype(np.float32) + sh.astype(np.float32) * sg).astype(np.float16)
    ulps = np.abs(got.view(np.int16).astype(np.int32) - want.view(np.int16).astype(np.int32))
    assert ulps.max() <= 1


def _block(v):
    from escha_mlx_amd import moe
    E, H = v["blk_gate_w"].shape
    gu = moe.EschaExperts(v["blk_gu_code"], v["blk_gu_rin"], v["blk_gu_rout"], device=DEV)
    dn = moe.EschaExperts(v["blk_dn_code"], v["blk_dn_rin"], v["blk_dn_rout"], device=DEV)
    shared = {f"{p}_{leaf}": v[f"blk_sh_{p}_{leaf}"] for p in ("gate", "up", "down")
              for leaf in ("w8", "scale")}
    return moe.EschaSparseMoeBlock(H, E, 2, gu, dn, v["blk_gate_w"], v["blk_shg_w"], shared)


def test_moe_block_vs_oracle_and_reference(ref_vectors):
    """The whole block against the oracle (same rounding points) and against
    ref.moe_block's own output (which keeps the routed sum in float64)."""
    v = ref_vectors
    blk = _block(v)
    x = _dev(v["blk_x"])
    y = blk(x)
    got = y.cpu().numpy()
    want = R.moe_block(v["blk_x"], moe_block_weights(v), 2)
    assert _rel(got, want) < 5e-3
    assert _rel(got, v["blk_y"]) < 5e-3
    assert torch.equal(blk(x), y)


@pytest.mark.parametrize("K", [256, 2048])
def test_q8_embed_bit_exact(K):
    """Embedding rows are the contract weights, bit for bit (the same rounding
    the w8a16 golden pins); an id outside the table gives a NaN row."""
    from escha_mlx_amd import quant
    rng = np.random.default_rng(K)
    N = 300
    w8 = rng.integers(-128, 128, size=(N, K), dtype=np.int8)
    scale = rng.uniform(1e-3, 5e-3, N).astype(np.float16)  # f16 scales, as exported
    emb = quant.make_embedding(w8, scale, device=DEV)
    ids = rng.integers(0, N, size=(2, 5))
    got = emb(torch.from_numpy(ids).to(DEV))
    assert got.shape == (2, 5, K) and got.dtype == torch.float16
    want = R.q8_embed(ids, w8, scale)
    assert np.array_equal(got.cpu().numpy().view(np.uint16), want.view(np.uint16))
    bad = emb(torch.tensor([0, N, -1, N - 1], device=DEV)).cpu().numpy()
    assert np.isnan(bad[1]).all() and np.isnan(bad[2]).all()
    assert np.array_equal(bad[[0, 3]].view(np.uint16), R.q8_embed(np.array([0, N - 1]), w8, scale).view(np.uint16))


# ---- many rows (k_rows_gemm, k_rows_gemm_lds at 64, 96 and 128 rows): one row
# past the smaller path, ragged rows and channels, few steps of K
@pytest.mark.parametrize("m,K,O", [(17, 128, 97), (33, 2048, 512), (130, 192, 64), (203, 576, 66),
                                   (500, 128, 4001), (260, 192, 20000), (700, 128, 8200)])
@pytest.mark.parametrize("q8", [True, False], ids=["int8", "f16"])
def test_many_rows_vs_f64(m, K, O, q8):
    """Within the other w8a16 paths' 2e-3 of each row's largest float64 value
    (f16 output, float32 sums), and one-hot rows bit-exact."""
    rng = np.random.default_rng(m + K + O)
    x = rng.standard_normal((m, K)).astype(np.float16)
    x[0] = 0
    x[0, K - 1] = 1.0  # one-hot: the output row is the weights' last column
    if q8:
        w8 = rng.integers(-128, 128, size=(O, K), dtype=np.int8)
        scale = rng.uniform(0.5, 1.5, O).astype(np.float32) * 1e-2
        wf = R.q8_dequant(w8, scale)
        y = ops().w8a16(_dev(x), _dev(w8), _dev(scale))
    else:
        wf = (rng.standard_normal((O, K)) * 0.05).astype(np.float16)
        y = ops().gemv_f16w(_dev(x), _dev(wf))
    got = y.cpu().numpy()
    want = x.astype(np.float64) @ wf.astype(np.float64).T
    assert np.array_equal(got[0].view(np.uint16), wf[:, K - 1].view(np.uint16))
    err = (np.abs(got - want).max(axis=1) / np.abs(want).max(axis=1)).max()
    assert err < 2e-3, err


# ---- the MoE block as one call: its few-token kernels at 1, 2, 3 and 4 tokens, the
# merged projections above; hidden sizes around a 512-input piece, shared widths of
# one piece, a ragged piece and two pieces per lane
@pytest.mark.parametrize("T,H,ish", [(1, 512, 128), (2, 640, 384), (3, 2048, 512), (4, 1664, 1152),
                                     (5, 640, 384), (40, 1024, 512)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32],
                         ids=["f16", "bf16", "f32"])
def test_moe_block_call_vs_separate_calls(T, H, ish, dtype):
    """Against the same module with a hook on its shared gate, which takes the
    separate calls: the same rounding points, float32 sums in another order, so
    single f16 roundings differ (the block tests' 5e-3 of the largest output)."""
    from escha_mlx_amd import moe
    E, I, k = 24, 256, 3
    rng = np.random.default_rng(T + H + ish)

    def experts(K, ic, oc):
        code = rng.integers(-32768, 32768, size=(E, ic // 16, oc // 16, 16 * K), dtype=np.int16)
        sign = lambda n: rng.choice([-1.0, 1.0], (E, n)).astype(np.float32)
        return moe.EschaExperts(code, sign(ic), sign(oc) * 0.04, device=DEV)

    gu, dn = experts(2, H, 2 * I), experts(3, I, H)
    q8 = lambda n, kk: rng.integers(-127, 128, size=(n, kk), dtype=np.int8)
    sc = lambda n, kk: (rng.uniform(0.5, 1.5, n) * 0.013 / np.sqrt(kk)).astype(np.float32)
    shared = {"gate_w8": q8(ish, H), "gate_scale": sc(ish, H), "up_w8": q8(ish, H),
              "up_scale": sc(ish, H), "down_w8": q8(H, ish), "down_scale": sc(H, ish)}
    blk = moe.EschaSparseMoeBlock(H, E, k, gu, dn, rng.standard_normal((E, H)) / np.sqrt(H),
                                  rng.standard_normal((1, H)) / np.sqrt(H), shared)
    x = torch.from_numpy(rng.standard_normal((T, H)).astype(np.float32)).to(dtype).to(DEV)
    y = blk(x)
    assert y.dtype == dtype and torch.equal(blk(x), y)
    handle = blk.sh_gate.register_forward_hook(lambda *a: None)
    want = blk(x)
    handle.remove()
    assert _rel(y.float().cpu().numpy(), want.float().cpu().numpy()) < 5e-3
