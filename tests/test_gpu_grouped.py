"""GPU parity of the many-row expert path: the grouped matrix-core GEMM with its
transforms and SwiGLU in the epilogues, at each of its row-block sizes, and the
grouping of many rows."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import ref_np as R

from .conftest import has_gpu
from .test_gpu_parity import _moe_case, _oracle_moe, dcode, ops

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not has_gpu(), reason="needs a ROCm GPU")]

DEV = "cuda"


def _args(c, K_gu, K_dn):
    dv = lambda n: torch.from_numpy(c[n]).to(DEV)
    return [dcode(c["gu_code"]), dv("gu_rin"), dv("gu_rout"), K_gu, dcode(c["dn_code"]),
            dv("dn_rin"), dv("dn_rout"), K_dn]


# rows per expert 20, 33, 66, 96 on average: 32-, 64-, 96- and 128-row groups;
# H of three 128-column blocks (half a workgroup unused in the down leg)
@pytest.mark.parametrize("E,T,k,H,I,K_gu,K_dn", [(4, 40, 2, 256, 128, 2, 3), (3, 50, 2, 384, 128, 3, 2),
                                                 (8, 66, 8, 256, 256, 2, 2), (2, 96, 2, 384, 128, 3, 3)],
                         ids=["rows32", "rows64_h384", "rows96", "rows128_h384"])
@pytest.mark.parametrize("skew", [False, True], ids=["spread", "skewed"])
def test_grouped_gemm_path_vs_oracle(E, T, k, H, I, K_gu, K_dn, skew):
    """f16 roundings at the oracle's points, float32 sums in another order: the
    bar of the other expert paths (5e-3 of the largest output).  Skewed: every
    token's first slot goes to expert 1, so some groups are full and others
    hold one row or none."""
    c = _moe_case(E, H, I, K_gu, K_dn, T, k, 70 + E + T)
    logits = c["logits"].copy()
    if skew:
        logits[:, 1] += 20.0
    ids, sc = ops().route_topk(torch.from_numpy(logits).to(DEV), k)
    x = torch.from_numpy(c["x"]).to(DEV)
    args = _args(c, K_gu, K_dn)
    ws = torch.zeros(ops().moe_expert_path_workspace(T, k, E, H, I), dtype=torch.uint8, device=DEV)
    y = ops().moe_expert_path(x, ids, sc, *args, ws=ws)
    ids_np, sc_np = ids.cpu().numpy(), sc.cpu().numpy()
    want = _oracle_moe(c, ids_np, sc_np, E, H, I, K_gu, K_dn, np.unique(ids_np)).astype(np.float32)
    got = y.cpu().numpy().astype(np.float32)
    assert np.abs(got - want).max() / np.abs(want).max() < 5e-3
    assert torch.equal(ops().moe_expert_path(x, ids, sc, *args, lut=True, ws=ws), y)


@pytest.mark.parametrize("m,E", [(1025, 256), (16384, 256), (5000, 512), (3000, 513), (1300, 2048)])
def test_build_groups_many_rows(m, E):
    """Both many-row forms (wave segments up to 512 experts, mask chunks above)
    against the oracle's model: a skewed expert, an empty one, a ragged end."""
    from escha_mlx_amd import moe
    rng = np.random.default_rng(m + E)
    re = rng.integers(0, E - 1, size=m).astype(np.int32)
    re[rng.random(m) < 0.3] = E // 2
    ng = moe.n_groups_bound(m, E, 16)
    rows_idx, group_expert = moe.build_groups(torch.from_numpy(re).to(DEV), E, 16, ng)
    ri, ge = R.build_groups(re, E, 16, ng)
    assert np.array_equal(rows_idx.cpu().numpy(), ri)
    assert np.array_equal(group_expert.cpu().numpy(), ge)


@pytest.mark.parametrize("T,E,k", [(2, 1, 1), (3, 64, 8), (2, 65, 32), (4, 256, 8), (2, 257, 2), (2, 1024, 32)])
def test_route_topk_edges(T, E, k):
    """Widths around each per-lane count, ties within and across lanes, masked
    logits (the type's lowest value, -inf) and NaN, which is never chosen: ids
    exact, scores as the router test's 2e-6."""
    rng = np.random.default_rng(T + E + k)
    lg = rng.integers(-6, 6, size=(T, E)).astype(np.float32)  # many ties
    free = np.arange(E) % 3 != 1
    if free.sum() >= k and E > 64:
        lg[0, ~free] = np.finfo(np.float32).min
        lg[1, ~free] = -np.inf
    ids, sc = ops().route_topk(torch.from_numpy(lg).to(DEV), k)
    want_ids, want_sc = R.route_topk(lg, k)
    assert np.array_equal(ids.cpu().numpy(), want_ids)
    assert np.allclose(sc.cpu().numpy(), want_sc, rtol=2e-6, atol=0)
    if E >= 2 * k:
        nan = rng.integers(-6, 6, size=(T, E)).astype(np.float32)
        nan[:, 1::2] = np.nan
        ids, _ = ops().route_topk(torch.from_numpy(nan).to(DEV), k)
        want, _ = R.route_topk(np.where(np.isnan(nan), -np.inf, nan), k)
        assert np.array_equal(ids.cpu().numpy(), want)


# 16,440 transforms of 8 lanes: past the size where a wave takes 8 of them; three
# 128-blocks per row, an odd top_k (the last slot of each token alone)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32],
                         ids=["f16", "bf16", "f32"])
def test_many_tokens_match_fewer(dtype):
    """A token's result does not depend on the tokens beside it: one call of 2740
    tokens has the bits of calls of 548, whose input transforms run one block a wave."""
    E, T, k, H, I, K_gu, K_dn = 4, 2740, 3, 384, 128, 2, 3
    c = _moe_case(E, H, I, K_gu, K_dn, T, k, 77)
    ids, sc = ops().route_topk(torch.from_numpy(c["logits"]).to(DEV), k)
    x = torch.from_numpy(c["x"]).to(DEV).to(dtype)
    args = _args(c, K_gu, K_dn)
    y = ops().moe_expert_path(x, ids, sc, *args)
    parts = [ops().moe_expert_path(*(t[i:i + 548].contiguous() for t in (x, ids, sc)), *args)
             for i in range(0, T, 548)]
    assert torch.equal(y, torch.cat(parts))
