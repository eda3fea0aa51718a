"""GPU parity of the top-k plan kernel against the numpy oracle: bit-exact indices and masks."""

import numpy as np
import pytest
import torch

from appcorr_amd import kernels as K
from oracle import plan as OP
from tests.util import assert_bits_equal

pytestmark = pytest.mark.gpu


def _check(dev, scores: np.ndarray, k: int, npre: int, ntok: int | None = None, dindice: np.ndarray | None = None):
    B, P = scores.shape
    if dindice is None:
        dindice = np.broadcast_to(np.arange(npre + P, dtype=np.int64), (B, npre + P)).copy()
    N = int(dindice.max()) + 1 if ntok is None else ntok
    got = K.topk_plan(torch.from_numpy(scores).to(dev), k, torch.from_numpy(dindice).to(dev), npre, N)
    ref = OP.build_plan(scores, k, dindice, npre, N)
    assert_bits_equal(got.update_indice, ref.update_indice, "update_indice")
    assert_bits_equal(got.active_batch_idx, ref.active_batch_idx, "active_batch_idx")
    assert_bits_equal(got.active_pos_idx, ref.active_pos_idx, "active_pos_idx")
    assert_bits_equal(got.active_token_idx, ref.active_token_idx, "active_token_idx")
    assert_bits_equal(got.active_patch_mask, ref.active_patch_mask.astype(np.uint8), "patch_mask")
    assert_bits_equal(got.active_rope_idx, ref.active_rope_idx, "rope_idx")
    assert_bits_equal(got.keep_mask, ref.keep_mask.astype(np.uint8), "keep_mask")
    assert_bits_equal(got.row_slot, ref.row_slot, "row_slot")


@pytest.mark.parametrize("B,P,ratio", [(16, 1024, 0.25), (16, 1024, 0.10), (16, 1024, 0.50), (8, 1024, 0.25),
                                       (1, 196, 0.5), (4, 4096, 0.10), (3, 100, 0.33), (2, 16384, 0.05)])
def test_topk_laplace_importance(dev, B, P, ratio):
    rng = np.random.default_rng(P + B)
    delta = rng.laplace(size=(B, P, 32)).astype(np.float32)
    scores = np.linalg.norm(delta, axis=-1).astype(np.float32)
    _check(dev, scores, OP.keep_count(P, ratio), 5)


@pytest.mark.parametrize("k", [0, 1, 7, 63, 64, 65, 127, 128])
def test_topk_edge_k(dev, k):
    rng = np.random.default_rng(k)
    scores = rng.standard_normal((3, 128)).astype(np.float32)
    _check(dev, scores, k, 5)


def test_topk_all_keep(dev):
    scores = np.random.default_rng(0).standard_normal((2, 196)).astype(np.float32)
    _check(dev, scores, 196, 5)


def test_topk_ties_lowest_index_wins(dev):
    scores = np.zeros((4, 300), dtype=np.float32)
    scores[1, ::3] = 1.0
    scores[2] = np.repeat(np.arange(30, dtype=np.float32), 10)
    scores[3, 5] = -0.0
    _check(dev, scores, 77, 5)


def test_topk_negative_inf_candidates_and_nan(dev):
    rng = np.random.default_rng(5)
    scores = rng.standard_normal((2, 200)).astype(np.float32)
    scores[0, 10:150] = -np.inf
    scores[1, [3, 17]] = np.nan
    scores[1, [4, 18]] = np.inf
    _check(dev, scores, 100, 5)


def test_topk_candidate_subset_dindice(dev):
    # Candidates are a strided group of patches (a correction group), not all patches.
    rng = np.random.default_rng(6)
    B, N, npre = 4, 1029, 5
    grp = np.arange(npre, N)[::4]
    dind = np.stack([np.concatenate([np.arange(npre), grp])] * B).astype(np.int64)
    scores = rng.standard_normal((B, grp.size)).astype(np.float32)
    _check(dev, scores, 64, npre, ntok=N, dindice=dind)



def _check_stats(dev, scores: np.ndarray, keep: np.ndarray):
    got = K.plan_stats(torch.from_numpy(scores).to(dev), torch.from_numpy(keep).to(dev)).cpu().numpy().astype(np.float64)
    ref = OP.plan_stats(scores, keep)
    # fp32 sums in a fixed order against the float64 oracle: |error| <= n * 2^-24 * sum|s|.
    bound = scores.size * 2.0 ** -24 * float(np.abs(scores[np.isfinite(scores)]).sum()) + 1e-30
    for i in range(2):
        if np.isnan(ref[i]) or np.isinf(ref[i]):
            assert (np.isnan(got[i]) and np.isnan(ref[i])) or got[i] == ref[i], (i, got[i], ref[i])
        else:
            assert abs(got[i] - ref[i]) <= bound, (i, got[i], ref[i], bound)
    np.testing.assert_array_equal(got[2:], ref[2:])


@pytest.mark.parametrize("B,P,ratio", [(16, 1024, 0.25), (1, 196, 0.5), (3, 100, 0.33), (2, 16384, 0.05)])
def test_plan_stats_against_oracle(dev, B, P, ratio):
    rng = np.random.default_rng(B * 7 + P)
    scores = np.abs(rng.laplace(size=(B, P))).astype(np.float32)
    k = OP.keep_count(P, ratio)
    got = K.topk_plan(torch.from_numpy(scores).to(dev), k,
                      torch.from_numpy(np.broadcast_to(np.arange(5 + P, dtype=np.int64), (B, 5 + P)).copy()).to(dev), 5)
    _check_stats(dev, scores, got.keep_mask.cpu().numpy().astype(bool))


def test_plan_stats_masked_and_special_values(dev):
    rng = np.random.default_rng(11)
    scores = rng.standard_normal((3, 300)).astype(np.float32)
    keep = rng.random((3, 300)) < 0.3
    _check_stats(dev, scores, keep)
    s2 = scores.copy()
    s2[0, ~keep[0]] = -np.inf           # masked candidates (candidate_valid_mask): NaN kept mass
    _check_stats(dev, s2, keep)
    s3 = scores.copy()
    s3[1, np.flatnonzero(keep[1])[:2]] = -np.inf  # only kept -inf: kept mass -inf
    _check_stats(dev, s3, keep)
    _check_stats(dev, np.zeros((2, 0), dtype=np.float32), np.zeros((2, 0), dtype=bool))


@pytest.mark.parametrize("B,P,gh,k,fusion,server,hint", [
    (2, 64, 100, 16, "SERVER", "fp", None), (16, 1024, 1024, 256, "GEO_MEAN", "fp", "patches"),
    (3, 759, 759, 379, "ADD", "fp", "tokens"), (1, 1, 5, 1, "MULTIPLY", "fp", "patches"),
    (4, 1025, 4096, 0, "MOBILE", None, "patches"), (2, 3000, 3000, 3000, "ADD", None, "tokens"),
    (2, 300, 300, 75, "GEO_MEAN", "wide", "patches")])
def test_plan_scores_equal_elementwise_steps(dev, B, P, gh, k, fusion, server, hint):
    """The candidate scores formed by the plan kernels equal torch's gathers and elementwise steps bit for bit
    (negative scores, infinities, NaN, -0, products that would contract to a fused multiply-add, strided score
    rows), and the fused top-k plan equals topk_plan of those scores; query_valid is all ones."""
    from appcorr_amd import _lib
    rng = np.random.default_rng(B * P + k)
    npre, N = 5, gh + 5
    cand = np.stack([np.sort(rng.permutation(gh)[:P]) + npre for _ in range(B)])
    dind = torch.from_numpy(np.concatenate([np.broadcast_to(np.arange(npre), (B, npre)), cand], 1).astype(np.int64)).to(dev)

    def rows(n):
        v = (rng.standard_normal((B, n)) * 10.0 ** rng.integers(-3, 3, (B, n))).astype(np.float32)
        special = np.array([np.inf, -np.inf, np.nan, -0.0, 0.0, 3e38, 1e-45], np.float32)
        at = rng.permutation(v.size)[: v.size // 16]
        v.ravel()[at] = special[rng.integers(0, special.size, at.size)]
        return torch.from_numpy(v).to(dev)

    sv = None if server is None else rows(N) if server == "fp" else rows(3 * N)[:, N: 2 * N]
    off = 0 if hint == "tokens" else npre
    ht = None if hint is None else rows(N - off)
    ws, wm = (0.0 if sv is None else 0.7), (1.0 if fusion == "MOBILE" else 1.3)
    src = K.CandidateScores(sv, ws, ht, off, wm, getattr(_lib, "FUSION_" + fusion))
    idx = dind[:, npre:]
    s_ref = torch.zeros((B, P), device=dev) if sv is None else sv.gather(1, idx)
    m_ref = None if ht is None else ht.gather(1, idx - off)
    c_ref = ws * s_ref
    if fusion == "MOBILE":
        c_ref = m_ref
    elif fusion != "SERVER":
        term = wm * m_ref
        c_ref = c_ref + term if fusion == "ADD" else c_ref * term
        if fusion == "GEO_MEAN":
            c_ref = torch.sqrt(torch.clamp(c_ref, min=0.0))

    def same(a, b, what):
        a, b = a.cpu().numpy(), b.cpu().numpy()
        nan = np.isnan(b)
        assert (np.isnan(a) == nan).all() and (a[~nan] == b[~nan]).all(), what

    tp, valid, *fused = K.topk_plan_scores(src, k, dind, npre, N)
    for got in (K.plan_scores(src, dind, npre), fused):
        for g, r, what in zip(got, (s_ref, m_ref, c_ref), ("server", "mobile", "combined")):
            assert (g is None) == (r is None), what
            if r is not None:
                same(g, r, what)
    ref = K.topk_plan(c_ref.contiguous(), k, dind, npre, N)
    for name in ("update_indice", "active_batch_idx", "active_pos_idx", "active_token_idx", "active_patch_mask",
                 "active_rope_idx", "keep_mask", "row_slot"):
        assert torch.equal(getattr(tp, name), getattr(ref, name)), name
    assert bool(valid.all()) and valid.shape == (B, npre + k)


@pytest.mark.parametrize("B", [0, 1])
@pytest.mark.parametrize("kw", [dict(), dict(server_pscore_weight=0.0), dict(token_keep_thres=-1.0, token_keep_cap=16),
                                dict(server_pscore_weight=0.0, token_keep_thres=-1.0, token_keep_cap=16),
                                dict(server_pscore_weight=0.0, token_keep_thres=-1.0),
                                dict(server_pscore_weight=0.0, mobile_pscore="residual_energy",
                                     mobile_pscore_weight=1.0)])
def test_correction_of_no_images(dev, B, kw):
    """An empty batch corrects to an empty batch with every kind of selection, with scores and without; one image
    of zero tokens beside it."""
    from appcorr_amd.dinov3 import SelfAttentionBlock
    N, C = 201, 384
    print(f"correction of {B} images {sorted(kw)}", flush=True)
    blk = SelfAttentionBlock(C, 6, ffn_ratio=4.0, qkv_bias=True, init_values=1.0, mask_k_bias=True)
    blk = blk.to(device=dev, dtype=torch.bfloat16)
    for t in (*blk.parameters(), *blk.buffers()):  # they come uninitialised
        t.data.zero_()
    x = torch.zeros(B, N, C, device=dev, dtype=torch.bfloat16)
    rope = (torch.zeros(N - 5, 64, device=dev), torch.ones(N - 5, 64, device=dev))
    cache = {"layer0_kv": x.new_zeros(B, N, 2, 6, 64), "layer0_blocks_out_sum": torch.zeros_like(x),
             "layer0_server_pscore": torch.zeros(B, N, device=dev)}
    dind = torch.arange(N, device=dev).unsqueeze(0).expand(B, -1).contiguous()
    if "mobile_pscore" in kw:
        kw = dict(kw, mobile_pscore_hint=torch.zeros(B, N - 5, device=dev))
    with torch.no_grad():
        y, _ = blk.correct(x, dind, rope, cache, "layer0", token_keep_ratio=0.5, **kw)
    assert y.shape == x.shape and bool(torch.isfinite(y).all())
