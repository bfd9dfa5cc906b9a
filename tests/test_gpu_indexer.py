"""FP8 indexer score (HIP) against the CPU oracle (model/attention/utils.py:
175-250 semantics).

Bar: bit-exact on small-integer codes with scales of the form 2^k (every
dot product, ReLU, weighted sum and key scale is exact in fp32); within
1e-5 relative of the float64 oracle (scaled by the row's largest |score|)
on random codes and scales; within 1e-4 on the act_quant ue8m0 pipeline,
whose codes span the whole e4m3 range (products up to 2e5 summed inside
the MFMA, which does not round like a sequential fp32 sum).  Cases: head dims 32 / 64 / 128, head
counts that are and are not multiples of 16, key counts across the 16-key
and 256-key chunk edges, a key slice of a longer FP8 cache, and the
reference's indexer pipeline (act_quant block 32 with ue8m0 scales).
"""
import numpy as np
import pytest
import torch

from llm_from_scratch_amd import kernels as K
from oracle import fp8 as F

pytestmark = pytest.mark.gpu
DEV = "cuda"


def codes(x):
    return torch.from_numpy(F.e4m3_encode(x)).view(torch.float8_e4m3fn).to(DEV)


@pytest.mark.parametrize("B,M,N,H,D", [(2, 5, 300, 64, 128), (1, 3, 17, 20, 64), (3, 2, 257, 16, 32)])
def test_fp8_index_exact_integers(B, M, N, H, D):
    rng = np.random.default_rng(B * M + N + H + D)
    ints = np.arange(-4, 5, dtype=np.float32)
    q = codes(rng.choice(ints, (B, M, H, D)))
    k = codes(rng.choice(ints, (B, N, D)))
    qs = torch.from_numpy(2.0 ** rng.integers(-3, 3, (B, M, H)).astype(np.float32)).to(DEV)
    ks = torch.from_numpy(2.0 ** rng.integers(-3, 3, (B, N)).astype(np.float32)).to(DEV)
    o = K.fp8_index(q, qs, k, ks)
    ref = F.fp8_index(q.view(torch.uint8).cpu().numpy(), qs.cpu().numpy(), k.view(torch.uint8).cpu().numpy(),
                      ks.cpu().numpy())
    np.testing.assert_array_equal(o.cpu().numpy(), ref.astype(np.float32))


def test_fp8_index_random_and_cache_slice():
    rng = np.random.default_rng(4)
    B, M, H, D, NMAX, N = 2, 4, 64, 128, 1000, 700
    q = codes(rng.standard_normal((B, M, H, D)) * 8)
    kcache = codes(rng.standard_normal((B, NMAX, D)) * 8)
    scache = torch.from_numpy(rng.uniform(1e-3, 1e-1, (B, NMAX)).astype(np.float32)).to(DEV)
    qs = torch.from_numpy(rng.uniform(1e-3, 1e-1, (B, M, H)).astype(np.float32)).to(DEV)
    k, ks = kcache[:, :N], scache[:, :N]  # the first N cached keys, no copy
    o = K.fp8_index(q, qs, k, ks).cpu().numpy()
    ref = F.fp8_index(q.view(torch.uint8).cpu().numpy(), qs.cpu().numpy(),
                      k.contiguous().view(torch.uint8).cpu().numpy(), ks.cpu().numpy())
    err = np.abs(o - ref) / np.abs(ref).max(axis=-1, keepdims=True)
    assert err.max() < 1e-5, err.max()


def test_fp8_index_reference_pipeline():
    """The reference indexer's inputs (DSA.py:92-105): q and k quantised by
    act_quant with block 32 and ue8m0 scales at head_dim 32 (one scale per
    head row and per key), head weights times the q scale."""
    g = torch.Generator(device=DEV).manual_seed(8)
    B, M, N, H, D = 2, 6, 130, 32, 32
    qx = torch.randn(B, M, H, D, generator=g, device=DEV).to(torch.bfloat16)
    kx = torch.randn(B, N, D, generator=g, device=DEV).to(torch.bfloat16)
    q8, q_scale = K.act_quant(qx, 32, "ue8m0")   # [B, M, H, 1]
    k8, k_scale = K.act_quant(kx, 32, "ue8m0")   # [B, N, 1]
    w = torch.rand(B, M, H, 1, generator=g, device=DEV) * H ** -0.5
    weights = w * q_scale * D ** -0.5
    o = K.fp8_index(q8, weights, k8, k_scale.squeeze(-1)).cpu().numpy()
    ref = F.fp8_index(q8.view(torch.uint8).cpu().numpy(), weights.squeeze(-1).cpu().numpy(),
                      k8.view(torch.uint8).cpu().numpy(), k_scale.squeeze(-1).cpu().numpy())
    err = np.abs(o - ref) / np.maximum(np.abs(ref).max(axis=-1, keepdims=True), 1e-30)
    assert err.max() < 1e-4, err.max()
    # approximates the bf16 score
    qf, kf = qx.float().cpu().numpy(), kx.float().cpu().numpy()
    full = np.maximum(np.einsum("bmhd,bnd->bmhn", qf, kf), 0) * (w * D ** -0.5).cpu().numpy()
    approx = full.sum(2)
    assert np.abs(o - approx).max() < 0.1 * np.abs(approx).max()


@pytest.mark.parametrize("B,M,N,H,D", [
    (1, 1, 129, 16, 128),     # one query: chunks of one tile
    (1, 2048, 1025, 16, 64),  # chunks of 256, the last of one key
    (2, 1024, 1500, 16, 32),  # 512
    (1, 4096, 2049, 32, 64),  # 1024
    (1, 8200, 130, 16, 128),  # 2048: one chunk, a part tile and a part workgroup of queries
])
def test_fp8_index_chunk_lengths(B, M, N, H, D):
    """Every key chunk length the sizes choose, at part tiles and chunks, with
    small and large head weights of both signs: a score depends on its own
    query and key alone, so the same bits as calls of a few queries over
    slices of the keys (one-tile chunks, which the tests above hold against
    the oracle)."""
    g = torch.Generator(device=DEV).manual_seed(M + N)
    q, k = ((torch.randn(*s, generator=g, device=DEV) * 100).clamp(-448, 448).to(torch.float8_e4m3fn)
            for s in ((B, M, H, D), (B, N, D)))
    for scale in (1.0, 2.0 ** -60, 2.0 ** 60):
        qs = (torch.rand(B, M, H, generator=g, device=DEV) - 0.2) * scale
        ks = torch.rand(B, N, generator=g, device=DEV)
        o = K.fp8_index(q, qs, k, ks)
        for m in (0, max(0, M // 2 - 3), max(0, M - 11)):
            for n in (0, max(0, N - 140)):
                part = K.fp8_index(q[:, m:m + 11].contiguous(), qs[:, m:m + 11], k[:, n:n + 140], ks[:, n:n + 140])
                assert torch.equal(o[:, m:m + 11, n:n + 140], part), (scale, m, n)
        assert torch.isfinite(o).all()


def test_fp8_index_nan_codes_score_zero():
    """A NaN code makes its products NaN, which the ReLU takes as 0."""
    g = torch.Generator(device=DEV).manual_seed(1)
    q, k = (torch.randn(*s, generator=g, device=DEV).to(torch.float8_e4m3fn) for s in ((1, 9, 32, 64), (1, 200, 64)))
    qs, ks = torch.rand(1, 9, 32, generator=g, device=DEV), torch.rand(1, 200, generator=g, device=DEV)
    want = K.fp8_index(q, qs, k, ks)
    k.view(torch.uint8)[0, 77, 5] = 0x7F
    k.view(torch.uint8)[0, 150, 60] = 0xFF
    o = K.fp8_index(q, qs, k, ks)
    want[0, :, [77, 150]] = 0
    assert torch.equal(o, want)


@pytest.mark.parametrize("e", [-140, -126, -110, -96, -95, 0, 94, 95, 110, 116])
def test_fp8_index_any_head_weight(e):
    """Weights over the whole fp32 range: one head of weight w and score s
    gives fp32(s * w) (the other heads add exact zeros: weight 0, or a score
    that the ReLU sets to 0 whatever its weight)."""
    rng = np.random.default_rng(e + 200)
    B, M, N, H, D = 1, 11, 150, 20, 64
    qi = rng.choice(np.arange(-4, 5, dtype=np.float32), (B, M, H, D))
    qi[:, :, 0] = -1  # only negative products
    ki = rng.choice(np.arange(1, 5, dtype=np.float32), (B, N, D))
    qi[:, :, 7, 0] = 4
    w = np.float32(np.ldexp(1 + 2.0 ** -23, e))
    qs = np.zeros((B, M, H), np.float32)
    qs[:, :, 7] = w
    qs[:, 1, 7] *= -1
    qs[:, ::2, 0] = np.float32(2.0 ** 120)  # a negative score under a huge weight
    qs[:, 3, 0] = np.float32(2.0 ** -130)
    o = K.fp8_index(codes(qi), torch.from_numpy(qs).to(DEV), codes(ki), torch.ones(B, N, device=DEV))
    s = np.maximum(np.einsum("bmd,bnd->bmn", qi[:, :, 7].astype(np.float64), ki), 0)
    np.testing.assert_array_equal(o.cpu().numpy(), (s * qs[:, :, 7, None].astype(np.float64)).astype(np.float32))
