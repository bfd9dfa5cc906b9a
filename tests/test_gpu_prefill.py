"""Varlen causal prefill attention (HIP) against the CPU oracle.

Bar: within 1e-2 relative / 2e-2 absolute of the float64 oracle on the same
bf16 inputs (P is rounded to bf16 for the P.V MFMA, accumulation is fp32).
Cases: D 64 and 128, GQA group sizes 1-8, sequence lengths across the
16-query and 32-key tile boundaries (1, 15, 16, 17, 31, 33, ...), contiguous
keys, paged keys with cached prefixes (lq < lk) at block sizes 16 and 256,
block tables with -1 padding past each sequence, and a pool whose slots past
every context hold NaN.
"""
import numpy as np
import pytest
import torch

from llm_from_scratch_amd import kernels as K
from oracle import paged_kv as P

pytestmark = pytest.mark.gpu
DEV = "cuda"
RTOL, ATOL = 1e-2, 2e-2


def f64(t):
    return t.double().cpu().numpy()


def assert_close(got, ref, what):
    err = np.abs(got - ref)
    bad = np.argwhere(err > ATOL + RTOL * np.abs(ref))
    assert bad.size == 0, f"{what}: {len(bad)} mismatches, worst {err.max():.4g}, first {bad[:3].tolist()}"


def bf16(rng, *shape, scale=1.0):
    return torch.from_numpy((rng.standard_normal(shape) * scale).astype(np.float32)).to(torch.bfloat16).to(DEV)


@pytest.mark.parametrize("Hq,Hkv,D", [(12, 4, 64), (32, 8, 128), (8, 8, 64), (16, 2, 128), (8, 1, 64)])
def test_prefill_contiguous(Hq, Hkv, D):
    rng = np.random.default_rng(Hq * 100 + Hkv + D)
    lens = [1, 15, 16, 17, 31, 33, 100, 257]
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32, device=DEV)
    T = int(sum(lens))
    q = bf16(rng, T, Hq, D)
    k = bf16(rng, T, Hkv, D)
    v = bf16(rng, T, Hkv, D)
    scale = 1.0 / np.sqrt(D)
    o = K.flash_attn_varlen_func(q, k, v, cu, cu, max(lens), max(lens), scale)
    ref = P.prefill_attention(f64(q), f64(k), f64(v), cu.cpu().numpy(), cu.cpu().numpy(), scale)
    assert_close(f64(o), ref, f"contiguous Hq={Hq} Hkv={Hkv} D={D}")


@pytest.mark.parametrize("BS", [16, 256])
@pytest.mark.parametrize("Hq,Hkv,D", [(12, 4, 64), (32, 8, 128)])
def test_prefill_paged_cached_prefix(BS, Hq, Hkv, D):
    """Keys from a randomly permuted pool through -1-padded block tables;
    sequences with a cached prefix (lq < lk), a whole prompt (lq == lk) and
    a single new token."""
    rng = np.random.default_rng(BS + Hq + D)
    lens_k = [300, 64, 17, 520, 1]
    lens_q = [44, 64, 1, 7, 1]
    B = len(lens_k)
    nblk = [-(-L // BS) for L in lens_k]
    NB = sum(nblk) + 7
    maxb = max(nblk) + 2
    perm = rng.permutation(NB)
    bt = np.full((B, maxb), -1, np.int32)
    pos = 0
    for i, n in enumerate(nblk):
        bt[i, :n] = perm[pos:pos + n]
        pos += n
    kc = bf16(rng, NB, BS, Hkv, D)
    vc = bf16(rng, NB, BS, Hkv, D)
    cu_q = torch.tensor(np.concatenate([[0], np.cumsum(lens_q)]), dtype=torch.int32, device=DEV)
    cu_k = torch.tensor(np.concatenate([[0], np.cumsum(lens_k)]), dtype=torch.int32, device=DEV)
    q = bf16(rng, int(sum(lens_q)), Hq, D)
    btd = torch.from_numpy(bt).to(DEV)
    o = K.flash_attn_varlen_func(q, kc, vc, cu_q, cu_k, max(lens_q), max(lens_k), 0.125, block_table=btd)
    ref = P.prefill_attention(f64(q), f64(kc), f64(vc), cu_q.cpu().numpy(), cu_k.cpu().numpy(), 0.125,
                              block_tables=bt)
    assert_close(f64(o), ref, f"paged BS={BS} Hq={Hq} Hkv={Hkv} D={D}")


@pytest.mark.parametrize("BS", [16, 64])
def test_prefill_paged_pool_poisoned_past_context(BS):
    """Pool slots that hold no key of any sequence (tails of the last
    blocks, unused blocks) are NaN: keys past a context are masked, and
    their V rows must not reach the output either (0 * NaN)."""
    rng = np.random.default_rng(BS + 7)
    Hq, Hkv, D = 12, 4, 64
    lens_k = [37, 20, 5, 70]
    lens_q = [37, 3, 5, 10]
    B = len(lens_k)
    nblk = [-(-L // BS) for L in lens_k]
    NB = sum(nblk) + 3
    perm = rng.permutation(NB)
    bt = np.full((B, max(nblk) + 1), -1, np.int32)
    kc = torch.full((NB, BS, Hkv, D), float("nan"), dtype=torch.bfloat16, device=DEV)
    vc = torch.full((NB, BS, Hkv, D), float("nan"), dtype=torch.bfloat16, device=DEV)
    pos = 0
    for i, n in enumerate(nblk):
        bt[i, :n] = perm[pos:pos + n]
        pos += n
        for t in range(lens_k[i]):  # only the context's own slots hold data
            blk, o = bt[i, t // BS], t % BS
            kc[blk, o] = bf16(rng, Hkv, D)
            vc[blk, o] = bf16(rng, Hkv, D)
    cu_q = torch.tensor(np.concatenate([[0], np.cumsum(lens_q)]), dtype=torch.int32, device=DEV)
    cu_k = torch.tensor(np.concatenate([[0], np.cumsum(lens_k)]), dtype=torch.int32, device=DEV)
    q = bf16(rng, int(sum(lens_q)), Hq, D)
    o = K.flash_attn_varlen_func(q, kc, vc, cu_q, cu_k, max(lens_q), max(lens_k), 0.125,
                                 block_table=torch.from_numpy(bt).to(DEV))
    assert torch.isfinite(o.float()).all(), "NaN from slots past a context"
    ref = P.prefill_attention(f64(q), np.nan_to_num(f64(kc)), np.nan_to_num(f64(vc)), cu_q.cpu().numpy(),
                              cu_k.cpu().numpy(), 0.125, block_tables=bt)
    assert_close(f64(o), ref, f"poisoned pool BS={BS}")


def test_prefill_long_prompt_and_graph_grid():
    """One 1000-token prompt next to short ones, with max_seqlen_q larger
    than every length (the grid only depends on it): rows of idle tiles are
    not written, every real row matches."""
    rng = np.random.default_rng(11)
    Hq, Hkv, D = 12, 4, 64
    lens = [1000, 3, 40]
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32, device=DEV)
    T = int(sum(lens))
    q, k, v = bf16(rng, T, Hq, D), bf16(rng, T, Hkv, D), bf16(rng, T, Hkv, D)
    o = K.flash_attn_varlen_func(q, k, v, cu, cu, 1100, 1100)
    ref = P.prefill_attention(f64(q), f64(k), f64(v), cu.cpu().numpy(), cu.cpu().numpy(), 1.0 / 8)
    assert_close(f64(o), ref, "long prompt")


@pytest.mark.parametrize("B,L,Hq,Hkv,D", [(8, 1024, 16, 8, 64), (16, 2048, 12, 4, 64)])
def test_prefill_large_grid_vs_torch_fp32(B, L, Hq, Hkv, D):
    """Grids of several workgroups per CU, tiles of 128 (query token, head)
    rows that begin within a token's heads or not (G = 2; G = 3: the bench
    shape): against causal attention computed per sequence in float32 with
    torch on the GPU (the float64 oracle is too slow at this size)."""
    g = torch.Generator(device=DEV).manual_seed(13)
    q = torch.randn(B * L, Hq, D, generator=g, device=DEV).to(torch.bfloat16)
    k = torch.randn(B * L, Hkv, D, generator=g, device=DEV).to(torch.bfloat16)
    v = torch.randn(B * L, Hkv, D, generator=g, device=DEV).to(torch.bfloat16)
    cu = torch.arange(0, (B + 1) * L, L, dtype=torch.int32, device=DEV)
    o = K.flash_attn_varlen_func(q, k, v, cu, cu, L, L)
    G = Hq // Hkv
    mask = torch.ones(L, L, device=DEV, dtype=torch.bool).tril()
    worst = 0.0
    for b in range(B):
        sl = slice(b * L, (b + 1) * L)
        qf = q[sl].float().permute(1, 0, 2).contiguous()                      # [Hq, L, D]
        kf = k[sl].float().repeat_interleave(G, 1).permute(1, 2, 0).contiguous()  # [Hq, D, L]
        vf = v[sl].float().repeat_interleave(G, 1).permute(1, 0, 2).contiguous()  # [Hq, L, D]
        s = torch.matmul(qf, kf) / D ** 0.5
        s = s.masked_fill(~mask, float("-inf"))
        ref = torch.matmul(torch.softmax(s, -1), vf).permute(1, 0, 2)
        err = (o[sl].float() - ref).abs()
        assert bool((err <= ATOL + RTOL * ref.abs()).all()), f"sequence {b}: worst {err.max().item():.4g}"
        worst = max(worst, err.max().item())


def _torch_causal_ref(qs, ks, vs, G, D, scale):
    """Causal attention of one sequence in float32 with torch on the GPU:
    qs [lq, Hq, D] are the last lq positions of ks / vs [lk, Hkv, D]."""
    lq, lk = qs.size(0), ks.size(0)
    qf = qs.float().permute(1, 0, 2).contiguous()                       # [Hq, lq, D]
    kf = ks.float().repeat_interleave(G, 1).permute(1, 2, 0).contiguous()  # [Hq, D, lk]
    vf = vs.float().repeat_interleave(G, 1).permute(1, 0, 2).contiguous()  # [Hq, lk, D]
    s = torch.matmul(qf, kf) * scale
    pos = torch.arange(lk - lq, lk, device=DEV)[:, None]
    s = s.masked_fill(torch.arange(lk, device=DEV)[None, :] > pos, float("-inf"))
    return torch.matmul(torch.softmax(s, -1), vf).permute(1, 0, 2)


def test_prefill_large_grid_d128():
    """D = 128 and G = 4 (the cfg4 heads, 32 / 8): 4 x 4096-token prompts are
    4096 workgroups of 128 rows, 16 per CU, of 1 to 64 key tiles.  Against
    causal attention per sequence in float32."""
    B, L, Hq, Hkv, D = 4, 4096, 32, 8, 128
    g = torch.Generator(device=DEV).manual_seed(14)
    q = torch.randn(B * L, Hq, D, generator=g, device=DEV).to(torch.bfloat16)
    k = torch.randn(B * L, Hkv, D, generator=g, device=DEV).to(torch.bfloat16)
    v = torch.randn(B * L, Hkv, D, generator=g, device=DEV).to(torch.bfloat16)
    cu = torch.arange(0, (B + 1) * L, L, dtype=torch.int32, device=DEV)
    o = K.flash_attn_varlen_func(q, k, v, cu, cu, L, L)
    for b in range(B):
        sl = slice(b * L, (b + 1) * L)
        ref = _torch_causal_ref(q[sl], k[sl], v[sl], Hq // Hkv, D, D ** -0.5)
        err = (o[sl].float() - ref).abs()
        assert bool((err <= ATOL + RTOL * ref.abs()).all()), f"sequence {b}: worst {err.max().item():.4g}"


@pytest.mark.parametrize("B,lq,cached,Hq,Hkv,D", [(16, 2048, 1536, 12, 4, 64), (8, 2048, 512, 32, 8, 128)])
def test_prefill_large_grid_paged_cached_prefix(B, lq, cached, Hq, Hkv, D):
    """The paged kernel (a prefix-cache hit: `cached` keys already in the
    pool) on a grid of several workgroups per CU: block size 256, a randomly
    permuted pool, -1-padded tables.  Against
    causal attention per sequence in float32 over the gathered keys."""
    BS = 256
    lk = cached + lq
    rng = np.random.default_rng(B + lq + D)
    nblk = -(-lk // BS)
    NB = B * nblk + 3
    perm = rng.permutation(NB)
    bt = np.full((B, nblk + 1), -1, np.int32)
    for b in range(B):
        bt[b, :nblk] = perm[b * nblk:(b + 1) * nblk]
    g = torch.Generator(device=DEV).manual_seed(15)
    kc = torch.randn(NB, BS, Hkv, D, generator=g, device=DEV).to(torch.bfloat16)
    vc = torch.randn(NB, BS, Hkv, D, generator=g, device=DEV).to(torch.bfloat16)
    q = torch.randn(B * lq, Hq, D, generator=g, device=DEV).to(torch.bfloat16)
    cu_q = torch.arange(0, (B + 1) * lq, lq, dtype=torch.int32, device=DEV)
    cu_k = torch.arange(0, (B + 1) * lk, lk, dtype=torch.int32, device=DEV)
    btd = torch.from_numpy(bt).to(DEV)
    scale = D ** -0.5
    o = K.flash_attn_varlen_func(q, kc, vc, cu_q, cu_k, lq, lk, scale, block_table=btd)
    for b in range(B):
        ids = torch.from_numpy(bt[b, :nblk].astype(np.int64)).to(DEV)
        ks = kc[ids].reshape(-1, Hkv, D)[:lk]
        vs = vc[ids].reshape(-1, Hkv, D)[:lk]
        sl = slice(b * lq, (b + 1) * lq)
        ref = _torch_causal_ref(q[sl], ks, vs, Hq // Hkv, D, scale)
        err = (o[sl].float() - ref).abs()
        assert bool((err <= ATOL + RTOL * ref.abs()).all()), f"sequence {b}: worst {err.max().item():.4g}"


@pytest.mark.parametrize("Hq,Hkv,D,B,BS,scale", [
    (12, 4, 64, 5, 0, 0.125),      # two row tiles of a kv head's XCD pair
    (15, 3, 64, 4, 48, 0.2),       # kv heads that do not divide 8, G = 5, blocks of 48
    (7, 1, 128, 3, 16, -0.1),      # one kv head over 8 XCDs, G = 7, a negative scale
    (16, 16, 64, 6, 32, 0.0),      # more kv heads than XCDs, equal weights
    (32, 8, 128, 64, 64, 0.09),    # as many sequences as lanes rank
    (32, 8, 128, 65, 0, 0.09),     # one more: tiles in index order
])
def test_prefill_ragged_work_items(Hq, Hkv, D, B, BS, scale):
    """Every (sequence, 128-row tile, kv head) is computed once whatever the
    order of the work: ragged lengths around the 64-key and 128-row edges,
    empty sequences, cached prefixes, and a max_seqlen_q above the longest.
    Bound as above (weights and output rounded to bf16)."""
    rng = np.random.default_rng(B + D + BS)
    G = Hq // Hkv
    edge = 128 // G
    pool = [0, 1, edge - 1, edge, edge + 1, 63, 64, 65, 128, 129, 2 * edge + 1, 200]
    lens_k = np.array([pool[(3 * b + 11) % 12] if b % 7 else 200 for b in range(B)])
    lens_q = np.array([n if BS == 0 or b % 3 == 0 else -(-n // (b % 3 + 1)) for b, n in enumerate(lens_k)])
    cu_q, cu_k = (torch.tensor(np.concatenate([[0], np.cumsum(n)]), dtype=torch.int32, device=DEV)
                  for n in (lens_q, lens_k))
    q = bf16(rng, int(lens_q.sum()), Hq, D)
    kw, bt = {}, None
    if BS:
        nblk = -(-lens_k // BS)
        perm = rng.permutation(int(nblk.sum()) + 2)
        bt = np.full((B, int(nblk.max()) + 1), -1, np.int32)
        at = 0
        for b, n in enumerate(nblk):
            bt[b, :n] = perm[at:at + n]
            at += n
        k, v = (bf16(rng, len(perm), BS, Hkv, D) for _ in range(2))
        kw = dict(block_table=torch.from_numpy(bt).to(DEV))
    else:
        k, v = (bf16(rng, int(lens_k.sum()), Hkv, D) for _ in range(2))
    o = K.flash_attn_varlen_func(q, k, v, cu_q, cu_k, int(lens_q.max()) + 70, int(lens_k.max()), scale, **kw)
    ref = P.prefill_attention(f64(q), f64(k), f64(v), cu_q.cpu().numpy(), cu_k.cpu().numpy(), scale,
                              **({"block_tables": bt} if BS else {}))
    assert_close(f64(o), ref, f"work items Hq={Hq} Hkv={Hkv} D={D} B={B} BS={BS}")


@pytest.mark.parametrize("Hq,Hkv,D", [(12, 4, 64), (10, 2, 128), (3, 3, 64), (7, 1, 64)])
def test_prefill_one_long_prompt_among_short(Hq, Hkv, D):
    """A prompt of 2001 tokens beside 63 of 0-70 (most work items are past the
    last tile; G and Hkv of 3, 5 and 7 divide by a rounded reciprocal), a batch
    of equal prompts, and one prompt alone (as long contexts, so that none goes
    to the short form): every sequence the same bits as by itself in index
    order (beside 64 empty ones, which the search passes by)."""
    rng = np.random.default_rng(Hq)
    long = [2001 if b == 40 else (7 * b) % 71 for b in range(64)]
    for lens in (long, [33] * 64, [130]):
        cu = np.concatenate([[0], np.cumsum(lens)])
        q, k, v = (bf16(rng, int(cu[-1]), h, D) for h in (Hq, Hkv, Hkv))
        c = torch.from_numpy(cu.astype(np.int32)).to(DEV)
        o = K.flash_attn_varlen_func(q, k, v, c, c, max(lens), 100000, 0.125)
        for a, b in list(zip(cu, cu[1:]))[::9]:
            alone = torch.tensor([0] * 65 + [b - a], dtype=torch.int32, device=DEV)
            if b > a:
                want = K.flash_attn_varlen_func(q[a:b], k[a:b], v[a:b], alone, alone, int(b - a), 100000, 0.125)
                assert torch.equal(o[a:b], want), (a, b)


@pytest.mark.parametrize("Hq,Hkv,D", [(3, 3, 64), (8, 4, 64), (12, 4, 64), (16, 4, 64), (5, 1, 64), (12, 2, 64),
                                      (7, 1, 64), (16, 2, 64), (8, 4, 128), (6, 2, 128), (8, 2, 128), (10, 2, 128),
                                      (6, 1, 128)])
@pytest.mark.parametrize("top", [1, 16, 63, 64, 65, 129, 250])
def test_prefill_short_prompts_same_bits(Hq, Hkv, D, top):
    """Short whole prompts and cached prefixes in token order (16-row tiles at
    these sizes) against the same call whose hint says that contexts are long,
    and the oracle; every group size that the short form is compiled for."""
    rng = np.random.default_rng(Hq * top + D)
    lens_k = np.array([top, max(1, top - 1), 0, (top + 1) // 2, min(top, 17)])
    lens_q = np.array([top, max(1, top // 3), 0, (top + 1) // 2, 1])
    cu_q, cu_k = (torch.tensor(np.concatenate([[0], np.cumsum(n)]), dtype=torch.int32, device=DEV) for n in (lens_q, lens_k))
    q = bf16(rng, int(lens_q.sum()), Hq, D)
    k, v = (bf16(rng, int(lens_k.sum()), Hkv, D) for _ in range(2))
    for scale in (0.125, -0.3):
        o = K.flash_attn_varlen_func(q, k, v, cu_q, cu_k, top, top, scale)
        assert torch.equal(o, K.flash_attn_varlen_func(q, k, v, cu_q, cu_k, top, 100000, scale))
        ref = P.prefill_attention(f64(q), f64(k), f64(v), cu_q.cpu().numpy(), cu_k.cpu().numpy(), scale)
        assert_close(f64(o), ref, f"short {Hq}/{Hkv} x {D}, {top}")


@pytest.mark.parametrize("Hq,Hkv,D", [(12, 4, 64), (8, 8, 64), (8, 1, 64), (32, 8, 128), (6, 1, 128)])
@pytest.mark.parametrize("BS", [16, 48])
def test_prefill_short_paged_same_bits(Hq, Hkv, D, BS):
    """Contexts of one 64-key tile through a block table (16-row tiles at these
    sizes), with cached prefixes, an entry out of range and a pool that holds
    NaN past every context: the long form's bits, and the oracle."""
    rng = np.random.default_rng(Hq + D + BS)
    lens_k, lens_q = np.array([64, 17, 33, 0, 48, 1]), np.array([64, 1, 20, 0, 16, 1])
    cu_q, cu_k = (torch.tensor(np.concatenate([[0], np.cumsum(n)]), dtype=torch.int32, device=DEV) for n in (lens_q, lens_k))
    nblk = -(-lens_k // BS)
    perm = rng.permutation(np.arange(1, int(nblk.sum()) + 3))
    bt = np.full((len(lens_k), int(nblk.max()) + 1), -1, np.int32)
    at = 0
    for b, n in enumerate(nblk):
        bt[b, :n] = perm[at:at + n]
        at += n
    q = bf16(rng, int(lens_q.sum()), Hq, D)
    k, v = (bf16(rng, len(perm) + 1, BS, Hkv, D) for _ in range(2))
    for pool in (k, v):
        for b, n in enumerate(lens_k):
            if n % BS:
                pool[int(bt[b, n // BS]), int(n % BS):] = float("nan")
    args = (q, k, v, cu_q, cu_k)
    o = K.flash_attn_varlen_func(*args, 64, 64, 0.125, block_table=torch.from_numpy(bt).to(DEV))
    assert torch.equal(o, K.flash_attn_varlen_func(*args, 64, 9999, 0.125, block_table=torch.from_numpy(bt).to(DEV)))
    ref = P.prefill_attention(f64(q), np.nan_to_num(f64(k)), np.nan_to_num(f64(v)), cu_q.cpu().numpy(), cu_k.cpu().numpy(),
                              0.125, block_tables=bt)
    assert_close(f64(o), ref, f"short paged {Hq}/{Hkv} x {D}, blocks of {BS}")
    bt[0, 0] = len(perm) + 7  # out of range: slot 0, on both forms
    o, long = (K.flash_attn_varlen_func(*args, 64, m, 0.125, block_table=torch.from_numpy(bt).to(DEV)) for m in (64, 9999))
    assert torch.equal(o, long)


def test_prefill_any_max_seqlen_k():
    """max_seqlen_k is a hint: absent, not a whole number, on the device (not
    read, so that the call can be captured), too small, negative or past 32
    bits, the result is the same."""
    rng = np.random.default_rng(5)
    cu = torch.tensor([0, 90, 91, 200], dtype=torch.int32, device=DEV)
    q, k, v = bf16(rng, 200, 12, 64), bf16(rng, 200, 4, 64), bf16(rng, 200, 4, 64)
    want = K.flash_attn_varlen_func(q, k, v, cu, cu, 109, 109)
    on_gpu = (cu[1:] - cu[:-1]).max()
    for m in (None, float("inf"), np.int64(109), 109.0, torch.tensor(109), on_gpu, 1, 0, -1, -2 ** 40, 2 ** 40):
        assert torch.equal(K.flash_attn_varlen_func(q, k, v, cu, cu, 109, m), want), str(m)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        o = K.flash_attn_varlen_func(q, k, v, cu, cu, 109, on_gpu)
    for _ in range(3):
        o.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, want)


@pytest.mark.parametrize("L,D,hint", [(70, 64, 70), (70, 64, 100000), (300, 64, 300), (140, 128, 140), (140, 128, 100000)])
def test_prefill_overflowed_rows_are_nan(L, D, hint):
    """A row whose scores are all -infinity (products past the fp32 range) has
    no softmax: NaN, on both tile forms; other rows, of the same token and
    wave too, are what they are without it."""
    rng = np.random.default_rng(L + D)
    Hq, Hkv = 12, 4
    q, k, v = bf16(rng, L, Hq, D), bf16(rng, L, Hkv, D).abs(), bf16(rng, L, Hkv, D)
    cu = torch.tensor([0, L], dtype=torch.int32, device=DEV)
    want = K.flash_attn_varlen_func(q, k, v, cu, cu, L, hint)
    bad = torch.zeros(L, Hq, dtype=torch.bool, device=DEV)
    for t, h in ((0, 0), (5, 7), (64, 2), (L - 1, 11)):
        bad[t, h] = True
    q[bad] = -3e38
    o = K.flash_attn_varlen_func(q, k, v, cu, cu, L, hint)
    assert bool(o[bad].isnan().all()) and torch.equal(o[~bad], want[~bad])


@pytest.mark.parametrize("max_q", [(1 << 20) - 100, 1 << 20])
def test_prefill_many_empty_workgroups(max_q):
    """Short prompts under a max_seqlen_q whose grid passes 2^20 workgroups
    (several grid rows) and 2^32 threads."""
    rng = np.random.default_rng(max_q)
    B, Hq, Hkv, D = 64, 32, 8, 64
    lens = rng.integers(1, 9, B)
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32, device=DEV)
    q, k, v = (bf16(rng, int(lens.sum()), h, D) for h in (Hq, Hkv, Hkv))
    o = K.flash_attn_varlen_func(q, k, v, cu, cu, max_q, max_q, 0.125)
    assert torch.equal(o, K.flash_attn_varlen_func(q, k, v, cu, cu, 8, 8, 0.125))
    c = cu.cpu().numpy()
    assert_close(f64(o), P.prefill_attention(f64(q), f64(k), f64(v), c, c, 0.125), f"max_seqlen_q {max_q}")


def test_prefill_argument_errors():
    q = torch.zeros(4, 8, 64, dtype=torch.bfloat16, device=DEV)
    kv = torch.zeros(4, 2, 64, dtype=torch.bfloat16, device=DEV)
    cu = torch.tensor([0, 4], dtype=torch.int32, device=DEV)
    with pytest.raises(TypeError):
        K.flash_attn_varlen_func(q, kv, kv, cu.long(), cu, 4, 4)
    with pytest.raises(AssertionError):
        K.flash_attn_varlen_func(q, kv, kv, cu, cu, 4, 4, causal=False)
    bad = torch.zeros(4, 3, 64, dtype=torch.bfloat16, device=DEV)  # 8 q heads over 3 kv heads
    with pytest.raises(ValueError):
        K.flash_attn_varlen_func(q, bad, bad, cu, cu, 4, 4)
