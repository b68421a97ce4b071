"""GPU parity tests: every HIP entry point, called through the C ABI, against the
CPU oracle on identical seeded inputs.

Bar: bit-exact for codes, nibbles, weights (bf16 bits), vote counts, candidate
lists and final top-k indices; rerank scores within 1e-5 relative of the oracle
(they are in fact evaluated in the same order, so equality is also asserted).
"""
import math

import numpy as np
import pytest
import torch

import workloads as W
from oracle import pkv_oracle as O

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from pariskv_amd import ops as _ops

    return _ops


@pytest.fixture(scope="module")
def wl_cfg1():
    return W.cfg1()


@pytest.fixture(scope="module")
def wl_cfg2():
    return W.cfg2()


@pytest.fixture(scope="module")
def wl_small_bf16():
    # ragged length (not a multiple of any tile), 2 sequences
    return W.make_workload("small", 2, 2, 4, 5000 + 37, 333, 100, O.BF16, 0.5, seed0=5)


def _say(msg):
    print(msg, flush=True)


# ------------------------------------------------------------------- encode


@pytest.mark.parametrize("dtype", [O.F32, O.BF16])
@pytest.mark.parametrize("layout", ["keymajor", "reference"])
def test_encode_append_bit_exact(ops, dtype, layout):
    _say(f"encode dtype={dtype} layout={layout}")
    bs, H, S = 2, 3, 1000 + 13
    tdt = torch.bfloat16 if dtype == O.BF16 else torch.float32
    signs = O.srht_signs(42)
    keys = np.stack([O.synth_keys(S, 100 + r, bf16=dtype == O.BF16) for r in range(bs * H)]).reshape(bs, H, S, 128)
    keys[0, 0, 5] = 0.0  # a zero key must not produce NaNs
    tk = torch.from_numpy(keys).to(tdt).to(DEV)
    if layout == "keymajor":
        _, _, _, cb, k4, kw = ops.alloc_keymajor(bs, H, S, DEV)
    else:
        cb = torch.zeros(bs, H, 16, S, dtype=torch.uint8, device=DEV)
        k4 = torch.zeros(bs, H, 16, S, 4, dtype=torch.uint8, device=DEV)
        kw = torch.zeros(bs, H, 16, S, dtype=torch.bfloat16, device=DEV)
    cc = torch.zeros(bs, H, 16, 256, dtype=torch.int32, device=DEV)
    ops.encode_append(tk, torch.from_numpy(signs).to(DEV), cb, k4, kw, cc)
    ops.encode_append(tk[:, :, :100], torch.from_numpy(signs).to(DEV), cb[..., :100], k4[:, :, :, :100], kw[..., :100], cc)
    torch.cuda.synchronize()
    for r in range(bs * H):
        b, h = divmod(r, H)
        codes, nib, w = O.encode(keys[b, h], signs, dtype)
        assert np.array_equal(cb[b, h].cpu().numpy().T, codes)
        assert np.array_equal(k4[b, h].cpu().numpy().transpose(1, 0, 2), nib)
        assert np.array_equal(kw[b, h].float().cpu().numpy().T, w)
        ref_cc = O.count_cluster_keys(codes)
        ref_cc = O.count_cluster_keys(codes[:100], ref_cc)  # += semantics
        assert np.array_equal(cc[b, h].cpu().numpy(), ref_cc)
    # count_cluster_keys on its own
    cc2 = torch.zeros_like(cc)
    ops.count_cluster_keys(cb, cc2)
    ops.count_cluster_keys(cb[..., :100], cc2)
    assert torch.equal(cc2, cc)


@pytest.mark.parametrize("dtype", [O.BF16, O.F32])
@pytest.mark.parametrize("S", [1, 15, 16, 17, 255, 256, 257, 300])
def test_encode_ragged_block_stays_inside_its_keys(ops, S, dtype):
    """The lanes past the end of a ragged block repeat its last key's stores: nothing beyond key S - 1 may change, and
    the cluster sizes count every key once."""
    _say(f"encode ragged S={S} dtype={dtype}")
    cap = S + 40
    signs = O.srht_signs(42)
    keys = O.synth_keys(S, 31 + S, bf16=dtype == O.BF16).reshape(1, 1, S, 128)
    codes_km, nib_km, w_km, cb, k4, kw = ops.alloc_keymajor(1, 2, cap, DEV)
    rec = nib_km.as_strided((1, 2, cap, 128), nib_km.stride(), nib_km.storage_offset())  # the whole 128-byte records
    codes_km.fill_(0xAB)
    rec.fill_(0xAB)
    cc = torch.zeros(1, 2, 16, 256, dtype=torch.int32, device=DEV)
    tk = torch.from_numpy(keys).to(torch.bfloat16 if dtype == O.BF16 else torch.float32).to(DEV)
    ops.encode_append(tk, torch.from_numpy(signs).to(DEV), cb[:, 1:, :, :S], k4[:, 1:, :, :S], kw[:, 1:, :, :S], cc[:, 1:])
    torch.cuda.synchronize()
    codes, nib, w = O.encode(keys[0, 0], signs, dtype)
    assert np.array_equal(cb[0, 1, :, :S].cpu().numpy().T, codes)
    assert np.array_equal(k4[0, 1, :, :S].cpu().numpy().transpose(1, 0, 2), nib)
    assert np.array_equal(kw[0, 1, :, :S].float().cpu().numpy().T, w)
    assert np.array_equal(cc[0, 1].cpu().numpy(), O.count_cluster_keys(codes)) and int(cc[0, 0].abs().sum()) == 0
    # untouched: head 0, the keys from S on of head 1, and bytes 96..127 of every record (the value-norm slot)
    assert bool((codes_km[0, 0] == 0xAB).all()) and bool((codes_km[0, 1, S:] == 0xAB).all())
    assert bool((rec[0, 0] == 0xAB).all()) and bool((rec[0, 1, S:] == 0xAB).all()) and bool((rec[0, 1, :, 96:] == 0xAB).all())


def _adversarial_keys(n, seed, bf16=True):
    """Keys that stress every rounding decision of the encoder: magnitudes from 2^-30 to 2^30, outlier dims,
    exact zeros and components far below the norm, powers of two, one-hot and constant vectors, tiny norms."""
    rng = np.random.default_rng(seed)
    k = rng.standard_normal((n, 128)).astype(np.float32)
    kind = np.arange(n) % 16
    k *= np.exp2(rng.integers(-30, 31, size=(n, 1))).astype(np.float32) * (kind[:, None] < 6) + (kind[:, None] >= 6)
    k[kind == 6] *= np.where(rng.random((int((kind == 6).sum()), 128)) < 0.05, 30.0, 1.0).astype(np.float32)   # outlier dims
    k[kind == 7] *= (rng.random((int((kind == 7).sum()), 128)) < 0.5)                                          # half zeros
    k[kind == 8] *= np.where(rng.random((int((kind == 8).sum()), 128)) < 0.1, 1e-30, 1.0).astype(np.float32)   # far below the norm
    k[kind == 9] = np.exp2(rng.integers(-8, 9, size=(int((kind == 9).sum()), 128))) * rng.choice([-1.0, 1.0], size=(int((kind == 9).sum()), 128))
    oh = np.where(kind == 10)[0]
    k[oh] = 0.0
    k[oh, rng.integers(0, 128, size=oh.size)] = rng.standard_normal(oh.size).astype(np.float32) + 3.0          # one-hot
    k[kind == 11] = (rng.standard_normal((int((kind == 11).sum()), 1)) * np.ones((1, 128))).astype(np.float32)  # constant
    k[kind == 12] *= 1e-9                                                                                      # norm below the 1e-8 clamp
    k[kind == 13] = np.round(k[kind == 13] * 4.0) / 4.0                                                        # many exact ties and zeros
    k[kind == 14] *= 3e-8                                                                                      # norm just above the clamp
    k = k.astype(np.float32)
    return O.bf16_round(k) if bf16 else k


def _adversarial_bf16_keys(n, seed):
    return _adversarial_keys(n, seed, True)


def test_encode_bf16_bit_exact_on_adversarial_keys(ops):
    """The bf16 encoder replaces divisions by reciprocals where that provably gives the same bf16 result and falls
    back to correctly rounded arithmetic per wave elsewhere; both routes must equal the oracle bit for bit."""
    H, S = 4, 16384 + 5
    signs = O.srht_signs(42)
    keys = np.stack([_adversarial_bf16_keys(S, 700 + h) for h in range(H)]).reshape(1, H, S, 128)
    _say(f"encode adversarial bf16 keys {keys.shape}")
    tk = torch.from_numpy(keys).to(torch.bfloat16).to(DEV)
    _, _, _, cb, k4, kw = ops.alloc_keymajor(1, H, S, DEV)
    cc = torch.zeros(1, H, 16, 256, dtype=torch.int32, device=DEV)
    ops.encode_append(tk, torch.from_numpy(signs).to(DEV), cb, k4, kw, cc)
    torch.cuda.synchronize()
    for h in range(H):
        codes, nib, w = O.encode(keys[0, h], signs, O.BF16)
        bad = np.where((cb[0, h].cpu().numpy().T != codes).any(axis=1))[0]
        assert bad.size == 0, f"codes differ at keys {bad[:8]} (kinds {bad[:8] % 16})"
        bad = np.where((k4[0, h].cpu().numpy().transpose(1, 0, 2) != nib).any(axis=(1, 2)))[0]
        assert bad.size == 0, f"4-bit codes differ at keys {bad[:8]} (kinds {bad[:8] % 16})"
        got_w = kw[0, h].float().cpu().numpy().T
        bad = np.where((got_w.view(np.uint32) != w.astype(np.float32).view(np.uint32)).any(axis=1))[0]
        assert bad.size == 0, f"weights differ at keys {bad[:8]} (kinds {bad[:8] % 16})"
        assert np.array_equal(cc[0, h].cpu().numpy(), O.count_cluster_keys(codes))


def test_encode_f32_bit_exact_on_adversarial_keys(ops):
    """The fp32 encoder shares one refined reciprocal among the quotients of a denominator and leaves out the range
    scaling of divisions and roots inside a checked range, falling back to the plain correctly rounded operations per
    wave elsewhere; both routes must equal the oracle bit for bit."""
    H, S = 4, 16384 + 5
    signs = O.srht_signs(42)
    keys = np.stack([_adversarial_keys(S, 900 + h, bf16=False) for h in range(H)]).reshape(1, H, S, 128)
    keys[0, 1] *= np.float32(2.0) ** np.random.default_rng(3).integers(-70, 50, size=(S, 1)).astype(np.float32)  # beyond the checked range too
    _say(f"encode adversarial fp32 keys {keys.shape}")
    tk = torch.from_numpy(keys).to(DEV)
    _, _, _, cb, k4, kw = ops.alloc_keymajor(1, H, S, DEV)
    cc = torch.zeros(1, H, 16, 256, dtype=torch.int32, device=DEV)
    ops.encode_append(tk, torch.from_numpy(signs).to(DEV), cb, k4, kw, cc)
    cb2 = torch.zeros(1, H, 16, S, dtype=torch.uint8, device=DEV)
    ops.encode_append(tk, torch.from_numpy(signs).to(DEV), cb2, None, None, None)  # codes only: the other kernel form
    torch.cuda.synchronize()
    for h in range(H):
        codes, nib, w = O.encode(keys[0, h], signs, O.F32)
        bad = np.where((cb[0, h].cpu().numpy().T != codes).any(axis=1))[0]
        assert bad.size == 0, f"codes differ at keys {bad[:8]} (kinds {bad[:8] % 16})"
        bad = np.where((cb2[0, h].cpu().numpy().T != codes).any(axis=1))[0]
        assert bad.size == 0, f"codes of the codes-only form differ at keys {bad[:8]} (kinds {bad[:8] % 16})"
        bad = np.where((k4[0, h].cpu().numpy().transpose(1, 0, 2) != nib).any(axis=(1, 2)))[0]
        assert bad.size == 0, f"4-bit codes differ at keys {bad[:8]} (kinds {bad[:8] % 16})"
        got_w = kw[0, h].float().cpu().numpy().T
        bad = np.where((got_w.view(np.uint32) != w.astype(np.float32).view(np.uint32)).any(axis=1))[0]
        assert bad.size == 0, f"weights differ at keys {bad[:8]} (kinds {bad[:8] % 16})"
        assert np.array_equal(cc[0, h].cpu().numpy(), O.count_cluster_keys(codes))


def test_encode_without_rabitq_outputs(ops):
    S = 300
    signs = O.srht_signs(42)
    keys = O.synth_keys(S, 9)
    cb = torch.zeros(1, 1, 16, S, dtype=torch.uint8, device=DEV)
    ops.encode_append(torch.from_numpy(keys).view(1, 1, S, 128).to(DEV), torch.from_numpy(signs).to(DEV), cb, None, None, None)
    assert np.array_equal(cb[0, 0].cpu().numpy().T, O.encode(keys, signs, O.F32)[0])


# --------------------------------------------------------------- query side


@pytest.mark.parametrize("wl_name", ["wl_cfg1", "wl_small_bf16"])
def test_query_prep_lut_bit_exact(ops, request, wl_name):
    w = request.getfixturevalue(wl_name)
    _say(f"query_prep_lut {w.name}")
    d = W.to_device(w, DEV, torch)
    qhat, qnorm, lut, ids = ops.query_prep_lut(d["queries"], w.H, d["signs"], d["cluster_counts"], w.tiers, want_sorted_ids=True)
    torch.cuda.synchronize()
    for r in range(w.R):
        st = W.oracle_stages(w, r)
        b, h = divmod(r, w.H)
        assert np.array_equal(qhat[b, h].cpu().numpy().view(np.uint32), st["qhat"].view(np.uint32))
        assert np.float32(qnorm[b, h].item()) == np.float32(st["qnorm"])
        assert np.array_equal(ids[b, h].cpu().numpy(), st["sorted_ids"])
        assert np.array_equal(lut[b, h].cpu().numpy(), st["lut"])


def test_query_prep_fp32_ranks_of_equal_scores(ops, wl_cfg1):
    """One-hot fp32 queries rotate into components of one magnitude, so that the 256 centroids of a subspace share nine scores:
    the ranks are decided by the ids, inside a wave's block of 64 ids and across blocks."""
    w = wl_cfg1
    signs = torch.from_numpy(np.ascontiguousarray(w.signs)).to(DEV)
    q = torch.zeros(1, 8, 128)
    for h in range(6):
        q[0, h, 23 * h] = 1.0 if h % 2 else -3.0
    q[0, 6] = torch.arange(128).remainder(4) - 1.5
    q[0, 7] = torch.randn(128, generator=torch.Generator().manual_seed(5))
    counts = torch.ones(1, 8, 16, 256, dtype=torch.int32, device=DEV)
    ids = ops.query_prep_lut(q.to(DEV), 8, signs, counts, [100], True)[3].cpu().numpy()
    for h in range(8):
        qh, _ = O.query_prep(q[0, h].numpy(), w.signs, O.F32)
        assert np.array_equal(ids[0, h], O.rank_centroids(qh, O.F32))


def test_query_prep_single_tier_and_group1(ops, wl_cfg1):
    w = wl_cfg1
    d = W.to_device(w, DEV, torch)
    q1 = d["queries"].view(w.bs, w.H, w.G, 128)[:, :, 0].contiguous()  # group size 1
    qhat, qnorm, lut, ids = ops.query_prep_lut(q1.view(w.bs, w.H, 128), w.H, d["signs"], d["cluster_counts"], [500], True)
    torch.cuda.synchronize()
    for r in range(w.R):
        qh, qn = O.query_prep(w.queries[0, r * w.G:r * w.G + 1], w.signs, w.dtype)
        lut_ref = O.tier_lut(O.rank_centroids(qh, w.dtype), w.cluster_counts[r], [500])
        assert np.array_equal(lut[0, r].cpu().numpy(), lut_ref) and lut_ref.max() == 1


def _collision_recipe(bs, kv_heads, kv_len, seed=42):
    """Input recipe of the reference's collision self-test (collision_fused/collision_test.py:16-53)."""
    torch.manual_seed(seed)
    ids = torch.stack([torch.stack([torch.stack([torch.randperm(256) for _ in range(16)])
                                    for _ in range(kv_heads)]) for _ in range(bs)]).to(torch.int64)
    counts = torch.randint(1, max(2, kv_len // 2), (bs, kv_heads, 16, 256), dtype=torch.int32)
    codebook = torch.randint(0, 256, (bs, kv_heads, 16, kv_len), dtype=torch.int32).to(torch.uint8)
    return ids, counts, codebook


@pytest.mark.parametrize("kv_len,ratio,ntier", [(2048, 0.2, 6), (4999, 0.5, 6), (2048, 0.3, 1), (70001, 0.2, 6)])
@pytest.mark.parametrize("layout", ["reference", "keymajor"])
def test_update_cache_cnt_interface(ops, kv_len, ratio, ntier, layout):
    from pariskv_amd.cache_hub.collision_fused import update_cache_cnt_cuda_interface

    _say(f"update_cache_cnt kv_len={kv_len} ntier={ntier} layout={layout}")
    bs, H = 2, 3
    ids, counts, codebook = _collision_recipe(bs, H, kv_len)
    ratios = list(O.TIER_RATIOS) if ntier == 6 else [1.0]
    tiers = O.tier_counts(kv_len, ratio, ratios)
    cb = codebook.to(DEV)
    if layout == "keymajor":
        cb = cb.permute(0, 1, 3, 2).contiguous().permute(0, 1, 3, 2)  # same logical tensor, key-major memory
    cnt = update_cache_cnt_cuda_interface(ids.to(DEV), counts.to(DEV), cb, tiers)
    torch.cuda.synchronize()
    assert cnt.dtype == torch.int32 and tuple(cnt.shape) == (bs, H, kv_len)
    for b in range(bs):
        for h in range(H):
            lut = O.tier_lut(ids[b, h].numpy(), counts[b, h].numpy(), tiers)
            ref = O.collision_count(np.ascontiguousarray(codebook[b, h].numpy().T), lut)
            assert np.array_equal(cnt[b, h].cpu().numpy(), ref)


def test_update_cache_cnt_sliced_views(ops):
    """The cache passes slices [.., start:end] of larger tensors (polar_cache.py:1051-1055)."""
    from pariskv_amd.cache_hub.collision_fused import update_cache_cnt_cuda_interface

    bs, H, cap, s, e = 1, 2, 3000, 129, 2777
    ids, counts, codebook = _collision_recipe(bs, H, cap)
    tiers = O.tier_counts(e - s, 0.5)
    for layout in ("reference", "keymajor"):
        cb = codebook.to(DEV)
        if layout == "keymajor":
            cb = cb.permute(0, 1, 3, 2).contiguous().permute(0, 1, 3, 2)
        cnt = update_cache_cnt_cuda_interface(ids.to(DEV), counts.to(DEV), cb[:, :, :, s:e], tiers)
        for h in range(H):
            lut = O.tier_lut(ids[0, h].numpy(), counts[0, h].numpy(), tiers)
            ref = O.collision_count(np.ascontiguousarray(codebook[0, h, :, s:e].numpy().T), lut)
            assert np.array_equal(cnt[0, h].cpu().numpy(), ref)


@pytest.mark.parametrize("layout", ["reference", "keymajor"])
def test_collision_scan_histograms(ops, layout):
    """Stand-alone scan from a ready table: u8 counts plus the per-chunk and per-row suffix histograms."""
    bs, H, N = 2, 2, 9001
    ids, counts, codebook = _collision_recipe(bs, H, N)
    tiers = O.tier_counts(N, 0.3)
    lut = np.stack([np.stack([O.tier_lut(ids[b, h].numpy(), counts[b, h].numpy(), tiers) for h in range(H)])
                    for b in range(bs)])
    cb = codebook.to(DEV)
    if layout == "keymajor":
        cb = cb.permute(0, 1, 3, 2).contiguous().permute(0, 1, 3, 2)
    cnt, (row_suf, chunk_suf), chunk = ops.collision_scan(cb, torch.from_numpy(lut).to(DEV), torch.uint8, want_hist=True)
    torch.cuda.synchronize()
    n_chunks = (N + chunk - 1) // chunk
    for b in range(bs):
        for h in range(H):
            r = b * H + h
            ref = O.collision_count(np.ascontiguousarray(codebook[b, h].numpy().T), lut[b, h])
            assert np.array_equal(cnt[b, h].cpu().numpy(), ref.astype(np.uint8))
            suf = lambda x: np.cumsum(np.bincount(x, minlength=128)[::-1])[::-1]
            assert np.array_equal(row_suf[r].cpu().numpy(), suf(ref))
            got = chunk_suf[r].cpu().numpy().astype(np.int64) & 0xFFFF
            for c in range(n_chunks):
                assert np.array_equal(got[c], suf(ref[c * chunk:(c + 1) * chunk]))


def test_update_cache_cnt_legacy(ops):
    from pariskv_amd.cache_hub.collision.collision import update_cache_cnt_cuda

    bs, H, N = 1, 4, 3001
    torch.manual_seed(42)  # recipe of collision/collision.py:11-26
    ids = torch.stack([torch.stack([torch.stack([torch.randperm(256) for _ in range(16)]) for _ in range(H)])
                       for _ in range(bs)]).to(torch.int32)
    topk_cnt = torch.randint(1, 256, (bs, H, 16), dtype=torch.int32)
    codebook = torch.randint(0, 256, (bs, H, 16, N), dtype=torch.int32)
    cnt = update_cache_cnt_cuda(ids.to(DEV), topk_cnt.to(DEV), codebook.to(DEV)).cpu()
    # membership form of collision/collision.py:29-45
    for h in range(H):
        ref = np.zeros(N, np.int32)
        for b in range(16):
            sel = set(ids[0, h, b, :int(topk_cnt[0, h, b])].tolist())
            ref += np.isin(codebook[0, h, b].numpy(), list(sel)).astype(np.int32)
        assert np.array_equal(cnt[0, h].numpy(), ref)


def test_interface_errors(ops):
    from pariskv_amd.cache_hub.collision_fused import update_cache_cnt_cuda_interface
    from pariskv_amd.cache_hub.topk import load_radix_topk_ext

    ids, counts, codebook = _collision_recipe(1, 1, 512)
    with pytest.raises(RuntimeError, match="uint8"):
        update_cache_cnt_cuda_interface(ids.to(DEV), counts.to(DEV), codebook.to(torch.int32).to(DEV), [10])
    with pytest.raises(RuntimeError, match="int64"):
        update_cache_cnt_cuda_interface(ids.to(torch.int32).to(DEV), counts.to(DEV), codebook.to(DEV), [10])
    with pytest.raises(RuntimeError, match="tier_num"):
        update_cache_cnt_cuda_interface(ids.to(DEV), counts.to(DEV), codebook.to(DEV), [])
    ext = load_radix_topk_ext()
    x = torch.zeros(2, 100, dtype=torch.int32, device=DEV)
    with pytest.raises(RuntimeError, match="exceed"):
        ext.bucket_topk(x, 101)
    with pytest.raises(RuntimeError, match="positive"):
        ext.radix_topk(x.float(), 0)
    with pytest.raises(RuntimeError, match="3D"):
        ext.radix_topk_3d(x, 5)


# --------------------------------------------------------------- selections


@pytest.mark.parametrize("rows,L,k", [(8, 8192, 1024), (3, 5037, 333), (2, 2048, 2048), (4, 100000, 5000), (1, 300, 1),
                                      (2, 4096, 4095)])
def test_bucket_and_radix_topk_on_counts(ops, rows, L, k):
    from pariskv_amd.cache_hub.topk import load_radix_topk_ext

    _say(f"bucket_topk rows={rows} L={L} k={k}")
    ext = load_radix_topk_ext()
    rng = np.random.default_rng(L + k)
    x = rng.binomial(96, 0.1, size=(rows, L)).astype(np.int32)
    tx = torch.from_numpy(x).to(DEV)
    out_b = ext.bucket_topk(tx, k).cpu().numpy()
    out_r = ext.radix_topk_3d(tx.view(1, rows, L), k).cpu().numpy()[0]  # hot call of polar_cache.py:1241
    assert out_b.dtype == np.int64
    for r in range(rows):
        ref, _ = O.select_candidates(x[r], k)
        assert np.array_equal(out_b[r], ref)
        assert np.array_equal(out_r[r], ref)
        tv = torch.topk(torch.from_numpy(x[r]), k).values.numpy()  # the reference's own check: same value multiset
        assert np.array_equal(np.sort(x[r][out_b[r]]), np.sort(tv))


@pytest.mark.parametrize("rows,N,k", [(1, 3, 1), (1, 255, 128), (2, 1026, 500), (8, 9001, 4000), (8, 20005, 20004), (33, 70003, 7000)])
def test_subspace_major_votes_and_coarse_filter_at_every_chunk_size(ops, rows, N, k):
    """Votes of a subspace-major codebook, four keys to a thread (rows of odd length: unaligned runs, one to three keys
    left over), and the coarse filter with 1, 4, 8 and 16 counts to a thread: whole numbers, exact."""
    from pariskv_amd.cache_hub.collision_fused import update_cache_cnt_cuda_interface

    _say(f"submajor votes rows={rows} N={N} k={k}")
    ids, counts, codebook = _collision_recipe(1, rows, N)
    tiers = O.tier_counts(N, 0.3)
    cnt = update_cache_cnt_cuda_interface(ids.to(DEV), counts.to(DEV), codebook.to(DEV), tiers)
    out = ops.bucket_topk(cnt.view(rows, N), k).cpu().numpy()
    for r in range(rows):
        ref = O.collision_count(np.ascontiguousarray(codebook[0, r].numpy().T), O.tier_lut(ids[0, r].numpy(), counts[0, r].numpy(), tiers))
        assert np.array_equal(cnt[0, r].cpu().numpy(), ref)
        assert np.array_equal(out[r], O.select_candidates(ref, k)[0])


def test_bucket_topk_all_equal_and_clamp(ops):
    x = torch.full((2, 3000), 7, dtype=torch.int32, device=DEV)
    assert torch.equal(ops.bucket_topk(x, 50).cpu(), torch.arange(50).expand(2, 50))
    y = torch.tensor([[500, -3, 4, 127, 128, 0, 9, 9]], dtype=torch.int32, device=DEV)
    assert ops.bucket_topk(y, 3).cpu().tolist() == [[0, 3, 4]]  # values clamp to [0,127]: 500,127,128 tie at 127


@pytest.mark.parametrize("rows,L,k", [(32, 4096, 1024), (8, 1024, 256), (3, 777, 100), (2, 8192, 8192), (4, 20000, 2048),
                                      (2, 105000, 2048), (1, 9000, 1), (5, 13107, 1024), (2, 16384, 8192), (3, 16385, 100)])
def test_topk_f32_exact(ops, rows, L, k):
    _say(f"topk_f32 rows={rows} L={L} k={k}")
    rng = np.random.default_rng(L * 7 + k)
    x = rng.standard_normal((rows, L)).astype(np.float32)
    x[:, ::5] = np.round(x[:, ::5], 1)  # exact ties
    ids = np.stack([rng.permutation(4 * L)[:L] for _ in range(rows)]).astype(np.int64)
    tx, tid = torch.from_numpy(x).to(DEV), torch.from_numpy(ids).to(DEV)
    out, vals = ops.topk_f32(tx, k, tid, want_values=True)
    out_pos = ops.topk_f32(tx, k)
    torch.cuda.synchronize()
    for r in range(rows):
        ref_ids, ref_pos = O.topk_f32(x[r], ids[r], k)
        assert np.array_equal(out[r].cpu().numpy(), ref_ids)
        assert np.array_equal(vals[r].cpu().numpy(), x[r][ref_pos])
        assert np.array_equal(out_pos[r].cpu().numpy(), O.topk_f32(x[r], None, k)[1])
    tv = torch.topk(tx, k, dim=-1).values  # same values, same order as torch.topk
    assert torch.equal(vals, tv)


def test_topk_f32_one_workgroup_score_distributions(ops):
    """Rows that one workgroup selects from (at most 8192 scores, k at most half of them) on score distributions
    that steer the kernel through each of its routes: evenly spread scores (bins of the row's own range, counting
    sort), a crowded winner bin (same bins, bitonic sort), a crowded threshold bin, a constant row, an outlier that
    stretches the range, infinities (radix select), exact ties decided by the ids, padded rows and k = 1."""
    rng = np.random.default_rng(2024)
    cases = []
    cases.append(("gaussian", rng.standard_normal((4, 4096)).astype(np.float32) * 20 + 30, 1024))
    x = rng.standard_normal((3, 4096)).astype(np.float32)
    x[:, 100:400] = np.float32(5.0)                                   # 300 winners in one bin
    cases.append(("crowded winner bin", x, 1024))
    x = rng.standard_normal((3, 4096)).astype(np.float32)
    x[:, :2000] = np.float32(0.5) + rng.integers(0, 3, (3, 2000)).astype(np.float32) * np.float32(2.0 ** -22)
    cases.append(("crowded threshold bin", x, 1500))
    cases.append(("constant", np.full((2, 4096), -3.5, np.float32), 700))
    x = rng.standard_normal((2, 4096)).astype(np.float32)
    x[0, 17], x[1, 4000] = 1e6, -1e6
    cases.append(("outlier", x, 1024))
    x = (rng.standard_normal((2, 4096)) * 100).astype(np.float32)
    x[0, 5], x[0, 77], x[1, 4095] = np.inf, -np.inf, np.inf
    cases.append(("infinities", x, 1000))
    cases.append(("ties by id", np.round(rng.standard_normal((3, 4096)) * 16).astype(np.float32) / 16, 1024))
    cases.append(("negative scores", -np.abs(rng.standard_normal((2, 4096))).astype(np.float32) - 1, 1024))
    cases.append(("padded row", rng.standard_normal((5, 3000)).astype(np.float32), 1))
    cases.append(("padded row, k=1500", rng.standard_normal((2, 3001)).astype(np.float32), 1500))
    cases.append(("2 keys per thread", rng.standard_normal((2, 2048)).astype(np.float32), 1024))
    cases.append(("8 keys per thread", rng.standard_normal((2, 8192)).astype(np.float32) ** 3, 4096))
    cases.append(("subnormal range", (rng.integers(0, 50, (2, 4096)).astype(np.float32) * np.float32(1e-45)), 512))
    for name, x, k in cases:
        _say(f"topk_f32 one workgroup: {name} {x.shape} k={k}")
        rows, L = x.shape
        ids = np.stack([rng.permutation(3 * L)[:L] for _ in range(rows)]).astype(np.int64)
        out, vals = ops.topk_f32(torch.from_numpy(x).to(DEV), k, torch.from_numpy(ids).to(DEV), want_values=True)
        torch.cuda.synchronize()
        for r in range(rows):
            ref_ids, ref_pos = O.topk_f32(x[r], ids[r], k)
            assert np.array_equal(out[r].cpu().numpy(), ref_ids), name
            assert np.array_equal(vals[r].cpu().numpy().view(np.uint32), x[r][ref_pos].view(np.uint32)), name


def test_topk_f32_wide_rows_edge_cases(ops):
    """Rows wider than one workgroup sorts (more than 8192 keys): the multi-workgroup histogram / compaction
    path with a threshold bin that holds the whole row (constant scores: every key ties, ids decide), one that
    holds more than 8192 keys, k = 8192, len = 8193, and mixed signs with infinities."""
    rng = np.random.default_rng(99)
    cases = []
    L = 30000
    cases.append(("constant", np.full((2, L), 1.25, np.float32), 700))
    x = rng.standard_normal((3, L)).astype(np.float32)
    x[:, : L // 2] = np.float32(0.75) + rng.integers(0, 4, (3, L // 2)).astype(np.float32) * np.float32(2.0 ** -20)
    cases.append(("crowded threshold bin", x, 9000 // 2))
    # the same with a list short enough for the one-binning selection + sort of the finish kernel, which must hand a
    # threshold bin this crowded (15 000 keys in four values) to the two-step path
    x2 = rng.standard_normal((3, L)).astype(np.float32)
    x2[:, : L // 2] = np.float32(2.5) + rng.integers(0, 4, (3, L // 2)).astype(np.float32) * np.float32(2.0 ** -20)
    cases.append(("crowded threshold bin, short list", x2, 1500))
    cases.append(("k=8192", rng.standard_normal((2, 70000)).astype(np.float32), 8192))
    cases.append(("len=8193", rng.standard_normal((5, 8193)).astype(np.float32), 100))
    y = (rng.standard_normal((2, 20001)) * 1e3).astype(np.float32)
    y[0, 5], y[0, 77], y[1, 20000] = np.inf, -np.inf, np.inf
    y[:, 100:4000] = -np.abs(y[:, 100:4000])
    cases.append(("signs and infinities", y, 3000))
    # scores that share their exponent: bins of fixed key bits would put the whole row into a few bins; the bins of
    # the row's own range keep the threshold bin small
    cases.append(("one binade", (rng.standard_normal((3, 52429)) * 2 + 100).astype(np.float32), 2048))
    cases.append(("narrow range", (rng.standard_normal((2, 20000)) * 1e-3 + 1.5).astype(np.float32), 1000))
    z = (rng.standard_normal((2, 30000)) * 5).astype(np.float32)
    z[0, 123] = 1e30                                   # an outlier stretches the range: everything else in one bin
    cases.append(("outlier", z, 512))
    # more slices than a row has range slots of its own: the control block is cleared by a launch and the slices'
    # ranges meet in two atomic words
    cases.append(("eighteen slices", rng.standard_normal((2, 140000)).astype(np.float32), 1500))
    for name, x, k in cases:
        _say(f"topk_f32 wide: {name} {x.shape} k={k}")
        rows, L = x.shape
        ids = np.stack([rng.permutation(3 * L)[:L] for _ in range(rows)]).astype(np.int64)
        out, vals = ops.topk_f32(torch.from_numpy(x).to(DEV), k, torch.from_numpy(ids).to(DEV), want_values=True)
        torch.cuda.synchronize()
        for r in range(rows):
            ref_ids, ref_pos = O.topk_f32(x[r], ids[r], k)
            assert np.array_equal(out[r].cpu().numpy(), ref_ids), name
            assert np.array_equal(vals[r].cpu().numpy(), x[r][ref_pos]), name
    with pytest.raises(RuntimeError, match="k up to"):
        ops.topk_f32(torch.zeros(1, 20000, device=DEV), 8193)


def test_radix_topk_float_api(ops):
    from pariskv_amd.cache_hub.topk import radix_topk, fast_topk, fast_topk_with_ratio

    g = torch.Generator().manual_seed(0)
    x = torch.rand(4, 3000, generator=g) * 96
    out = radix_topk(x.to(DEV), 64).cpu()
    assert torch.equal(torch.gather(x, 1, out), torch.topk(x, 64).values)
    xi = (x * 1).to(torch.int32)
    assert fast_topk(xi.to(DEV), 64).shape == (4, 64)
    assert fast_topk_with_ratio(xi.to(DEV).view(2, 2, 3000), 0.05).shape == (2, 2, 150)


# ------------------------------------------------------------------- rerank


@pytest.mark.parametrize("layout", ["keymajor", "reference"])
def test_partial_rerank_parity(ops, wl_small_bf16, layout):
    from pariskv_amd.cache_hub.rerank.rerank import partial_rerank_cuda

    w = wl_small_bf16
    _say(f"rerank layout={layout}")
    d = W.to_device(w, DEV, torch)
    k4 = d["nib_km"].view(w.bs, w.H, w.N, 16, 4).permute(0, 1, 3, 2, 4)
    kw = d["w_km"].permute(0, 1, 3, 2)
    if layout == "reference":
        k4, kw = k4.contiguous(), kw.contiguous()
    rng = np.random.default_rng(1)
    cand = np.stack([rng.permutation(w.N)[:w.C] for _ in range(w.R)]).astype(np.int64).reshape(w.bs, w.H, w.C)
    stages = [W.oracle_stages(w, r) for r in range(w.R)]
    q_blocks = torch.from_numpy(np.stack([s["qhat"] for s in stages])).view(w.bs, w.H, 16, 8).to(torch.bfloat16).to(DEV)
    q_norm = torch.tensor([s["qnorm"] for s in stages]).view(w.bs, w.H, 1).to(torch.bfloat16).to(DEV)
    centers = torch.tensor(ops.MAG_CENTERS, dtype=torch.bfloat16, device=DEV)
    scores, v4b = partial_rerank_cuda(torch.from_numpy(cand).to(DEV), k4, kw, q_blocks, q_norm, centers, 16, 8)
    torch.cuda.synchronize()
    assert scores.dtype == torch.float32 and tuple(v4b.shape) == (w.bs, w.H, 16, w.C, 8)
    th, ce = O.mag_constants()
    for r in range(w.R):
        b, h = divmod(r, w.H)
        ref = O.rerank(cand[b, h], w.nib[r], w.weight[r], stages[r]["qhat"], stages[r]["qnorm"])
        got = scores[b, h].cpu().numpy()
        np.testing.assert_allclose(got, ref, rtol=1e-5, atol=1e-5 * np.abs(ref).max())  # the stated tolerance
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))                 # and in fact identical
        # unpacked values (reference's second output): +-centers by nibble
        nibs = w.nib[r][cand[b, h]]  # [C,16,4]
        v = np.stack([nibs & 0x0F, nibs >> 4], axis=-1).reshape(w.C, 16, 8)
        ref_v = np.where(v & 8, 1.0, -1.0).astype(np.float32) * ce[v & 7]
        assert np.array_equal(v4b[b, h].float().cpu().numpy(), ref_v.transpose(1, 0, 2))


def test_rerank_out_of_range_candidate_is_masked(ops, wl_small_bf16):
    w = wl_small_bf16
    d = W.to_device(w, DEV, torch)
    k4 = d["nib_km"].view(w.bs, w.H, w.N, 16, 4).permute(0, 1, 3, 2, 4)
    kw = d["w_km"].permute(0, 1, 3, 2)
    cand = torch.tensor([0, w.N - 1, w.N, -1, 5], dtype=torch.int64, device=DEV).expand(w.bs, w.H, 5).contiguous()
    qhat = torch.zeros(w.bs, w.H, 128, device=DEV)
    scores, _ = ops.rerank4(cand, k4, kw, qhat, torch.ones(w.bs, w.H, device=DEV), ops.mag_centers(DEV))
    s = scores[0, 0].cpu()
    assert torch.isinf(s[2]) and torch.isinf(s[3]) and s[0] == 0 and s[1] == 0 and s[4] == 0


# ------------------------------------------------------------------ gathers


def test_h2d_gather_kv_matches_index_select(ops):
    from pariskv_amd.cache_hub.gather_trans import h2d_gather_kv

    bs, heads, kv_len, topk, max_topk = 2, 8, 32 * 1024, 100, 160  # shape of trans_h2d.py:108-120
    g = torch.Generator().manual_seed(0)
    src_k = torch.randn(bs, heads, kv_len, 128, generator=g).to(torch.bfloat16).pin_memory()
    src_v = torch.randn(bs, heads, kv_len, 128, generator=g).to(torch.bfloat16).pin_memory()
    idx = torch.randint(0, kv_len, (bs, heads, topk), generator=g)
    dst_k = torch.zeros(bs, heads, max_topk, 128, dtype=torch.bfloat16, device=DEV)
    dst_v = torch.zeros_like(dst_k)
    h2d_gather_kv(src_k, src_v, idx.to(DEV), dst_k, dst_v)
    torch.cuda.synchronize()
    ek = torch.gather(src_k, 2, idx.unsqueeze(-1).expand(-1, -1, -1, 128))
    ev = torch.gather(src_v, 2, idx.unsqueeze(-1).expand(-1, -1, -1, 128))
    assert torch.equal(dst_k[:, :, :topk].cpu().view(torch.int16), ek.view(torch.int16))
    assert torch.equal(dst_v[:, :, :topk].cpu().view(torch.int16), ev.view(torch.int16))
    assert not dst_k[:, :, topk:].any()  # rows beyond topk untouched
    # oracle gather on one row
    ref = O.gather_rows(src_k[1, 3].view(torch.int16).numpy(), idx[1, 3].numpy())
    assert np.array_equal(dst_k[1, 3, :topk].cpu().view(torch.int16).numpy(), ref)
    with pytest.raises(AssertionError):
        h2d_gather_kv(src_k.clone(), src_v, idx.to(DEV), dst_k, dst_v)  # unpinned source


def test_gather_hbm_with_offset_and_bounds(ops):
    bs, H, n, k = 1, 2, 500, 40
    g = torch.Generator().manual_seed(1)
    sk = torch.randn(bs, H, n, 128, generator=g).to(torch.bfloat16).to(DEV)
    sv = torch.randn(bs, H, n, 128, generator=g).to(torch.bfloat16).to(DEV)
    idx = torch.randint(0, n - 20, (bs, H, k), generator=g)
    idx[0, 0, 0] = n  # out of range after the offset -> zero row, no fault
    dk = torch.ones(bs, H, 64, 128, dtype=torch.bfloat16, device=DEV)
    dv = torch.ones_like(dk)
    ops.gather_hbm(sk, sv, idx.to(DEV), dk, dv, idx_offset=20, dst_row0=8)
    torch.cuda.synchronize()
    exp = torch.gather(sk.cpu(), 2, (idx + 20).clamp(max=n - 1).unsqueeze(-1).expand(-1, -1, -1, 128))
    exp[0, 0, 0] = 0
    assert torch.equal(dk[:, :, 8:8 + k].cpu(), exp) and (dk[:, :, :8] == 1).all() and (dk[:, :, 8 + k:] == 1).all()


def test_gather_uva_packed_layout(ops):
    """Ragged gather contract of polar_cache_adaptivek_varlen.py:1573-1644."""
    bs, H, n, sl_end = 2, 2, 1000, 6
    V = bs * H
    g = torch.Generator().manual_seed(2)
    ks = torch.tensor([5, 0, 17, 9])
    src_k = torch.randn(bs, H, n, 128, generator=g).to(torch.bfloat16).pin_memory()
    src_v = torch.randn(bs, H, n, 128, generator=g).to(torch.bfloat16).pin_memory()
    idx_packed = torch.randint(0, n, (int(ks.sum()),), generator=g)
    cu_topk = torch.zeros(V + 1, dtype=torch.int32)
    cu_topk[1:] = torch.cumsum(ks, 0)
    cu_k = torch.zeros(V + 1, dtype=torch.int32)
    cu_k[1:] = torch.cumsum(ks + sl_end, 0)
    total = int(cu_k[-1])
    kp = torch.zeros(total, 128, dtype=torch.bfloat16, device=DEV)
    vp = torch.zeros_like(kp)
    ops.gather_uva_packed(src_k, src_v, kp, vp, idx_packed.to(DEV), cu_topk.to(DEV), cu_k.to(DEV), sl_end, int(ks.max()))
    torch.cuda.synchronize()
    exp_k = torch.zeros(total, 128, dtype=torch.bfloat16)
    exp_v = torch.zeros_like(exp_k)
    for v in range(V):
        b, h = divmod(v, H)
        for s in range(int(ks[v])):
            src = int(idx_packed[int(cu_topk[v]) + s])
            exp_k[int(cu_k[v]) + sl_end + s] = src_k[b, h, src]
            exp_v[int(cu_k[v]) + sl_end + s] = src_v[b, h, src]
    assert torch.equal(kp.cpu(), exp_k) and torch.equal(vp.cpu(), exp_v)


# ------------------------------------------------------- fused decode step


def _run_fused(ops, w, gather_host=False):
    d = W.to_device(w, DEV, torch)
    plan = ops.RetrievePlan(w.bs, w.H, w.G, w.N, DEV, w.N, w.C, w.K)
    scores = torch.empty(w.bs, w.H, w.K, dtype=torch.float32, device=DEV)
    out = plan.run(d["queries"], d["signs"], d["centers"], d["cluster_counts"], d["codes_km"], d["nib_km"], d["w_km"], 0,
                   w.N, w.tiers, w.C, w.K, out_scores=scores)
    torch.cuda.synchronize()
    return plan, out, scores


def _any_order_model(scores, ids, k):
    """The order in which the one-workgroup top-k writes its k winners when the final sort is left out, restated:
    512 even bins of [row min, row max] (bin = min(511, floor((x - lo) * (512 / (hi - lo)))), fp32 operations); the
    threshold bin b* is the one in which the k-th largest score lies; the winners of the bins above b* come first,
    ordered by the wave that loaded them (element i is loaded by thread i % 1024 as its (i // 1024)-th element), then
    by element, then by lane; the winners inside b* follow in descending (score, smaller id first) order.  None
    where the kernel takes another route (more than 256 scores in b*, or no positive finite range)."""
    x = scores.astype(np.float32)
    lo, hi = x.min(), x.max()
    rng = np.float32(hi - lo)
    if not (np.isfinite(rng) and rng > 0):
        return None
    scale = np.float32(512.0) / rng
    t = ((x - lo) * scale).astype(np.float32)
    b = np.minimum(511, t.astype(np.int64))
    hist = np.bincount(b, minlength=512)
    above = np.cumsum(hist[::-1])[::-1] - hist          # scores in the bins above b
    bstar = int(np.max(np.nonzero((above < k) & (above + hist >= k))[0]))
    if hist[bstar] > 256:
        return None
    need = k - int(above[bstar])
    i = np.arange(len(x))
    tid, e = i % 1024, i // 1024
    first = np.nonzero(b > bstar)[0]
    first = first[np.lexsort((tid[first] % 64, e[first], tid[first] // 64))]
    inside = np.nonzero(b == bstar)[0]
    inside = inside[np.lexsort((ids[inside], -x[inside].astype(np.float64)))][:need]
    return np.concatenate([ids[first], ids[inside]])


@pytest.mark.parametrize("wl_name", ["wl_cfg1", "wl_cfg2", "wl_small_bf16"])
def test_retrieve_any_order_is_the_same_set_in_a_fixed_order(ops, request, wl_name):
    """any_order leaves the final sort out: the k ids are the sorted mode's ids exactly (as a set, scores attached
    to the right ids), they come in the documented order of their candidate-list positions (restated by
    _any_order_model), and two runs agree bit for bit."""
    w = request.getfixturevalue(wl_name)
    _say(f"retrieve any_order {w.name}")
    d = W.to_device(w, DEV, torch)
    plan = ops.RetrievePlan(w.bs, w.H, w.G, w.N, DEV, w.N, w.C, w.K)
    args = (d["queries"], d["signs"], d["centers"], d["cluster_counts"], d["codes_km"], d["nib_km"], d["w_km"], 0, w.N, w.tiers,
            w.C, w.K)
    s_sorted = torch.empty(w.bs, w.H, w.K, dtype=torch.float32, device=DEV)
    s_any = torch.empty_like(s_sorted)
    ids_sorted = plan.run(*args, out_scores=s_sorted).clone()
    ids_any = plan.run(*args, out_scores=s_any, any_order=True).clone()
    cand = plan.view("cand", w.N, w.C, w.K, torch.int64).view(w.R, w.C).cpu().numpy()
    ids_again = plan.run(*args, any_order=True)
    torch.cuda.synchronize()
    assert torch.equal(ids_any, ids_again)
    a, b_ = ids_sorted.view(w.R, w.K).cpu().numpy(), ids_any.view(w.R, w.K).cpu().numpy()
    sa, sb = s_sorted.view(w.R, w.K).cpu().numpy(), s_any.view(w.R, w.K).cpu().numpy()
    for r in range(w.R):
        assert np.array_equal(np.sort(a[r]), np.sort(b_[r]))
        assert dict(zip(a[r].tolist(), sa[r].tolist())) == dict(zip(b_[r].tolist(), sb[r].tolist()))
        if 2048 <= w.C <= 8192 and 4 * w.K <= w.C:
            # the select kernel without its sort: the documented order, restated from the candidate list and its scores
            sc_all = plan.view("scores", w.N, w.C, w.K, torch.float32).view(w.R, w.C)[r].cpu().numpy()
            want = _any_order_model(sc_all, cand[r], w.K)
            if want is not None:
                assert np.array_equal(b_[r], want), f"any-order ids of row {r} are not in the documented order"
        else:                                         # other shapes keep the descending-score order
            assert np.array_equal(a[r], b_[r])


@pytest.mark.parametrize("wl_name", ["wl_cfg1", "wl_cfg2", "wl_small_bf16"])
def test_retrieve_fused_matches_oracle(ops, request, wl_name):
    w = request.getfixturevalue(wl_name)
    _say(f"retrieve {w.name}: R={w.R} N={w.N} C={w.C} K={w.K}")
    plan, out, scores = _run_fused(ops, w)
    cnt_stride = (w.N + 15) // 16 * 16
    cnt = plan.view("cnt_u8", w.N, w.C, w.K, torch.uint8).view(w.R, cnt_stride)[:, :w.N].cpu().numpy()
    cand = plan.view("cand", w.N, w.C, w.K, torch.int64).view(w.R, w.C).cpu().numpy()
    sc = plan.view("scores", w.N, w.C, w.K, torch.float32).view(w.R, w.C).cpu().numpy()
    suf = plan.view("chunk_suffix_hist", w.N, w.C, w.K, torch.int16).view(w.R, -1, 128).cpu().numpy().astype(np.int64) & 0xFFFF
    row_suf = plan.view("row_suffix_hist", w.N, w.C, w.K, torch.int32).view(w.R, 128).cpu().numpy().astype(np.int64)
    for r in range(w.R):
        b, h = divmod(r, w.H)
        st = W.oracle_stages(w, r)
        assert np.array_equal(cnt[r], st["cnt"].astype(np.uint8)), f"vote counts differ in row {r}"
        ref_suf = np.cumsum(np.bincount(st["cnt"], minlength=128)[::-1])[::-1]  # keys with count >= t
        assert np.array_equal(suf[r].sum(axis=0), ref_suf) and np.array_equal(row_suf[r], ref_suf), f"histogram row {r}"
        assert np.array_equal(cand[r], st["cand"]), f"candidate list differs in row {r}"
        np.testing.assert_allclose(sc[r], st["scores"], rtol=1e-5, atol=1e-5 * np.abs(st["scores"]).max())
        assert np.array_equal(out[b, h].cpu().numpy(), st["final"]), f"final top-k differs in row {r}"
        assert np.array_equal(scores[b, h].cpu().numpy(), st["final_scores"])
        # whole-row oracle entry point agrees as well
        q = w.queries[b, h * w.G:(h + 1) * w.G]
        whole = O.retrieve_row(q, w.signs, w.dtype, w.codes[r], w.nib[r], w.weight[r], w.cluster_counts[r], w.tiers, w.C, w.K)
        assert np.array_equal(out[b, h].cpu().numpy(), whole)


@pytest.mark.parametrize("H,N,C", [(2, 255, 254), (2, 257, 100), (8, 769, 385), (8, 8192, 4096), (8, 8193, 900), (8, 16385, 1639),
                                   (1, 32769, 1500)])
def test_retrieve_short_rows_chunk_edges(ops, H, N, C):
    """Rows scanned in chunks of 256, 512 and 1024 keys, at and beside the sizes where the chunk size changes and with
    ragged last chunks: vote counts, histograms, candidate list and final ids against the oracle."""
    w = W.make_workload(f"short{N}", 1, H, 4, N, C, min(100, C), O.BF16, 0.3, seed0=N, with_values=False)
    _say(f"retrieve short rows H={H} N={N} C={C}")
    plan, out, scores = _run_fused(ops, w)
    cnt = plan.view("cnt_u8", w.N, w.C, w.K, torch.uint8).view(w.R, (N + 15) // 16 * 16)[:, :N].cpu().numpy()
    cand = plan.view("cand", w.N, w.C, w.K, torch.int64).view(w.R, w.C).cpu().numpy()
    suf = plan.view("chunk_suffix_hist", w.N, w.C, w.K, torch.int16).view(w.R, -1, 128).cpu().numpy().astype(np.int64) & 0xFFFF
    for r in range(w.R):
        st = W.oracle_stages(w, r)
        assert np.array_equal(cnt[r], st["cnt"].astype(np.uint8))
        chunk = 256 << next(i for i in range(4) if -(-N // (256 << i)) == suf.shape[1])   # the chunk size that was taken
        for c in range(suf.shape[1]):
            hist = np.bincount(st["cnt"][c * chunk:(c + 1) * chunk], minlength=128)
            assert np.array_equal(suf[r, c], np.cumsum(hist[::-1])[::-1])
        assert np.array_equal(cand[r], st["cand"])
        assert np.array_equal(out[0, r].cpu().numpy(), st["final"])
        assert np.array_equal(scores[0, r].cpu().numpy(), st["final_scores"])


@pytest.mark.parametrize("wl_name", ["wl_cfg1", "wl_cfg2", "wl_small_bf16"])
def test_one_launch_plan_equals_three_launches(ops, request, wl_name):
    """pkv_retrieve_args.launch_plan = PKV_PLAN_ONE_LAUNCH (query prep, scan and select + rerank as one launch whose
    workgroups hand the vote table and the histogram over) against the three launches: every intermediate and every
    output bit for bit, and against the oracle; with the flag area full of garbage before the first launch, three
    launches back to back on one workspace, no workgroup giving up a wait."""
    from pariskv_amd import _lib

    w = request.getfixturevalue(wl_name)
    _say(f"one-launch plan {w.name}: R={w.R} N={w.N} C={w.C} K={w.K}")
    d = W.to_device(w, DEV, torch)
    args = (d["queries"], d["signs"], d["centers"], d["cluster_counts"], d["codes_km"], d["nib_km"], d["w_km"], 0, w.N, w.tiers,
            w.C, w.K)
    names = (("qhat", torch.float32), ("qnorm", torch.float32), ("lut", torch.uint8), ("chunk_suffix_hist", torch.int16),
             ("row_suffix_hist", torch.int32), ("cand", torch.int64), ("scores", torch.float32))
    cnt_stride = (w.N + 15) // 16 * 16
    plan = ops.RetrievePlan(w.bs, w.H, w.G, w.N, DEV, w.N, w.C, w.K)
    ref_sc = torch.empty(w.bs, w.H, w.K, dtype=torch.float32, device=DEV)
    ref_ids = plan.run(*args, out_scores=ref_sc).clone()
    ref = {n: plan.view(n, w.N, w.C, w.K, dt).clone() for n, dt in names}
    ref_cnt = plan.view("cnt_u8", w.N, w.C, w.K, torch.uint8).view(w.R, cnt_stride)[:, :w.N].clone()
    plan.launch_plan = _lib.PLAN_ONE_LAUNCH
    plan.ws.fill_(0xA5)
    for rep in range(3):
        plan.skip_vote_counts = rep == 2
        if rep == 2:
            plan.view("cnt_u8", w.N, w.C, w.K, torch.uint8).zero_()
        sc = torch.empty_like(ref_sc)
        ids = plan.run(*args, out_scores=sc)
        torch.cuda.synchronize()
        assert int(plan.view("handover_status", w.N, w.C, w.K, torch.int32)[0]) == 0
        assert torch.equal(ids, ref_ids) and torch.equal(sc, ref_sc)
        for n, dt in names:
            assert torch.equal(plan.view(n, w.N, w.C, w.K, dt), ref[n]), f"{n} differs in launch {rep}"
        cnt = plan.view("cnt_u8", w.N, w.C, w.K, torch.uint8).view(w.R, cnt_stride)[:, :w.N]
        if rep == 2:
            assert not bool(cnt.any())  # the counts stayed on chip
        else:
            assert torch.equal(cnt, ref_cnt)
    for r in range(w.R):
        b, h = divmod(r, w.H)
        assert np.array_equal(ids[b, h].cpu().numpy(), W.oracle_stages(w, r)["final"])


def test_retrieve_large_rows_strided_pieces(ops):
    """Rows long enough for 8192-key chunks (8 rows x 600 000 keys): the collision scan and the select + rerank then
    work on four pieces per chunk spread over the row.  Keys with a drifting mean (candidates bunch in bands) and a
    ragged last chunk; candidate list, scores and final ids of three rows against the oracle, all rows against the
    one-launch plan (whole chunks)."""
    from pariskv_amd import _lib

    bs, H, G, N, C, K = 1, 8, 4, 600_000, 30_000, 512
    _say(f"strided pieces: N={N} C={C} K={K}")
    assert ops.pick_chunk_keys(bs * H, N) == 8192
    g = torch.Generator(device=DEV).manual_seed(11)
    keys = torch.randn(bs, H, N, 128, generator=g, device=DEV)
    keys[..., [7, 31, 64, 101]] *= 10.0
    ang = torch.arange(N, device=DEV, dtype=torch.float32) * (5.0 / 1000.0) * (math.pi / 180.0)
    keys[..., 0] += 2.0 * torch.cos(ang)
    keys[..., 1] += 2.0 * torch.sin(ang)
    keys = keys.to(torch.bfloat16)
    q = (keys[:, :, -2048:].float().mean(dim=2, keepdim=True) + 0.5 * torch.randn(bs, H, G, 128, generator=g, device=DEV))
    q = q.to(torch.bfloat16).view(bs, 1, H * G, 128).contiguous()
    signs, centers = ops.srht_signs(DEV), ops.mag_centers(DEV)
    codes_km, nib_km, w_km, cb, k4, kw = ops.alloc_keymajor(bs, H, N, DEV)
    cc = torch.zeros(bs, H, 16, 256, dtype=torch.int32, device=DEV)
    ops.encode_append(keys, signs, cb, k4, kw, cc)
    tiers = O.tier_counts(N, 0.2)
    plan = ops.RetrievePlan(bs, H, G, N, DEV, N, C, K)
    args = (q, signs, centers, cc, codes_km, nib_km, w_km, 0, N, tiers, C, K)
    sc = torch.empty(bs, H, K, device=DEV)
    ids = plan.run(*args, out_scores=sc).clone()
    cand = plan.view("cand", N, C, K, torch.int64).view(H, C).clone()
    csc = plan.view("scores", N, C, K, torch.float32).view(H, C).clone()
    per_chunk = torch.bincount(cand[0] // 8192, minlength=(N + 8191) // 8192)
    assert int(per_chunk.max()) > 1.5 * C / per_chunk.numel()  # the data does bunch
    plan.launch_plan = _lib.PLAN_ONE_LAUNCH
    ids1 = plan.run(*args)
    torch.cuda.synchronize()
    assert int(plan.view("handover_status", N, C, K, torch.int32)[0]) == 0
    assert torch.equal(ids, ids1)
    assert torch.equal(plan.view("cand", N, C, K, torch.int64).view(H, C), cand)
    assert torch.equal(plan.view("scores", N, C, K, torch.float32).view(H, C), csc)
    sg = signs.cpu().numpy()
    for r in (0, 4, 7):
        qh, qn = O.query_prep(q.view(bs, H, G, 128)[0, r].float().cpu().numpy(), sg, O.BF16)
        lut = O.tier_lut(O.rank_centroids(qh, O.BF16), cc[0, r].cpu().numpy(), tiers)
        cand_ref, _ = O.select_candidates(O.collision_count(codes_km[0, r].cpu().numpy(), lut), C)
        assert np.array_equal(cand[r].cpu().numpy(), cand_ref), f"candidate list of row {r}"
        sc_ref = O.rerank(cand_ref, nib_km[0, r].cpu().numpy().reshape(N, 16, 4), w_km[0, r].float().cpu().numpy(), qh, qn)
        np.testing.assert_allclose(csc[r].cpu().numpy(), sc_ref, rtol=1e-5, atol=1e-5 * np.abs(sc_ref).max())
        final, _ = O.topk_f32(sc_ref, cand_ref, K)
        assert np.array_equal(ids[0, r].cpu().numpy(), final), f"final ids of row {r}"


def test_retrieve_subrange_and_candidates_equal_keys(ops, wl_small_bf16):
    """Retrieval zone = [key0, key0+n) of a larger capacity; and C == N (identity candidates)."""
    w = wl_small_bf16
    d = W.to_device(w, DEV, torch)
    key0, n = 64, 2000
    plan = ops.RetrievePlan(w.bs, w.H, w.G, w.N, DEV, w.N, w.N, 64)
    tiers = O.tier_counts(n, 0.5)
    out = plan.run(d["queries"], d["signs"], d["centers"], d["cluster_counts"], d["codes_km"], d["nib_km"], d["w_km"], key0,
                   n, tiers, 200, 64)
    out_all = plan.run(d["queries"], d["signs"], d["centers"], d["cluster_counts"], d["codes_km"], d["nib_km"], d["w_km"],
                       key0, n, tiers, n, 64)
    torch.cuda.synchronize()
    for r in range(w.R):
        b, h = divmod(r, w.H)
        q = w.queries[b, h * w.G:(h + 1) * w.G]
        sl = slice(key0, key0 + n)
        ref = O.retrieve_row(q, w.signs, w.dtype, w.codes[r][sl], w.nib[r][sl], w.weight[r][sl], w.cluster_counts[r], tiers, 200, 64)
        assert np.array_equal(out[b, h].cpu().numpy(), ref)
        qhat, qn = O.query_prep(q, w.signs, w.dtype)
        s_all = O.rerank(np.arange(n), w.nib[r][sl], w.weight[r][sl], qhat, qn)
        assert np.array_equal(out_all[b, h].cpu().numpy(), O.topk_f32(s_all, None, 64)[0])


def test_retrieve_with_uva_gather(ops, wl_small_bf16):
    w = wl_small_bf16
    d = W.to_device(w, DEV, torch)
    kcpu = torch.from_numpy(w.keys.reshape(w.bs, w.H, w.N, 128)).to(torch.bfloat16).pin_memory()
    vcpu = torch.from_numpy(w.values.reshape(w.bs, w.H, w.N, 128)).to(torch.bfloat16).pin_memory()
    dk = torch.zeros(w.bs, w.H, w.K + 3, 128, dtype=torch.bfloat16, device=DEV)
    dv = torch.zeros_like(dk)
    plan = ops.RetrievePlan(w.bs, w.H, w.G, w.N, DEV, w.N, w.C, w.K)
    out = plan.run(d["queries"], d["signs"], d["centers"], d["cluster_counts"], d["codes_km"], d["nib_km"], d["w_km"], 0,
                   w.N, w.tiers, w.C, w.K,
                   gather=dict(src_k=kcpu, src_v=vcpu, from_host=True, dst_k=dk, dst_v=dv, dst_row0=3))
    torch.cuda.synchronize()
    idx = out.cpu().unsqueeze(-1).expand(-1, -1, -1, 128)
    assert torch.equal(dk[:, :, 3:].cpu(), torch.gather(kcpu, 2, idx))
    assert torch.equal(dv[:, :, 3:].cpu(), torch.gather(vcpu, 2, idx))
    for r in range(w.R):
        b, h = divmod(r, w.H)
        assert np.array_equal(out[b, h].cpu().numpy(), W.oracle_stages(w, r)["final"])


def test_retrieve_argument_errors(ops, wl_small_bf16):
    w = wl_small_bf16
    d = W.to_device(w, DEV, torch)
    plan = ops.RetrievePlan(w.bs, w.H, w.G, w.N, DEV, w.N, w.C, w.K)
    args = (d["queries"], d["signs"], d["centers"], d["cluster_counts"], d["codes_km"], d["nib_km"], d["w_km"])
    with pytest.raises(RuntimeError):
        plan.run(*args, 0, w.N, w.tiers, w.C, w.C + 1)        # k > n_cand
    with pytest.raises(RuntimeError):
        plan.run(*args, 10, w.N, w.tiers, w.C, w.K)           # zone exceeds capacity
    with pytest.raises(RuntimeError):
        plan.run(*args, 0, w.N, w.tiers, w.N + 1, w.K)        # n_cand > n_keys


# ------------------------------------------------ full-size property checks


@pytest.mark.parametrize("N,R,C,K", [(131072, 32, 4096, 1024)])
def test_full_size_properties(ops, N, R, C, K):
    """BASELINE config 3 at full size on GPU-generated inputs (batch 4, an independent seed per sequence, K/V in
    pinned host memory): size-independent properties of the whole step, the UVA gather of all 32 x 1024 selected rows
    bit for bit against torch.gather on the pinned tensors, and 8 rows spread over the four sequences against the
    oracle (GPU-encoded index copied back to the host; the encode of those rows against the oracle's too).  Both
    launch plans."""
    from pariskv_amd import _lib

    _say(f"full-size N={N} R={R} C={C} K={K}")
    bs, H, G = 4, 8, 4
    signs = ops.srht_signs(DEV)
    codes_km, nib_km, w_km, cb, k4, kw = ops.alloc_keymajor(bs, H, N, DEV)
    cc = torch.zeros(bs, H, 16, 256, dtype=torch.int32, device=DEV)
    q = torch.empty(bs, 1, H * G, 128, dtype=torch.bfloat16, device=DEV)
    keys = torch.empty(bs, H, N, 128, dtype=torch.bfloat16, device=DEV)
    kcpu = torch.empty(bs, H, N, 128, dtype=torch.bfloat16, pin_memory=True)
    vcpu = torch.empty(bs, H, N, 128, dtype=torch.bfloat16, pin_memory=True)
    for b in range(bs):
        g = torch.Generator(device=DEV).manual_seed(1000 * 3 + b)  # one seed per sequence
        kf = torch.randn(1, H, N, 128, generator=g, device=DEV, dtype=torch.float32)
        kf[..., [7, 31, 64, 101]] *= 10
        keys[b] = kf[0].to(torch.bfloat16)
        q[b, 0] = (kf.mean(dim=2, keepdim=True) + 0.5 * torch.randn(1, H, G, 128, generator=g, device=DEV)).view(H * G, 128).to(torch.bfloat16)
        ops.encode_append(keys[b:b + 1], signs, cb[b:b + 1], k4[b:b + 1], kw[b:b + 1], cc[b:b + 1])
        kcpu[b].copy_(keys[b])
        vcpu[b].copy_(torch.randn(H, N, 128, generator=g, device=DEV).to(torch.bfloat16))
        del kf
    assert int(cc.sum()) == R * N * 16 and bool((cc.sum(dim=-1) == N).all())  # every key lands in one cluster per subspace
    tiers = O.tier_counts(N, 0.2)
    plan = ops.RetrievePlan(bs, H, G, N, DEV, N, C, K)
    sc = torch.empty(bs, H, K, device=DEV)
    dk = torch.zeros(bs, H, K, 128, dtype=torch.bfloat16, device=DEV)
    dv = torch.zeros_like(dk)
    gather = dict(src_k=kcpu, src_v=vcpu, from_host=True, dst_k=dk, dst_v=dv)
    out1 = plan.run(q, signs, ops.mag_centers(DEV), cc, codes_km, nib_km, w_km, 0, N, tiers, C, K, out_scores=sc, gather=gather).clone()
    cand = plan.view("cand", N, C, K, torch.int64).view(R, C).clone()
    cnt = plan.view("cnt_u8", N, C, K, torch.uint8).view(R, N).clone()
    out2 = plan.run(q, signs, ops.mag_centers(DEV), cc, codes_km, nib_km, w_km, 0, N, tiers, C, K)
    plan.launch_plan = _lib.PLAN_ONE_LAUNCH
    out3 = plan.run(q, signs, ops.mag_centers(DEV), cc, codes_km, nib_km, w_km, 0, N, tiers, C, K).clone()
    out4 = plan.run(q, signs, ops.mag_centers(DEV), cc, codes_km, nib_km, w_km, 0, N, tiers, C, K)
    torch.cuda.synchronize()
    assert int(plan.view("handover_status", N, C, K, torch.int32)[0]) == 0
    assert torch.equal(out1, out2) and torch.equal(out1, out3) and torch.equal(out1, out4)  # deterministic, both plans
    assert torch.equal(plan.view("cand", N, C, K, torch.int64).view(R, C), cand)
    # the gather of every selected row out of pinned host memory
    idx = out1.cpu().unsqueeze(-1).expand(-1, -1, -1, 128)
    assert torch.equal(dk.cpu(), torch.gather(kcpu, 2, idx)) and torch.equal(dv.cpu(), torch.gather(vcpu, 2, idx))
    assert bool((sc[..., :-1] >= sc[..., 1:]).all())                 # descending scores
    assert bool((out1 >= 0).all()) and bool((out1 < N).all())
    srt = out1.sort(dim=-1).values
    assert bool((srt[..., 1:] != srt[..., :-1]).all())               # no duplicates
    # candidates: distinct, and every non-candidate has a count <= every candidate's
    cs = cand.sort(dim=-1).values
    assert bool((cs[:, 1:] != cs[:, :-1]).all())
    cand_cnt = torch.gather(cnt, 1, cand)
    mask = torch.ones_like(cnt, dtype=torch.bool).scatter_(1, cand, False)
    rest_max = torch.where(mask, cnt, torch.zeros_like(cnt)).max(dim=1).values
    assert bool((cand_cnt.min(dim=1).values >= rest_max).all())
    # final ids are a subset of the candidates
    assert bool(torch.isin(out1.view(R, K), cand).all())
    # rows of every sequence against the oracle, using the GPU-encoded index
    sg = signs.cpu().numpy()
    for r in (0, 5, 10, 13, 19, 22, 28, 31):
        b, h = divmod(r, H)
        ref = O.retrieve_row(q.view(bs, H, G, 128)[b, h].float().cpu().numpy(), sg, O.BF16,
                             codes_km[b, h].cpu().numpy(), nib_km[b, h].cpu().numpy().reshape(N, 16, 4),
                             w_km[b, h].float().cpu().numpy(), cc[b, h].cpu().numpy(), tiers, C, K)
        assert np.array_equal(out1[b, h].cpu().numpy(), ref), f"row {r}"
    for r in (0, 13, 31):  # and the GPU encode of these rows equals the oracle's encode
        b, h = divmod(r, H)
        codes, nib, wt = O.encode(keys[b, h].float().cpu().numpy(), sg, O.BF16)
        assert np.array_equal(codes_km[b, h].cpu().numpy(), codes)
        assert np.array_equal(nib_km[b, h].cpu().numpy().reshape(N, 16, 4), nib)
        assert np.array_equal(w_km[b, h].float().cpu().numpy(), wt)


# --------------------------------------------------------------- adaptive-k


def _adaptive_recipe(bs, kv_heads, sl_len, cand_len, seed, head_dim=128):
    """Seeded input recipe of the reference's adaptive-k self-test (adaptive_topk.py:178-249), on the CPU."""
    torch.manual_seed(seed)
    q = (torch.randn(bs, kv_heads, head_dim) * 0.1).to(torch.bfloat16)
    slk = (torch.randn(bs, kv_heads, sl_len, head_dim) * 0.1).to(torch.bfloat16)
    sl_vnorm = torch.rand(bs, kv_heads, sl_len) + 0.5
    base = math.sqrt(head_dim)
    cs = torch.randn(bs, kv_heads, cand_len) * (0.3 * base)
    rng = torch.Generator().manual_seed(seed)
    heavy = torch.randint(16, 1025, (bs, kv_heads), generator=rng).tolist()
    for b in range(bs):
        for h in range(kv_heads):
            n = min(heavy[b][h], cand_len)
            cs[b, h, :n] += torch.rand(n) * 5.0 * base + 3.0 * base
    ci = torch.stack([torch.stack([torch.randperm(cand_len) for _ in range(kv_heads)]) for _ in range(bs)])
    cv = torch.rand(bs, kv_heads, cand_len) + 0.5
    return q, slk, sl_vnorm, cs.to(torch.bfloat16), ci, cv, 1.0 / base


@pytest.mark.parametrize("cfg", [dict(bs=1, kv_heads=8, sl_len=320, cand_len=12500, topk_cap=2048, threshold=0.95, seed=42),
                                 dict(bs=1, kv_heads=8, sl_len=832, cand_len=5000, topk_cap=2048, threshold=0.95, seed=7),
                                 dict(bs=2, kv_heads=8, sl_len=576, cand_len=8000, topk_cap=2048, threshold=0.85, seed=123),
                                 dict(bs=1, kv_heads=16, sl_len=320, cand_len=15000, topk_cap=2048, threshold=0.95, seed=99),
                                 dict(bs=1, kv_heads=2, sl_len=64, cand_len=700, topk_cap=2048, threshold=0.95, seed=5),
                                 dict(bs=1, kv_heads=2, sl_len=320, cand_len=104858, topk_cap=2048, threshold=0.95, seed=6)])
def test_adaptive_topk_matches_oracle(ops, cfg):
    """The reference's four seeded shapes (adaptive_topk.py:492-497) + a short and a 1M-context-sized one.
    Its acceptance rule is `k exact, first-k index sets equal`; with the fixed tie rule the whole list is compared."""
    from pariskv_amd.cache_hub.adaptive_k_fused import adaptive_topk_cuda

    _say(f"adaptive_topk {cfg}")
    q, slk, slv, cs, ci, cv, scale = _adaptive_recipe(cfg["bs"], cfg["kv_heads"], cfg["sl_len"], cfg["cand_len"], cfg["seed"])
    ak, ids = adaptive_topk_cuda(q.to(DEV), slk.to(DEV), slv.to(DEV), cs.to(DEV), ci.to(DEV), cv.to(DEV), scale,
                                 cfg["threshold"], cfg["topk_cap"])
    torch.cuda.synchronize()
    k_out = min(cfg["topk_cap"], cfg["cand_len"])
    assert tuple(ids.shape) == (cfg["bs"], cfg["kv_heads"], k_out) and ak.dtype == torch.int64
    # same dense logits expression as the call under test, evaluated by torch on the GPU
    sl_logits = (torch.einsum("bhd,bhkd->bhk", q.to(DEV), slk.to(DEV)).to(torch.float32) * scale).cpu().numpy()
    for b in range(cfg["bs"]):
        for h in range(cfg["kv_heads"]):
            lc = (cs[b, h].float() * np.float32(scale)).numpy()
            k_ref, ids_ref = O.adaptive_topk(sl_logits[b, h], slv[b, h].numpy(), lc, cv[b, h].numpy(), ci[b, h].numpy(),
                                             cfg["threshold"], k_out)
            assert int(ak[b, h]) == k_ref, (b, h, int(ak[b, h]), k_ref)
            assert np.array_equal(ids[b, h].cpu().numpy(), ids_ref)
    assert int(ak.min()) >= 1 and int(ak.max()) <= k_out


def test_adaptive_topk_value_norm_gather_and_edges(ops):
    """v2 form: bf16 scores scaled in the kernel, ||v|| gathered at cand_idx + sink (varlen call site :1741-1753);
    plus total <= 0 -> 1 and never reached -> k_out."""
    bs, H, sl, Cn, cap, sink = 1, 3, 100, 3000, 5000, 64
    q, slk, slv, cs, ci, cv, scale = _adaptive_recipe(bs, H, sl, Cn, 11)
    vn = torch.rand(bs, H, cap) + 0.5
    sl_logits = (torch.einsum("bhd,bhkd->bhk", q, slk).float() * scale)
    ak, ids = ops.adaptive_topk(sl_logits.to(DEV), slv.to(DEV), cs.to(DEV), scale, ci.to(DEV), 0.9, 1024,
                                value_norm=vn.to(DEV), vn_offset=sink)
    for h in range(H):
        cvn = vn[0, h][ci[0, h] + sink]
        k_ref, ids_ref = O.adaptive_topk(sl_logits[0, h].numpy(), slv[0, h].numpy(), (cs[0, h].float() * np.float32(scale)).numpy(),
                                         cvn.numpy(), ci[0, h].numpy(), 0.9, 1024)
        assert int(ak[0, h]) == k_ref and np.array_equal(ids[0, h].cpu().numpy(), ids_ref)
    z = torch.zeros(1, 1, 50, device=DEV)
    ak, _ = ops.adaptive_topk(z[..., :5], z[..., :5], z, 1.0, torch.arange(50, device=DEV).view(1, 1, 50), 0.95, 10, cand_vnorm=z)
    assert int(ak) == 1
    one = torch.ones(1, 1, 50, device=DEV)
    ak, ids = ops.adaptive_topk(z[..., :1], one[..., :1], z, 1.0, torch.arange(50, device=DEV).flip(0).view(1, 1, 50).contiguous(),
                                0.95, 10, cand_vnorm=one)
    assert int(ak) == 10 and ids[0, 0].cpu().tolist() == list(range(49, 39, -1))


@pytest.mark.parametrize("sl,Cn,k_out,thr,mode", [(9000, 3000, 3000, 0.97, "cv"),       # dense sum over two slices, k_out == n_cand
                                                  (0, 20000, 4096, 0.5, "cv"),          # no dense tokens, wide path, early k
                                                  (300, 40000, 8192, 0.999, "gather"),  # wide path, largest k_out, norm gather
                                                  (300, 8192, 1000, 0.6, "gather"),     # widest one-workgroup row
                                                  (300, 8193, 1000, 0.6, "gather"),     # narrowest multi-workgroup row
                                                  (50, 30000, 500, 0.9, "ties")])       # quantised benefits: crowded bins
def test_adaptive_topk_shapes_and_orders(ops, sl, Cn, k_out, thr, mode):
    """Adaptive-k against the CPU checker on shapes that exercise each summation / selection branch: k exact,
    ids identical (both follow the same fixed orders)."""
    _say(f"adaptive_topk sl={sl} C={Cn} k_out={k_out} thr={thr} {mode}")
    g = torch.Generator().manual_seed(sl * 31 + Cn)
    H, cap, off = 3, 50000, 17
    sc = torch.randn(1, H, Cn, generator=g) * 6 + 4
    if mode == "ties":
        sc = torch.round(sc)
    sll = torch.randn(1, H, sl, generator=g) * 2 + 6
    slv = torch.rand(1, H, sl, generator=g) + 0.5
    ci = torch.stack([torch.randperm(cap - off, generator=g)[:Cn] for _ in range(H)]).view(1, H, Cn)
    scale = 0.25
    if mode == "gather":
        vn = torch.rand(1, H, cap, generator=g) + 0.5
        ak, ids = ops.adaptive_topk(sll.to(DEV), slv.to(DEV), sc.to(DEV), scale, ci.to(DEV), thr, k_out,
                                    value_norm=vn.to(DEV), vn_offset=off)
        cv = torch.stack([vn[0, h][ci[0, h] + off] for h in range(H)]).view(1, H, Cn)
    else:
        cv = torch.rand(1, H, Cn, generator=g) + 0.5 if mode == "cv" else torch.ones(1, H, Cn)
        ak, ids = ops.adaptive_topk(sll.to(DEV), slv.to(DEV), sc.to(DEV), scale, ci.to(DEV), thr, k_out, cand_vnorm=cv.to(DEV))
    torch.cuda.synchronize()
    ks = []
    for h in range(H):
        k_ref, ids_ref = O.adaptive_topk(sll[0, h].numpy(), slv[0, h].numpy(), (sc[0, h] * np.float32(scale)).numpy(),
                                         cv[0, h].numpy(), ci[0, h].numpy(), thr, k_out)
        assert int(ak[0, h]) == k_ref
        assert np.array_equal(ids[0, h].cpu().numpy(), ids_ref)
        ks.append(k_ref)
    if thr <= 0.6:
        assert max(ks) < k_out  # the threshold is reached inside the list in these cases


def test_adaptive_topk_config4_rows_land_at_different_k(ops):
    """BASELINE config 4's adaptive-k shape (8 rows x ceil(0.05 * 2^20) candidates, list 2048, mass 0.95, clamp
    [256, 2048], value norms gathered from a 2^20-entry table) on scores whose mass is spread differently per row:
    benefits decay like exp(-rank / tau_r), so the 0.95 mass is reached near 3 tau_r and every row stops at its own
    k strictly inside the clamp.  k and the whole id list against the CPU checker."""
    H, N, sink, sl = 8, 1 << 20, 64, 64 + 512
    Cn, k_out, thr, k_min, k_max = int(math.ceil(N * 0.05)), 2048, 0.95, 256, 2048
    taus = [110.0, 170.0, 240.0, 320.0, 400.0, 480.0, 560.0, 630.0]
    g = torch.Generator().manual_seed(44)
    scale = 1.0 / math.sqrt(128)
    sc = torch.empty(1, H, Cn)
    ci = torch.empty(1, H, Cn, dtype=torch.int64)
    for h in range(H):
        rank = torch.randperm(Cn, generator=g).float()                          # rank of candidate i in its row
        sc[0, h] = (-(rank / taus[h]) + 0.3 * torch.rand(Cn, generator=g)) / scale
        ci[0, h] = torch.sort(torch.randperm(N, generator=g)[:Cn]).values       # sorted positions, as the select emits them
    sll = torch.randn(1, H, sl, generator=g) * 0.5 - 6.0                          # the dense tokens hold a small share of the mass
    slv = torch.rand(1, H, sl, generator=g) + 0.5
    vn = torch.rand(1, H, N + sink, generator=g) * 0.2 + 0.9
    _say(f"adaptive-k config 4 shape: {H} rows x {Cn} candidates")
    ak, ids, rk = ops.adaptive_topk(sll.to(DEV), slv.to(DEV), sc.to(DEV), scale, ci.to(DEV), thr, k_out,
                                    value_norm=vn.to(DEV), vn_offset=sink, k_min=k_min, k_max=k_max, row_keys_base=sl)
    torch.cuda.synchronize()
    rk = rk.view(-1)
    ks = []
    for h in range(H):
        cvn = vn[0, h][ci[0, h] + sink]
        k_ref, ids_ref = O.adaptive_topk(sll[0, h].numpy(), slv[0, h].numpy(), (sc[0, h] * np.float32(scale)).numpy(),
                                         cvn.numpy(), ci[0, h].numpy(), thr, k_out)
        assert k_min < k_ref < k_max, (h, k_ref)
        assert int(ak[0, h]) == k_ref and int(rk[h]) == sl + k_ref
        assert np.array_equal(ids[0, h].cpu().numpy(), ids_ref)
        ks.append(k_ref)
    assert len(set(ks)) == H and ks == sorted(ks), ks
    _say(f"adaptive k per row: {ks}")


def test_adaptive_topk_wide_zero_mass(ops):
    """total <= 0 on the multi-workgroup path: k = 1 (adaptive_topk.py:304-306); ids still ordered by position."""
    Cn = 10000
    z = torch.zeros(1, 2, Cn, device=DEV)
    ci = torch.arange(Cn, device=DEV).flip(0).expand(1, 2, Cn).contiguous()
    ak, ids = ops.adaptive_topk(z[..., :7], z[..., :7], z, 1.0, ci, 0.95, 300, cand_vnorm=z)
    assert ak.flatten().tolist() == [1, 1]
    assert ids[0, 1].cpu().tolist() == list(range(Cn - 1, Cn - 301, -1))


# ---------------------------------- 1M keys, adaptive-k, packed gather


def test_million_key_adaptive_pipeline(ops):
    """Llama-3-8B head shape, batch 1, 1M cached keys per head with a slowly drifting key mean (0.5 degrees per 1K
    tokens), bucket top-k over 1M vote counts, rerank of all candidates, adaptive-k (k clamped to [256, 2048], mass
    0.95), packed UVA gather.  Every stage of two sampled rows is compared with the oracle; the rest by properties."""
    from pariskv_amd.cache_hub.topk import load_radix_topk_ext

    _say("cfg4: N=2^20")
    bs, H, G, N = 1, 8, 4, 1 << 20
    sink, sl = 64, 64 + 512
    Cn = int(math.ceil(N * 0.05))
    cap_k, min_k, thr = 2048, 256, 0.95
    g = torch.Generator(device=DEV).manual_seed(4)
    keys = torch.randn(bs, H, N, 128, generator=g, device=DEV)
    keys[..., [7, 31, 64, 101]] *= 10.0
    ang = torch.arange(N, device=DEV, dtype=torch.float32) * (0.5 / 1000.0) * (math.pi / 180.0)
    keys[..., 0] += 3.0 * torch.cos(ang)
    keys[..., 1] += 3.0 * torch.sin(ang)
    keys = keys.to(torch.bfloat16)
    q = (keys[:, :, -4096:].float().mean(dim=2, keepdim=True) + 0.5 * torch.randn(bs, H, G, 128, generator=g, device=DEV))
    q = q.to(torch.bfloat16).view(bs, 1, H * G, 128).contiguous()
    signs = ops.srht_signs(DEV)
    codes_km, nib_km, w_km, cb, k4, kw = ops.alloc_keymajor(bs, H, N, DEV)
    cc = torch.zeros(bs, H, 16, 256, dtype=torch.int32, device=DEV)
    ops.encode_append(keys, signs, cb, k4, kw, cc)
    tiers = O.tier_counts(N, 0.2)
    assert tiers == [10486, 31458, 62915, 104858, 157287, 209716]
    qhat, qnorm, lut, _ = ops.query_prep_lut(q, H, signs, cc, tiers)
    cnt, _, _ = ops.collision_scan(cb, lut, out_dtype=torch.int32)
    cand = load_radix_topk_ext().radix_topk_3d(cnt, Cn)          # "radix top-k over 1M scores" (polar_cache.py:1241)
    scores, _ = ops.rerank4(cand, k4, kw, qhat, qnorm, ops.mag_centers(DEV))
    # dense side of adaptive-k: logits and value norms of sink + local tokens, ||v|| of every cached token
    sl_logits = torch.randn(bs, H, sl, generator=g, device=DEV) * 0.5
    sl_vnorm = torch.rand(bs, H, sl, generator=g, device=DEV) + 0.5
    value_norm = torch.rand(bs, H, N + sink, generator=g, device=DEV) + 0.5
    scale = 1.0 / math.sqrt(128)
    k_out = min(cap_k, Cn)
    ak, ids = ops.adaptive_topk(sl_logits, sl_vnorm, scores, scale, cand, thr, k_out, value_norm=value_norm, vn_offset=sink)
    ak = ak.clamp(min=max(1, min_k), max=max(1, cap_k))           # polar_cache_adaptivek_varlen.py:1759
    torch.cuda.synchronize()
    sg = signs.cpu().numpy()
    for r in (1, 6):
        codes = codes_km[0, r].cpu().numpy()
        ec, en, ew = O.encode(keys[0, r].float().cpu().numpy(), sg, O.BF16)
        assert np.array_equal(codes, ec) and np.array_equal(nib_km[0, r].cpu().numpy().reshape(N, 16, 4), en)
        assert np.array_equal(w_km[0, r].float().cpu().numpy(), ew)
        assert np.array_equal(cc[0, r].cpu().numpy(), O.count_cluster_keys(ec))
        qh, qn = O.query_prep(q.view(bs, H, G, 128)[0, r].float().cpu().numpy(), sg, O.BF16)
        lut_ref = O.tier_lut(O.rank_centroids(qh, O.BF16), cc[0, r].cpu().numpy(), tiers)
        cnt_ref = O.collision_count(ec, lut_ref)
        assert np.array_equal(cnt[0, r].cpu().numpy(), cnt_ref)
        cand_ref, _ = O.select_candidates(cnt_ref, Cn)
        assert np.array_equal(cand[0, r].cpu().numpy(), cand_ref)
        sc_ref = O.rerank(cand_ref, en, ew, qh, qn)
        got = scores[0, r].cpu().numpy()
        np.testing.assert_allclose(got, sc_ref, rtol=1e-5, atol=1e-5 * np.abs(sc_ref).max())
        vn = value_norm[0, r].cpu().numpy()[cand_ref + sink]
        k_ref, ids_ref = O.adaptive_topk(sl_logits[0, r].cpu().numpy(), sl_vnorm[0, r].cpu().numpy(), got * np.float32(scale), vn,
                                         cand_ref, thr, k_out)
        assert int(ak[0, r]) == min(max(k_ref, min_k), cap_k)
        assert np.array_equal(ids[0, r].cpu().numpy(), ids_ref)
    assert int(ak.min()) >= min_k and int(ak.max()) <= cap_k
    # pack the per-head prefixes (polar_cache_adaptivek_varlen.py:1817-1832) and gather them raggedly out of host memory
    V = bs * H
    mask = torch.arange(k_out, device=DEV).unsqueeze(0) < ak.view(V, 1)
    packed = ids.view(V, k_out)[mask].contiguous()
    cu_topk = torch.zeros(V + 1, dtype=torch.int32, device=DEV)
    cu_topk[1:] = torch.cumsum(ak.view(V), 0)
    cu_k = torch.zeros(V + 1, dtype=torch.int32, device=DEV)
    cu_k[1:] = torch.cumsum(ak.view(V) + sl, 0)
    total = int(cu_k[-1])
    kcpu = torch.empty(bs, H, N, 128, dtype=torch.bfloat16, pin_memory=True)
    vcpu = torch.empty(bs, H, N, 128, dtype=torch.bfloat16, pin_memory=True)
    kcpu.copy_(keys)
    vcpu.copy_(-keys)
    kp = torch.zeros(total, 128, dtype=torch.bfloat16, device=DEV)
    vp = torch.zeros_like(kp)
    ops.gather_uva_packed(kcpu, vcpu, kp, vp, packed, cu_topk, cu_k, sl, int(ak.max()))
    torch.cuda.synchronize()
    for v in range(V):
        n = int(ak.view(V)[v])
        sel = ids.view(V, k_out)[v, :n]
        base = int(cu_k[v]) + sl
        assert torch.equal(kp[base:base + n], keys[0, v][sel]) and torch.equal(vp[base:base + n], -keys[0, v][sel])
        assert not kp[int(cu_k[v]):base].any()   # the sink/local slots are the caller's to fill


# ------------------------------------------------------- decode attention


@pytest.mark.parametrize("dtype,group,lens", [
    (torch.bfloat16, 4, (64, 1024, 512)),          # sink | gathered top-k | local window
    (torch.bfloat16, 4, (64, 300, 1000, 37)),      # four ragged segments
    (torch.bfloat16, 1, (5,)),                     # fewer keys than one workgroup step
    (torch.bfloat16, 8, (2000,)),
    (torch.float32, 2, (129, 64)),
    (torch.bfloat16, 7, (64, 500)),                # 28 query / 4 KV heads
])
def test_decode_attention_segments_vs_oracle(ops, dtype, group, lens):
    """softmax(q k^T / sqrt(128)) v over row segments read in place, against the double-precision
    CPU oracle on the same (bf16-exact) inputs.  Tolerance 2e-2 absolute in bf16, 1e-4 in fp32."""
    bs, H = 2, 3
    _say(f"decode attention dtype={dtype} G={group} segments={lens}")
    g = torch.Generator(device=DEV).manual_seed(11)
    q = (torch.randn(bs, 1, H * group, 128, generator=g, device=DEV) * 1.5).to(dtype)
    segs, ks, vs = [], [], []
    for i, n in enumerate(lens):
        cap = n + 17 + i
        row0 = 3 + i
        k = torch.randn(bs, H, cap, 128, generator=g, device=DEV).to(dtype)
        v = torch.randn(bs, H, cap, 128, generator=g, device=DEV).to(dtype)
        if i == 1:  # a sliced parent tensor: batch/head strides larger than rows * 128
            big_k = torch.randn(bs, H + 1, cap + 5, 128, generator=g, device=DEV).to(dtype)
            big_v = torch.randn(bs, H + 1, cap + 5, 128, generator=g, device=DEV).to(dtype)
            k, v = big_k[:, :H, :cap], big_v[:, :H, :cap]
        segs.append((k, v, row0, n))
        ks.append(k[:, :, row0:row0 + n])
        vs.append(v[:, :, row0:row0 + n])
    att = ops.DecodeAttention(bs, H, group, sum(lens), DEV)
    out = att.run(q, segs)
    torch.cuda.synchronize()
    assert out.shape == q.shape and out.dtype == dtype
    kc = torch.cat(ks, dim=2).float().cpu().numpy()
    vc = torch.cat(vs, dim=2).float().cpu().numpy()
    qc = q.float().cpu().numpy().reshape(bs, H, group, 128)
    got = out.float().cpu().numpy().reshape(bs, H, group, 128)
    tol = 2e-2 if dtype == torch.bfloat16 else 1e-4
    for b in range(bs):
        for h in range(H):
            ref = O.attention(qc[b, h], kc[b, h], vc[b, h])
            assert np.abs(got[b, h] - ref).max() <= tol, (b, h, np.abs(got[b, h] - ref).max())


@pytest.mark.parametrize("dtype,group,K", [(torch.bfloat16, 4, 300), (torch.bfloat16, 8, 77), (torch.bfloat16, 1, 1500),
                                           (torch.float32, 4, 130), (torch.float32, 7, 64)])
def test_decode_attention_indexed_segment_equals_gathered(ops, dtype, group, K):
    """A segment given as an index list (rows row0 + idx[b,h,j], read in place) against the same rows gathered into a
    buffer first (reference polar_cache.py:1089-1095 + 1097-1105): the two outputs are identical, and both match the
    CPU oracle.  Sink and local segments surround the indexed one, as in the no-offload decode step; a ragged
    row_keys case and out-of-range indices (clamped, no fault) are included."""
    bs, H, cap, sink, tail0, tail = 2, 3, 2500, 5, 2300, 140
    _say(f"indexed attention dtype={dtype} G={group} K={K}")
    g = torch.Generator(device=DEV).manual_seed(21)
    q = (torch.randn(bs, 1, H * group, 128, generator=g, device=DEV) * 1.5).to(dtype)
    kk = torch.randn(bs, H, cap, 128, generator=g, device=DEV).to(dtype)
    vv = torch.randn(bs, H, cap, 128, generator=g, device=DEV).to(dtype)
    idx = torch.stack([torch.randperm(tail0 - sink, generator=g, device=DEV)[:K + 9] for _ in range(bs * H)]).view(bs, H, K + 9)
    gk = torch.empty(bs, H, K, 128, dtype=dtype, device=DEV)
    gv = torch.empty_like(gk)
    ops.gather_hbm(kk, vv, idx[:, :, :K].contiguous(), gk, gv, idx_offset=sink)
    att = ops.DecodeAttention(bs, H, group, sink + K + tail, DEV)
    for row_keys in (None, torch.tensor([[sink + K + tail, sink + 3, sink + K], [40 if K > 40 else K, sink + K + 1, 1]],
                                        dtype=torch.int32, device=DEV)):
        a = att.run(q, [(kk, vv, 0, sink), (kk, vv, sink, K, idx), (kk, vv, tail0, tail)], row_keys=row_keys).clone()
        b_ = att.run(q, [(kk, vv, 0, sink), (gk, gv, 0, K), (kk, vv, tail0, tail)], row_keys=row_keys).clone()
        torch.cuda.synchronize()
        assert torch.equal(a, b_)
    kc = torch.cat([kk[:, :, :sink], gk, kk[:, :, tail0:tail0 + tail]], dim=2).float().cpu().numpy()
    vc = torch.cat([vv[:, :, :sink], gv, vv[:, :, tail0:tail0 + tail]], dim=2).float().cpu().numpy()
    full = att.run(q, [(kk, vv, 0, sink), (kk, vv, sink, K, idx), (kk, vv, tail0, tail)])
    got = full.float().cpu().numpy().reshape(bs, H, group, 128)
    qc = q.float().cpu().numpy().reshape(bs, H, group, 128)
    tol = 2e-2 if dtype == torch.bfloat16 else 1e-4
    for b in range(bs):
        for h in range(H):
            assert np.abs(got[b, h] - O.attention(qc[b, h], kc[b, h], vc[b, h])).max() <= tol
    wild = idx.clone()
    wild[:, :, ::7] = 10 ** 9          # far outside the tensor: clamped to its last row, must not fault
    wild[:, :, 3::11] = -5
    out = att.run(q, [(kk, vv, sink, K, wild)])
    torch.cuda.synchronize()
    assert bool(torch.isfinite(out.float()).all())
    with pytest.raises(RuntimeError, match="segment indices"):
        att.run(q, [(kk, vv, sink, K, idx.to(torch.int32))])


@pytest.mark.parametrize("group", [3, 4, 5, 7, 8])
def test_decode_attention_fp32_head_groups(ops, group):
    """fp32 query heads in workgroups of four side by side: every head count around that limit, ragged rows, against the
    oracle (fp32 sums of at most 333 keys: 1e-4, as in the segment test)."""
    bs, H, n = 2, 2, 333
    g = torch.Generator(device=DEV).manual_seed(group)
    q = torch.randn(bs, 1, H * group, 128, generator=g, device=DEV) * 1.5
    k, v = (torch.randn(bs, H, n, 128, generator=g, device=DEV) for _ in range(2))
    row_keys = torch.tensor([[n, 1], [33, n - 1]], dtype=torch.int32, device=DEV)
    out = ops.DecodeAttention(bs, H, group, n, DEV).run(q, [(k, v, 0, n)], row_keys=row_keys).cpu().numpy().reshape(bs, H, group, 128)
    for b in range(bs):
        for h in range(H):
            rk = int(row_keys[b, h])
            ref = O.attention(q.cpu().numpy().reshape(bs, H, group, 128)[b, h], k[b, h, :rk].cpu().numpy(), v[b, h, :rk].cpu().numpy())
            assert np.abs(out[b, h] - ref).max() <= 1e-4, (b, h)


def test_decode_attention_argument_errors(ops):
    att = ops.DecodeAttention(1, 2, 4, 64, DEV)
    q = torch.zeros(1, 1, 8, 128, dtype=torch.bfloat16, device=DEV)
    k = torch.zeros(1, 2, 64, 128, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(RuntimeError, match="out of range"):
        att.run(q, [(k, k, 10, 60)])
    with pytest.raises(RuntimeError, match="share a dtype"):
        att.run(q, [(k.float(), k.float(), 0, 8)])
    with pytest.raises(RuntimeError, match="no keys"):
        att.run(q, [(k, k, 0, 0)])
    bad = ops.DecodeAttention(1, 2, 9, 64, DEV)
    with pytest.raises(RuntimeError, match="group must be"):
        bad.run(torch.zeros(1, 1, 18, 128, dtype=torch.bfloat16, device=DEV), [(k, k, 0, 8)])


# --------------------------------------------------- randomised small shapes


def test_retrieve_random_shapes_vs_oracle(ops):
    """Whole retrieval on 16 seeded shapes (ragged key counts, group sizes 1-7, candidate counts from 1 to
    every key, k from 1 to the candidate count, both dtype chains): final indices bit-exact against the oracle."""
    rng = np.random.default_rng(2024)
    shapes = [(1, 1, 1, 50, 1, 1), (1, 2, 7, 333, 333, 17), (2, 1, 3, 4097, 4096, 4096), (1, 1, 4, 8193, 5000, 1),
              (1, 2, 4, 30000, 12000, 3000), (1, 1, 2, 20000, 20000, 8192)]   # candidate rows wider than one workgroup sorts
    while len(shapes) < 16:
        N = int(rng.integers(60, 20000))
        C = int(rng.integers(1, N + 1))
        shapes.append((int(rng.integers(1, 3)), int(rng.integers(1, 3)), int(rng.integers(1, 8)), N, C,
                       int(rng.integers(1, C + 1))))
    for i, (bs, H, G, N, C, K) in enumerate(shapes):
        dtype = O.BF16 if i % 3 else O.F32
        _say(f"random shape {i}: bs={bs} H={H} G={G} N={N} C={C} K={K} dtype={dtype}")
        w = W.make_workload(f"rand{i}", bs, H, G, N, C, K, dtype, float(rng.choice([0.2, 0.3, 0.5])), seed0=100 + i,
                            with_values=False)
        plan, out, scores = _run_fused(ops, w)
        for r in range(w.R):
            b, h = divmod(r, w.H)
            ref = O.retrieve_row(w.queries[b, h * G:(h + 1) * G], w.signs, w.dtype, w.codes[r], w.nib[r], w.weight[r],
                                 w.cluster_counts[r], w.tiers, C, K)
            assert np.array_equal(out[b, h].cpu().numpy(), ref), f"shape {i} row {r}"
            s = scores[b, h].cpu().numpy()
            assert np.all(s[:-1] >= s[1:])


def test_decode_step_single_call_equals_separate_calls(ops, wl_small_bf16):
    """pkv_decode_step (retrieve + gather + attention from one host call) against the three separate entry points."""
    w = wl_small_bf16
    d = W.to_device(w, DEV, torch)
    g = torch.Generator(device=DEV).manual_seed(3)
    src_k = torch.randn(w.bs, w.H, w.N, 128, generator=g, device=DEV).to(torch.bfloat16)
    src_v = torch.randn(w.bs, w.H, w.N, 128, generator=g, device=DEV).to(torch.bfloat16)
    dense_k = torch.randn(w.bs, w.H, 40, 128, generator=g, device=DEV).to(torch.bfloat16)
    dense_v = torch.randn(w.bs, w.H, 40, 128, generator=g, device=DEV).to(torch.bfloat16)
    plan = ops.RetrievePlan(w.bs, w.H, w.G, w.N, DEV, w.N, w.C, w.K)
    att = ops.DecodeAttention(w.bs, w.H, w.G, 40 + w.K, DEV)
    outs = []
    for fused in (False, True):
        dst_k = torch.zeros(w.bs, w.H, w.K, 128, dtype=torch.bfloat16, device=DEV)
        dst_v = torch.zeros_like(dst_k)
        gather = dict(src_k=src_k, src_v=src_v, from_host=False, dst_k=dst_k, dst_v=dst_v)
        segs = [(dense_k, dense_v, 0, 8), (dst_k, dst_v, 0, w.K), (dense_k, dense_v, 8, 32)]
        args = (d["queries"], d["signs"], d["centers"], d["cluster_counts"], d["codes_km"], d["nib_km"], d["w_km"], 0, w.N,
                w.tiers, w.C, w.K)
        if fused:
            ids = plan.run(*args, gather=gather, attention=(att, segs, None))
            out = plan.attn_out
        else:
            ids = plan.run(*args, gather=gather)
            out = att.run(d["queries"], segs)
        torch.cuda.synchronize()
        outs.append((ids.clone(), out.clone(), dst_k.clone()))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][2], outs[1][2])
    assert torch.equal(outs[0][1], outs[1][1]) and outs[1][1].shape == d["queries"].shape
    # and the attention agrees with the oracle on the gathered rows of one (b, h)
    b, h = 1, 0
    sel = outs[1][0][b, h].cpu()
    kk = torch.cat([dense_k[b, h, :8].cpu(), src_k[b, h].cpu()[sel], dense_k[b, h, 8:40].cpu()]).float().numpy()
    vv = torch.cat([dense_v[b, h, :8].cpu(), src_v[b, h].cpu()[sel], dense_v[b, h, 8:40].cpu()]).float().numpy()
    qq = d["queries"][b, 0, h * w.G:(h + 1) * w.G].float().cpu().numpy()
    got = outs[1][1][b, 0, h * w.G:(h + 1) * w.G].float().cpu().numpy()
    assert np.abs(got - O.attention(qq, kk, vv)).max() <= 2e-2


def test_decode_step_replays_from_a_captured_graph(ops, wl_small_bf16):
    """The launch sequence allocates nothing, synchronises nothing and records no memset: it can be captured into
    a graph once and replayed.  Three replays with different queries and eager work in between, each checked
    against the eager result of the same inputs."""
    w = wl_small_bf16
    d = W.to_device(w, DEV, torch)
    g = torch.Generator(device=DEV).manual_seed(4)
    src_k = torch.randn(w.bs, w.H, w.N, 128, generator=g, device=DEV).to(torch.bfloat16)
    src_v = torch.randn(w.bs, w.H, w.N, 128, generator=g, device=DEV).to(torch.bfloat16)
    plan = ops.RetrievePlan(w.bs, w.H, w.G, w.N, DEV, w.N, w.C, w.K)
    att = ops.DecodeAttention(w.bs, w.H, w.G, w.K, DEV)
    dst_k = torch.zeros(w.bs, w.H, w.K, 128, dtype=torch.bfloat16, device=DEV)
    dst_v = torch.zeros_like(dst_k)
    gather = dict(src_k=src_k, src_v=src_v, from_host=False, dst_k=dst_k, dst_v=dst_v)
    q_static = d["queries"].clone()
    ids_static = torch.zeros(w.bs, w.H, w.K, dtype=torch.int64, device=DEV)
    out_static = torch.zeros_like(q_static)

    def step():
        plan.run(q_static, d["signs"], d["centers"], d["cluster_counts"], d["codes_km"], d["nib_km"], d["w_km"], 0, w.N,
                 w.tiers, w.C, w.K, out_ids=ids_static, gather=gather, attention=(att, [(dst_k, dst_v, 0, w.K)], out_static))

    step()  # warm-up outside the capture (module load, workspace sizing)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for rep in range(3):
        q_new = (d["queries"].float() + 0.3 * torch.randn(d["queries"].shape, generator=g, device=DEV)).to(torch.bfloat16)
        q_static.copy_(q_new)
        ids_static.zero_(), out_static.zero_(), dst_k.zero_()
        graph.replay()
        torch.cuda.synchronize()
        got_ids, got_out = ids_static.clone(), out_static.clone()
        scratch = torch.randn(1 << 20, device=DEV).sum().item()  # unrelated eager work between replays
        ids_static.zero_(), out_static.zero_()
        step()
        torch.cuda.synchronize()
        assert torch.equal(got_ids, ids_static), f"replay {rep}: indices differ from the eager run"
        assert torch.equal(got_out, out_static), f"replay {rep}: attention differs from the eager run"
        assert scratch == scratch


def test_rerank_rabitq_fused_helper(ops, wl_small_bf16):
    """rerank_rabitq_fused (reference rerank.py:266-293): coarse filter + rerank + final top-k from the vote counts."""
    from pariskv_amd.cache_hub.rerank.rerank import rerank_rabitq_fused

    w = wl_small_bf16
    d = W.to_device(w, DEV, torch)
    codes_km, nib_km, w_km = d["codes_km"], d["nib_km"], d["w_km"]
    k4 = nib_km.view(w.bs, w.H, w.N, 16, 4).permute(0, 1, 3, 2, 4)   # reference-shaped views of key-major memory
    kw = w_km.permute(0, 1, 3, 2)
    cb = codes_km.permute(0, 1, 3, 2)
    qhat, qnorm, lut, _ = ops.query_prep_lut(d["queries"], w.H, d["signs"], d["cluster_counts"], w.tiers)
    cnt, _, _ = ops.collision_scan(cb, lut, out_dtype=torch.int32)
    ratio, final_k = 0.05, 40
    ids, scores, v4b = rerank_rabitq_fused(cnt, k4, kw, qhat.view(w.bs, w.H, 16, 8), qnorm.view(w.bs, w.H, 1),
                                           ops.mag_centers(DEV), ratio, final_k, 16, 8)
    torch.cuda.synchronize()
    n_cand = int(math.ceil(w.N * ratio))
    assert ids.shape == (w.bs, w.H, final_k) and scores.shape == (w.bs, w.H, n_cand)
    for r in range(w.R):
        b, h = divmod(r, w.H)
        st = W.oracle_stages(w, r)
        cand, _ = O.select_candidates(st["cnt"], n_cand)
        sc = O.rerank(cand, w.nib[r], w.weight[r], st["qhat"], st["qnorm"])
        final, _ = O.topk_f32(sc, cand, final_k)
        assert np.array_equal(ids[b, h].cpu().numpy(), final)
    # candidate set not larger than final_topk: the coarse indices come back, nothing is scored
    ids2, s2, v2 = rerank_rabitq_fused(cnt, k4, kw, qhat.view(w.bs, w.H, 16, 8), qnorm.view(w.bs, w.H, 1),
                                       ops.mag_centers(DEV), 0.001, 40, 16, 8)
    assert s2 is None and v2 is None and ids2.shape[2] == int(math.ceil(w.N * 0.001))


def test_srht_signs_equal_the_device_generator_draw(ops):
    """The reference draws the SRHT diagonal from torch's device generator (polar_cache.py:57-63); the host
    restatement used here must give the same vector, for the shipped seed and others, and leave the generators alone."""
    cpu_state, dev_state = torch.get_rng_state(), torch.cuda.get_rng_state(0)
    for seed in (42, 0, 7, 123456789012):
        before = torch.get_rng_state(), torch.cuda.get_rng_state(0)
        mine = ops.srht_signs(DEV, seed)
        assert torch.equal(torch.get_rng_state(), before[0]) and torch.equal(torch.cuda.get_rng_state(0), before[1])
        torch.manual_seed(seed)
        ref = torch.randint(0, 2, (128,), device=DEV, dtype=torch.bfloat16) * 2 - 1   # the reference's expression
        assert torch.equal(mine, ref.float())
        assert np.array_equal(O.srht_signs(seed), mine.cpu().numpy())
    torch.set_rng_state(cpu_state)
    torch.cuda.set_rng_state(dev_state, 0)


def test_gather_uva_ragged_moves_only_each_rows_prefix(ops):
    """pkv_gather_uva_ragged: row (b, h) fetches its first row_counts[b, h] selected rows; the rest of dst is untouched;
    counts 0 and K included."""
    g = torch.Generator().manual_seed(8)
    bs, H, N, K, D = 2, 3, 500, 40, 128
    sk = torch.randn(bs, H, N, D, generator=g).to(torch.bfloat16).pin_memory()
    sv = torch.randn(bs, H, N, D, generator=g).to(torch.bfloat16).pin_memory()
    idx = torch.stack([torch.randperm(N, generator=g)[:K] for _ in range(bs * H)]).view(bs, H, K)
    counts = torch.tensor([[0, K, 7], [1, 39, 20]], dtype=torch.int64)
    dk = torch.full((bs, H, K + 5, D), 3.0, dtype=torch.bfloat16, device=DEV)
    dv = torch.full((bs, H, K + 5, D), 5.0, dtype=torch.bfloat16, device=DEV)
    want_k, want_v = dk.cpu().clone(), dv.cpu().clone()
    ops.gather_uva_ragged(sk, sv, idx.to(DEV), counts.to(DEV), dk, dv, dst_row0=2)
    torch.cuda.synchronize()
    for b in range(bs):
        for h in range(H):
            c = int(counts[b, h])
            want_k[b, h, 2:2 + c] = sk[b, h][idx[b, h, :c]]
            want_v[b, h, 2:2 + c] = sv[b, h][idx[b, h, :c]]
    assert torch.equal(dk.cpu(), want_k) and torch.equal(dv.cpu(), want_v)


def test_append_kv_equals_indexed_assignment(ops):
    """pkv_append_kv against the two indexed assignments it replaces (reference polar_cache.py:848-856), with
    contiguous and strided new rows and a strided (sliced-batch) store."""
    g = torch.Generator().manual_seed(5)
    bs, H, cap, D = 3, 4, 37, 128
    for dtype in (torch.bfloat16, torch.float32):
        kg = torch.randn(bs + 1, H, cap, D, generator=g).to(dtype).to(DEV)
        vg = torch.randn(bs + 1, H, cap, D, generator=g).to(dtype).to(DEV)
        dk, dv = kg[1:], vg[1:]
        fused = torch.randn(bs, 1, 3 * H, D, generator=g).to(dtype).to(DEV)   # rows of a fused projection: strided heads
        for k1, v1 in ((fused[:, :, :H], fused[:, :, 2 * H:]),
                       (fused[:, :, H:2 * H].contiguous(), fused[:, :, :H].contiguous())):
            for slot in (0, 17, cap - 1):
                wk, wv = dk.clone(), dv.clone()
                wk[:, :, slot, :] = k1[:, 0]
                wv[:, :, slot, :] = v1[:, 0]
                ops.append_kv(k1, v1, dk, dv, slot)
                torch.cuda.synchronize()
                assert torch.equal(dk, wk) and torch.equal(dv, wv)
        with pytest.raises(RuntimeError, match="slot"):
            ops.append_kv(fused[:, :, :H], fused[:, :, H:2 * H], dk, dv, cap)
    with pytest.raises(RuntimeError):
        ops.append_kv(fused[:, :, :H], fused[:, :, H:2 * H + 1], dk, dv, 0)


def test_append_kv_value_norm(ops):
    """The value norm written by pkv_append_kv (adaptive-k bookkeeping, reference polar_cache_adaptivek_varlen.py:1179):
    bit-equal to the oracle's fixed-order restatement, within one step of the dtype of torch's vector_norm; the other
    slots of the norm table stay untouched."""
    g = torch.Generator().manual_seed(8)
    bs, H, cap, D = 3, 4, 21, 128
    for dtype, odt, rtol in ((torch.bfloat16, O.BF16, 2.0 ** -7), (torch.float32, O.F32, 2e-6)):
        dk = torch.zeros(bs, H, cap, D, dtype=dtype, device=DEV)
        dv = torch.zeros_like(dk)
        table = torch.full((bs + 1, H, cap + 3), -1.0, device=DEV)
        vn = table[1:]                                         # a batch slice: strided rows
        fused = (torch.randn(bs, 1, 3 * H, D, generator=g) * torch.rand(bs, 1, 3 * H, 1, generator=g) * 4).to(dtype).to(DEV)
        for slot, (k1, v1) in ((5, (fused[:, :, :H], fused[:, :, 2 * H:])), (cap - 1, (fused[:, :, H:2 * H], fused[:, :, :H]))):
            ops.append_kv(k1, v1, dk, dv, slot, vnorm=vn)
            torch.cuda.synchronize()
            assert torch.equal(dv[:, :, slot], v1[:, 0]) and torch.equal(dk[:, :, slot], k1[:, 0])
            want = O.value_norm(v1[:, 0].float().cpu().numpy().reshape(-1, D), odt).reshape(bs, H)
            assert np.array_equal(vn[:, :, slot].cpu().numpy(), want)
            ref = torch.linalg.vector_norm(v1[:, 0], dim=-1).float()
            assert torch.allclose(vn[:, :, slot], ref, rtol=rtol, atol=0)
        untouched = torch.ones(cap + 3, dtype=torch.bool)
        untouched[[5, cap - 1]] = False
        assert (vn[:, :, untouched] == -1).all() and (table[0] == -1).all()
    with pytest.raises(RuntimeError, match="vnorm"):
        ops.append_kv(fused[:, :, :H], fused[:, :, H:2 * H], dk, dv, 0, vnorm=vn[:, :, :0])


@pytest.mark.parametrize("bs,H,G,rows,n", [(1, 8, 4, 700, 700), (2, 2, 7, 100, 33), (3, 1, 1, 17, 17), (1, 4, 12, 2000, 1999)])
def test_dense_logits_match_oracle(ops, bs, H, G, rows, n):
    """pkv_dense_logits (reference polar_cache_adaptivek_varlen.py:1418-1419 + :1731): bit-equal to the oracle's
    fixed-order restatement in both rounding chains, and within one bf16 step / 2e-6 of the torch expressions; rows
    beyond n and the padding of a longer output row are not written."""
    g = torch.Generator().manual_seed(bs * 100 + G)
    scale = 1.0 / math.sqrt(128)
    for dtype, odt, rtol in ((torch.bfloat16, O.BF16, 2.0 ** -7), (torch.float32, O.F32, 2e-6)):
        q = torch.randn(bs, 1, H * G, 128, generator=g).to(dtype).to(DEV)
        store = (torch.randn(bs + 1, H, rows, 128, generator=g) * 1.5).to(dtype).to(DEV)
        k = store[1:]                                           # strided batch
        out = torch.full((bs, H, rows + 5), 7.0, device=DEV)
        got = ops.dense_logits(q, k, n, scale, out=out)
        torch.cuda.synchronize()
        assert got.data_ptr() == out.data_ptr() and (out[:, :, n:] == 7.0).all()
        qc, kc = q.float().cpu().numpy().reshape(bs, H, G, 128), k.float().cpu().numpy()
        for b in range(bs):
            for h in range(H):
                want = O.dense_logits(qc[b, h], kc[b, h, :n], scale, odt)
                assert np.array_equal(out[b, h, :n].cpu().numpy(), want), (b, h)
        ref = torch.einsum("bhd,bhkd->bhk", q[:, 0].view(bs, H, G, 128).mean(dim=2), k[:, :, :n]).to(torch.float32) * scale
        assert torch.allclose(out[:, :, :n], ref, rtol=rtol, atol=rtol * float(ref.abs().max()))
        fresh = ops.dense_logits(q, k, n, scale)
        assert fresh.shape == (bs, H, n) and torch.equal(fresh, out[:, :, :n])
    with pytest.raises(RuntimeError):
        ops.dense_logits(q, k, rows + 1, scale)


def test_adaptive_topk_clamp_and_row_keys(ops):
    """The clamp of k (reference polar_cache_adaptivek_varlen.py:1759) and the per-row key count folded into the
    adaptive-k kernels, on the one-workgroup and the multi-workgroup path: equal to clamping the unclamped result."""
    for Cn, k_out in ((3000, 800), (20000, 800)):
        bs, H, sl = 2, 3, 200
        q, slk, slv, cs, ci, cv, scale = _adaptive_recipe(bs, H, sl, Cn, 23)
        sl_logits = (torch.einsum("bhd,bhkd->bhk", q, slk).float() * scale).to(DEV)
        args = (sl_logits, slv.to(DEV), cs.to(DEV), scale, ci.to(DEV))
        for thr in (0.3, 0.9, 0.9999):
            ak0, ids0 = ops.adaptive_topk(*args, thr, k_out, cand_vnorm=cv.to(DEV))
            ak1, ids1, rk = ops.adaptive_topk(*args, thr, k_out, cand_vnorm=cv.to(DEV), k_min=100, k_max=500, row_keys_base=sl + 7)
            assert torch.equal(ids0, ids1)
            assert torch.equal(ak1, ak0.clamp(min=100, max=500))
            assert rk.dtype == torch.int32 and torch.equal(rk.long(), ak1 + sl + 7)
        assert len({int(v) for v in ak0.flatten()} | {int(v) for v in ak1.flatten()}) > 1
    with pytest.raises(RuntimeError, match="clamp"):
        ops.adaptive_topk(*args, 0.9, k_out, cand_vnorm=cv.to(DEV), k_min=600, k_max=500)


def test_uniform_k_is_the_row_maximum(ops):
    """pkv_uniform_k: max over all rows, broadcast, plus the attention's key count (the reference reads
    adaptive_k.max().item() on the host, polar_cache_atten_value_indices_adaptive_k.py:1585)."""
    g = torch.Generator().manual_seed(2)
    for shape in ((1, 1), (2, 3), (8, 8), (40, 64)):   # up to 2560 rows: more than one pass of the 1024 threads
        ak = torch.randint(1, 5000, shape, generator=g).to(DEV)
        uk, rk = ops.uniform_k(ak, row_keys_base=77)
        assert uk.shape == ak.shape and (uk == ak.max()).all()
        assert rk.dtype == torch.int32 and (rk == int(ak.max()) + 77).all()
        assert torch.equal(ops.uniform_k(ak), uk)


@pytest.mark.parametrize("engine", ["kernel", "dma", "dma-one-command"])
def test_offload_rows_equals_sliced_copy(ops, engine):
    """pkv_offload_rows / pkv_offload_rows_dma against the sliced copy_ it replaces (reference polar_cache.py:457-471, :778-799): rows read in
    place from the model's [bs,seq,h,d] layout and from a partly filled staging buffer, into a batch slice of the pinned
    store; rows outside the written window stay untouched."""
    kw = {"kernel": {}, "dma": {"dma": True}, "dma-one-command": {"dma": True, "dma_flags": ops.OFFLOAD_ONE_COMMAND}}[engine]
    g = torch.Generator().manual_seed(3)
    bs, H, cap, D = 3, 4, 50, 128
    kc = torch.randn(bs + 1, H, cap, D, generator=g).to(torch.bfloat16).pin_memory()
    vc = torch.randn(bs + 1, H, cap, D, generator=g).to(torch.bfloat16).pin_memory()
    want_k, want_v = kc.clone(), vc.clone()
    model_k = torch.randn(bs, 40, H, D, generator=g).to(torch.bfloat16).to(DEV)    # [bs, seq, h, d]
    model_v = torch.randn(bs, 40, H, D, generator=g).to(torch.bfloat16).to(DEV)
    src_k, src_v = model_k[:, 5:33].permute(0, 2, 1, 3), model_v[:, 5:33].permute(0, 2, 1, 3)
    ops.offload_rows(src_k, src_v, kc[1:], vc[1:], 7, **kw)
    want_k[1:, :, 7:35] = src_k.cpu()
    want_v[1:, :, 7:35] = src_v.cpu()
    stage_k = torch.randn(bs, H, 16, D, generator=g).to(torch.bfloat16).to(DEV)   # staging buffer, first 9 rows valid
    stage_v = torch.randn(bs, H, 16, D, generator=g).to(torch.bfloat16).to(DEV)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    ops.offload_rows(stage_k[:, :, :9], stage_v[:, :, :9], kc[:bs], vc[:bs], cap - 9, stream=side, **kw)
    want_k[:bs, :, cap - 9:] = stage_k[:, :, :9].cpu()
    want_v[:bs, :, cap - 9:] = stage_v[:, :, :9].cpu()
    torch.cuda.synchronize()
    assert torch.equal(kc, want_k) and torch.equal(vc, want_v)
    with pytest.raises(RuntimeError, match="outside the host store"):
        ops.offload_rows(stage_k, stage_v, kc[:bs], vc[:bs], cap - 9, **kw)
    with pytest.raises(RuntimeError):
        ops.offload_rows(stage_k, stage_v, kc[:bs].clone(), vc[:bs], 0, **kw)   # not pinned


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n_sink,n_enc,n_tail", [(0, 1, 0), (4, 255, 3), (64, 256, 64), (65, 2049, 129), (70, 0, 0), (3, 4097, 1)])
def test_prefill_store_rows_index_and_norms(ops, dtype, n_sink, n_enc, n_tail):
    """pkv_prefill_store at and beside its workgroup sizes (256 encoded, 64 dense tokens): rows copied bit for bit to
    their places and nowhere else, the index equal to pkv_encode_append's on the same keys, value norms equal to a
    restatement of their summation order."""
    bs, H, S = 2, 3, n_sink + n_enc + n_tail
    _say(f"prefill_store {dtype} {n_sink}+{n_enc}+{n_tail}")
    gen = torch.Generator().manual_seed(S)
    k = torch.randn(bs, S, H, 128, generator=gen).to(dtype).to(DEV)
    v = torch.randn(bs, S, H, 128, generator=gen).to(dtype).to(DEV)
    kp, vp = k.permute(0, 2, 1, 3), v.permute(0, 2, 1, 3)
    signs = ops.srht_signs(DEV)
    gap, cap = 2, n_enc + 5                                # rows between the sink and the tail, spare rows behind
    tail0 = n_sink + gap
    dk = torch.full((bs, H, tail0 + n_tail + 3, 128), 7.0, dtype=dtype, device=DEV)
    zk = torch.full((bs, H, cap, 128), 7.0, dtype=dtype, device=DEV)
    dv, zv = dk.clone(), zk.clone()
    dn = torch.full(dk.shape[:3], 7.0, device=DEV)
    zn2 = torch.full((bs, H, cap), 7.0, device=DEV)
    codes, nib, w, cb, k4, kw = ops.alloc_keymajor(bs, H, cap, DEV)
    zn = ops.record_value_norm_view(nib)
    cc = torch.ones(bs, H, 16, 256, dtype=torch.int32, device=DEV)
    sl = slice(0, n_enc)
    ops.prefill_store(kp, vp, n_sink, n_enc, signs, (dk, dv), tail0, (zk, zv),
                      (cb[..., sl], k4[:, :, :, sl], kw[..., sl], cc) if n_enc else None, dense_vnorm=dn,
                      zone_vnorm=zn[..., sl], zone_vnorm2=zn2)
    quads = vp.float().cpu().contiguous().view(bs, H, S, 32, 4) ** 2
    norm = ((quads[..., 0] + quads[..., 1]) + quads[..., 2]) + quads[..., 3]
    while norm.shape[-1] > 1:
        norm = norm[..., 0::2] + norm[..., 1::2]
    norm = torch.from_numpy(np.sqrt(norm[..., 0].numpy())).to(dtype).float().to(DEV)   # correctly rounded, as torch's CPU root is not
    for src, dense, zone in ((kp, dk, zk), (vp, dv, zv)):
        want_d, want_z = torch.full_like(dense, 7.0), torch.full_like(zone, 7.0)
        want_d[:, :, :n_sink], want_d[:, :, tail0:tail0 + n_tail] = src[:, :, :n_sink], src[:, :, n_sink + n_enc:]
        want_z[:, :, :n_enc] = src[:, :, n_sink:n_sink + n_enc]
        assert torch.equal(dense, want_d) and torch.equal(zone, want_z)
    want = torch.full_like(dn, 7.0)
    want[:, :, :n_sink], want[:, :, tail0:tail0 + n_tail] = norm[:, :, :n_sink], norm[:, :, n_sink + n_enc:]
    assert torch.equal(dn, want)
    if n_enc:
        codes2, nib2, w2, cb2, k42, kw2 = ops.alloc_keymajor(bs, H, cap, DEV)
        cc2 = torch.ones_like(cc)
        ops.encode_append(kp[:, :, n_sink:n_sink + n_enc], signs, cb2[..., sl], k42[:, :, :, sl], kw2[..., sl], cc2)
        assert torch.equal(codes, codes2) and torch.equal(nib, nib2) and torch.equal(w.view(torch.int16), w2.view(torch.int16))
        assert torch.equal(cc, cc2)
        assert torch.equal(zn[..., sl], norm[:, :, n_sink:n_sink + n_enc]) and torch.equal(zn2[..., sl], norm[:, :, n_sink:n_sink + n_enc])
        assert torch.all(zn[..., n_enc:] == 0) and torch.all(zn2[..., n_enc:] == 7.0)


@pytest.mark.parametrize("same_tensor", [True, False])
@pytest.mark.parametrize("lens,indexed", [((1,), ()), ((1, 31, 1), (1,)), ((5, 64, 33), (1,)), ((127, 130), (0,)), ((63, 1, 64, 3), (3,)),
                                          ((20, 40, 17), (0, 2)), ((9000,), ()), ((40, 8300), (1,))])
def test_decode_attention_places_of_keys(ops, same_tensor, lens, indexed):
    """Segments of one K/V tensor (places as 32-bit offsets), of several tensors, with no, one and two indexed segments, at the
    edges of waves and splits: against attention over the same rows in 64 bits."""
    bs, H, group = 2, 3, 5
    g = torch.Generator(device=DEV).manual_seed(sum(lens) + 2 * len(indexed) + same_tensor)
    rows = max(lens) + 50
    pool = [[torch.randn(bs, H, rows, 128, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2)] for _ in lens]
    q = torch.randn(bs, 1, H * group, 128, generator=g, device=DEV).to(torch.bfloat16)
    segs, K, V = [], [], []
    for i, n in enumerate(lens):
        k, v = pool[0 if same_tensor else i]
        row0 = 7 + 3 * i
        if i in indexed:
            idx = torch.randint(0, rows - row0, (bs, H, n + 2), generator=g, device=DEV)
            segs.append((k, v, row0, n, idx))
            at = (idx[:, :, :n] + row0)[..., None].expand(-1, -1, -1, 128)
            K.append(k.gather(2, at)), V.append(v.gather(2, at))
        else:
            segs.append((k, v, row0, n))
            K.append(k[:, :, row0:row0 + n]), V.append(v[:, :, row0:row0 + n])
    out = ops.DecodeAttention(bs, H, group, sum(lens), DEV).run(q, segs)
    K, V = torch.cat(K, dim=2).double(), torch.cat(V, dim=2).double()
    p = torch.softmax(q.double().view(bs, H, group, 128) @ K.transpose(2, 3).contiguous() / math.sqrt(128), dim=-1)
    ref = (p @ V).view(bs, 1, H * group, 128)
    # probabilities and the result are rounded to bf16 (2^-9 relative each); values up to ~4.5
    assert (out.double() - ref).abs().max().item() < 2e-2


@pytest.mark.parametrize("same_tensor", [True, False])
@pytest.mark.parametrize("lens,indexed", [((1,), ()), ((1, 31, 1), (1,)), ((5, 64, 33), (1,)), ((63, 1, 64, 3), (3,)), ((20, 40, 17), (0, 2)),
                                          ((9000,), ()), ((40, 8300), (1,))])
def test_decode_attention_fp32_places_of_keys(ops, same_tensor, lens, indexed):
    """The same for fp32 rows, whose places are found for 64 keys of a workgroup at a time."""
    bs, H, group = 2, 3, 5
    g = torch.Generator(device=DEV).manual_seed(sum(lens) + 2 * len(indexed) + same_tensor)
    rows = max(lens) + 50
    pool = [[torch.randn(bs, H, rows, 128, generator=g, device=DEV) for _ in range(2)] for _ in lens]
    q = torch.randn(bs, 1, H * group, 128, generator=g, device=DEV)
    segs, K, V = [], [], []
    for i, n in enumerate(lens):
        k, v = pool[0 if same_tensor else i]
        row0 = 7 + 3 * i
        if i in indexed:
            idx = torch.randint(0, rows - row0, (bs, H, n + 2), generator=g, device=DEV)
            segs.append((k, v, row0, n, idx))
            at = (idx[:, :, :n] + row0)[..., None].expand(-1, -1, -1, 128)
            K.append(k.gather(2, at)), V.append(v.gather(2, at))
        else:
            segs.append((k, v, row0, n))
            K.append(k[:, :, row0:row0 + n]), V.append(v[:, :, row0:row0 + n])
    out = ops.DecodeAttention(bs, H, group, sum(lens), DEV).run(q, segs)
    K, V = torch.cat(K, dim=2).double(), torch.cat(V, dim=2).double()
    p = torch.softmax(q.double().view(bs, H, group, 128) @ K.transpose(2, 3).contiguous() / math.sqrt(128), dim=-1)
    ref = (p @ V).view(bs, 1, H * group, 128)
    # a score's 128 products and a result's weighted mean, each rounded at 2^-24: a few 1e-6 of values up to ~4.5
    assert (out.double() - ref).abs().max().item() < 2e-5


@pytest.mark.parametrize("rows,n,k", [(1, 300, 150), (8, 3520, 1760), (8, 6000, 3), (8, 32000, 3200), (16, 20001, 4001),
                                      (64, 40000, 4000), (32, 70001, 7000)])
def test_select_rerank_at_every_chunk_size(ops, rows, n, k):
    """Candidates and scores of the fused select + rerank for chunks of 256, 1024, 2048 and 4096 keys (one to sixteen counts per
    thread), with a ragged last chunk: the candidate list is the stand-alone select's, the scores the stand-alone rerank's."""
    bs, H, G = (rows // 8, 8, 2) if rows >= 8 else (1, rows, 2)
    g = torch.Generator(device=DEV).manual_seed(n + k)
    keys = torch.randn(bs, H, n, 128, generator=g, device=DEV).to(torch.bfloat16)
    signs, centers = ops.srht_signs(DEV), ops.mag_centers(DEV)
    codes_km, nib_km, w_km, cb, k4, kw = ops.alloc_keymajor(bs, H, n, DEV)
    cc = torch.zeros(bs, H, 16, 256, dtype=torch.int32, device=DEV)
    ops.encode_append(keys, signs, cb, k4, kw, cc)
    q = torch.randn(bs, 1, H * G, 128, generator=g, device=DEV).to(torch.bfloat16)
    tiers = [int(math.ceil(n * 0.3 * r)) for r in ops.TIER_RATIOS]
    plan = ops.RetrievePlan(bs, H, G, n, DEV, n, k, 1)
    cand, scores = plan.run_candidates(q, signs, centers, cc, codes_km, nib_km, w_km, 0, n, tiers, k)
    qhat, qnorm, lut, _ = ops.query_prep_lut(q, H, signs, cc, tiers)
    cnt = ops.collision_scan(cb, lut)
    cnt = cnt[0] if isinstance(cnt, tuple) else cnt
    want = ops.bucket_topk(cnt.view(bs * H, n), k).view(bs, H, k)
    assert torch.equal(cand.view(bs, H, k), want)
    ref = ops.rerank4(want, k4, kw, qhat.view(bs, H, 16, 8), qnorm.view(bs, H, 1), centers)
    ref = ref[0] if isinstance(ref, tuple) else ref
    assert torch.equal(scores.view(bs, H, k), ref.view(bs, H, k))


@pytest.mark.parametrize("N", [1, 7, 1027, 5000])
def test_scan_counts_of_any_table(ops, N):
    """Votes of a table with any entries (the retrieval's hold at most 127 in all): int32 counts are the sums, byte counts
    their low eight bits, in every code layout."""
    bs, H = 1, 3
    g = torch.Generator(device=DEV).manual_seed(N)
    lut = torch.randint(0, 256, (bs, H, 16, 256), generator=g, device=DEV).to(torch.uint8)
    code = torch.randint(0, 256, (bs, H, 16, N), generator=g, device=DEV).to(torch.uint8)
    want = lut.int().gather(3, code.long()).sum(dim=2)
    for layout in (code, code.permute(0, 1, 3, 2).contiguous().permute(0, 1, 3, 2)):   # subspace-major, key-major
        assert torch.equal(ops.collision_scan(layout, lut, torch.int32)[0], want.int())
        assert torch.equal(ops.collision_scan(layout, lut, torch.uint8)[0], (want & 255).to(torch.uint8))


def test_prefill_store_beyond_2_to_the_23_tokens(ops):
    """One head with more than 2^23 tokens: all rows in their places, the index of the last keys equal to pkv_encode_append's,
    every key counted once."""
    n_sink, n_tail, last = 5, 70, 1000
    n = (1 << 23) + 301
    S = n_sink + n + n_tail
    g = torch.Generator(device=DEV).manual_seed(8)
    k, v = (torch.randn(1, 1, S, 128, generator=g, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    signs = ops.srht_signs(DEV)
    dk, zk = torch.zeros(1, 1, n_sink + n_tail, 128, dtype=k.dtype, device=DEV), torch.zeros(1, 1, n, 128, dtype=k.dtype, device=DEV)
    dv, zv = torch.zeros_like(dk), torch.zeros_like(zk)
    codes, nib, w, cb, k4, kw = ops.alloc_keymajor(1, 1, n, DEV)
    cc = torch.zeros(1, 1, 16, 256, dtype=torch.int32, device=DEV)
    ops.prefill_store(k, v, n_sink, n, signs, (dk, dv), n_sink, (zk, zv), (cb, k4, kw, cc))
    for src, dense, zone in ((k, dk, zk), (v, dv, zv)):
        assert torch.equal(zone, src[:, :, n_sink:n_sink + n])
        assert torch.equal(dense, torch.cat([src[:, :, :n_sink], src[:, :, n_sink + n:]], dim=2))
    assert torch.all(cc.sum(dim=3) == n)
    codes2, nib2, w2, cb2, k42, kw2 = ops.alloc_keymajor(1, 1, last, DEV)
    ops.encode_append(k[:, :, n_sink + n - last:n_sink + n], signs, cb2, k42, kw2, torch.zeros_like(cc))
    assert torch.equal(codes[:, :, -last:], codes2) and torch.equal(nib[:, :, -last:], nib2)
    assert torch.equal(w[:, :, -last:].view(torch.int16), w2.view(torch.int16))


def test_bound_append_refuses_a_slot_behind_the_norms(ops):
    """The kept append refuses what append_kv refuses: a slot that the K/V rows have and the value norms have not."""
    dk, dv = (torch.zeros(1, 2, 8, 128, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    k, v = (torch.ones(1, 1, 2, 128, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    vn = torch.zeros(1, 2, 5, device=DEV)
    bound = ops.BoundAppend(dk, dv, vnorm=vn)
    bound.launch(k, v, 4)
    assert torch.equal(vn[:, :, 4], torch.full((1, 2), float(torch.tensor(128.0).sqrt().to(torch.bfloat16)), device=DEV))
    for slot in (5, 7, 8, -1):
        with pytest.raises(RuntimeError):
            bound.launch(k, v, slot)
    bound = ops.BoundAppend(dk, dv)
    bound.launch(k, v, 7)
    for slot in (8, -1):
        with pytest.raises(RuntimeError):
            bound.launch(k, v, slot)
    torch.cuda.synchronize()
    assert torch.all(dk[:, :, [4, 7]] == 1) and torch.all(dk[:, :, [0, 1, 2, 3, 5, 6]] == 0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("layout", ["subspace", "packed", "records"])
@pytest.mark.parametrize("norms", [False, True])
@pytest.mark.parametrize("n_enc", [1, 255, 257, 1033])
def test_prefill_store_index_layouts(ops, dtype, layout, norms, n_enc):
    """The index layouts that pkv_prefill_store takes beside whole key records with their norms: subspace-major and packed
    tensors with norms in a tensor of their own (or none), records with none or with norms elsewhere.  Index, rows and norms
    equal pkv_encode_append's and the records form's; what lies behind the encoded keys stays as it was."""
    bs, H, n_sink, n_tail, cap = 2, 3, 3, 66, n_enc + 5
    _say(f"prefill_store {dtype} {layout} norms={norms} {n_enc}")
    gen = torch.Generator().manual_seed(n_enc)
    k, v = (torch.randn(bs, n_sink + n_enc + n_tail, H, 128, generator=gen).to(dtype).to(DEV).permute(0, 2, 1, 3) for _ in range(2))
    signs = ops.srht_signs(DEV)

    def index(form):
        if form == "records":
            _, nib, w, cb, k4, kw = ops.alloc_keymajor(bs, H, cap, DEV)
            return cb, k4, kw
        if form == "subspace":
            return (torch.zeros(bs, H, 16, cap, dtype=torch.uint8, device=DEV), torch.zeros(bs, H, 16, cap, 4, dtype=torch.uint8, device=DEV),
                    torch.zeros(bs, H, 16, cap, dtype=torch.bfloat16, device=DEV))
        return (torch.zeros(bs, H, cap, 16, dtype=torch.uint8, device=DEV).permute(0, 1, 3, 2),
                torch.zeros(bs, H, cap, 16, 4, dtype=torch.uint8, device=DEV).permute(0, 1, 3, 2, 4),
                torch.zeros(bs, H, cap, 16, dtype=torch.bfloat16, device=DEV).permute(0, 1, 3, 2))

    def store(form, **kw_norms):
        cb, k4, kw = index(form)
        cc = torch.ones(bs, H, 16, 256, dtype=torch.int32, device=DEV)
        dk, zk = (torch.full((bs, H, n, 128), 7.0, dtype=dtype, device=DEV) for n in (n_sink + n_tail + 2, cap))
        dv, zv = dk.clone(), zk.clone()
        ops.prefill_store(k, v, n_sink, n_enc, signs, (dk, dv), n_sink, (zk, zv),
                          (cb[..., :n_enc], k4[:, :, :, :n_enc], kw[..., :n_enc], cc), **kw_norms)
        return cb, k4, kw.contiguous().view(torch.int16), cc, dk, dv, zk, zv

    # the form the caches use, for rows and norms
    _, nib, _, cb, k4, kw = ops.alloc_keymajor(bs, H, cap, DEV)
    want_n = ops.record_value_norm_view(nib)
    dn = torch.zeros(bs, H, n_sink + n_tail, device=DEV)
    rows = [torch.full((bs, H, n, 128), 7.0, dtype=dtype, device=DEV) for n in (n_sink + n_tail + 2, cap) for _ in range(2)]
    ops.prefill_store(k, v, n_sink, n_enc, signs, rows[:2], n_sink, rows[2:],
                      (cb[..., :n_enc], k4[:, :, :, :n_enc], kw[..., :n_enc], torch.zeros(bs, H, 16, 256, dtype=torch.int32, device=DEV)),
                      dense_vnorm=dn, zone_vnorm=want_n[..., :n_enc])
    cb2, k42, kw2 = index(layout)
    cc2 = torch.ones(bs, H, 16, 256, dtype=torch.int32, device=DEV)
    ops.encode_append(k[:, :, n_sink:n_sink + n_enc], signs, cb2[..., :n_enc], k42[:, :, :, :n_enc], kw2[..., :n_enc], cc2)
    extra, zn = {}, torch.full((bs, H, cap, 3), 7.0, device=DEV)   # every third word: any key stride
    if norms:
        extra = dict(zone_vnorm=zn[:, :, :n_enc, 1])
    got = store(layout, **extra)
    for a, b in zip(got, (cb2, k42, kw2.contiguous().view(torch.int16), cc2, *rows)):
        assert torch.equal(a, b)
    want = torch.full_like(zn, 7.0)
    if norms:
        want[:, :, :n_enc, 1] = want_n[..., :n_enc]
    assert torch.equal(zn, want)


@pytest.mark.parametrize("group,k,sink,tail,keys,cand", [(*c, 3000, 1500) for c in (
    (4, 100, 64, 529), (1, 1, 0, 1), (3, 15, 3, 0), (5, 16, 64, 64), (8, 17, 64, 1100), (2, 33, 95, 30), (6, 256, 1, 130), (4, 256, 64, 700),
    (7, 257, 0, 0), (4, 512, 64, 700), (8, 100, 64, 1300), (6, 1024, 64, 1300), (4, 64, 31, 1), (2, 31, 129, 65), (4, 192, 64, 700), (8, 162, 33, 0))] + [
    (4, 100, 64, 529, 20000, 8193), (3, 129, 31, 65, 20000, 9001), (2, 200, 64, 1, 20000, 9001), (4, 192, 64, 529, 20000, 9001)])
def test_decode_step_in_place_attends_in_two_parts(ops, group, k, sink, tail, keys, cand):
    """The step whose attention reads selected rows where they lie: the other rows beside the query side, selected rows in the
    top-k's workgroups.  The same ids and the same sums, bit for bit, as the top-k and the attention called one by one; and the
    attention against 64 bits: probabilities and output are rounded to 8 bits, 2^-9 of the largest value each."""
    _say(f"two-part attention group {group} k {k} sink {sink} tail {tail} candidates {cand} of {keys}")
    w = W.make_workload("two_parts", 2, 2, group, keys, cand, k, O.BF16, 0.5, seed0=11, with_values=False)
    d = W.to_device(w, DEV, torch)
    g = torch.Generator(device=DEV).manual_seed(5)
    rows = sink + w.N + tail
    kk, vv = (torch.randn(w.bs, w.H, rows, 128, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
    plan = ops.RetrievePlan(w.bs, w.H, w.G, w.N, DEV, w.N, w.C, w.K)
    att = ops.DecodeAttention(w.bs, w.H, w.G, rows, DEV)
    args = (d["queries"], d["signs"], d["centers"], d["cluster_counts"], d["codes_km"], d["nib_km"], d["w_km"], 0, w.N, w.tiers, w.C, w.K)
    want_ids = plan.run(*args, any_order=True)  # more than 8192 candidates come out sorted all the same
    ids = torch.zeros_like(want_ids)
    segs = [s for s in [(kk, vv, 0, sink), (kk, vv, sink, k, ids), (kk, vv, sink + w.N, tail)] if s[3]]
    blocks = (sink + k - 1) // 32 - sink // 32 + 1
    assert _step_form(ops, plan, att, d["queries"], args, segs) == (
        1 if blocks <= 6 and sink + k + tail <= 11 * 128 else 2 if cand <= 8192 else 0)
    plan.run(*args, out_ids=ids, attention=(att, segs, None), any_order=True)
    torch.cuda.synchronize()
    got = plan.attn_out.clone()
    assert torch.equal(ids, want_ids)
    assert torch.equal(got, att.run(d["queries"], segs))
    want = _near_attention_in_64_bits(got, d["queries"], kk, vv, sink, w.N, ids)
    err = (got.view(w.bs, w.H, group, 128).double() - want).abs().max().item()
    assert err <= vv.abs().max().item() * 2.0 ** -8, err


def _step_form(ops, plan, att, q, args, segs):
    """How pkv_decode_step takes plan.run(*args, out_ids=segs' ids, attention=(att, segs, None), any_order=True)."""
    import ctypes

    ids = next(s[4] for s in segs if len(s) > 4)
    a = plan._fill(*args, ids, None, None, False, any_order=True)
    aa, out = att.c_args(q, segs)
    return ops._lib.lib().pkv_decode_step_form(ctypes.byref(a), plan.ws.data_ptr(), ctypes.byref(aa))


def _near_attention_in_64_bits(got, queries, kk, vv, sink, n, ids):
    """The attention over rows 0 .. sink, sink + ids and sink + n .. in 64 bits, close to `got`: probabilities are rounded to bf16
    before they meet the values and the output is, 2^-8 relative each; scores and sums are fp32 (1e-5)."""
    bs, H, rows, _ = kk.shape
    group = queries.numel() // (bs * H * 128)
    sel = torch.cat([torch.arange(sink, device=DEV).expand(bs, H, -1), sink + ids,
                     torch.arange(sink + n, rows, device=DEV).expand(bs, H, -1)], dim=2)[..., None].expand(-1, -1, -1, 128)
    ks, vs = (t.gather(2, sel).double() for t in (kk, vv))
    p = torch.softmax(queries.view(bs, H, group, 128).double() @ ks.transpose(2, 3).contiguous() / 128 ** 0.5, dim=-1)
    want, weight = p @ vs, p @ vs.abs()
    err = (got.view(bs, H, group, 128).double() - want).abs()
    assert (err <= (weight + want.abs()) * 2.0 ** -8 + 1e-5 * weight).all(), (err / weight).max().item()
    return want


@pytest.mark.parametrize("bs,H,group,k,sink,tail,keys,cand,form", [
    # candidates per thread: 2, 4, 8; one workgroup a row and several
    (2, 2, 4, 100, 64, 529, 5000, 3000, 1), (2, 2, 4, 100, 64, 529, 9000, 8192, 1), (2, 2, 4, 512, 64, 529, 5000, 4096, 2),
    (2, 2, 8, 1024, 64, 529, 9000, 8192, 2), (1, 3, 5, 300, 1, 40, 9000, 5001, 2),
    # two and three splits to a workgroup, the last workgroup's not all there
    (8, 8, 4, 512, 64, 300, 3000, 1500, 2), (8, 8, 4, 1024, 64, 300, 5000, 2500, 2), (9, 8, 4, 800, 64, 300, 5000, 2500, 2),
    (9, 8, 3, 800, 50, 0, 9000, 8000, 2), (64, 4, 8, 512, 64, 129, 3000, 1500, 2), (40, 4, 1, 1024, 64, 1, 5000, 4096, 2),
    # six to eight blocks by one workgroup a row: over two splits, over three, with a split that is selected whole
    (16, 8, 4, 200, 64, 300, 3000, 1500, 1), (16, 8, 4, 250, 64, 300, 5000, 3000, 1), (17, 8, 4, 225, 127, 300, 3000, 1500, 1),
    (17, 8, 8, 256, 0, 70, 3000, 1500, 1), (16, 8, 2, 230, 40, 900, 9000, 8192, 1), (16, 8, 4, 225, 127, 529, 20000, 9001, 1),
    # refused: a second round of workgroups that select again
    (12, 8, 4, 1024, 64, 300, 5000, 2500, 0)])
def test_decode_step_in_two_parts_by_number_of_rows(ops, bs, H, group, k, sink, tail, keys, cand, form):
    """The forms that depend on the rows and the candidates: as the top-k and the attention called one by one, bit for bit."""
    _say(f"two-part attention {bs}x{H} rows group {group} k {k} sink {sink} tail {tail} candidates {cand} of {keys}")
    _two_parts(ops, bs, H, group, k, sink, tail, keys, cand, form)


@pytest.mark.parametrize("scores", ["equal", "few", "infinite"])
@pytest.mark.parametrize("bs,k,keys,cand,form", [(2, 100, 3000, 1500, 1), (2, 512, 5000, 3000, 2), (32, 512, 5000, 5000 - 1, 2),
                                                 (2, 100, 20000, 9001, 1)])
def test_decode_step_in_two_parts_where_scores_tie(ops, scores, bs, k, keys, cand, form):
    """Selections that no bins of the scores' range separate (all scores equal, a few values, infinite ones): the ids that the
    attention goes on with are those of the top-k."""
    _say(f"two-part attention, scores {scores}, {bs * 2} rows k {k} candidates {cand} of {keys}")
    _two_parts(ops, bs, 2, 4, k, 64, 100, keys, cand, form, scores)


@pytest.mark.parametrize("k,keys,cand,form", [(100, 4000, 1500, 1), (512, 5000, 3000, 2), (100, 20000, 9001, 1)])
def test_decode_step_in_two_parts_replays_from_a_captured_graph(ops, k, keys, cand, form):
    """Captured once, replayed with other queries and eager work in between: each replay as the eager step."""
    _say(f"two-part attention captured, k {k} candidates {cand} of {keys}")
    _two_parts(ops, 2, 2, 4, k, 64, 100, keys, cand, form, replays=4)


def _two_parts(ops, bs, H, group, k, sink, tail, keys, cand, form, scores=None, replays=0):
    g = torch.Generator(device=DEV).manual_seed(7)
    rows = sink + keys + tail
    kk, vv = (torch.randn(bs, H, rows, 128, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
    zone = kk[:, :, sink:sink + keys]
    if scores in ("equal", "few"):  # one key, or four, again and again in the index (the attended rows stay apart)
        zone = zone[:, :, :1 if scores == "equal" else 4].repeat(1, 1, keys, 1)[:, :, :keys].contiguous()
    signs, centers = torch.from_numpy(O.srht_signs(42)).to(DEV), torch.from_numpy(O.mag_constants()[1]).to(DEV)
    codes, nib, wt, cb, k4, kw = ops.alloc_keymajor(bs, H, keys, DEV)
    cc = torch.zeros(bs, H, 16, 256, dtype=torch.int32, device=DEV)
    ops.encode_append(zone, signs, cb, k4, kw, cc)
    if scores == "infinite":
        wt[:, :, ::7] = float("inf")
    q = torch.randn(bs, 1, H * group, 128, generator=g, device=DEV).to(torch.bfloat16)
    plan = ops.RetrievePlan(bs, H, group, keys, DEV, keys, cand, k)
    att = ops.DecodeAttention(bs, H, group, rows, DEV)
    args = (q, signs, centers, cc, codes, nib, wt, 0, keys, O.tier_counts(keys, 0.5), cand, k)
    want_ids = plan.run(*args, any_order=True)
    ids = torch.zeros_like(want_ids)
    segs = [s for s in [(kk, vv, 0, sink), (kk, vv, sink, k, ids), (kk, vv, sink + keys, tail)] if s[3]]
    assert _step_form(ops, plan, att, q, args, segs) == form
    plan.run(*args, out_ids=ids, attention=(att, segs, None), any_order=True)
    torch.cuda.synchronize()
    got = plan.attn_out.clone()
    assert torch.equal(ids, want_ids)
    assert (ids.sort(dim=2).values.diff(dim=2) > 0).all() and int(ids.min()) >= 0 and int(ids.max()) < keys
    assert torch.equal(got, att.run(q, segs))
    _near_attention_in_64_bits(got, q, kk, vv, sink, keys, ids)
    if not replays:
        return
    out = torch.zeros_like(q)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        plan.run(*args, out_ids=ids, attention=(att, segs, out), any_order=True)
    for _ in range(replays):
        q.copy_(torch.randn(q.shape, generator=g, device=DEV))
        ids.zero_(), out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        got_ids, got = ids.clone(), out.clone()
        torch.randn(1 << 20, device=DEV).sum().item()  # unrelated eager work between replays
        assert torch.equal(got_ids, plan.run(*args, any_order=True))
        assert torch.equal(got, att.run(q, segs))


@pytest.mark.parametrize("k,keys,cand", [(100, 3000, 1500), (512, 3000, 1500), (100, 20000, 9001)])
def test_decode_step_with_one_scratch_buffer(ops, k, keys, cand):
    """Retrieval and attention with the same scratch memory, and with the output over the queries: as with buffers of their own."""
    _say(f"decode step in one scratch buffer, k {k} candidates {cand} of {keys}")
    w = W.make_workload("one_scratch", 2, 2, 4, keys, cand, k, O.BF16, 0.5, seed0=12, with_values=False)
    d = W.to_device(w, DEV, torch)
    g = torch.Generator(device=DEV).manual_seed(6)
    rows = 64 + w.N + 529
    kk, vv = (torch.randn(w.bs, w.H, rows, 128, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
    plan = ops.RetrievePlan(w.bs, w.H, w.G, w.N, DEV, w.N, w.C, w.K)
    att = ops.DecodeAttention(w.bs, w.H, w.G, rows, DEV)

    def step(q, out=None):
        ids = torch.zeros(w.bs, w.H, k, dtype=torch.int64, device=DEV)
        segs = [(kk, vv, 0, 64), (kk, vv, 64, k, ids), (kk, vv, 64 + w.N, 529)]
        plan.run(q, d["signs"], d["centers"], d["cluster_counts"], d["codes_km"], d["nib_km"], d["w_km"], 0, w.N, w.tiers, w.C, w.K,
                 out_ids=ids, attention=(att, segs, out), any_order=True)
        torch.cuda.synchronize()
        return ids, plan.attn_out.clone()

    want_ids, want = step(d["queries"])
    q = d["queries"].clone()
    ids, got = step(q, q)
    assert torch.equal(ids, want_ids) and torch.equal(got, want)
    plan.ws = att.ws = torch.empty(plan.ws.numel() + att.ws.numel(), dtype=torch.uint8, device=DEV)
    for _ in range(3):
        ids, got = step(d["queries"])
        assert torch.equal(ids, want_ids) and torch.equal(got, want)


@pytest.mark.parametrize("rows,L,k", [(3, 8193, 1), (2, 8193, 2048), (2, 16384, 2048), (2, 16385, 100), (2, 24577, 1025), (2, 32767, 1024),
                                      (2, 32768, 2048), (2, 32769, 100), (300, 9000, 64)])
@pytest.mark.parametrize("kind", ["spread", "ties", "few values", "crowded bin", "constant", "infinite", "nan", "lowest"])
def test_topk_f32_of_long_rows(ops, rows, L, k, kind):
    """Rows of 8193 to 32768 scores, which one workgroup selects from: both ends of its two forms, a last thread without all its keys,
    and scores that the bins of their range do not separate.  Ids and scores exactly as the oracle's, ties by id."""
    _say(f"topk_f32 long {rows}x{L} k={k} {kind}")
    rng = np.random.default_rng(L + k)
    x = (rng.standard_normal((rows, L)) * 10 + 3).astype(np.float32)
    if kind == "ties":
        x = np.round(x * 8).astype(np.float32) / 8
    elif kind == "few values":
        x = rng.integers(0, 4, (rows, L)).astype(np.float32)
    elif kind == "crowded bin":
        x[:, 50:50 + 400] = np.float32(90.0)
        x[:, 9:L:3] = np.float32(12.0)
    elif kind == "constant":
        x[:] = np.float32(-2.5)
    elif kind == "infinite":
        x[:, ::1000], x[0, 7] = np.inf, -np.inf
    elif kind == "nan":
        x[:, 11::2000] = np.nan
    elif kind == "lowest":
        x[:, L // 2:] = np.finfo(np.float32).min
    some = sorted({0, rows // 2, rows - 1})
    ids = np.stack([rng.permutation(2 * L)[:L] for _ in range(rows)]).astype(np.int64)
    out, vals = ops.topk_f32(torch.from_numpy(x).to(DEV), k, torch.from_numpy(ids).to(DEV), want_values=True)
    pos = ops.topk_f32(torch.from_numpy(x).to(DEV), k)
    torch.cuda.synchronize()
    for r in some:
        ref_ids, ref_pos = O.topk_f32(x[r], ids[r], k)
        assert np.array_equal(out[r].cpu().numpy(), ref_ids)
        assert np.array_equal(vals[r].cpu().numpy().view(np.uint32), x[r][ref_pos].view(np.uint32))
        assert np.array_equal(pos[r].cpu().numpy(), O.topk_f32(x[r], None, k)[1])


@pytest.mark.parametrize("L,k", [(8193, 1), (8193, 2048), (16384, 256), (16385, 257), (26000, 1024), (32768, 2048)])
@pytest.mark.parametrize("kind", ["log-normal", "outlier", "two outliers", "lowest outlier", "half zero", "many infinite", "infinite only", "few finite",
                                  "nan of both signs", "tie 256", "tie 257", "tie taken whole", "equal ids", "neighbours"])
def test_topk_f32_of_long_rows_narrows_the_edge(ops, L, k, kind):
    """Scores that the bins of a long row's range leave together: binned again, by their bits and then by the ids of those that tie, up to
    the most keys that are ranked one by one (256) and beyond.  Ids and scores exactly as the oracle's."""
    _say(f"topk_f32 long, edge {L} k={k} {kind}")
    rng = np.random.default_rng(L * 31 + k)
    x = rng.standard_normal((2, L)).astype(np.float32)
    ids = np.stack([rng.permutation(2 * L)[:L] for _ in range(2)]).astype(np.int64)
    if kind == "log-normal":
        x = np.exp(4 * x)
    elif kind == "outlier":
        x[:, L // 3] = 1e30
    elif kind == "two outliers":
        x[:, L // 3], x[:, L - 1] = 1e30, 1e9
    elif kind == "lowest outlier":
        x[:, 5] = np.finfo(np.float32).min
    elif kind == "half zero":
        x = np.maximum(x, np.float32(0))
        x[:, ::3] = -0.0
    elif kind == "many infinite":
        x[0, ::5], x[1, ::7] = np.inf, -np.inf
    elif kind == "infinite only":
        x[0], x[1] = np.where(x[0] > 0, np.inf, -np.inf), np.inf
    elif kind == "few finite":
        x[:, 300:] = -np.inf
    elif kind == "nan of both signs":
        x[:, 3::40] = np.nan
        x.view(np.uint32)[:, 4::50] = 0xffc00001
        x[:, 6::60] = -np.inf
    elif kind.startswith("tie"):   # k - 1 scores above the tied ones, or (taken whole) as many above as leave all of them winners
        n = {"tie 256": 256, "tie 257": 257, "tie taken whole": 300}[kind]
        above = max(0, k - (n if n == 300 else 1))
        for r in range(2):
            order = rng.permutation(L)
            x[r] = -np.abs(x[r]) - 1
            x[r, order[:above]] = 100 + rng.random(above).astype(np.float32)
            x[r, order[above:above + n]] = 50
    elif kind == "equal ids":
        x[:] = np.where(x > 1, 2.0, 0.5)
        ids[:] = 7
    elif kind == "neighbours":   # one part in 2^23 apart, beside one far away
        x = (np.float32(1.0).view(np.uint32) + rng.integers(0, 900, (2, L)).astype(np.uint32)).view(np.float32)
        x[:, 0] = -1e5
    out, vals = ops.topk_f32(torch.from_numpy(x).to(DEV), k, torch.from_numpy(ids).to(DEV), want_values=True)
    pos = ops.topk_f32(torch.from_numpy(x).to(DEV), k)
    torch.cuda.synchronize()
    for r in range(2):
        ref_ids, ref_pos = O.topk_f32(x[r], ids[r], k)
        assert np.array_equal(out[r].cpu().numpy(), ref_ids)
        assert np.array_equal(vals[r].cpu().numpy().view(np.uint32), x[r][ref_pos].view(np.uint32))
        assert np.array_equal(pos[r].cpu().numpy(), O.topk_f32(x[r], None, k)[1])


def test_topk_f32_of_long_rows_with_infinities_is_no_cliff(ops):
    """A few infinities among the scores of a long row cost no more than three times a row without (1.9; a selection that reads scores and ids
    from memory in each of eight passes, 6.3).  The best of several replays of a graph."""
    _say("topk_f32 long, time of infinities")
    x = torch.randn(8, 32768, generator=torch.Generator(device=DEV).manual_seed(0), device=DEV)
    y, ids = x.clone(), torch.arange(32768, device=DEV).repeat(8, 1)
    y[:, ::1000] = float("inf")
    took = []
    for s in (x, y):
        ops.topk_f32(s, 100, ids)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(20):
                ops.topk_f32(s, 100, ids)
        graph.replay()
        best = float("inf")
        for _ in range(10):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            graph.replay()
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        took.append(best)
    assert took[1] <= 3 * took[0], took


@pytest.mark.parametrize("scores", [None, "equal", "infinite"])
@pytest.mark.parametrize("bs,group,k,keys,cand", [(2, 4, 100, 40000, 16384), (1, 8, 192, 40000, 16385), (2, 3, 1, 60000, 32768)])
def test_decode_step_merges_after_the_selection_from_a_long_row(ops, bs, group, k, keys, cand, scores):
    """The attention behind that selection, in the selecting workgroup: as top-k and attention called one by one, bit for bit."""
    _say(f"two-part attention behind a long row, {bs} x 2 rows group {group} k {k} candidates {cand} of {keys} scores {scores}")
    _two_parts(ops, bs, 2, group, k, 64, 300, keys, cand, 1, scores, replays=3 if scores is None else 0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind", ["spread", "ties", "one dim", "zero subspaces", "tiny"])
def test_query_prep_ranks_equal_and_zero_scores_by_id(ops, dtype, kind):
    """The ranking by pairs of antipodal centroids where scores tie, vanish or differ in sign alone: as the oracle's, ids and votes."""
    _say(f"query prep ranking {dtype} {kind}")
    bs, H, group = 2, 3, 4
    g = torch.Generator().manual_seed(5)
    q = torch.randn(bs, 1, H * group, 128, generator=g)
    if kind == "ties":
        q = torch.where(q > 0, 1.0, -1.0)
    elif kind == "one dim":
        q[..., 1:] = 0
    elif kind == "zero subspaces":   # the rotation undone: the rotated query has zeros in whole subspaces
        had = torch.ones(1, 1)
        for _ in range(7):
            had = torch.cat([torch.cat([had, had], 1), torch.cat([had, -had], 1)], 0)
        want = torch.zeros(128)
        want[:24] = torch.tensor([1.0, 2.0, -1.0, 0.5, 0.0, -2.0, 1.0, 1.0]).repeat(3)
        q = ((want @ had) * torch.from_numpy(O.srht_signs(42)) / 128).expand(bs, 1, H * group, 128).clone()
    elif kind == "tiny":
        q = q * 1e-20
    q = q.to(dtype)
    signs = torch.from_numpy(O.srht_signs(42))
    cc = torch.randint(0, 40, (bs, H, 16, 256), generator=g, dtype=torch.int32)
    tiers = [200, 400, 800, 1200, 2000, 3000]
    qhat, _, lut, ids = ops.query_prep_lut(q.to(DEV), H, signs.to(DEV), cc.to(DEV), tiers, want_sorted_ids=True)
    torch.cuda.synchronize()
    od = O.BF16 if dtype == torch.bfloat16 else O.F32
    for b in range(bs):
        for h in range(H):
            want_ids = O.rank_centroids(qhat[b, h].cpu().numpy(), od)
            assert np.array_equal(ids[b, h].cpu().numpy(), want_ids), (b, h)
            assert np.array_equal(lut[b, h].cpu().numpy(), O.tier_lut(want_ids, cc[b, h].numpy(), tiers)), (b, h)


@pytest.mark.parametrize("dtype,rows", [(torch.bfloat16, 8), (torch.float32, 5)])
@pytest.mark.parametrize("n_enc", [129, 300, 513])
@pytest.mark.parametrize("layout", ["records", "subspace"])
def test_prefill_store_of_many_keys(ops, dtype, rows, n_enc, layout):
    """A call that moves more than 576 MiB spreads a workgroup's keys over its head; rows, index, cluster sizes and norms are
    those of calls for a few samples each, which keep them together.  One run and a remainder of keys per head up to three
    workgroups of two runs."""
    es, cap = (2, n_enc + 3) if dtype == torch.bfloat16 else (4, n_enc + 3)
    bs = (576 << 20) // ((512 * es + 144) * rows * n_enc) + 1
    _say(f"prefill_store of many keys {dtype} bs={bs} heads={rows} {n_enc} {layout}")
    gen = torch.Generator(device=DEV).manual_seed(n_enc)
    k, v = (torch.randn(bs, 2 + n_enc + 1, rows, 128, generator=gen, device=DEV).to(dtype).permute(0, 2, 1, 3) for _ in range(2))
    signs = ops.srht_signs(DEV)

    def store(step):
        zk, zv = (torch.full((bs, rows, cap, 128), 7.0, dtype=dtype, device=DEV) for _ in range(2))
        dk, dv = (torch.full((bs, rows, 3, 128), 7.0, dtype=dtype, device=DEV) for _ in range(2))
        cc = torch.zeros(bs, rows, 16, 256, dtype=torch.int32, device=DEV)
        if layout == "records":
            _, nib, _, cb, k4, kw = ops.alloc_keymajor(bs, rows, cap, DEV)
            zn = ops.record_value_norm_view(nib)
        else:
            cb, k4 = (torch.zeros(bs, rows, 16, cap, *e, dtype=torch.uint8, device=DEV) for e in ((), (4,)))
            kw, zn = torch.zeros(bs, rows, 16, cap, dtype=torch.bfloat16, device=DEV), torch.zeros(bs, rows, cap, device=DEV)
        zn2 = torch.zeros(bs, rows, cap, device=DEV)
        for b in range(0, bs, step):
            s = slice(b, b + step)
            ops.prefill_store(k[s], v[s], 2, n_enc, signs, (dk[s], dv[s]), 2, (zk[s], zv[s]),
                              (cb[s, ..., :n_enc], k4[s, :, :, :n_enc], kw[s, ..., :n_enc], cc[s]),
                              zone_vnorm=zn[s, :, :n_enc], zone_vnorm2=zn2[s, :, :n_enc])
        return zk, zv, dk, dv, cc, cb, k4, kw.view(torch.int16), zn, zn2

    for a, b in zip(store(bs), store(bs // 3 + 1)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype,group", [(torch.bfloat16, 4), (torch.bfloat16, 8), (torch.bfloat16, 1), (torch.float32, 2), (torch.float32, 7)])
@pytest.mark.parametrize("n", [1, 127, 129, 2048, 2049, 6000])
def test_bound_attention_merges_in_its_own_launch(ops, dtype, group, n):
    """The kept dense attention (the last workgroup of a row merges, while the splits are few) and the two launches of
    DecodeAttention.run: the same bits, launch after launch and in a replayed graph, and the counters are zero again."""
    _say(f"bound attention {dtype} group={group} {n}")
    bs, H = 2, 3
    g = torch.Generator(device=DEV).manual_seed(n + group)
    k, v = (torch.randn(bs, H, n + 9, 128, generator=g, device=DEV).to(dtype) for _ in range(2))
    att = ops.DecodeAttention(bs, H, group, n + 9, DEV)
    qs = [torch.randn(bs, 1, H * group, 128, generator=g, device=DEV).to(dtype) for _ in range(3)]
    bound = ops.BoundAttention(att, qs[0], [(k, v, 2, n)])
    for q, m in zip(qs, (n, max(1, n - 60), n)):
        bound.segs[0].n_rows = m
        got = bound.launch(q)
        assert torch.equal(got, att.run(q, [(k, v, 2, m)]))
        assert not torch.any(att.arrivals)
    # counters that overlapping launches left behind (the call after them may be spoiled as well) are gone two calls later
    att.arrivals.fill_(1)
    for _ in range(2):
        bound.launch(qs[0])
    assert not torch.any(att.arrivals) or n > 2048 or dtype == torch.float32   # two launches there, which count nothing
    att.arrivals.zero_()
    assert torch.equal(bound.launch(qs[1]), att.run(qs[1], [(k, v, 2, n)]))
    graph, q = torch.cuda.CUDAGraph(), qs[0].clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        bound.launch(q)
    torch.cuda.current_stream().wait_stream(side)
    with torch.cuda.graph(graph):
        out = bound.launch(q)
    for other in qs:
        q.copy_(other)
        graph.replay()
        want = att.run(other, [(k, v, 2, n)])
        torch.cuda.synchronize()
        assert torch.equal(out, want) and not torch.any(att.arrivals)
    # nor does a graph, which would count in the same half for good, depend on what they hold
    att.arrivals.fill_(1)
    for other in qs:
        q.copy_(other)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, att.run(other, [(k, v, 2, n)])) and torch.all(att.arrivals == 1)


@pytest.mark.parametrize("rows,L", [(3, 1), (2, 3), (3, 64), (2, 4095), (2, 4096), (3, 4097), (1, 12287), (2, 20480), (5, 24573), (2, 24577),
                                    (64, 24577), (65, 28673), (64, 32768), (64, 32769)])
def test_bucket_topk_of_rows_of_every_length(ops, rows, L):
    """One workgroup a row up to 24576 values (32768 from 64 rows on) and two launches beyond: the oracle's indices, in order, for
    rows at any alignment, values outside [0, 127], few distinct values and every kind of k."""
    _say(f"bucket_topk rows={rows} L={L}")
    g = torch.Generator().manual_seed(rows * L)
    wide = torch.randint(-40, 200, (rows, L + 3), generator=g, dtype=torch.int32)
    for x in (wide[:, :L], torch.randint(3, 6, (rows, L), generator=g, dtype=torch.int32), torch.full((rows, L), 127, dtype=torch.int32)):
        clamped = x.clamp(0, 127).numpy()
        dev = wide.to(DEV)[:, 1:L + 1].copy_(x.to(DEV))   # rows an odd number of words apart, one word in
        for k in sorted({1, (L + 1) // 2, max(1, L - 1), max(1, L // 7)}):
            out = ops.bucket_topk(dev, k).cpu().numpy()
            for r in {0, rows - 1}:
                assert np.array_equal(out[r], np.arange(L) if k == L else O.select_candidates(clamped[r], k)[0])


@pytest.mark.parametrize("bs,H,N,n_tiers", [(1, 1, 1, 6), (1, 3, 5, 1), (2, 3, 1027, 6), (1, 5, 20011, 3), (1, 1, 1 << 20, 6), (1, 1, (1 << 20) + 3, 6)])
def test_votes_of_a_ranking_with_repeats_in_any_layout(ops, bs, H, N, n_tiers):
    """Subspace-major codes (one launch while rows x keys <= 2^20, each workgroup building the table) and key-major ones (the table
    first): the same votes from rankings that name a centroid twice, from slices of wider tensors."""
    _say(f"votes of a ranking {bs} x {H} x {N}, {n_tiers} tiers")
    g = torch.Generator(device=DEV).manual_seed(N)
    ids = torch.randint(0, 256, (bs, H + 1, 18, 256), generator=g, device=DEV)[:, 1:, 1:17]
    counts = torch.randint(0, N // 100 + 2, (bs, H, 17, 256), generator=g, device=DEV, dtype=torch.int32)[:, :, 1:]
    code = torch.randint(0, 256, (bs, H, 16, N + 2), generator=g, device=DEV).to(torch.uint8)[..., 1:N + 1]
    tiers = [max(1, N * (t + 1) // (2 * n_tiers)) for t in range(n_tiers)]
    got = ops.update_cache_cnt(ids, counts, code, tiers)
    want = ops.update_cache_cnt(ids, counts, code.permute(0, 1, 3, 2).contiguous().permute(0, 1, 3, 2), tiers)
    assert torch.equal(got, want)
    assert N < 100 or got.max() > 0   # the few keys of a short row may all have unranked codes


@pytest.mark.parametrize("group", [1, 4, 7, 8])
@pytest.mark.parametrize("n", [130, 700, 1280, 2048])
def test_bound_attention_of_infinite_values(ops, group, n):
    """The merge in the attention's own launch, 2 to 16 splits: an infinite value makes its dimension infinite, with its sign, and no
    other one, as the merge by a launch of its own has it, in whatever split it lies."""
    _say(f"bound attention, infinite values, group={group} {n}")
    bs, H = 1, 3
    g = torch.Generator(device=DEV).manual_seed(n)
    k, v = (torch.randn(bs, H, n, 128, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
    at = {3: (0, float("inf")), 40: (127, float("-inf")), 64: (128, float("inf")), 90: (n // 2, float("-inf")), 127: (n - 2, float("inf"))}
    for d, (key, x) in at.items():
        v[:, :, key, d] = x
    att = ops.DecodeAttention(bs, H, group, n, DEV)
    q = torch.randn(bs, 1, H * group, 128, generator=g, device=DEV).to(torch.bfloat16)
    got = ops.BoundAttention(att, q, [(k, v, 0, n)]).launch(q)
    for d in range(128):
        if d in at:
            assert (got[..., d] == at[d][1]).all(), d
        else:
            assert torch.isfinite(got[..., d]).all(), d
    assert torch.equal(got, att.run(q, [(k, v, 0, n)]))


@pytest.mark.parametrize("what", ["votes", "bucket"])
def test_captured_operators_take_their_faster_launches(ops, what):
    """Votes from a ranking and the bucket top-k of a row that one launch is as long as two for: replayed, the same results as eagerly, in
    the two launches that are faster where no host waits (one launch writes nothing into the table's workspace or the counts')."""
    from pariskv_amd import _lib

    _say(f"captured {what}")
    g = torch.Generator(device=DEV).manual_seed(3)
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    if what == "votes":
        bs, H, N = 2, 3, 3001
        ids = torch.randint(0, 256, (bs, H, 16, 256), generator=g, device=DEV)
        counts = torch.randint(0, 40, (bs, H, 16, 256), generator=g, device=DEV, dtype=torch.int32)
        code = torch.randint(0, 256, (bs, H, 16, N), generator=g, device=DEV).to(torch.uint8)
        ws, out = torch.zeros(bs * H * 4096, dtype=torch.uint8, device=DEV), torch.zeros(bs, H, N, dtype=torch.int32, device=DEV)
        tiers, nt = ops._tiers([300, 700, 1500])

        def call():
            _lib.check(_lib.lib().pkv_update_cache_cnt(
                ids.data_ptr(), *ids.stride()[:3], counts.data_ptr(), *counts.stride()[:3], code.data_ptr(), code.stride(0), code.stride(1),
                code.stride(3), code.stride(2), bs, H, N, tiers, nt, ws.data_ptr(), out.data_ptr(), torch.cuda.current_stream().cuda_stream))

        def want():
            return ops.update_cache_cnt(ids, counts, code, [300, 700, 1500])

        change = ids
    else:
        rows, L, k = 3, 24000, 2000
        x = torch.randint(0, 90, (rows, L), generator=g, device=DEV, dtype=torch.int32)
        n = _lib.lib().pkv_bucket_topk_ws_bytes(rows, L)
        ws, out = torch.zeros(n, dtype=torch.uint8, device=DEV), torch.zeros(rows, k, dtype=torch.int64, device=DEV)

        def call():
            _lib.check(_lib.lib().pkv_bucket_topk(x.data_ptr(), L, rows, L, k, out.data_ptr(), ws.data_ptr(), n,
                                                  torch.cuda.current_stream().cuda_stream))

        def want():
            return ops.bucket_topk(x, k)

        change = x
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(out, want()) and not ws.any()
    with torch.cuda.graph(graph):
        call()
    for _ in range(3):
        change.copy_(change.flip(-1))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want()) and ws.any()


@pytest.mark.parametrize("what", ["topk values", "topk ids", "bucket", "votes over the ranking", "votes over the counts"])
def test_results_over_the_inputs(ops, what):
    """Results written over the operator's own inputs, the first rows' over the last ones', with more rows than run at once: the results of
    separate buffers.  The forms in which a row's workgroup writes while others still read stay out of such calls."""
    from pariskv_amd import _lib

    _say(f"results over the inputs, {what}")
    lib, s = _lib.lib(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device=DEV).manual_seed(11)

    def at_end(n_bytes, tail):   # `tail` bytes at the end of a buffer of n_bytes, as its address
        buf = torch.empty(n_bytes, dtype=torch.uint8, device=DEV)
        return buf, buf.data_ptr() + n_bytes - tail

    if what.startswith("topk") or what == "bucket":
        rows, L, k = (3000, 8200, 512) if what != "bucket" else (3000, 5000, 512)
        if what == "bucket":
            x = torch.randint(0, 100, (rows, L), generator=g, device=DEV, dtype=torch.int32)
            want = ops.bucket_topk(x, k)
            n = lib.pkv_bucket_topk_ws_bytes(rows, L)
            ws = torch.empty(n, dtype=torch.uint8, device=DEV)
            buf, out = at_end(rows * L * 4, rows * k * 8)
            buf.view(torch.int32).view(rows, L).copy_(x)
            _lib.check(lib.pkv_bucket_topk(buf.data_ptr(), L, rows, L, k, out, ws.data_ptr(), n, s))
            assert torch.equal(buf[-rows * k * 8:].view(torch.int64).view(rows, k), want)
            return
        x = torch.randn(rows, L, generator=g, device=DEV)
        ids = torch.arange(L, device=DEV).repeat(rows, 1).flip(1).contiguous()
        want_ids, want = ops.topk_f32(x, k, ids, want_values=True)
        n = lib.pkv_topk_f32_ws_bytes(rows, L, k)
        ws = torch.empty(n, dtype=torch.uint8, device=DEV)
        ids_out, vals = torch.empty(rows, k, dtype=torch.int64, device=DEV), torch.empty(rows, k, device=DEV)
        if what == "topk values":
            buf, out = at_end(rows * L * 4, rows * k * 4)
            buf.view(torch.float32).view(rows, L).copy_(x)
            _lib.check(lib.pkv_topk_f32(buf.data_ptr(), L, ids.data_ptr(), L, rows, L, k, ids_out.data_ptr(), out, ws.data_ptr(), n, s))
            vals = buf[-rows * k * 4:].view(torch.float32).view(rows, k)
        else:
            buf, out = at_end(rows * L * 8, rows * k * 8)
            buf.view(torch.int64).view(rows, L).copy_(ids)
            _lib.check(lib.pkv_topk_f32(x.data_ptr(), L, buf.data_ptr(), L, rows, L, k, out, vals.data_ptr(), ws.data_ptr(), n, s))
            ids_out = buf[-rows * k * 8:].view(torch.int64).view(rows, k)
        assert torch.equal(ids_out, want_ids) and torch.equal(vals, want)
        return
    bs, H, N = 187, 8, 700
    ids = torch.stack([torch.randperm(256, generator=g, device=DEV) for _ in range(64)]).repeat(bs * H * 16 // 64, 1).view(bs, H, 16, 256)
    counts = torch.randint(0, 40, (bs, H, 16, 256), generator=g, device=DEV, dtype=torch.int32)
    code = torch.randint(0, 256, (bs, H, 16, N), generator=g, device=DEV).to(torch.uint8)
    want = ops.update_cache_cnt(ids, counts, code, [300, 700, 1500])
    tiers, nt = ops._tiers([300, 700, 1500])
    lut = torch.empty(bs * H * 4096, dtype=torch.uint8, device=DEV)
    src = ids if what.endswith("ranking") else counts
    buf, out = at_end(src.numel() * src.element_size(), bs * H * N * 4)
    buf.view(src.dtype).view(src.shape).copy_(src)
    i, c = (buf.data_ptr(), counts.data_ptr()) if src is ids else (ids.data_ptr(), buf.data_ptr())
    _lib.check(lib.pkv_update_cache_cnt(i, *ids.stride()[:3], c, *counts.stride()[:3], code.data_ptr(), code.stride(0), code.stride(1), 1,
                                        code.stride(2), bs, H, N, tiers, nt, lut.data_ptr(), out, s))
    assert torch.equal(buf[-bs * H * N * 4:].view(torch.int32).view(bs, H, N), want)


def test_bound_attention_on_another_stream_than_its_counters(ops):
    """Counters made behind a long queue of one stream are zero for a launch on another one, which shares no data with it and does not wait."""
    _say("bound attention, counters of another stream")
    bs, H, group, n = 1, 4, 4, 700
    g = torch.Generator(device=DEV).manual_seed(1)
    k, v = (torch.randn(bs, H, n, 128, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
    q = torch.randn(bs, 1, H * group, 128, generator=g, device=DEV).to(torch.bfloat16)
    want = ops.DecodeAttention(bs, H, group, n, DEV).run(q, [(k, v, 0, n)])
    a = torch.randn(8192, 8192, generator=g, device=DEV).to(torch.bfloat16)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    used = [torch.full((2 * bs * H,), 5, dtype=torch.int32, device=DEV) for _ in range(64)]   # what the counters' memory held before
    del used
    torch.cuda.synchronize()
    for _ in range(10):
        a @ a
    att = ops.DecodeAttention(bs, H, group, n, DEV)
    with torch.cuda.stream(side):
        got = ops.BoundAttention(att, q, [(k, v, 0, n)]).launch(q)
    side.synchronize()
    assert torch.equal(got, want)
    torch.cuda.synchronize()


@pytest.mark.parametrize("bs,H,group,lens,base", [(2, 3, 4, (700, 300), 9), (1, 5, 5, (1, 1300), 0), (3, 2, 7, (513, 512, 30), 4), (2, 2, 6, (64, 1, 900), 1),
                                                  (4, 4, 4, (1000, 1048), 3), (4, 4, 4, (1000, 1049), 3), (16, 4, 4, (500, 12), 0), (16, 4, 4, (501, 12), 0),
                                                  (17, 4, 3, (200, 200), 2), (1, 1, 8, (2048,), 0)])
def test_bound_attention_of_several_tensors(ops, bs, H, group, lens, base):
    """The merge in the attention's own launch where the keys lie in tensors of different strides, for query heads that fill a turn of its
    loop in part, and on both sides of its limits (16 splits a row, 256 workgroups): the two launches' bits."""
    _say(f"bound attention, several tensors, {bs} x {H} group {group} {lens}")
    g = torch.Generator(device=DEV).manual_seed(sum(lens) + group)
    segs = []
    for i, n in enumerate(lens):
        k, v = (torch.randn(bs, H, n + base + 5 * i, 128, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
        segs.append((k, v, base, n))
    att = ops.DecodeAttention(bs, H, group, sum(lens), DEV)
    q = torch.randn(bs, 1, H * group, 128, generator=g, device=DEV).to(torch.bfloat16)
    bound = ops.BoundAttention(att, q, segs)
    for _ in range(3):
        q.normal_(generator=g)
        assert torch.equal(bound.launch(q), att.run(q, segs)) and not torch.any(att.arrivals)


def test_votes_of_a_ranking_refuse_an_unaligned_table(ops):
    """Whether the scan builds the table itself or not."""
    from pariskv_amd import _lib

    _say("votes of a ranking, unaligned table")
    ids = torch.arange(256, device=DEV).repeat(1, 1, 16, 1)
    counts = torch.ones(1, 1, 16, 256, dtype=torch.int32, device=DEV)
    ws, tiers = torch.zeros(4096 + 4, dtype=torch.uint8, device=DEV), ops._tiers([10])
    for code in (torch.zeros(1, 1, 16, 100, dtype=torch.uint8, device=DEV), torch.zeros(1, 1, 100, 16, dtype=torch.uint8, device=DEV).transpose(2, 3)):
        out = torch.full((1, 1, 100), -1, dtype=torch.int32, device=DEV)
        rc = _lib.lib().pkv_update_cache_cnt(
            ids.data_ptr(), *ids.stride()[:3], counts.data_ptr(), *counts.stride()[:3], code.data_ptr(), code.stride(0), code.stride(1),
            code.stride(3), code.stride(2), 1, 1, 100, *tiers, ws.data_ptr() + 1, out.data_ptr(), torch.cuda.current_stream().cuda_stream)
        with pytest.raises(RuntimeError, match="aligned"):
            _lib.check(rc)
        assert torch.all(out == -1)
