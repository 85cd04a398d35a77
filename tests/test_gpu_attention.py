"""GPU parity of the block-sparse attention kernel through every entry point.

Reference: the fp32 oracle (``oracle/attention.py``) on the same bf16-rounded
inputs.  Tolerance (bf16 output vs fp32 reference):
max |err| <= 2e-2 and mean |err| <= 2e-3.  Inputs follow the BASELINE recipe:
one CPU generator, seed 0, fp32 randn drawn in order q, k, v, then text q,
k, v, shapes [B, N, H, D], rounded to the compute dtype.
"""

import ctypes as C
import dataclasses
import math

import pytest
import torch

import longvideosparseattention_amd as lv
from longvideosparseattention_amd import _capi as capi
from longvideosparseattention_amd import hip_ops
from oracle import attention as oa
from oracle import lvsa_mask as om

pytestmark = pytest.mark.gpu

MAX_ABS = 2e-2
MEAN_ABS = 2e-3


def _draw(shapes, seed=0, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(*s, generator=g, dtype=torch.float32).to(dtype) for s in shapes]


def _close(got, ref, what, max_abs=MAX_ABS, mean_abs=MEAN_ABS):
    ref = ref.to(got.device)
    sel = torch.isfinite(ref)
    err = (got.float()[sel] - ref[sel]).abs()
    assert err.numel() > 0
    mx, mn = err.max().item(), err.mean().item()
    assert mx <= max_abs and mn <= mean_abs, f"{what}: max {mx:.3e} mean {mn:.3e}"


def _meta(T, P, W, n, kfi, off=0, rank=0, world=1, guards=None):
    return lv.LVSAMetadata.build(total_latent_frames=T, num_patches=P, window_size=W, n_first_frames=n,
                                 key_frame_interval=kfi, rank=rank, world=world, keyframe_offset=off,
                                 boundary_guards=guards)


SMALL = [
    # T, P, W, n, kfi, off, H, Hkv, D, n_txt, dtype
    (9, 256, 1, 1, 4, 3, 2, 2, 128, 0, torch.bfloat16),
    (9, 256, 1, 1, 4, 3, 2, 2, 64, 0, torch.bfloat16),
    (10, 4, 0, 2, 3, 0, 2, 2, 128, 0, torch.bfloat16),       # W=0, tiny frames -> generic masks
    (21, 30, 3, 3, 4, 2, 4, 1, 128, 0, torch.bfloat16),      # GQA 4:1, frames < block
    (9, 200, 1, 1, 4, 1, 4, 4, 128, 37, torch.bfloat16),     # text keys + text queries
    (13, 150, 1, 1, 4, 0, 3, 3, 64, 26, torch.float16),      # fp16, D=64, text
    (24, 130, 2, 1, 8, 5, 2, 2, 128, 0, torch.bfloat16),
    (6, 8, 2, 1, 1, 0, 8, 2, 128, 16, torch.bfloat16),       # kfi=1: dense
    (5, 30, 10, 1, None, 0, 2, 2, 64, 0, torch.bfloat16),    # W > T: dense
    (1, 77, 0, 1, None, 0, 2, 2, 128, 3, torch.bfloat16),    # single frame
    (17, 129, 2, 2, 5, 4, 2, 2, 128, 129, torch.float16),    # odd sizes, text tail
    (9, 200, 1, 1, 4, 1, 4, 2, 96, 37, torch.bfloat16),      # D=96 (native, 256-row tiles), GQA, text
    (13, 150, 1, 1, 4, 0, 3, 3, 96, 26, torch.float16),      # D=96, fp16, text
    (9, 256, 1, 1, 4, 3, 2, 2, 192, 0, torch.bfloat16),      # D=192 (native, 128-row tiles)
    (13, 150, 1, 1, 4, 0, 4, 2, 192, 26, torch.float16),     # D=192, fp16, GQA, text
    (9, 200, 1, 1, 4, 1, 4, 4, 256, 37, torch.bfloat16),     # D=256, text
    (13, 150, 1, 1, 4, 0, 3, 3, 256, 26, torch.float16),     # D=256, fp16, text
]


@pytest.mark.parametrize("block_q", [128, 256], ids=["tile128", "tile256"])
@pytest.mark.parametrize("cfg", SMALL, ids=[str(c[:10]) for c in SMALL])
def test_fused_attention_small(cfg, block_q, gpu, monkeypatch):
    """Both kernels (128-row tiles: 4 waves; 256-row tiles: 8 waves in two
    alternating groups) on every small configuration."""
    monkeypatch.setenv("LVSA_ATTN_BLOCK_Q", str(block_q))
    T, P, W, n, kfi, off, H, Hkv, D, n_txt, dt = cfg
    N = T * P
    m = _meta(T, P, W, n, kfi, off)
    q, k, v, qt, kt, vt = _draw([(1, N, H, D), (1, N, Hkv, D), (1, N, Hkv, D), (1, n_txt, H, D),
                                 (1, n_txt, Hkv, D), (1, n_txt, Hkv, D)], dtype=dt)
    ref_rows = [set(r) for r in om.build_frame_mask(T, P, W, n, kfi, offset=off).rows]
    args = dict(k_text=kt.to(gpu), v_text=vt.to(gpu), q_text=qt.to(gpu)) if n_txt else {}
    res = lv.lvsa_attention(q.to(gpu), k.to(gpu), v.to(gpu), m, return_lse=True, **args)
    ro, rl = oa.per_frame_sdpa(q.float(), k.float(), v.float(), ref_rows, P,
                               k_extra=kt.float() if n_txt else None, v_extra=vt.float() if n_txt else None)
    if n_txt:
        o, ot, lse, lse_t = res
        rto, rtl = oa.text_row_attention(qt.float(), k.float(), v.float(), kt.float(), vt.float())
        _close(ot, rto, "text rows")
        torch.testing.assert_close(lse_t.cpu(), rtl, atol=2e-2, rtol=0)
    else:
        o, lse = res
    assert o.dtype == dt and o.shape == q.shape
    _close(o, ro, "video rows")
    torch.testing.assert_close(lse.cpu(), rl, atol=2e-2, rtol=0)


def _random_cfg(seed):
    """A seeded random geometry: frame sizes on and off the 64-key blocks,
    every head size, GQA, text tokens, both dtypes and both tile heights."""
    g = torch.Generator().manual_seed(1000 + seed)
    pick = lambda xs: xs[int(torch.randint(len(xs), (1,), generator=g))]  # noqa: E731
    T = int(torch.randint(1, 17, (1,), generator=g))
    P = int(torch.randint(1, 301, (1,), generator=g))
    W = pick([0, 1, 1, 2, 2, 3, 4])
    n = pick([1, 1, 2, 3])
    kfi = pick([None, 1, 2, 3, 4, 5, 8])
    off = int(torch.randint(0, 8, (1,), generator=g)) % (kfi or 1)
    D = pick([64, 96, 128, 192, 256])
    Hkv = pick([1, 2, 3])
    H = Hkv * pick([1, 2])
    n_txt = pick([0, 0, 1, 17, 64, 100])
    dt = pick([torch.bfloat16, torch.float16])
    block_q = pick([128, 256])
    return T, P, W, n, kfi, off, H, Hkv, D, n_txt, dt, block_q


@pytest.mark.parametrize("seed", range(24))
def test_random_geometries(seed, gpu, monkeypatch):
    """Seeded random geometries through ``lvsa_attention`` against the fp32
    oracle (video rows, text rows and both LSEs)."""
    T, P, W, n, kfi, off, H, Hkv, D, n_txt, dt, block_q = _random_cfg(seed)
    monkeypatch.setenv("LVSA_ATTN_BLOCK_Q", str(block_q))
    N = T * P
    m = _meta(T, P, W, n, kfi, off)
    q, k, v, qt, kt, vt = _draw([(1, N, H, D), (1, N, Hkv, D), (1, N, Hkv, D), (1, n_txt, H, D),
                                 (1, n_txt, Hkv, D), (1, n_txt, Hkv, D)], seed=seed, dtype=dt)
    rows = [set(r) for r in om.build_frame_mask(T, P, W, n, kfi, offset=off).rows]
    args = dict(k_text=kt.to(gpu), v_text=vt.to(gpu), q_text=qt.to(gpu)) if n_txt else {}
    res = lv.lvsa_attention(q.to(gpu), k.to(gpu), v.to(gpu), m, return_lse=True, **args)
    ro, rl = oa.per_frame_sdpa(q.float(), k.float(), v.float(), rows, P,
                               k_extra=kt.float() if n_txt else None, v_extra=vt.float() if n_txt else None)
    what = f"seed {seed}: T={T} P={P} W={W} n={n} kfi={kfi} off={off} H={H}/{Hkv} D={D} txt={n_txt} {dt} bq={block_q}"
    if n_txt:
        o, ot, lse, lse_t = res
        rto, rtl = oa.text_row_attention(qt.float(), k.float(), v.float(), kt.float(), vt.float())
        _close(ot, rto, what + " text rows")
        torch.testing.assert_close(lse_t.cpu(), rtl, atol=2e-2, rtol=0, msg=what)
    else:
        o, lse = res
    assert o.dtype == dt and o.shape == q.shape
    _close(o, ro, what)
    torch.testing.assert_close(lse.cpu(), rl, atol=2e-2, rtol=0, msg=what)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("cfg", [
    # T, P, W, kfi, off, H, Hkv, D, n_txt: frames shorter than a key block or a tile
    (300, 3, 2, 8, 5, 2, 1, 64, 0),      # 10 relation words: rows looked up in global memory
    (256, 1, 1, 4, 3, 1, 1, 128, 5),     # 8 words: the most that LDS holds; one token per frame
    (257, 2, 1, 4, 0, 1, 1, 128, 0),     # 9 words
    (12, 63, 1, 4, 2, 2, 2, 128, 0),     # three frames in some blocks
    (12, 64, 1, 4, 1, 2, 2, 64, 9),      # frames on the block grid
    (7, 65, 2, 3, 1, 2, 2, 96, 0),       # block edges one token into a frame
    (3, 254, 1, None, 0, 2, 2, 128, 3),  # the longest frames with generic blocks in 256-row tiles
], ids=str)
def test_generic_masks_short_frames(cfg, dt, gpu):
    T, P, W, kfi, off, H, Hkv, D, n_txt = cfg
    N = T * P
    q, k, v, qt, kt, vt = _draw([(1, N, H, D), (1, N, Hkv, D), (1, N, Hkv, D), (1, n_txt, H, D),
                                 (1, n_txt, Hkv, D), (1, n_txt, Hkv, D)], seed=P, dtype=dt)
    m = _meta(T, P, W, 1, kfi, off)
    args = dict(k_text=kt.to(gpu), v_text=vt.to(gpu)) if n_txt else {}
    out, lse = lv.lvsa_attention(q.to(gpu), k.to(gpu), v.to(gpu), m, return_lse=True, **args)
    rows = [set(r) for r in om.build_frame_mask(T, P, W, 1, kfi, offset=off).rows]
    ro, rl = oa.per_frame_sdpa(q.float(), k.float(), v.float(), rows, P, k_extra=kt.float() if n_txt else None,
                               v_extra=vt.float() if n_txt else None)
    tol = dict(max_abs=FP32_MAX_ABS, mean_abs=FP32_MEAN_ABS) if dt == torch.float32 else {}
    _close(out, ro, str(cfg), **tol)
    torch.testing.assert_close(lse.cpu(), rl, atol=2e-5 if dt == torch.float32 else 2e-2, rtol=1e-6)


def test_repeat_call_is_bitwise_identical(gpu):
    T, P, H, D = 12, 300, 4, 128
    m = _meta(T, P, 2, 1, 4, 1)
    q, k, v = (x.to(gpu) for x in _draw([(1, T * P, H, D)] * 3))
    a = lv.lvsa_attention(q, k, v, m)
    b = lv.lvsa_attention(q, k, v, m)
    assert torch.equal(a, b)


def test_lvsa_sdpa_with_k_global_and_text(gpu):
    # The reference call path: build_global_kv + text appended -> lvsa_sdpa.
    T, P, W, H, Hkv, D, n_txt = 11, 160, 2, 4, 2, 128, 40
    m = _meta(T, P, W, 1, 4, 2)
    q, k, v, kt, vt = (x.to(gpu) for x in _draw([(1, T * P, H, D), (1, T * P, Hkv, D), (1, T * P, Hkv, D),
                                                 (1, n_txt, Hkv, D), (1, n_txt, Hkv, D)]))
    kg, vg = lv.build_global_kv(k, v, m.global_indices, P)
    kg, vg = torch.cat([kg, kt], 1), torch.cat([vg, vt], 1)
    out = lv.lvsa_sdpa(q, k, v, kg, vg, m)
    out2 = lv.sparse_windowed_attention(q, k, v, kg, vg, m, backend="sdpa")
    assert torch.equal(out, out2)
    ref = om.build_frame_mask(T, P, W, 1, 4, offset=2)
    ro, _ = oa.per_frame_sdpa(q.float(), k.float(), v.float(), om.window_only_relation(ref), P,
                              k_extra=kg.float(), v_extra=vg.float())
    _close(out, ro, "lvsa_sdpa")
    fused = lv.lvsa_attention(q, k, v, m, k_text=kt, v_text=vt)
    _close(fused, ro, "fused vs lvsa_sdpa reference")


CP_SHARDS = [
    # T, P, W, kfi, off, H, D, world, rank
    (12, 50, 2, 5, 3, 2, 128, 2, 1),
    # P >= 255 (single-stream kernels) with the shard's short last key block
    # [256, 312) crossing the frame boundary at 260: planned "generic", so
    # these run the compiler-built kernels
    (6, 260, 1, 3, 1, 2, 128, 5, 0),
    (6, 260, 1, 3, 1, 2, 64, 5, 0),
    (6, 260, 1, 3, 1, 2, 192, 5, 0),
    # P >= 383 (where head size 64 may run 384-row tiles) with a crossing
    # last block: keys [384, 440), boundary at 385
    (8, 385, 1, 3, 2, 2, 64, 7, 0),
]


@pytest.mark.parametrize("cfg", CP_SHARDS, ids=[str(c) for c in CP_SHARDS])
def test_lvsa_sdpa_context_parallel_shard(cfg, gpu):
    # one rank: local queries/keys, globals assembled from the full sequence.
    T, P, W, kfi, off, H, D, world, rank = cfg
    guards = lv.compute_boundary_guard_frames(T, T * P // world, P, world, W)
    m = _meta(T, P, W, 1, kfi, off, rank=rank, world=world, guards=guards)
    q, k, v = _draw([(1, T * P, H, D)] * 3)
    s, e = m.global_token_start, m.global_token_start + m.local_seq
    kg = torch.cat([k[:, g * P:(g + 1) * P] for g in m.global_indices], 1)
    vg = torch.cat([v[:, g * P:(g + 1) * P] for g in m.global_indices], 1)
    out = lv.lvsa_sdpa(q[:, s:e].to(gpu), k[:, s:e].to(gpu), v[:, s:e].to(gpu), kg.to(gpu), vg.to(gpu), m)
    # Oracle: the reference loop over local frames (lvsa/sparse_attention.py:674-704).
    ref = torch.full((1, m.local_seq, H, D), float("nan"))
    for f, qs, qe in m.local_frames:
        parts_k = [kg.float()] + [k[:, s + a:s + b].float() for a, b in m.window_ctx[f]]
        parts_v = [vg.float()] + [v[:, s + a:s + b].float() for a, b in m.window_ctx[f]]
        o, _ = oa.dense_attention(q[:, s + qs:s + qe].float(), torch.cat(parts_k, 1), torch.cat(parts_v, 1))
        ref[:, qs:qe] = o
    _close(out, ref, "cp shard")


def test_flashinfer_backend_and_wrapper(gpu):
    T, P, W, H, D = 9, 96, 1, 4, 128
    m = _meta(T, P, W, 1, 4, 3)
    m.ensure_device(gpu)
    q, k, v = (x.to(gpu) for x in _draw([(1, T * P, H, D)] * 3))
    kg, vg = lv.build_global_kv(k, v, m.global_indices, P)
    ck = q.new_zeros(1, m.fi_N, H, D)
    cv = q.new_zeros(1, m.fi_N, H, D)
    for src, dst in m.fi_global_copies:
        ck[:, dst:dst + P], cv[:, dst:dst + P] = kg[:, src:src + P], vg[:, src:src + P]
    for src, dst in m.fi_local_copies:
        ck[:, dst:dst + P], cv[:, dst:dst + P] = k[:, src:src + P], v[:, src:src + P]
    w = lv.BlockSparseAttentionWrapper(torch.empty(1, dtype=torch.uint8, device=gpu))
    w.plan(m.fi_indptr, m.fi_indices, M=m.fi_M, N=m.fi_N, R=P, C=P, num_qo_heads=H, num_kv_heads=H,
           head_dim=D, q_data_type="bfloat16")
    out = lv.sparse_windowed_attention(q, k, v, kg, vg, m, backend="flashinfer", k_compact=ck, v_compact=cv,
                                       fi_wrapper=w)
    rows = [set(r) for r in om.build_frame_mask(T, P, W, 1, 4, offset=3).rows]
    ro, rl = oa.per_frame_sdpa(q.float(), k.float(), v.float(), rows, P)
    _close(out, ro, "flashinfer backend")
    o2, lse2 = w.run(q[0], ck[0], cv[0], return_lse=True)
    torch.testing.assert_close(lse2.cpu(), (rl[0].transpose(0, 1) / math.log(2.0)).cpu(), atol=3e-2, rtol=0)


def test_flashinfer_backend_batch_of_two(gpu):
    """B = 2 (classifier-free guidance): the backend runs the batch in one
    launch (run_batched), bit for bit what one run() per element gives, and
    matches the oracle per element."""
    T, P, W, H, Hkv, D = 9, 96, 1, 4, 2, 128
    m = _meta(T, P, W, 1, 4, 2)
    m.ensure_device(gpu)
    q = _draw([(2, T * P, H, D)], seed=11)[0].to(gpu)
    k, v = (x.to(gpu) for x in _draw([(2, T * P, Hkv, D)] * 2, seed=12))
    kg, vg = lv.build_global_kv(k, v, m.global_indices, P)
    ck = k.new_zeros(2, m.fi_N, Hkv, D)
    cv = k.new_zeros(2, m.fi_N, Hkv, D)
    for src, dst in m.fi_global_copies:
        ck[:, dst:dst + P], cv[:, dst:dst + P] = kg[:, src:src + P], vg[:, src:src + P]
    for src, dst in m.fi_local_copies:
        ck[:, dst:dst + P], cv[:, dst:dst + P] = k[:, src:src + P], v[:, src:src + P]
    w = lv.BlockSparseAttentionWrapper(torch.empty(1, dtype=torch.uint8, device=gpu))
    w.plan(m.fi_indptr, m.fi_indices, M=m.fi_M, N=m.fi_N, R=P, C=P, num_qo_heads=H, num_kv_heads=Hkv,
           head_dim=D, q_data_type="bfloat16")
    qp = q.new_zeros(2, m.fi_M, H, D)
    qp[:, :m.local_seq] = q
    out = lv.sparse_windowed_attention(qp, k, v, kg, vg, m, backend="flashinfer", k_compact=ck, v_compact=cv,
                                       fi_wrapper=w)
    assert out.shape == (2, m.local_seq, H, D)
    rows = [set(r) for r in om.build_frame_mask(T, P, W, 1, 4, offset=2).rows]
    for b in range(2):
        assert torch.equal(out[b], w.run(qp[b], ck[b], cv[b])[:m.local_seq])
        ro, _ = oa.per_frame_sdpa(q[b:b + 1].float(), k[b:b + 1].float(), v[b:b + 1].float(), rows, P)
        _close(out[b:b + 1], ro, f"flashinfer backend batch element {b}")


def test_dual_stream_runner_gqa(gpu):
    # lvsa-vllm-omni/tests/test_flashinfer_runner.py: H=8, Hkv=2, D=128, P=8, 16 und tokens.
    H, HKV, D, P, S_UND = 8, 2, 128, 8, 16
    for T_lat, ref_frames, kfi in [(24, 6, None), (6, 6, 1)]:
        if kfi is None:
            kfi = lv.compute_auto_kfi(T_lat, 2, 1, reference_frames=ref_frames)
        m = lv.LVSAMetadata.build(total_latent_frames=T_lat, num_patches=P, window_size=2, n_first_frames=1,
                                  key_frame_interval=kfi, rank=0, world=1, reference_frames=ref_frames)
        q, k, v, ku, vu = (x.to(gpu) for x in _draw([(1, T_lat * P, H, D), (1, T_lat * P, HKV, D),
                                                     (1, T_lat * P, HKV, D), (1, S_UND, HKV, D),
                                                     (1, S_UND, HKV, D)], seed=T_lat))
        kg, vg = lv.build_global_kv(k, v, m.global_indices, P)
        kg, vg = torch.cat([kg, ku], 1), torch.cat([vg, vu], 1)
        out = lv.get_shared_runner().run(q, k, v, kg, vg, m)
        assert out.shape == q.shape and torch.isfinite(out.float()).all()
        rows = [set(r) for r in om.build_frame_mask(T_lat, P, 2, 1, kfi).rows]
        ro, _ = oa.per_frame_sdpa(q.float(), k.float(), v.float(), rows, P, k_extra=ku.float(), v_extra=vu.float())
        _close(out, ro, f"runner T={T_lat}")
        if kfi == 1:
            dense, _ = oa.dense_attention(q.float(), torch.cat([k, ku], 1).float(), torch.cat([v, vu], 1).float())
            rel = ((out.float() - dense).norm() / dense.norm()).item()
            assert rel < 2e-2


def test_build_global_kv_exact(gpu):
    # lvsa-vllm-omni/tests/test_global_kv.py
    B, T, P, H, D = 1, 5, 2, 1, 8
    k = torch.arange(T * P, dtype=torch.float32).view(1, T * P, 1, 1).expand(B, T * P, H, D).contiguous().to(gpu)
    kg, _ = lv.build_global_kv(k, k.clone(), [1, 3], P)
    assert kg[0, :, 0, 0].tolist() == [2, 3, 6, 7]
    kb = torch.randn(3, 8 * 4, 2, 8, device=gpu, dtype=torch.bfloat16)
    kg, vg = lv.build_global_kv(kb, kb, [0, 4], 4)
    for b in range(3):
        assert torch.equal(kg[b, :4], kb[b, :4]) and torch.equal(kg[b, 4:], kb[b, 16:20])
    e, _ = lv.build_global_kv(kb, kb, [], 4)
    assert e.shape == (3, 0, 2, 8)
    full, _ = lv.build_global_kv(kb, kb, list(range(8)), 4)
    assert torch.equal(full, kb)


@pytest.mark.parametrize("D", [128, 64, 96, 192, 256])
def test_single_prefill_dense(D, gpu):
    """Dense prefill at every head size (head size 192: 256-row tiles on the
    dual-wide map, which a dense plan takes whatever its length)."""
    q, k, v = (x.to(gpu) for x in _draw([(1, 300, 4, D), (1, 333, 2, D), (1, 333, 2, D)]))
    o, lse = lv.single_prefill_with_kv_cache(q[0], k[0], v[0], causal=False, return_lse=True)
    ro, rl = oa.dense_attention(q.float(), k.float(), v.float())
    _close(o.unsqueeze(0), ro, f"single_prefill D={D}")
    torch.testing.assert_close(lse.cpu(), rl[0].transpose(0, 1).cpu() / math.log(2.0), atol=3e-2, rtol=0)


def test_batch_views_and_fp32_inputs(gpu):
    T, P, W, H, D = 8, 64, 1, 2, 64
    m = _meta(T, P, W, 1, 3, 1)
    qkv = torch.randn(2, T * P, 3 * H * D, device=gpu, dtype=torch.bfloat16)
    q, k, v = (t.unflatten(-1, (H, D)) for t in qkv.chunk(3, dim=-1))   # strided views
    out = lv.lvsa_attention(q, k, v, m)
    rows = [set(r) for r in om.build_frame_mask(T, P, W, 1, 3, offset=1).rows]
    for b in range(2):
        ro, _ = oa.per_frame_sdpa(q[b:b + 1].float(), k[b:b + 1].float(), v[b:b + 1].float(), rows, P)
        _close(out[b:b + 1], ro, f"batch {b}")
    out32 = lv.lvsa_attention(q.float(), k.float(), v.float(), m)   # fp32 kernel, strided fp32 copies
    assert out32.dtype == torch.float32
    for b in range(2):
        ro, _ = oa.per_frame_sdpa(q[b:b + 1].float(), k[b:b + 1].float(), v[b:b + 1].float(), rows, P)
        _close(out32[b:b + 1], ro, f"fp32 batch {b}", max_abs=FP32_MAX_ABS, mean_abs=FP32_MEAN_ABS)


# fp32 callers compute in fp32 (fp32 MFMA products and accumulation, exact
# online softmax): tolerance against the fp32 oracle about 400x tighter
# than the 16-bit path's.
FP32_MAX_ABS = 5e-5
FP32_MEAN_ABS = 5e-6


def test_fp32_baseline_config_1(gpu):
    """BASELINE config 1 (fp32, 12 heads, D 128, 9 frames x 256 tokens, 1
    anchor, keyframe stride 4 rotated by step 3, window 1) through
    lvsa_sdpa and lvsa_attention, against the fp32 oracle on the CPU."""
    T, P, W, kfi, off, H, D = 9, 256, 1, 4, 3, 12, 128
    N = T * P
    q, k, v = _draw([(1, N, H, D)] * 3, dtype=torch.float32)
    m = _meta(T, P, W, 1, kfi, off)
    rows = [set(r) for r in om.build_frame_mask(T, P, W, 1, kfi, offset=off).rows]
    ro, rl = oa.per_frame_sdpa(q, k, v, rows, P)
    o, lse = lv.lvsa_attention(q.to(gpu), k.to(gpu), v.to(gpu), m, return_lse=True)
    assert o.dtype == torch.float32
    _close(o, ro, "fp32 lvsa_attention", max_abs=FP32_MAX_ABS, mean_abs=FP32_MEAN_ABS)
    torch.testing.assert_close(lse.cpu(), rl, atol=2e-5, rtol=1e-6)
    # the reference's lvsa_sdpa semantics: pre-gathered globals + window frames
    kd, vd = k.to(gpu), v.to(gpu)
    kg, vg = lv.build_global_kv(kd, vd, m.global_indices, P)
    o2 = lv.lvsa_sdpa(q.to(gpu), kd, vd, kg, vg, m)
    _close(o2, ro, "fp32 lvsa_sdpa", max_abs=FP32_MAX_ABS, mean_abs=FP32_MEAN_ABS)
    # the bf16 path on the same data is within the 16-bit tolerance only
    ob = lv.lvsa_attention(*(x.to(gpu, torch.bfloat16) for x in (q, k, v)), m)
    assert (ob.float().cpu() - ro).abs().max().item() > 20 * FP32_MAX_ABS


@pytest.mark.parametrize("cfg", SMALL, ids=[str(c[:10]) for c in SMALL])
def test_fp32_small_configs(cfg, gpu):
    """fp32 over the small grid: every head size, GQA, text keys and text
    queries, W = 0 and frames below a tile (generic masks), kfi = 1."""
    T, P, W, n, kfi, off, H, Hkv, D, n_txt, _ = cfg
    N = T * P
    q, k, v, qt, kt, vt = _draw([(1, N, H, D), (1, N, Hkv, D), (1, N, Hkv, D), (1, n_txt, H, D),
                                 (1, n_txt, Hkv, D), (1, n_txt, Hkv, D)], seed=4, dtype=torch.float32)
    m = _meta(T, P, W, n, kfi, off)
    g = [x.to(gpu) for x in (q, k, v, qt, kt, vt)]
    rows = [set(r) for r in om.build_frame_mask(T, P, W, n, kfi, offset=off).rows]
    ro, rl = oa.per_frame_sdpa(q, k, v, rows, P, k_extra=kt if n_txt else None, v_extra=vt if n_txt else None)
    if n_txt:
        o, ot, lse, lse_t = lv.lvsa_attention(g[0], g[1], g[2], m, k_text=g[4], v_text=g[5], q_text=g[3],
                                              return_lse=True)
        rto, rtl = oa.text_row_attention(qt, k, v, kt, vt)
        _close(ot, rto, "fp32 text rows", max_abs=FP32_MAX_ABS, mean_abs=FP32_MEAN_ABS)
        torch.testing.assert_close(lse_t.cpu(), rtl, atol=2e-5, rtol=1e-6)
    else:
        o, lse = lv.lvsa_attention(g[0], g[1], g[2], m, return_lse=True)
    _close(o, ro, f"fp32 D={D}", max_abs=FP32_MAX_ABS, mean_abs=FP32_MEAN_ABS)
    torch.testing.assert_close(lse.cpu(), rl, atol=2e-5, rtol=1e-6)


@pytest.mark.parametrize("D", [64, 96, 128, 192, 256])
@pytest.mark.parametrize("P,H,n_txt", [
    (70, 2, 9),       # few tiles: two key groups per work-group (D <= 128), odd key tails
    (256, 12, 0),
    (300, 60, 130),   # more tiles than compute units; text tiles in chunks at T = 40
])
def test_fp32_split_is_no_further_from_float64(P, H, n_txt, D, gpu):
    """fp32 inputs on the split fp16 MFMAs: error against float64 attention at
    most that of the fp32-MFMA kernel (``scratch=False``), video rows, text
    rows and LSE."""
    if H == 60 and D != 128:
        H = 30
    T = 40 if (P == 300 and D == 64) else 8
    m = _meta(T, P, 1, 1, 4, 2)
    N = T * P
    q, k, v, qt, kt, vt = (x.to(gpu) for x in _draw(
        [(1, N, H, D), (1, N, H // 2, D), (1, N, H // 2, D), (1, n_txt, H, D), (1, n_txt, H // 2, D),
         (1, n_txt, H // 2, D)], seed=D + P, dtype=torch.float32))
    plan = m.full_plan(gpu, N, N, n_txt, n_txt, D, torch.float32)
    kw = dict(kx=kt, vx=vt, qt=qt) if n_txt else {}
    split = hip_ops.attn_fwd(q, k, v, plan, return_lse=True, **kw)
    plain = hip_ops.attn_fwd(q, k, v, plan, return_lse=True, scratch=False, **kw)
    rows = [set(r) for r in om.build_frame_mask(T, P, 1, 1, 4, offset=2).rows]
    heads = [0, H - 1]
    for hd in heads:
        kk, vv = k[0, :, hd // 2].double(), v[0, :, hd // 2].double()
        if n_txt:
            kk, vv = torch.cat([kk, kt[0, :, hd // 2].double()]), torch.cat([vv, vt[0, :, hd // 2].double()])
        frame = torch.arange(N, device=gpu) // P
        ok = torch.zeros(T, T, dtype=torch.bool)
        for f, r in enumerate(rows):
            ok[f, sorted(r)] = True
        seen = ok.to(gpu)[frame][:, frame]
        seen = torch.cat([seen, torch.ones(N, n_txt, dtype=torch.bool, device=gpu)], 1)
        s = (q[0, :, hd].double() @ kk.T / D ** 0.5).masked_fill(~seen, float("-inf"))
        want = [torch.softmax(s, -1) @ vv, torch.logsumexp(s, -1)]
        if n_txt:
            st = qt[0, :, hd].double() @ kk.T / D ** 0.5
            want += [torch.softmax(st, -1) @ vv, torch.logsumexp(st, -1)]

        def errors(res):
            o, ot, lse, lse_t = res
            got = [o[0, :, hd], lse[0, hd]] + ([ot[0, :, hd], lse_t[0, hd]] if n_txt else [])
            return [((g.double() - w).norm() / w.norm()).item() for g, w in zip(got, want)]

        for a, b in zip(errors(split), errors(plain)):
            # 1e-7: one rounding of the fp32 result (2^-24), which both share
            assert a <= max(b, 1e-7), (errors(split), errors(plain))


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("kind", ["k_inf", "k_nan", "v_inf", "q_ninf", "huge", "v_far", "tiny_v", "zeros"])
def test_fp32_split_range(kind, D, gpu):
    """Inputs outside the split's range give what the fp32-MFMA kernel gives:
    non-finite values, products that overflow, V blocks of very different
    size; and small or zero blocks keep fp32's relative accuracy."""
    T, P, H = 6, 130, 2
    m = _meta(T, P, 1, 1, 3, 1)
    N = T * P
    q, k, v = _draw([(1, N, H, D)] * 3, seed=D, dtype=torch.float32)
    if kind == "k_inf":
        k[0, 300, 0, 5] = float("-inf")
    elif kind == "k_nan":
        k[0, 10, 1, 3] = float("nan")
    elif kind == "v_inf":
        v[0, 500, 0, 7] = float("inf")
    elif kind == "q_ninf":
        q[0, 200, 0, 1] = float("-inf")
    elif kind == "huge":
        q[0, 200] *= 1e19
        k[0, 150] *= 1e20
    elif kind == "v_far":
        v[0, :P] *= 1e-9
    elif kind == "tiny_v":
        v *= 1e-25
    else:
        k[0, :128] = 0
        v[0, 64:256] = 0
    plan = m.full_plan(gpu, N, N, 0, 0, D, torch.float32)
    q, k, v = q.to(gpu), k.to(gpu), v.to(gpu)
    a, _, la, _ = hip_ops.attn_fwd(q, k, v, plan, return_lse=True)
    b, _, lb, _ = hip_ops.attn_fwd(q, k, v, plan, return_lse=True, scratch=False)
    tol = 2e-5 * b[torch.isfinite(b)].abs().max().item()
    torch.testing.assert_close(a, b, atol=tol, rtol=2e-5, equal_nan=True)
    torch.testing.assert_close(la, lb, atol=2e-5, rtol=1e-6, equal_nan=True)


OUTLIERS = ["k_inf", "k_ninf", "k_nan", "k_1e6", "k_1e8", "k_1e20", "k_rows_1e8", "k_frame_1e10", "k_small_rows",
            "v_inf", "v_1e6", "v_1e8", "v_1e20", "v_rows_1e8", "v_frame_2^8", "v_frame_2^11", "v_frame_2^13",
            "v_frame_2^16", "v_frame_2^130", "v_channel", "qk_channel", "kq_channel", "q_channel"]


def _plant(kind, q, k, v, P):
    """Outliers at the first and the last key of frame 5, in the whole frame or in one channel."""
    first, last, frame = 5 * P, 6 * P - 1, slice(5 * P, 6 * P)
    name, _, what = kind.partition("_")
    t = {"k": k, "v": v}.get(name)
    if what == "channel":
        {"v": lambda: v[..., 3].mul_(1e9),
         "qk": lambda: (q[..., 3].mul_(1e9), k[..., 3].mul_(1e-9)),
         "kq": lambda: (k[..., 3].mul_(1e9), q[..., 3].mul_(1e-9)),
         "q": lambda: (q[..., 3].mul_(1e9), k[..., 3].zero_())}[name]()
    elif what == "small_rows":
        k[0, ::3] *= 1e-6
        q *= 1e5
    elif what == "rows_1e8":
        t[0, first] *= 1e8
        t[0, last] *= 1e8
    elif what == "frame_1e10":
        t[0, frame] *= 1e10
    elif what.startswith("frame_2^"):
        n = int(what[8:])
        t[0, frame] *= 2.0 ** (n - n // 2)
        t *= 2.0 ** -(n // 2)
        t[0, frame] *= 2.0 ** (n // 2)
    else:
        t[0, first, 0, 9] = t[0, last, 1, 9] = float(what.replace("ninf", "-inf"))


@pytest.mark.parametrize("D", [64, 96, 128, 192, 256])
@pytest.mark.parametrize("kind", OUTLIERS)
def test_fp32_split_outliers(kind, D, gpu):
    """fp32 inputs of a wide range: rows that do not attend the outlier but
    share a key block with it are no further from float64 than the fp32-MFMA
    kernel (``scratch=False``), and rows that attend it give what that kernel
    gives.  Frames of 130 tokens, so frame 5 shares its first and last key
    block with frames 4 and 6; only frames 4 to 6 attend it, so a tile holds
    rows of both kinds."""
    T, P, H = 20, 130, 2
    N = T * P
    m = _meta(T, P, 1, 1, 8, 3)
    rows = om.build_frame_mask(T, P, 1, 1, 8, offset=3).rows
    assert [f for f in range(T) if 5 in rows[f]] == [4, 5, 6]
    q, k, v = (x.to(gpu) for x in _draw([(1, N, H, D)] * 3, seed=D, dtype=torch.float32))
    _plant(kind, q, k, v, P)
    plan = m.full_plan(gpu, N, N, 0, 0, D, torch.float32)
    split, _, lse_s, _ = hip_ops.attn_fwd(q, k, v, plan, return_lse=True)
    plain, _, lse_p, _ = hip_ops.attn_fwd(q, k, v, plan, return_lse=True, scratch=False)
    frame = torch.arange(N, device=gpu) // P
    ok = torch.zeros(T, T, dtype=torch.bool, device=gpu)
    for f, r in enumerate(rows):
        ok[f, sorted(r)] = True
    away = torch.ones(N, dtype=torch.bool, device=gpu) if kind.endswith("channel") or "small" in kind else \
        (frame < 4) | (frame > 6)
    for h in range(H):
        s = q[0, :, h].double() @ k[0, :, h].double().T / D ** 0.5
        s.masked_fill_(~ok[frame][:, frame], float("-inf"))
        p = torch.softmax(s, -1)
        vh = v[0, :, h].double()
        want, size, want_lse = p @ vh, p @ vh.abs(), torch.logsumexp(s, -1)
        a, b, la, lb = split[0, :, h], plain[0, :, h], lse_s[0, h], lse_p[0, h]

        def errors(o, lse):
            # relative to the sum of |P V|; all, the worst row and the worst channel
            e = ((o.double() - want) / size)[away] ** 2
            return [x.item() for x in (e.mean().sqrt(), e.mean(1).max().sqrt(), e.mean(0).max().sqrt(),
                                       ((lse.double() - want_lse) / want_lse)[away].abs().max())]

        if kind != "v_inf":                   # 0 * inf is NaN on both kernels
            got, ref = errors(a, la), errors(b, lb)
            # the extremes may be half as much again, all rows 1%: tiles in parts round at other points
            assert all(x <= f * y for x, y, f in zip(got, ref, [1.01, 1.5, 1.5, 1.5])), (kind, h, got, ref)
        for x, y in ((a, b), (la, lb)):
            # the rows of k_frame_1e10 that attend it: scores of 1e10 round by hundreds, so exp2 may overflow on either
            assert kind == "k_frame_1e10" or (torch.equal(torch.isnan(x), torch.isnan(y)) and
                                              torch.equal(torch.isinf(x), torch.isinf(y))), kind
        if kind in ("k_inf", "k_ninf") or (kind.startswith("v") and kind != "v_inf"):
            sel = torch.isfinite(b) & torch.isfinite(size)
            assert ((a - b).abs()[sel] <= 2e-5 * size[sel]).all(), kind


@pytest.mark.parametrize("D", [64, 128, 256])
def test_fp32_split_v_rise(D, gpu, monkeypatch):
    """The last V blocks 2^130 above the others, attended by some rows of a
    tile only: the other rows keep their result.  Frames of 192 tokens lie on
    the key blocks; a tile holds rows of frames 6 and 7, frame 7 attends the
    last frame and frame 6 does not."""
    T, P, H = 9, 192, 2
    N = T * P
    m = _meta(T, P, 1, 1, None)
    rows = om.build_frame_mask(T, P, 1, 1, None).rows
    assert 8 in rows[7] and 8 not in rows[6] and 7 * P % 128 == 64
    q, k, v = (x.to(gpu) for x in _draw([(1, N, H, D)] * 3, seed=D, dtype=torch.float32))
    monkeypatch.setenv("LVSA_VIDEO_SPLIT", "0")   # no part that holds the last frame alone
    v *= 2.0 ** -65
    v[:, 8 * P:] *= 2.0 ** 65
    v[:, 8 * P:] *= 2.0 ** 65
    plan = m.full_plan(gpu, N, N, 0, 0, D, torch.float32)
    split = hip_ops.attn_fwd(q, k, v, plan)[0][0, 7 * P - 64:7 * P].double()
    plain = hip_ops.attn_fwd(q, k, v, plan, scratch=False)[0][0, 7 * P - 64:7 * P].double()
    seen = torch.cat([torch.arange(f * P, (f + 1) * P) for f in sorted(rows[6])]).to(gpu)
    for h in range(H):
        s = q[0, 7 * P - 64:7 * P, h].double() @ k[0, seen, h].double().T / D ** 0.5
        want = torch.softmax(s, -1) @ v[0, seen, h].double()
        err = [((x[:, h] - want).norm() / want.norm()).item() for x in (split, plain)]
        assert err[0] <= 1.01 * err[1], err


def test_fp32_smaller_workspace_runs_the_fp32_kernel(gpu):
    """A workspace too small for the split operands (1 KiB was enough for any
    fp32 call) still runs, on the fp32 MFMAs: bit for bit the call without."""
    T, P, H, D = 5, 100, 2, 64
    m = _meta(T, P, 1, 1, 3, 1)
    q, k, v = (x.to(gpu) for x in _draw([(1, T * P, H, D)] * 3, dtype=torch.float32))
    plan = m.full_plan(gpu, T * P, T * P, 0, 0, D, torch.float32)
    want = hip_ops.attn_fwd(q, k, v, plan, scratch=False)[0]
    call = hip_ops.attn_args(q, k, v, plan)
    ws = torch.empty(1024, dtype=torch.uint8, device=gpu)
    call.args.workspace, call.args.workspace_bytes = ws.data_ptr(), 1024
    capi.check("lvsa_attn_fwd", capi.lib().lvsa_attn_fwd(C.byref(call.args), hip_ops._stream(call.out.device)))
    assert torch.equal(call.out, want)


@pytest.mark.parametrize("R,Cf,MB,NB", [(128, 128, 1, 40), (70, 100, 3, 60), (200, 1, 2, 1100), (64, 64, 5, 33)], ids=str)
def test_fp32_split_leaves_unattended_blocks_out(R, Cf, MB, NB, gpu):
    """Fewer query rows than keys: only key blocks that some row attends are
    split (the exponents of the others stay as the scratch held them)."""
    H, Hkv, D = 2, 1, 64
    N = NB * Cf
    g = torch.Generator().manual_seed(NB)
    rows = [sorted({0 if r else NB - 1} | set(torch.randperm(NB, generator=g)[:3].tolist())) for r in range(MB)]
    indptr = torch.tensor([0] + [len(r) for r in rows]).cumsum(0).int().to(gpu)
    indices = torch.tensor(sum(rows, []), dtype=torch.int32, device=gpu)
    w = lv.BlockSparseAttentionWrapper()
    w.plan(indptr, indices, MB * R, N, R, Cf, H, Hkv, D, q_data_type=torch.float32)
    q, k, v = (x.to(gpu) for x in _draw([(1, MB * R, H, D), (1, N, Hkv, D), (1, N, Hkv, D)], dtype=torch.float32))
    plain = hip_ops.attn_fwd(q, k, v, w._plan, scratch=False)[0]
    call = hip_ops.attn_args(q, k, v, w._plan)
    n = C.c_int64()
    capi.check("lvsa_attn_workspace_query", capi.lib().lvsa_attn_workspace_query(C.byref(call.args), C.byref(n)))
    blocks = -(-N // 64)
    ws = torch.full((n.value // 4,), 77, dtype=torch.int32, device=gpu)
    call.args.workspace, call.args.workspace_bytes = ws.data_ptr(), n.value
    capi.check("lvsa_attn_fwd", capi.lib().lvsa_attn_fwd(C.byref(call.args), hip_ops._stream(call.out.device)))
    _close(call.out, plain, "split", max_abs=FP32_MAX_ABS, mean_abs=FP32_MEAN_ABS)
    listed = {key // 64 for r in rows for b in r for key in range(b * Cf, (b + 1) * Cf)}
    split = (ws[-2 * blocks:].reshape(blocks, 2) != 77).cpu()
    assert [b for b in range(blocks) if split[b].any()] == sorted(listed) and len(listed) < blocks


def test_fp32_without_memory_for_the_scratch(gpu):
    """Where memory for the fp16 pairs of K and V is short, an fp32 call runs
    without them (on the fp32 MFMAs) instead of failing."""
    T, P, H, D = 16, 1024, 8, 128
    m = _meta(T, P, 1, 1, 4, 1)
    q, k, v = (x.to(gpu) for x in _draw([(1, T * P, H, D)] * 3, dtype=torch.float32))   # 64 MiB each
    plan = m.full_plan(gpu, T * P, T * P, 0, 0, D, torch.float32)
    want = hip_ops.attn_fwd(q, k, v, plan, scratch=False)[0]
    out = torch.empty_like(q)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    limit = torch.cuda.memory_reserved(gpu) + (64 << 20)
    torch.cuda.set_per_process_memory_fraction(limit / torch.cuda.get_device_properties(gpu).total_memory, gpu)
    try:
        with pytest.raises(torch.cuda.OutOfMemoryError):
            torch.empty(128 << 20, dtype=torch.uint8, device=gpu)
        hip_ops.attn_fwd(q, k, v, plan, out=out)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, gpu)
    assert torch.equal(out, want)


def test_fp32_wrapper_and_prefill(gpu):
    """fp32 through the block-sparse wrapper (planned for fp16, run in fp32:
    the wrapper re-plans for 128-row tiles) and the dense prefill."""
    R, C, nb, H, D = 64, 64, 6, 2, 128
    g = torch.Generator().manual_seed(9)
    indptr = torch.tensor([0, 2, 3, 6, 6, 8, 9], dtype=torch.int32)
    indices = torch.tensor([0, 3, 1, 5, 2, 0, 4, 1, 3], dtype=torch.int32)
    q, k, v = (torch.randn(nb * R, H, D, generator=g) for _ in range(3))
    w = lv.BlockSparseAttentionWrapper()
    w.plan(indptr.to(gpu), indices.to(gpu), nb * R, nb * C, R, C, H, H, D)
    o = w.run(q.to(gpu), k.to(gpu), v.to(gpu))
    assert o.dtype == torch.float32
    for i in range(nb):
        cols = indices[indptr[i]:indptr[i + 1]].tolist()
        rows = slice(i * R, (i + 1) * R)
        if not cols:
            assert (o[rows] == 0).all()
            continue
        kk = torch.cat([k[c * C:(c + 1) * C] for c in cols])
        vv = torch.cat([v[c * C:(c + 1) * C] for c in cols])
        ro, _ = oa.dense_attention(q[rows].unsqueeze(0), kk.unsqueeze(0), vv.unsqueeze(0))
        _close(o[rows].unsqueeze(0), ro, f"fp32 wrapper row block {i}", max_abs=FP32_MAX_ABS,
               mean_abs=FP32_MEAN_ABS)
    qd, kd, vd = (torch.randn(*s, generator=g) for s in ((70, 4, 64), (3000, 2, 64), (3000, 2, 64)))
    od = lv.single_prefill_with_kv_cache(qd.to(gpu), kd.to(gpu), vd.to(gpu))
    rd, _ = oa.dense_attention(qd.unsqueeze(0), kd.unsqueeze(0), vd.unsqueeze(0))
    _close(od.unsqueeze(0), rd, "fp32 prefill", max_abs=FP32_MAX_ABS, mean_abs=FP32_MEAN_ABS)


EXTREME = ["hot", "cold", "cold_then_hot", "hot_then_cold"]


@pytest.mark.parametrize("block_q", [128, 256], ids=["tile128", "tile256"])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("D", [64, 96, 128, 192, 256])
@pytest.mark.parametrize("pattern", EXTREME)
@pytest.mark.parametrize("P", [96, 300])
def test_extreme_logits(P, pattern, D, dt, block_q, gpu, monkeypatch):
    """Logits far from N(0,1), where the exponent offset of a row has to move.

    * hot: |s * scale| up to hundreds, so 2^(s * scale * log2 e) overflows fp32 without an offset.
    * cold: every logit very negative, so the exponentials underflow without an offset.
    * cold_then_hot / hot_then_cold: the key frames switch between the two, so a row's offset
      first settles low and must move up, or must stay while later blocks vanish.

    Frames of 300 tokens put D = 128 on the single-stream kernel, whose softmax
    skips the row max unless a block raises it (its rare path).
    """
    monkeypatch.setenv("LVSA_ATTN_BLOCK_Q", str(block_q))
    T, W, n, kfi, off, H = 9, 1, 1, 4, 1, 2
    N = T * P
    amp = 12.0 if dt == torch.bfloat16 else 5.0
    g = torch.Generator().manual_seed(7)
    q = torch.randn(1, N, H, D, generator=g)
    k = torch.randn(1, N, H, D, generator=g)
    v = torch.randn(1, N, H, D, generator=g)
    hot_q, hot_k = amp * q, amp * k
    cold_q, cold_k = amp * (q.abs() + 0.5), -amp * (k.abs() + 0.5)
    key_frame = torch.arange(N) // P
    if pattern == "hot":
        q, k = hot_q, hot_k
    elif pattern == "cold":
        q, k = cold_q, cold_k
    else:
        first_cold = pattern == "cold_then_hot"
        early = (key_frame < T // 2).view(1, N, 1, 1)
        q = cold_q if first_cold else hot_q.abs() + 0.5
        k_cold, k_hot = cold_k, amp * (k.abs() + 0.5)
        k = torch.where(early, k_cold, k_hot) if first_cold else torch.where(early, k_hot, k_cold)
    q, k, v = q.to(dt), k.to(dt), v.to(dt)
    m = _meta(T, P, W, n, kfi, off)
    o, lse = lv.lvsa_attention(q.to(gpu), k.to(gpu), v.to(gpu), m, return_lse=True)
    rows = [set(r) for r in om.build_frame_mask(T, P, W, n, kfi, offset=off).rows]
    ro, rl = oa.per_frame_sdpa(q.float(), k.float(), v.float(), rows, P)
    assert torch.isfinite(o.float()).all() and torch.isfinite(lse).all()
    _close(o, ro, f"{pattern} D={D}")
    torch.testing.assert_close(lse.cpu(), rl, atol=2e-2, rtol=1e-5)


def test_rejects_unsupported_head_dim(gpu):
    m = _meta(4, 16, 1, 1, 2)
    q = torch.randn(1, 64, 2, 80, device=gpu, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="head_dim 80"):
        lv.lvsa_attention(q, q, q, m)


# ── BASELINE shapes at full size ─────────────────────────────────────────────

BASELINE = [
    # name, T, P, W, kfi, off, H, D, n_txt, dtype, spot frames
    ("cpu", 9, 256, 1, 4, 3, 12, 128, 0, torch.float32, None),
    ("wan4x_off0", 84, 1560, 2, 8, 0, 12, 128, 0, torch.bfloat16, [0, 1, 41, 42, 82, 83]),
    ("wan4x_off5", 84, 1560, 2, 8, 5, 12, 128, 0, torch.bfloat16, [1, 13, 50, 83]),
    ("wan6x_w1", 121, 1560, 1, 8, 3, 12, 128, 0, torch.bfloat16, [0, 60, 120]),
    ("cog", 13, 1350, 1, 4, 0, 48, 64, 226, torch.bfloat16, [0, 5, 12]),
    ("hv_off2", 49, 1590, 2, 8, 2, 16, 128, 256, torch.bfloat16, [0, 24, 48]),
]


@pytest.mark.parametrize("cfg", BASELINE, ids=[c[0] for c in BASELINE])
def test_baseline_config_parity(cfg, gpu):
    name, T, P, W, kfi, off, H, D, n_txt, dt, frames = cfg
    N = T * P
    q, k, v, qt, kt, vt = _draw([(1, N, H, D), (1, N, H, D), (1, N, H, D), (1, n_txt, H, D),
                                 (1, n_txt, H, D), (1, n_txt, H, D)], dtype=dt)
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    m = _meta(T, P, W, 1, kfi, off)
    if n_txt:
        o, ot = lv.lvsa_attention(qd, kd, vd, m, k_text=kt.to(gpu), v_text=vt.to(gpu), q_text=qt.to(gpu))
    else:
        o = lv.lvsa_attention(qd, kd, vd, m)
    # size-independent properties: finite, convex combination of value rows
    vmax = v.abs().max().item() if not n_txt else max(v.abs().max().item(), vt.abs().max().item())
    assert torch.isfinite(o.float()).all()
    assert o.float().abs().max().item() <= vmax * 1.01
    rows = [set(r) for r in om.build_frame_mask(T, P, W, 1, kfi, offset=off).rows]
    ro, _ = oa.per_frame_sdpa(qd.float(), kd.float(), vd.float(), rows, P,
                              k_extra=kt.to(gpu).float() if n_txt else None,
                              v_extra=vt.to(gpu).float() if n_txt else None, frames=frames)
    _close(o, ro, name)
    if n_txt:
        rto, _ = oa.text_row_attention(qt.to(gpu).float(), kd.float(), vd.float(), kt.to(gpu).float(),
                                       vt.to(gpu).float())
        _close(ot, rto, name + " text rows")


SWEEP = [
    # name, T, P, W, kfi, H, D, n_txt, offsets (full BASELINE sizes, bf16)
    ("wan4x", 84, 1560, 2, 8, 12, 128, 0, tuple(range(8))),
    ("hv", 49, 1590, 2, 8, 16, 128, 256, tuple(range(8))),
    ("wan6x_w2", 121, 1560, 2, 8, 12, 128, 0, (0, 3, 6)),
    ("wan6x_w4", 121, 1560, 4, 8, 12, 128, 0, (1, 7)),
]


def _sweep_frames(T, P, kfi, off):
    """Query frames to compare: first / last, the rotated keyframes and their
    neighbours (rows that gain or lose a global frame with the offset), and
    the frames whose first row lies nearest above a 256-row tile edge and a
    128-row block edge."""
    fs = {0, 1, T - 1, off % T, (off + 1) % T, (off - 1) % T}
    mid = off + kfi * ((T // kfi) // 2)
    fs |= {mid % T, (mid + 1) % T}
    fs.add(min(range(1, T), key=lambda f: (f * P) % 256))
    fs.add(min(range(1, T), key=lambda f: (-(f * P)) % 128))
    return sorted(fs)


@pytest.mark.parametrize("cfg", SWEEP, ids=[c[0] for c in SWEEP])
def test_baseline_sweep_spot_frames(cfg, gpu):
    """Every keyframe rotation of Wan 4x and HunyuanVideo and the window
    sweep of Wan 6x, at full size through lvsa_attention: about 9 query
    frames per offset against the fp32 oracle, all frames by properties."""
    name, T, P, W, kfi, H, D, n_txt, offsets = cfg
    N = T * P
    g = torch.Generator(device=gpu).manual_seed(11)
    q, k, v = (torch.randn(1, N, H, D, generator=g, device=gpu).to(torch.bfloat16) for _ in range(3))
    qt, kt, vt = (torch.randn(1, n_txt, H, D, generator=g, device=gpu).to(torch.bfloat16) for _ in range(3))
    qf, kf, vf = q.float(), k.float(), v.float()
    vmax = max(v.abs().max().item(), vt.abs().max().item() if n_txt else 0.0)
    for off in offsets:
        m = _meta(T, P, W, 1, kfi, off)
        if n_txt:
            o, ot = lv.lvsa_attention(q, k, v, m, k_text=kt, v_text=vt, q_text=qt)
        else:
            o = lv.lvsa_attention(q, k, v, m)
        assert torch.isfinite(o.float()).all() and o.float().abs().max().item() <= vmax * 1.01
        rows = [set(r) for r in om.build_frame_mask(T, P, W, 1, kfi, offset=off).rows]
        frames = _sweep_frames(T, P, kfi, off)
        ro, _ = oa.per_frame_sdpa(qf, kf, vf, rows, P, k_extra=kt.float() if n_txt else None,
                                  v_extra=vt.float() if n_txt else None, frames=frames)
        _close(o, ro, f"{name} offset {off} frames {frames}")
        if n_txt and off == offsets[0]:
            rto, _ = oa.text_row_attention(qt.float(), kf, vf, kt.float(), vt.float())
            _close(ot, rto, f"{name} text rows")


ALL_FRAMES = [
    # name, T, P, W, kfi, offsets, H, D, n_txt[, dtype[, Hkv]] (full BASELINE sizes, bf16 and Hkv = H
    # unless given).  Wan 4x, Wan 6x (window +-2), HunyuanVideo and CogVideoX at every keyframe
    # rotation; the Wan 6x window sweep points +-1 and +-4 at four rotations each.
    ("wan4x_all_offsets", 84, 1560, 2, 8, tuple(range(8)), 12, 128, 0),
    ("wan6x_w1_four_offsets", 121, 1560, 1, 8, (0, 3, 5, 7), 12, 128, 0),
    ("wan6x_w2_all_offsets", 121, 1560, 2, 8, tuple(range(8)), 12, 128, 0),
    ("wan6x_w4_four_offsets", 121, 1560, 4, 8, (1, 2, 6, 7), 12, 128, 0),
    ("hv_all_offsets", 49, 1590, 2, 8, tuple(range(8)), 16, 128, 256),
    ("cog_all_offsets", 13, 1350, 1, 4, tuple(range(4)), 48, 64, 226),
    # the plugin's other head sizes at the Wan 4x geometry (96: D = 128 LDS layout; 192: dual-wide map,
    # 256-row tiles; 256: wide map), and 192 with text rows (HunyuanVideo geometry), fp16 and GQA
    ("wan4x_d96_off6", 84, 1560, 2, 8, (6,), 12, 96, 0),
    ("wan4x_d192_off1", 84, 1560, 2, 8, (1,), 12, 192, 0),
    ("hv_d192_off3", 49, 1590, 2, 8, (3,), 16, 192, 256),
    ("wan4x_d192_f16_gqa3_off4", 84, 1560, 2, 8, (4,), 12, 192, 0, torch.float16, 4),
    ("wan4x_d256_off7", 84, 1560, 2, 8, (7,), 12, 256, 0),
    # fp16 inputs (the loops' f16 variants)
    ("wan4x_f16_off0", 84, 1560, 2, 8, (0,), 12, 128, 0, torch.float16),
    ("cog_f16_off2", 13, 1350, 1, 4, (2,), 48, 64, 226, torch.float16),
    # grouped K/V heads (3 query heads per K/V head), read in place
    ("wan4x_gqa3_off2", 84, 1560, 2, 8, (2,), 12, 128, 0, torch.bfloat16, 4),
    # batch of two (classifier-free guidance in the plugin): the batch index is a grid dimension
    ("cog_b2_off0", 13, 1350, 1, 4, (0,), 48, 64, 226, torch.bfloat16, 48, 2),
    ("wan4x_b2_off5", 84, 1560, 2, 8, (5,), 12, 128, 0, torch.bfloat16, 12, 2),
]


@pytest.mark.parametrize("cfg", ALL_FRAMES, ids=[c[0] for c in ALL_FRAMES])
def test_baseline_all_frames(cfg, gpu):
    """Every query frame (not a sample) at full size against the fp32 oracle
    (its per-frame gather and dense attention run on the GPU in fp32), with
    the LSE; text rows too.  Each listed keyframe rotation rebuilds the
    pattern (lvsa/lvsa_processor.py:317-331) on the same inputs."""
    name, T, P, W, kfi, offsets, H, D, n_txt = cfg[:9]
    dt = cfg[9] if len(cfg) > 9 else torch.bfloat16
    Hkv = cfg[10] if len(cfg) > 10 else H
    B = cfg[11] if len(cfg) > 11 else 1
    N = T * P
    g = torch.Generator(device=gpu).manual_seed(37)
    q = torch.randn(B, N, H, D, generator=g, device=gpu).to(dt)
    k, v = (torch.randn(B, N, Hkv, D, generator=g, device=gpu).to(dt) for _ in range(2))
    qt = torch.randn(B, n_txt, H, D, generator=g, device=gpu).to(dt)
    kt, vt = (torch.randn(B, n_txt, Hkv, D, generator=g, device=gpu).to(dt) for _ in range(2))
    args = dict(k_text=kt, v_text=vt, q_text=qt) if n_txt else {}
    for off in offsets:
        tag = f"{name} offset {off}"
        print(f"  {tag}", flush=True)
        m = _meta(T, P, W, 1, kfi, off)
        res = lv.lvsa_attention(q, k, v, m, return_lse=True, **args)
        o, lse = (res[0], res[2]) if n_txt else res
        rows = [set(r) for r in om.build_frame_mask(T, P, W, 1, kfi, offset=off).rows]
        ro, rl = oa.per_frame_sdpa(q.float(), k.float(), v.float(), rows, P,
                                   k_extra=kt.float() if n_txt else None, v_extra=vt.float() if n_txt else None)
        assert not torch.isnan(ro).any()
        _close(o, ro, tag)
        torch.testing.assert_close(lse.float(), rl, atol=2e-2, rtol=0, msg=tag)
        del ro, rl
        if n_txt and off == offsets[0]:
            rto, _ = oa.text_row_attention(qt.float(), k.float(), v.float(), kt.float(), vt.float())
            _close(res[1], rto, tag + " text rows")


SUPPORT = [
    # name, T, P, W, kfi, H, D, n_txt, offsets (full BASELINE sizes, bf16; T + 1 <= D)
    ("wan4x", 84, 1560, 2, 8, 12, 128, 0, tuple(range(8))),
    ("wan6x_w0", 121, 1560, 0, 8, 12, 128, 0, (2,)),
    ("wan6x_w1", 121, 1560, 1, 8, 12, 128, 0, (3,)),
    ("wan6x_w2", 121, 1560, 2, 8, 12, 128, 0, (0, 5)),
    ("wan6x_w3", 121, 1560, 3, 8, 12, 128, 0, (6,)),
    ("wan6x_w4", 121, 1560, 4, 8, 12, 128, 0, (1, 7)),
    ("cog", 13, 1350, 1, 4, 48, 64, 226, tuple(range(4))),
    ("hv", 49, 1590, 2, 8, 16, 128, 256, tuple(range(8))),
]


@pytest.mark.parametrize("cfg", SUPPORT, ids=[c[0] for c in SUPPORT])
def test_baseline_frame_support_every_row(cfg, gpu):
    """Every query row at full size, every listed keyframe rotation: with the
    value rows of key frame t equal to the unit vector e_t (text keys: e_T),
    output coordinate d of a row is the softmax weight its row gives key
    frame d.  So a row's nonzero coordinates must be exactly the frames the
    reference's frame rule lets its query frame attend (plus the text
    keys), each weight positive, every other coordinate exactly 0 (masked
    keys and skipped blocks contribute nothing), and the weights sum to 1.
    Text-query rows attend every frame and the text."""
    name, T, P, W, kfi, H, D, n_txt, offsets = cfg
    assert T + 1 <= D
    N = T * P
    g = torch.Generator(device=gpu).manual_seed(29)
    q, k = (torch.randn(1, N, H, D, generator=g, device=gpu).to(torch.bfloat16) for _ in range(2))
    fidx = torch.arange(N, device=gpu) // P
    v = torch.zeros(1, N, H, D, device=gpu, dtype=torch.bfloat16)
    v[0, torch.arange(N, device=gpu), :, fidx] = 1.0
    args = {}
    if n_txt:
        qt, kt = (torch.randn(1, n_txt, H, D, generator=g, device=gpu).to(torch.bfloat16) for _ in range(2))
        vt = torch.zeros(1, n_txt, H, D, device=gpu, dtype=torch.bfloat16)
        vt[..., T] = 1.0
        args = dict(k_text=kt, v_text=vt, q_text=qt)
    for off in offsets:
        m = _meta(T, P, W, 1, kfi, off)
        res = lv.lvsa_attention(q, k, v, m, **args)
        o = (res[0] if n_txt else res)[0].float()                    # [N, H, D]
        allowed = torch.zeros(T, D, dtype=torch.bool)
        for i, r in enumerate(om.build_frame_mask(T, P, W, 1, kfi, offset=off).rows):
            allowed[i, sorted(r)] = True
        if n_txt:
            allowed[:, T] = True
        keep = allowed.to(gpu)[fidx][:, None, :]                      # [N, 1, D]
        what = f"{name} offset {off}"
        assert o.masked_fill(keep, 0.0).abs().max().item() == 0.0, what + ": weight on a frame outside the rule"
        assert o.masked_fill(~keep, 1.0).min().item() > 1e-4, what + ": an allowed frame got no weight"
        assert (o.sum(-1) - 1.0).abs().max().item() < 1e-2, what + ": weights do not sum to 1"
        if n_txt:
            ot = res[1][0].float()
            assert ot[..., T + 1:].abs().max().item() == 0.0 and ot[..., :T + 1].min().item() > 1e-4, what
            assert (ot.sum(-1) - 1.0).abs().max().item() < 1e-2, what


SPLIT = [
    # T, P, H, Hkv, D, n_txt, dtype, B   (text tiles of more than 128 key blocks: split into chunks)
    (8, 1100, 2, 2, 128, 100, torch.bfloat16, 1),   # 140 blocks: 2 chunks
    (24, 1100, 2, 1, 128, 300, torch.bfloat16, 2),  # 418 blocks: 4 chunks, GQA, batch 2
    (13, 1350, 3, 3, 64, 226, torch.float16, 1),    # CogVideoX frame size
    (9, 1000, 2, 2, 96, 37, torch.bfloat16, 1),
    (9, 1000, 2, 2, 256, 37, torch.bfloat16, 1),    # 128-row tiles
]


@pytest.mark.parametrize("cfg", SPLIT, ids=[str(c[:6]) for c in SPLIT])
def test_text_split_parity(cfg, gpu, monkeypatch):
    """Text-query tiles split into key-range chunks (scratch + log-sum-exp
    merge launch) against the fp32 oracle and against the unsplit launch."""
    monkeypatch.setenv("LVSA_VIDEO_SPLIT", "0")   # video tiles whole: their rows compare bit for bit
    T, P, H, Hkv, D, n_txt, dt, B = cfg
    N = T * P
    m = _meta(T, P, 1, 1, 4, 1)
    q, k, v, qt, kt, vt = _draw([(B, N, H, D), (B, N, Hkv, D), (B, N, Hkv, D), (B, n_txt, H, D),
                                 (B, n_txt, Hkv, D), (B, n_txt, Hkv, D)], seed=3, dtype=dt)
    g = [x.to(gpu) for x in (q, k, v, qt, kt, vt)]
    plan = m.full_plan(gpu, N, N, n_txt, n_txt, D)
    o1, ot1, l1, lt1 = hip_ops.attn_fwd(g[0], g[1], g[2], plan, kx=g[4], vx=g[5], qt=g[3], return_lse=True)
    o0, ot0, l0, lt0 = hip_ops.attn_fwd(g[0], g[1], g[2], plan, kx=g[4], vx=g[5], qt=g[3], return_lse=True,
                                        scratch=False)
    assert torch.equal(o1, o0) and torch.equal(l1, l0)   # video rows do not depend on the split
    for b in range(B):
        rto, rtl = oa.text_row_attention(qt[b:b + 1].float(), k[b:b + 1].float(), v[b:b + 1].float(),
                                         kt[b:b + 1].float(), vt[b:b + 1].float())
        _close(ot1[b:b + 1], rto, f"split text rows, batch {b}")
        _close(ot0[b:b + 1], rto, f"unsplit text rows, batch {b}")
        torch.testing.assert_close(lt1[b:b + 1].cpu(), rtl, atol=2e-2, rtol=0)
    _close(ot1, ot0.float(), "split vs unsplit", max_abs=8e-3, mean_abs=5e-4)


QUEUED = [
    # T, P, H, Hkv, D, n_txt, B   (well over 256 work items: the persistent work-queue launch)
    (24, 1100, 8, 2, 128, 300, 2),   # 1664 video tiles + split text chunks, GQA, batch 2
    (13, 1350, 24, 24, 64, 226, 1),  # CogVideoX frame size and text length, half the heads
    (13, 1350, 16, 4, 64, 226, 2),   # the same, GQA (16 query heads over 4) and batch 2: split tiles of both
    (40, 1560, 12, 12, 128, 0, 1),   # Wan frame size, video only
    (24, 1100, 8, 2, 192, 300, 2),   # head size 192 (the dual-wide map), GQA, split text chunks, batch 2
]


@pytest.mark.parametrize("cfg", QUEUED, ids=[str(c) for c in QUEUED])
def test_work_queues_match_static_grid(cfg, gpu, monkeypatch):
    """The single-stream kernel over the work queues (persistent work-groups,
    items stolen across XCDs) computes every whole item exactly as the launch
    with one work-group per item: with the video split off, video rows and
    LSE bit for bit (the text rows differ only by their split).  With the
    split on (the dual map of head size 64: each queue's last video tiles run
    as key-range halves merged by log-sum-exp), rows of split tiles differ by
    rounding only; spot frames, the last ones (split tiles) among them,
    against the fp32 oracle."""
    T, P, H, Hkv, D, n_txt, B = cfg
    N = T * P
    m = _meta(T, P, 2, 1, 8, 3)
    q, k, v, qt, kt, vt = _draw([(B, N, H, D), (B, N, Hkv, D), (B, N, Hkv, D), (B, n_txt, H, D),
                                 (B, n_txt, Hkv, D), (B, n_txt, Hkv, D)], seed=21)
    g = [x.to(gpu) for x in (q, k, v, qt, kt, vt)]
    plan = m.full_plan(gpu, N, N, n_txt, n_txt, D)
    kw = dict(kx=g[4], vx=g[5], qt=g[3]) if n_txt else {}
    o1, ot1, l1, lt1 = hip_ops.attn_fwd(g[0], g[1], g[2], plan, return_lse=True, **kw)
    o0, ot0, l0, lt0 = hip_ops.attn_fwd(g[0], g[1], g[2], plan, return_lse=True, scratch=False, **kw)
    monkeypatch.setenv("LVSA_VIDEO_SPLIT", "0")
    oq, otq, lq, ltq = hip_ops.attn_fwd(g[0], g[1], g[2], plan, return_lse=True, **kw)
    monkeypatch.delenv("LVSA_VIDEO_SPLIT")
    assert torch.equal(oq, o0) and torch.equal(lq, l0)
    # the split tiles: rounding of the two-way merge at most
    assert (o1.float() - o0.float()).abs().max().item() <= 4e-3, "split video tiles differ beyond rounding"
    assert (l1 - l0).abs().max().item() <= 1e-3, "split video tiles: LSE"
    assert torch.equal(o1, o0) != (D == 64), "the dual map (only) splits video tiles"
    rows = [set(r) for r in om.build_frame_mask(T, P, 2, 1, 8, offset=3).rows]
    for b in range(B):
        ro, _ = oa.per_frame_sdpa(g[0][b:b + 1].float(), g[1][b:b + 1].float(), g[2][b:b + 1].float(), rows, P,
                                  k_extra=g[4][b:b + 1].float() if n_txt else None,
                                  v_extra=g[5][b:b + 1].float() if n_txt else None, frames=[0, T // 2, T - 1])
        _close(o1[b:b + 1], ro, f"queued, batch {b}")
    if n_txt:
        _close(ot1, ot0.float(), "queued text vs unsplit", max_abs=8e-3, mean_abs=5e-4)
        rto, _ = oa.text_row_attention(g[3][:1].float(), g[1][:1].float(), g[2][:1].float(), g[4][:1].float(),
                                       g[5][:1].float())
        _close(ot1[:1], rto, "queued text rows")


def _scratch_bytes(q, k, v, m, kt=None, vt=None, qt=None):
    """What lvsa_attn_workspace_query asks for the fused call."""
    n_t = 0 if kt is None else kt.shape[1]
    plan = m.full_plan(q.device, q.shape[1], k.shape[1], n_t, 0 if qt is None else n_t, q.shape[3], q.dtype)
    call = hip_ops.attn_args(q, k, v, plan, kx=kt, vx=vt, qt=qt)
    n = C.c_int64()
    capi.check("lvsa_attn_workspace_query", capi.lib().lvsa_attn_workspace_query(C.byref(call.args), C.byref(n)))
    return n.value


def _partials(tiles, parts, rows, D):
    """Bytes of the video split's partials."""
    return 8 * tiles * parts * rows * (D + 2) * 4


@pytest.mark.parametrize("cfg,want", [
    # T, P, W, kfi, H, Hkv, D, n_txt: partials in bytes (256 compute units)
    ((13, 600, 1, 4, 24, 24, 64, 226), _partials(32, 2, 256, 64)),       # the dual map's halves, text tiles whole
    ((6, 300, 1, 4, 12, 6, 96, 11), 0),                             # the text tile is as long as the video tiles
    ((24, 445, 1, 8, 8, 8, 128, 123), 2 * 8 * 123 * (128 + 2) * 4),  # long text in two chunks, no parts beside them
    ((6, 390, 2, 4, 12, 12, 128, 200), 0),
    ((24, 130, 2, 8, 12, 12, 128, 37), 3 * 12 * 37 * (128 + 2) * 4),  # a text tile three times as long: chunks
    ((33, 390, 2, 8, 12, 12, 128, 0), _partials(13, 2, 256, 128)),       # 100 tiles in the last round: halves
], ids=str)
def test_splits_only_where_the_launch_ends_sooner(cfg, want, gpu):
    """Text chunks and key-range parts by the scratch that a call asks for.
    The calls without were 6% to 40% slower with them."""
    if torch.cuda.get_device_properties(gpu).multi_processor_count != 256:
        pytest.skip("counts of a GPU of 256 compute units")
    T, P, W, kfi, H, Hkv, D, n_txt = cfg
    m = _meta(T, P, W, 1, kfi, 1)
    q, k, v = (torch.empty(1, T * P, h, D, dtype=torch.bfloat16, device=gpu) for h in (H, Hkv, Hkv))
    text = [torch.empty(1, n_txt, h, D, dtype=torch.bfloat16, device=gpu) for h in (Hkv, Hkv, H)] if n_txt else []
    assert _scratch_bytes(q, k, v, m, *text) == -(-want // 256) * 256 + 1024


PARTS = [
    # T, P, H, Hkv, D, n_txt, dtype: fewer rounds than kSplitRounds with a part-filled last one
    (9, 512, 2, 1, 128, 0, torch.bfloat16),     # the half map on a 256-row plan, no queues
    (25, 300, 12, 12, 128, 40, torch.float16),  # 360 tiles: the work queues, text chunks
    (9, 600, 2, 1, 64, 0, torch.bfloat16),      # the half map of D = 64
    (9, 600, 3, 3, 96, 5, torch.bfloat16),
    (9, 500, 4, 2, 192, 0, torch.bfloat16),     # dual-wide map
    (9, 500, 2, 2, 256, 9, torch.float16),      # wide map, 128-row tiles
    (50, 200, 3, 3, 96, 0, torch.bfloat16),     # ping-pong kernel, generic masks
    (50, 126, 1, 1, 256, 0, torch.bfloat16),    # 4-wave kernel
    (9, 500, 2, 1, 128, 0, torch.float32),      # fp32, two key groups
    (13, 900, 9, 9, 64, 70, torch.float32),     # fp32, more tiles than concurrent work-groups
    (9, 500, 2, 1, 256, 0, torch.float32),
]


@pytest.mark.parametrize("cfg", PARTS, ids=[str(c[:6]) for c in PARTS])
def test_video_tiles_in_parts(cfg, gpu, monkeypatch):
    """Last-round tiles as key-range parts merged by log-sum-exp, against whole
    tiles (LVSA_VIDEO_SPLIT=0): O and LSE within the rounding of the merge."""
    T, P, H, Hkv, D, n_txt, dt = cfg
    N = T * P
    m = _meta(T, P, 2, 1, 8, 3)
    q, k, v, qt, kt, vt = (x.to(gpu) for x in _draw(
        [(1, N, H, D), (1, N, Hkv, D), (1, N, Hkv, D), (1, n_txt, H, D), (1, n_txt, Hkv, D), (1, n_txt, Hkv, D)],
        seed=33, dtype=dt))
    kw = dict(k_text=kt, v_text=vt, q_text=qt) if n_txt else {}
    parts = lv.lvsa_attention(q, k, v, m, return_lse=True, **kw)
    text = (kt, vt, qt) if n_txt else ()
    split = _scratch_bytes(q, k, v, m, *text)
    monkeypatch.setenv("LVSA_VIDEO_SPLIT", "0")
    # (the outputs can differ without parts: LVSA_VIDEO_SPLIT=0 also turns the two key groups off)
    assert split >= _scratch_bytes(q, k, v, m, *text) + _partials(1, 2, 128, D), "no tile is split"
    whole = lv.lvsa_attention(q, k, v, m, return_lse=True, **kw)
    assert not torch.equal(parts[0], whole[0]), "no tile was split"
    # one rounding of the output type (|O| < 1) each; fp32: a few of the merge
    tol = {torch.bfloat16: 4e-3, torch.float16: 1e-3, torch.float32: 2e-6}[dt]
    for a, b in zip(parts, whole):
        torch.testing.assert_close(a.float(), b.float(), atol=tol, rtol=tol)


HALF = [
    # T, P, H, Hkv, n_txt, dtype, B: the half map's plans
    (9, 127, 2, 1, 5, torch.bfloat16, 1),     # shortest frames, 128-row plan; a last tile of 119 rows
    (7, 254, 3, 3, 0, torch.float16, 2),      # longest frames with a 128-row plan
    (11, 128, 2, 2, 130, torch.bfloat16, 1),  # frames on the tiles; two text tiles
    (5, 255, 2, 2, 3, torch.bfloat16, 1),     # 256-row plan, two tiles per entry list, row splits in both halves
    (5, 385, 4, 2, 200, torch.float16, 1),    # ... text tiles of both halves; an odd number of 128-row tiles
    (1, 257, 1, 1, 0, torch.bfloat16, 1),     # one row in the last plan tile
    (40, 200, 16, 4, 37, torch.bfloat16, 1),  # more tiles than two per CU: the work queues
]


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("cfg", HALF, ids=[str(c[:5]) for c in HALF])
def test_half_map(cfg, D, gpu):
    """The half map (D = 64 and 128, 128-row tiles) against the fp32 oracle."""
    T, P, H, Hkv, n_txt, dt, B = cfg
    N = T * P
    m = _meta(T, P, 1, 1, 4, 2)
    q, k, v, qt, kt, vt = _draw([(B, N, H, D), (B, N, Hkv, D), (B, N, Hkv, D), (B, n_txt, H, D),
                                 (B, n_txt, Hkv, D), (B, n_txt, Hkv, D)], seed=P, dtype=dt)
    g = [x.to(gpu) for x in (q, k, v, qt, kt, vt)]
    kw = dict(k_text=g[4], v_text=g[5], q_text=g[3]) if n_txt else {}
    res = lv.lvsa_attention(g[0], g[1], g[2], m, return_lse=True, **kw)
    o, lse = (res[0], res[2]) if n_txt else res
    rows = [set(r) for r in om.build_frame_mask(T, P, 1, 1, 4, offset=2).rows]
    frames = None if T < 20 else [0, 1, T // 2, T - 1]
    ro, rl = oa.per_frame_sdpa(g[0].float(), g[1].float(), g[2].float(), rows, P,
                               k_extra=g[4].float() if n_txt else None, v_extra=g[5].float() if n_txt else None,
                               frames=frames)
    _close(o, ro, str(cfg))
    if frames is None:
        torch.testing.assert_close(lse, rl.to(gpu), atol=2e-2, rtol=0)
    if n_txt:
        rto, rtl = oa.text_row_attention(g[3].float(), g[1].float(), g[2].float(), g[4].float(), g[5].float())
        _close(res[1], rto, str(cfg) + " text rows")
        torch.testing.assert_close(res[3], rtl.to(gpu), atol=2e-2, rtol=0)


@pytest.mark.parametrize("D", [64, 96, 128, 192, 256])
@pytest.mark.parametrize("rest", [1, 15, 16, 17, 31, 32])
def test_output_stores_end_at_the_last_row(rest, D, gpu):
    """Lanes of a stream-kernel wave store parts of each other's rows: every remainder of a wave's 32 rows
    against the oracle, in a strided output whose rows past the end and heads beside it stay untouched."""
    P, H = 384 + rest, 2
    m = _meta(1, P, 1, 1, 4)
    q, k, v = (x.to(gpu) for x in _draw([(1, P, H, D)] * 3, seed=rest))
    buf = torch.full((1, P + 40, H + 1, D), 7.0, dtype=q.dtype, device=gpu)
    out = buf[:, :P, :H]
    hip_ops.attn_fwd(q, k, v, m.full_plan(q.device, P, P, 0, 0, D, q.dtype), out=out)
    ro, _ = oa.per_frame_sdpa(q.float(), k.float(), v.float(), [{0}], P)
    _close(out, ro, f"{P} rows, D {D}")
    assert (buf[:, P:] == 7).all() and (buf[:, :, H:] == 7).all()


TALL = [
    # T, P, W, kfi, off, H, Hkv, D, n_txt, dtype, B  (head size 64, frames >= 383 rows: 384-row tiles possible)
    (13, 1350, 1, 4, 0, 6, 6, 64, 226, torch.bfloat16, 1),     # CogVideoX frame and text sizes
    (9, 383, 2, 4, 1, 4, 2, 64, 37, torch.bfloat16, 2),        # smallest frame for 384 rows, GQA, batch 2
    (21, 700, 1, 3, 2, 3, 3, 64, 0, torch.float16, 1),         # fp16, video only, frames straddling tiles
    (16, 1500, 2, 8, 5, 8, 4, 64, 300, torch.float16, 1),      # more than 256 items: work queues
]


@pytest.mark.parametrize("cfg", TALL, ids=[str(c[:9]) for c in TALL])
def test_head64_maps_agree(cfg, gpu, monkeypatch):
    """Head size 64 has three single-stream maps for frames of >= 383 rows:
    the dual map (the default: 256-row tiles, 4 waves of 64 rows, two
    work-groups per CU), 8 waves of 32 rows on the same plan
    (LVSA_D64_WAVES=8) and 12 waves on 384-row tiles.  Per query row the
    8- and 12-wave kernels walk the same key blocks in the same order
    (blocks masked out for a row add exact zeros), so their O and LSE agree
    bit for bit.  The dual map computes each 32-row half as the 8-wave kernel
    does, except that a half also takes the exact-max path when the other
    half of its wave needs it (a rescale, rounding only).  Spot frames and
    text rows are checked against the fp32 oracle."""
    T, P, W, kfi, off, H, Hkv, D, n_txt, dt, B = cfg
    monkeypatch.setenv("LVSA_VIDEO_SPLIT", "0")   # whole tiles: the maps split different tiles
    N = T * P
    m = _meta(T, P, W, 1, kfi, off)
    q, k, v, qt, kt, vt = _draw([(B, N, H, D), (B, N, Hkv, D), (B, N, Hkv, D), (B, n_txt, H, D),
                                 (B, n_txt, Hkv, D), (B, n_txt, Hkv, D)], seed=17, dtype=dt)
    g = [x.to(gpu) for x in (q, k, v, qt, kt, vt)]
    plan = m.full_plan(gpu, N, N, n_txt, n_txt, D, dt)
    assert plan.block_q == 256
    st = m.device_state(gpu)
    plan384 = hip_ops.plan_build(st.mask.rel_full, n_q=N, n_k=N, n_x=n_txt, n_tq=n_txt, R=P, Cf=P,
                                 max_row_frames=max(1, m.max_row_frames), block_q=384)
    kw = dict(kx=g[4], vx=g[5], qt=g[3]) if n_txt else {}
    od, otd, ld, ltd = hip_ops.attn_fwd(g[0], g[1], g[2], plan, return_lse=True, **kw)
    o12, ot12, l12, lt12 = hip_ops.attn_fwd(g[0], g[1], g[2], plan384, return_lse=True, **kw)
    monkeypatch.setenv("LVSA_D64_WAVES", "8")
    o8, ot8, l8, lt8 = hip_ops.attn_fwd(g[0], g[1], g[2], plan, return_lse=True, **kw)
    monkeypatch.delenv("LVSA_D64_WAVES")
    assert torch.equal(o12, o8) and torch.equal(l12, l8), "video rows differ between 384- and 256-row tiles"
    if n_txt:
        assert torch.equal(ot12, ot8) and torch.equal(lt12, lt8), "text rows differ"
    # dual map against 8 waves: rounding of an extra rescale at most
    assert (od.float() - o8.float()).abs().max().item() <= 2e-3 and (ld - l8).abs().max().item() <= 1e-4
    if n_txt:
        assert (otd.float() - ot8.float()).abs().max().item() <= 2e-3 and (ltd - lt8).abs().max().item() <= 1e-4
    rows = [set(r) for r in om.build_frame_mask(T, P, W, 1, kfi, offset=off).rows]
    for b in range(B):
        ro, _ = oa.per_frame_sdpa(g[0][b:b + 1].float(), g[1][b:b + 1].float(), g[2][b:b + 1].float(), rows, P,
                                  k_extra=g[4][b:b + 1].float() if n_txt else None,
                                  v_extra=g[5][b:b + 1].float() if n_txt else None, frames=[0, 1, T // 2, T - 1])
        _close(od[b:b + 1], ro, f"dual map, batch {b}")
        _close(o12[b:b + 1], ro, f"384-row tiles, batch {b}")
    if n_txt:
        rto, _ = oa.text_row_attention(g[3][:1].float(), g[1][:1].float(), g[2][:1].float(), g[4][:1].float(),
                                       g[5][:1].float())
        _close(otd[:1], rto, "dual map, text rows")
        _close(ot12[:1], rto, "384-row tiles, text rows")


@pytest.mark.parametrize("D", [128, 192])
def test_single_prefill_long_keys_split(D, gpu):
    """Dense prefill over more than 128 key blocks runs split (chunks + merge)."""
    q, k, v = (x.to(gpu) for x in _draw([(1, 70, 4, D), (1, 20000, 2, D), (1, 20000, 2, D)], seed=5))
    o, lse = lv.single_prefill_with_kv_cache(q[0], k[0], v[0], causal=False, return_lse=True)
    ro, rl = oa.dense_attention(q.float(), k.float(), v.float())
    _close(o.unsqueeze(0), ro, f"single_prefill split D={D}")
    torch.testing.assert_close(lse.cpu(), rl[0].transpose(0, 1).cpu() / math.log(2.0), atol=3e-2, rtol=0)


def test_plan_overflow_and_block_k_are_rejected(gpu):
    """A plan whose entry capacity is too small (max_row_frames below the
    relation's row maximum) raises at first use; so does a plan built for key
    blocks other than the kernels' 64 rows."""
    T, P, H, D = 12, 300, 2, 128
    m = _meta(T, P, 2, 1, 4, 1)
    m.ensure_device(gpu)
    st = m.device_state(gpu)
    q, k, v = (x.to(gpu) for x in _draw([(1, T * P, H, D)] * 3))
    bad = hip_ops.plan_build(st.mask.rel_full, n_q=T * P, n_k=T * P, R=P, Cf=P, max_row_frames=1)
    with pytest.raises(RuntimeError, match="exceed the capacity"):
        hip_ops.attn_fwd(q, k, v, bad)
    wide = hip_ops.plan_build(st.mask.rel_full, n_q=T * P, n_k=T * P, R=P, Cf=P,
                              max_row_frames=m.max_row_frames, block_k=128)
    with pytest.raises(ValueError, match="block_k=128"):
        hip_ops.attn_fwd(q, k, v, wide)
    good = hip_ops.plan_build(st.mask.rel_full, n_q=T * P, n_k=T * P, R=P, Cf=P, max_row_frames=m.max_row_frames)
    out, _, _, _ = hip_ops.attn_fwd(q, k, v, good)
    assert torch.equal(out, lv.lvsa_attention(q, k, v, m))


@pytest.mark.parametrize("change", [dict(window_size=9), dict(max_row_frames=1), dict(n_first_frames=20)], ids=str)
def test_replaced_metadata_fields_cannot_truncate_a_plan(change, gpu):
    """Fields replaced on a built instance leave max_row_frames behind: the
    plan's capacity is checked, as for any other caller of plan_build."""
    T, P, H, D = 24, 300, 2, 128
    m = dataclasses.replace(_meta(T, P, 1, 1, 8, 1), _device_state={}, **change)
    q, k, v = (x.to(gpu) for x in _draw([(1, T * P, H, D)] * 3))
    with pytest.raises(RuntimeError, match="exceed the capacity"):
        lv.lvsa_attention(q, k, v, m)


def test_wrapper_rejects_out_of_range_columns(gpu):
    w = lv.BlockSparseAttentionWrapper()
    indptr = torch.tensor([0, 2, 3], dtype=torch.int32)
    indices = torch.tensor([0, 5, 1], dtype=torch.int32)  # column 5 of 2
    w.plan(indptr, indices, M=128, N=128, R=64, C=64, num_qo_heads=2, num_kv_heads=2, head_dim=128)
    q, k, v = (x.to(gpu) for x in _draw([(128, 2, 128)] * 3))
    with pytest.raises(ValueError, match="outside"):
        w.run(q, k, v)


def _stream_cfg(seed, p_min=255):
    """Random geometries the single-stream kernel serves (frames of at least
    p_min tokens): window / keyframe patterns, text, GQA, both dtypes."""
    g = torch.Generator().manual_seed(2000 + seed)
    pick = lambda xs: xs[int(torch.randint(len(xs), (1,), generator=g))]  # noqa: E731
    T = int(torch.randint(1, 14, (1,), generator=g))
    P = int(torch.randint(p_min, 700, (1,), generator=g))
    W = pick([0, 1, 2, 3])
    n = pick([1, 1, 2])
    kfi = pick([None, 1, 2, 3, 4, 8])
    off = int(torch.randint(0, 8, (1,), generator=g)) % (kfi or 1)
    Hkv = pick([1, 2])
    H = Hkv * pick([1, 2])
    n_txt = pick([0, 0, 1, 37, 64, 300])
    dt = pick([torch.bfloat16, torch.float16])
    return T, P, W, n, kfi, off, H, Hkv, n_txt, dt


@pytest.mark.parametrize("D", [128, 64, 96, 192, 256])
@pytest.mark.parametrize("seed", range(16))
def test_stream_kernel_random_geometries(seed, D, gpu, monkeypatch):
    """D = 64, 96 and 128 on frames of >= 255 tokens, and D = 192 and 256 (the
    wide map, 128-row tiles) on frames of >= 127, run the hand-scheduled
    single-stream kernel; against the fp32 oracle, and the ping-pong (D >= 192:
    4-wave) kernel within bf16 rounding."""
    # the wide map's 128-row tiles take frames from 127 tokens on
    T, P, W, n, kfi, off, H, Hkv, n_txt, dt = _stream_cfg(seed, 127 if D >= 192 else 255)
    N = T * P
    m = _meta(T, P, W, n, kfi, off)
    q, k, v, qt, kt, vt = _draw([(1, N, H, D), (1, N, Hkv, D), (1, N, Hkv, D), (1, n_txt, H, D),
                                 (1, n_txt, Hkv, D), (1, n_txt, Hkv, D)], seed=seed, dtype=dt)
    rows = [set(r) for r in om.build_frame_mask(T, P, W, n, kfi, offset=off).rows]
    args = dict(k_text=kt.to(gpu), v_text=vt.to(gpu), q_text=qt.to(gpu)) if n_txt else {}
    res = lv.lvsa_attention(q.to(gpu), k.to(gpu), v.to(gpu), m, return_lse=True, **args)
    monkeypatch.setenv("LVSA_ATTN_KERNEL", "pp")
    res_pp = lv.lvsa_attention(q.to(gpu), k.to(gpu), v.to(gpu), m, return_lse=True, **args)
    ro, rl = oa.per_frame_sdpa(q.float(), k.float(), v.float(), rows, P,
                               k_extra=kt.float() if n_txt else None, v_extra=vt.float() if n_txt else None)
    what = f"seed {seed}: D={D} T={T} P={P} W={W} n={n} kfi={kfi} off={off} H={H}/{Hkv} txt={n_txt} {dt}"
    o, lse = (res[0], res[2]) if n_txt else res
    _close(o, ro, what)
    torch.testing.assert_close(lse.cpu(), rl, atol=2e-2, rtol=0, msg=what)
    _close(o, (res_pp[0] if n_txt else res_pp[0]).float(), what + " vs ping-pong", max_abs=8e-3, mean_abs=5e-4)
    if n_txt:
        rto, _ = oa.text_row_attention(qt.float(), k.float(), v.float(), kt.float(), vt.float())
        _close(res[1], rto, what + " text rows")


def test_shared_pattern_across_streams(gpu):
    """LVSAMetadata.build shares one pattern per set of arguments: built (mask
    and plan) on one stream and then used on another, the second stream waits
    for the build and registers itself with the allocator, and both give the
    same output bit for bit."""
    T, P, W, kfi, off, H, D = 11, 264, 1, 4, 2, 2, 128
    m = _meta(T, P, W, 1, kfi, off)
    q, k, v = (x.to(gpu) for x in _draw([(1, T * P, H, D)] * 3, seed=5))
    s1, s2 = torch.cuda.Stream(gpu), torch.cuda.Stream(gpu)
    s1.wait_stream(torch.cuda.current_stream(gpu))
    s2.wait_stream(torch.cuda.current_stream(gpu))
    with torch.cuda.stream(s1):
        o1 = lv.lvsa_attention(q, k, v, m)
    with torch.cuda.stream(s2):
        o2 = lv.lvsa_attention(q, k, v, m)
    torch.cuda.synchronize(gpu)
    st = m.device_state(gpu)
    assert st.joined.get(s1.cuda_stream) == st.version and st.joined.get(s2.cuda_stream) == st.version
    assert torch.equal(o1, o2)
    rows = [set(r) for r in om.build_frame_mask(T, P, W, 1, kfi, offset=off).rows]
    ro, _ = oa.per_frame_sdpa(q.float(), k.float(), v.float(), rows, P)
    _close(o2, ro, "second stream")
