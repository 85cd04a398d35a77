"""The attention work a user of this package has it do, as measurable cases.

Each case is one call (or one short chain of calls) through the public entry
points: the fused attention at the video models' shapes, the same through the
reference's two backends, small and tiny calls, fp32 callers, frames shorter
than a query tile, the larger head sizes, and the first call of a new pattern.

Geometry of a case: ``T`` latent frames of ``P`` tokens, window ``W``,
``n_first`` anchor frames, keyframe interval ``kfi`` (0: none) at ``offset``,
``text`` joint text tokens, ``B`` x ``H`` (``Hkv``) x ``D`` heads.
"""

import contextlib
import io
import math

import torch

import longvideosparseattention_amd as lv
from longvideosparseattention_amd import sparse_attention as sa
from longvideosparseattention_amd.processor import DistributedLVSAProcessor

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _case(name, kind, T, P, W, kfi, offset, H, D, dtype="bf16", Hkv=0, B=1, text=0, n_first=1, lse=False,
          layout="plain"):
    return {"name": name, "kind": kind, "T": T, "P": P, "W": W, "kfi": kfi, "offset": offset, "n_first": n_first,
            "B": B, "H": H, "Hkv": Hkv or H, "D": D, "dtype": dtype, "text": text, "lse": lse, "layout": layout}


def listed():
    return [
        # Wan 2.1 1.3B self-attention at four times its trained length: the long-video call itself.
        _case("wan_4x", "fused", 84, 1560, 2, 8, 3, 12, 128),
        # HunyuanVideo 1.5 480p dual-stream attention: video and text rows are views of one joint sequence.
        _case("hunyuan_joint", "fused", 49, 1590, 2, 8, 2, 16, 128, text=256, layout="text_last"),
        # CogVideoX-5B joint attention, text first, small heads.
        _case("cog_joint", "fused", 13, 1350, 1, 4, 0, 48, 64, text=226, layout="text_first"),
        # A caller of the reference's default backend: global K/V gathered, then lvsa_sdpa, with the two
        # batch elements of classifier-free guidance.
        _case("wan_sdpa_cfg", "sdpa", 21, 1560, 2, 8, 1, 12, 128, B=2),
        # The plugin's largest head size with grouped K/V heads, fp16.
        _case("head256_gqa", "fused", 21, 1560, 2, 8, 5, 12, 256, dtype="f16", Hkv=4),
        # The reference's FlashInfer backend: its block CSR planned and run, one layer's call; low-resolution frames.
        _case("flashinfer_plan_run", "flashinfer", 33, 390, 2, 8, 4, 12, 128),
        # A low-resolution preview with a text encoder stream through the processor: frames shorter than a query tile.
        _case("preview_processor", "processor", 24, 130, 2, 8, 5, 12, 128, text=37),
        # The reference's CPU-sized configuration as a 16-bit caller runs it, with the log-sum-exp (nine frames).
        _case("nine_frames", "fused", 9, 256, 1, 4, 3, 12, 128, lse=True),
        # The same in fp32, as the reference quotes it.
        _case("nine_frames_f32", "fused", 9, 256, 1, 4, 3, 12, 128, dtype="f32"),
        # An fp32 caller at a video model's frame size, text included.
        _case("video_f32", "fused", 13, 1350, 1, 4, 2, 6, 64, dtype="f32", text=226),
        # The smallest call: a unit-test-sized clip with eight text tokens; nothing but latency.
        _case("tiny_clip", "fused", 9, 16, 1, 4, 3, 2, 64, text=8),
        # A new denoising step's pattern: mask, CSR and plan built, then the first attention call on it.
        _case("new_pattern", "new_pattern", 33, 256, 2, 8, 6, 12, 128),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more call of the listed ranges: every entry point, head size and dtype, odd frame sizes included."""
    most = _cost(listed()[0])
    while True:
        kind = rng.choice(["video", "video", "joint", "joint", "sdpa", "heads", "heads", "flashinfer", "short", "short",
                           "small", "small", "f32", "f32", "tiny", "new_pattern"])
        W, n_first, kfi = rng.randint(1, 4), rng.choice([1, 1, 2]), rng.choice([4, 5, 8, 8])
        H, D, text, dtype, B, group = rng.choice([4, 8, 12, 16]), 128, 0, rng.choice(["bf16", "bf16", "f16"]), 1, 1
        layout, entry, lse = rng.choice(["plain", "packed"]), "fused", rng.random() < 0.25
        if kind == "video":
            T, P = _log_int(rng, 13, 121), _log_int(rng, 390, 1600)
        elif kind == "joint":
            T, P, D = _log_int(rng, 9, 49), _log_int(rng, 390, 1600), rng.choice([64, 128])
            text, layout = _log_int(rng, 16, 512), rng.choice(["text_last", "text_first"])
        elif kind == "sdpa":
            T, P, B, entry, lse = _log_int(rng, 9, 42), _log_int(rng, 256, 1600), rng.choice([1, 2]), "sdpa", False
        elif kind == "heads":
            T, P, D, group = _log_int(rng, 9, 42), _log_int(rng, 256, 1600), rng.choice([64, 96, 192, 256]), rng.choice([1, 2, 4])
        elif kind == "flashinfer":
            T, P, entry, lse, layout = _log_int(rng, 9, 48), _log_int(rng, 64, 1560), "flashinfer", False, "plain"
            D, group, B = rng.choice([64, 128]), rng.choice([1, 2]), rng.choice([1, 2])
        elif kind == "short":
            T, P, D = _log_int(rng, 6, 48), _log_int(rng, 30, 254), rng.choice([64, 128, 128, 192, 256])
            text, entry, lse, layout = rng.choice([0, 17, 37, 128]), "processor", False, "plain"
        elif kind == "small":
            T, P, D, group = _log_int(rng, 4, 21), _log_int(rng, 255, 600), rng.choice([64, 128]), rng.choice([1, 1, 2])
            text = rng.choice([0, 0, 77])
        elif kind == "f32":
            T, P, D, dtype = _log_int(rng, 4, 16), _log_int(rng, 100, 1400), rng.choice([64, 96, 128, 128]), "f32"
            H, text = rng.choice([2, 4, 6, 12]), rng.choice([0, 0, 77, 226])
        elif kind == "tiny":
            T, P, D, H, text = rng.randint(2, 9), _log_int(rng, 4, 60), rng.choice([64, 128]), rng.choice([1, 2, 4]), rng.choice([0, 8])
        else:
            T, P, entry, lse = _log_int(rng, 9, 84), _log_int(rng, 128, 600), "new_pattern", False
        case = _case("", entry, T, P, W, kfi, rng.randrange(kfi), H, D, dtype, H // group, B, text, n_first, lse,
                     "plain" if text and layout == "packed" else layout)
        del case["name"]
        if _cost(case) <= most:
            return case


# ── geometry, in plain Python ────────────────────────────────────────────────


def _rows(case):
    """Attended frames of every query frame (the frame rule of the package's documentation)."""
    T, W, kfi = case["T"], case["W"], case["kfi"]
    anchors = set(range(min(case["n_first"], T)))
    if kfi:
        anchors |= {(case["offset"] + i * kfi) % T for i in range(-(-T // kfi))}
    want = min(2 * W + 1, T - len(anchors))
    rows = []
    for f in range(T):
        lo = max(0, min(f - W, T - 1 - 2 * W))
        hi = min(T - 1, max(f + W, 2 * W))
        left = True
        while W and sum(x not in anchors for x in range(lo, hi + 1)) < want and (lo > 0 or hi < T - 1):
            if left:
                lo = max(0, lo - 1)
            else:
                hi = min(T - 1, hi + 1)
            left = not left
        rows.append(sorted(anchors | set(range(lo, hi + 1) if W else ())))
    return rows


def _pairs(case):
    """(query, key) token pairs of one head, text included."""
    n = case["T"] * case["P"]
    return sum(map(len, _rows(case))) * case["P"] ** 2 + n * case["text"] + case["text"] * (n + case["text"])


def _cost(case):
    """Matrix operations of a pass, fp32 ones weighted by the matrix cores' rates (and frames shorter than a tile
    by the work their masks add), to keep drawn cases below the largest listed one."""
    ops = 4 * case["B"] * case["H"] * case["D"] * _pairs(case)
    return ops * (32 if case["dtype"] == "f32" else 1) * (16 if case["P"] < 255 else 1)


def work(case):
    size = torch.empty(0, dtype=DTYPES[case["dtype"]]).element_size()
    n, t, bd = case["T"] * case["P"], case["text"], case["B"] * case["D"]
    n_k = n
    if case["kind"] == "flashinfer":
        n_k = len(set().union(*_rows(case))) * case["P"]
    moved = 2 * bd * case["H"] * (n + t) + 2 * bd * case["Hkv"] * (n_k + t)     # Q and O, K and V
    lse = 4 * case["B"] * case["H"] * (n + t) if case["lse"] else 0
    return {"bytes": size * moved + lse, "flops": 4 * bd * case["H"] * _pairs(case)}


# ── the calls ────────────────────────────────────────────────────────────────


def _metadata(case):
    return lv.LVSAMetadata.build(
        total_latent_frames=case["T"], num_patches=case["P"], window_size=case["W"], n_first_frames=case["n_first"],
        key_frame_interval=case["kfi"] or None, rank=0, world=1, keyframe_offset=case["offset"])


def _inputs(case, seed):
    """Q, K, V ~ N(0, 1) of the video tokens and the text tokens (None without text)."""
    B, n, t = case["B"], case["T"] * case["P"], case["text"]
    H, Hkv, D, dt = case["H"], case["Hkv"], case["D"], DTYPES[case["dtype"]]
    g = torch.Generator(device="cuda").manual_seed(seed)
    n_k = n
    if case["kind"] == "flashinfer":                       # the compact K/V of the attended frames
        n_k = len(set().union(*_rows(case))) * case["P"]

    def rand(rows, heads):
        return torch.randn(B, rows, heads, D, generator=g, device="cuda", dtype=torch.float32).to(dt)

    if case["layout"] == "packed" and H == Hkv:            # one fused projection: Q, K, V interleaved per token
        qkv = torch.randn(B, n, 3, H, D, generator=g, device="cuda", dtype=torch.float32).to(dt)
        return [qkv[:, :, i] for i in range(3)], [None] * 3
    video, words = [], []
    for rows, heads in ((n, H), (n_k, Hkv), (n_k, Hkv)):
        x = rand(rows + t, heads)
        first = case["layout"] == "text_first"
        video.append(x[:, t:] if first else x[:, :rows])
        words.append(None if not t else x[:, :t] if first else x[:, rows:])
    if case["layout"] == "plain":
        video = [x.contiguous() for x in video]
        words = [None if x is None else x.contiguous() for x in words]
    return video, words


def prepare(case, seed):
    (q, k, v), (qt, kt, vt) = _inputs(case, seed)
    state = {"case": case, "q": q, "k": k, "v": v, "qt": qt, "kt": kt, "vt": vt}
    kind = case["kind"]
    if kind == "processor":
        with contextlib.redirect_stdout(io.StringIO()):    # its one-line summary
            proc = DistributedLVSAProcessor(
                total_num_latent_frames=case["T"], num_patches=case["P"], window_size=case["W"],
                n_first_frames=case["n_first"], key_frame_interval=case["kfi"], rank=0, world=1)
        proc.set_step(case["offset"])
        state["proc"] = proc
    elif kind != "new_pattern":
        state["meta"] = _metadata(case)
        state["meta"].ensure_device(q.device)
    if kind == "flashinfer":
        state["wrapper"] = lv.BlockSparseAttentionWrapper(torch.empty(1 << 20, dtype=torch.uint8, device=q.device))
    return state


def run(state):
    case, q, k, v = state["case"], state["q"], state["k"], state["v"]
    kind = case["kind"]
    if kind == "fused":
        out = lv.lvsa_attention(q, k, v, state["meta"], k_text=state["kt"], v_text=state["vt"], q_text=state["qt"],
                                return_lse=case["lse"])
        return list(out) if isinstance(out, tuple) else [out]
    if kind == "sdpa":
        m = state["meta"]
        kg, vg = lv.build_global_kv(k, v, m.global_indices, m.num_patches)
        return [lv.lvsa_sdpa(q, k, v, kg, vg, m)]
    if kind == "flashinfer":
        m, w = state["meta"], state["wrapper"]
        w.plan(m.fi_indptr, m.fi_indices, M=m.fi_M, N=m.fi_N, R=m.num_patches, C=m.num_patches,
               num_qo_heads=case["H"], num_kv_heads=case["Hkv"], head_dim=case["D"], q_data_type=q.dtype)
        return [lv.sparse_windowed_attention(q, k, v, None, None, m, backend="flashinfer", k_compact=k, v_compact=v,
                                             fi_wrapper=w)]
    if kind == "processor":
        out, text = state["proc"].attention(q, k, v, state["qt"], state["kt"], state["vt"])
        return [out] if text is None else [out, text]
    sa.clear_metadata_cache()                              # a step whose pattern no earlier call has built
    m = _metadata(case)
    out = lv.lvsa_attention(q, k, v, m)
    return [m.fi_indptr, m.fi_indices, out]


# ── the answer in 64 bits ────────────────────────────────────────────────────


def _attend(q, k, v, scale):
    """[n, D] queries of one head over [m, D] keys, by rows to bound memory: output and log-sum-exp."""
    outs, lses = [], []
    for a in range(0, q.shape[0], 4096):
        s = (q[a:a + 4096] @ k.T) * scale
        lse = torch.logsumexp(s, -1)
        outs.append(torch.exp(s.sub_(lse[:, None])) @ v)
        lses.append(lse)
    return torch.cat(outs), torch.cat(lses)


def exact(case, seed):
    (q, k, v), (qt, kt, vt) = _inputs(case, seed)
    T, P, D, t = case["T"], case["P"], case["D"], case["text"]
    rows = _rows(case)
    ids = {f: f for f in range(T)}
    if case["kind"] == "flashinfer":
        ids = {f: i for i, f in enumerate(sorted(set().union(*rows)))}
    scale, group = 1.0 / math.sqrt(D), case["H"] // case["Hkv"]
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    lse = torch.empty(case["B"], case["H"], q.shape[1], dtype=torch.float64, device=q.device)
    if t:
        out_t = torch.empty(qt.shape, dtype=torch.float64, device=q.device)
        lse_t = torch.empty(case["B"], case["H"], t, dtype=torch.float64, device=q.device)
    for b in range(case["B"]):
        for h in range(case["H"]):
            kh, vh = k[b, :, h // group].double(), v[b, :, h // group].double()
            qh = q[b, :, h].double()
            if t:
                kth, vth = kt[b, :, h // group].double(), vt[b, :, h // group].double()
                o, s = _attend(qt[b, :, h].double(), torch.cat([kh, kth]), torch.cat([vh, vth]), scale)
                out_t[b, :, h], lse_t[b, h] = o, s
            for f in range(T):
                tok = torch.cat([torch.arange(ids[x] * P, (ids[x] + 1) * P, device=q.device) for x in rows[f]])
                kk, vv = kh[tok], vh[tok]
                if t:
                    kk, vv = torch.cat([kk, kth]), torch.cat([vv, vth])
                at = slice(f * P, (f + 1) * P)
                out[b, at, h], lse[b, h, at] = _attend(qh[at], kk, vv, scale)
    if case["kind"] == "new_pattern":
        return [None, None, out]
    res = [out] + ([out_t] if t else [])
    if case["lse"]:
        res += [lse] + ([lse_t] if t else [])
    return res


def tolerance(case):
    """Largest relative error another correct implementation at the same precision would show.

    16 bit: the probabilities and the output are rounded to bf16 (fp16) once each, which puts a result 0.0024
    (0.0003) off the 64-bit one.  fp32: sums over up to 10,000 keys in another order; measured 0.9e-6 to 2.5e-6.
    Four times what was measured."""
    return {"rel": {"bf16": 1e-2, "f16": 1.2e-3, "f32": 1e-5}[case["dtype"]]}
