"""The attention layer's work that is timed: impl forwards of engine steps and cache writes.

A case is one call a serving engine makes on one FULL-attention layer (one TP
rank's share): `forward` of a step (decode, MTP verification, prefill, mixed
batches), `forward` without fresh K/V (the DecodeOnly read), or
`do_kv_cache_update` of a batch of tokens.  A step is written as text, one
`new@history` entry per request: "4@24579" is one request with 4 new tokens
over 24579 cached ones.

Everything the layer holds before the call (INT2 pages, window arena, block
table) is computed here with plain torch in float64, so that a change of the
framework's own write path does not change what its read path is given.
"""
from __future__ import annotations

import dataclasses
import math
import os
from types import SimpleNamespace

import numpy as np
import torch

os.environ.setdefault("OSCAR_ASCEND_VERBOSE", "0")

D = 256                               # the head size the framework is built for
OUTLIERS = (7, 71, 135, 199)          # K/V channels of 8 times the others' scale
SLOT_BYTES_READ = 136                 # 8 metadata + 64 K code + 64 V code bytes a cached token and head
MOST_FLOPS = 1.14e12                  # of a drawn case: the largest listed one's
DEVICE = "cuda:0"

# The deployment's options: window of 128 sink and 256 recent tokens, clipping
# on, 128-token pages in the int8 cache geometry, 6 query heads on one K/V head.
DEPLOYED = {"heads": 6, "kv_heads": 1, "page": 128, "slot": 256, "sink": 128, "recent": 256, "staging": 8192,
            "clip_k": 0.96, "clip_v": 0.92}

# Histories of 32 concurrent requests, spread over [2048, 16384].
CONCURRENT = (4171, 13250, 9002, 2311, 15777, 6640, 11893, 3527, 14608, 8215, 5099, 12346, 2998, 16201, 7433, 10560,
              4822, 9671, 13999, 3210, 6011, 15102, 8888, 2555, 11047, 7019, 12877, 5450, 10013, 14250, 3777, 9333)


def _case(name, kind, requests, **options):
    return {"name": name, "kind": kind, "requests": requests, **{**DEPLOYED, **options}}


def _write_case(name, tokens, skipped, **options):
    return {"name": name, "kind": "write", "tokens": tokens, "skipped": skipped, **{**DEPLOYED, **options}}


def listed():
    return [
        # One user, a short chat, no speculation: the smallest step there is.
        _case("decode 1x1 1K", "step", "1@1024"),
        # One user with a long document, four MTP tokens verified at once.
        _case("mtp 1x4 24K", "step", "4@24579"),
        # A busy server: 32 users verifying four MTP tokens each.
        _case("mtp 32x4 2-16K", "step", ",".join(f"4@{h}" for h in CONCURRENT)),
        # Long-context decoding of a few users without speculation.
        _case("decode 8x1 32K", "step", ",".join(["1@32768"] * 8)),
        # A ragged batch (draft lengths, histories down to a few tokens) of a
        # rank with two K/V heads, 64-token pages in the bf16 cache geometry.
        _case("mtp ragged 2 kv heads", "step", "1@3,4@130,2@8191,16@517,3@12000,1@777,5@40", heads=12, kv_heads=2,
              page=64, slot=512),
        # The same long contexts read by an engine's DecodeOnly state.
        _case("decode-only 8x32K", "decode_only", ",".join(["1@32768"] * 8)),
        # A new prompt.
        _case("prefill 3001", "step", "3001@0"),
        # A long prompt's last chunk over its cached part.
        _case("prefill 9256 over 15K", "step", "9256@15360"),
        # A follow-up question on a cached document (a prefix-cache hit).
        _case("prefill 77 over 20K", "step", "77@20011"),
        # Chunked prefill: one prompt's chunk beside seven users' MTP steps.
        _case("mixed chunk + 7x4", "step", "4@5000,4@2711,1024@4096,4@900,4@16000,4@333,4@7777,4@12001"),
        # A bulk cache write with padding slots, in scattered slots.
        _write_case("write 65536", 65536, 0.0625),
        # The cache write of one MTP step.
        _write_case("write 4", 4, 0.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    heads, kv_heads = rng.choice(((6, 1), (6, 1), (6, 1), (12, 2), (8, 1), (12, 1), (16, 2), (4, 4)))
    options = {"heads": heads, "kv_heads": kv_heads, "page": rng.choice((128, 128, 128, 64, 32)),
               "slot": rng.choice((256, 256, 512))}
    if rng.random() < 0.2:            # no window
        options["staging"] = 0
    elif rng.random() < 0.2:          # the defaults of the environment
        options["sink"] = 64
    if rng.random() < 0.2:            # no clipping
        options["clip_k"] = options["clip_v"] = 0.0
    kind = rng.choice(("step", "step", "step", "step", "decode_only", "prefill", "prefill", "prefill", "mixed", "mixed",
                       "write", "write"))
    if kind == "write":
        case = _write_case("", _log(rng, 1, 65536 // kv_heads), rng.choice((0.0, 0.0625)), **options)
        del case["name"]
        return case

    def histories(count, lo, total):
        most = max(lo + 1, min(32768, total // (count * kv_heads)))
        return [_log(rng, lo, most) for _ in range(count)]

    requests = []
    if kind in ("step", "decode_only"):
        count = _log(rng, 1, 32)
        new = 1 if kind == "decode_only" else rng.choice((1, 2, 4, 4, 8, 0))
        requests = [(new or rng.randint(1, 16), h) for h in histories(count, 16, 280000)]
    else:
        for h in histories(rng.randint(1, 3) if kind == "prefill" else 1, 16, 32768):
            requests.append((_log(rng, 17, 9256), 0 if rng.random() < 0.3 else h))
        if kind == "mixed":
            requests += [(rng.choice((1, 2, 4)), h) for h in histories(rng.randint(1, 16), 16, 120000)]
            rng.shuffle(requests)
        flops = 4 * D * heads * sum(_visible(n, h) for n, h in requests)
        if flops > MOST_FLOPS:
            requests = [(max(1, int(n * MOST_FLOPS / flops)), h) for n, h in requests]
    case = _case("", "decode_only" if kind == "decode_only" else "step", ",".join(f"{n}@{h}" for n, h in requests),
                 **options)
    del case["name"]
    return case


def _visible(new, history):
    """Keys that a request's new tokens attend to, summed over the tokens."""
    return new * history + new * (new + 1) // 2


def _requests(case):
    return [tuple(int(x) for x in r.split("@")) for r in case["requests"].split(",")]


def work(case):
    hq, hk = case["heads"], case["kv_heads"]
    rotations = 4 * D * D
    if case["kind"] == "write":
        written = int(case["tokens"] * (1 - case["skipped"]))
        return {"bytes": case["tokens"] * (hk * 2 * D * 2 + 8) + written * hk * SLOT_BYTES_READ + 2 * rotations,
                "flops": case["tokens"] * hk * 2 * 2 * D * D}
    reqs = _requests(case)
    new = sum(n for n, _ in reqs)
    only = case["kind"] == "decode_only"
    cached = sum(h for _, h in reqs) + (new if only else 0)
    nbytes = cached * hk * SLOT_BYTES_READ + new * hq * D * 2 * 2 + 3 * rotations
    flops = 4 * D * hq * sum(_visible(n, h) for n, h in reqs) + new * hq * 2 * 2 * D * D
    if not only:
        nbytes += new * (hk * (2 * D * 2 + SLOT_BYTES_READ) + 8)
        flops += new * hk * 2 * 2 * D * D
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["kind"] == "write":
        return {"rel": 0.0, "differ": DIFFER}
    if case["kind"] == "step" and any(n > 16 for n, _ in _requests(case)):
        return {"rel": 8e-3, "max": 0.2, "differ": DIFFER}
    return {"rel": 7e-3, "max": 0.03, "differ": DIFFER}


# Four times what the framework shows against float64: bf16 outputs (relative
# error 1.5e-3 .. 2.1e-3, largest 5e-3 for decode and 5e-2 for prefill), and
# the share of cache bytes whose codes round the other way when the rotation's
# sums run in another order or through bf16 high and low parts (2.8e-5).
DIFFER = 1.2e-4


# ------------------------------------------------------------------ plain torch
def _normal(generator, *shape):
    return torch.randn(*shape, generator=generator, device=DEVICE, dtype=torch.float32)


def _kv(generator, n, hk):
    scale = torch.ones(D, device=DEVICE)
    scale[list(OUTLIERS)] = 8.0
    return [(_normal(generator, n, hk, D) * scale).to(torch.bfloat16) for _ in range(2)]


def _rotation(seed):
    g = torch.Generator().manual_seed(seed)
    return torch.linalg.qr(torch.randn(D, D, generator=g)).Q.contiguous().to(DEVICE)


def _slot_parts(rotated, clip):
    """(scale, zero) fp16 bit patterns and packed codes of float32 vectors [.., D]."""
    x = rotated
    if clip > 0:
        rank = min(int(clip * D), D - 1)
        bound = x.abs().sort(dim=-1).values[..., rank:rank + 1]
        x = torch.maximum(torch.minimum(x, bound), -bound)
    low = x.amin(-1, keepdim=True)
    scale = ((x.amax(-1, keepdim=True) - low) / 3).clamp_min(2.0 ** -14).half()
    zero = low.half()
    codes = ((x - zero.float()) / scale.float() + 0.5).floor().clamp(0, 3).to(torch.uint8)
    c = codes.view(*codes.shape[:-1], D // 4, 4)
    packed = c[..., 0] | (c[..., 1] << 2) | (c[..., 2] << 4) | (c[..., 3] << 6)
    return scale, zero, packed


def _store(caches, slots, k_rot, v_rot, case):
    """Quantize and write rotated vectors [n, Hk, D] to cache slots."""
    for a in range(0, slots.numel(), 32768):
        s, kr, vr = slots[a:a + 32768], k_rot[a:a + 32768].float(), v_rot[a:a + 32768].float()
        ks, kz, kp = _slot_parts(kr, case["clip_k"])
        vs, vz, vp = _slot_parts(vr, case["clip_v"])
        meta = torch.cat((ks, kz, vs, vz), -1).contiguous().view(torch.uint8)
        rows_k, rows_v = (c.view(torch.uint8).view(-1, *c.view(torch.uint8).shape[2:]) for c in caches)
        rows_k[s, :, :8] = meta
        rows_k[s, :, 32:96] = kp
        rows_v[s, :, :64] = vp


def _load(caches, slots):
    """Dequantized float64 (k, v) [n, Hk, D] of cache slots."""
    rows_k, rows_v = (c.view(torch.uint8).view(-1, *c.view(torch.uint8).shape[2:]) for c in caches)
    k8, v8 = rows_k[slots], rows_v[slots]
    meta = k8[..., :8].contiguous().view(torch.float16).double()
    out = []
    for i, packed in enumerate((k8[..., 32:96], v8[..., :64])):
        codes = torch.stack([(packed >> (2 * e)) & 3 for e in range(4)], -1).flatten(-2).double()
        out.append(codes * meta[..., 2 * i:2 * i + 1] + meta[..., 2 * i + 1:2 * i + 2])
    return out


def _window_rows(case):
    page, sink, recent, staging = case["page"], case["sink"], case["recent"], case["staging"]
    if staging <= 0 or (sink <= 0 and recent <= 0):
        return 0
    return max(-(-staging // page), sink // page + -(-recent // page) + 1 + 2)


def _claim(arena, case, slots, keep, k_rot, v_rot):
    """A step's window write: the last token of a seat takes it, kept or as empty."""
    page, rows = case["page"], arena["owner"].shape[0]
    live = np.flatnonzero(slots >= 0)
    seats = (slots[live] // page % rows) * page + slots[live] % page
    seat, last = np.unique(seats[::-1], return_index=True)
    token = live[::-1][last]
    owner = np.where(keep[token], slots[token] // page, -1)
    arena["owner"].view(-1)[torch.from_numpy(seat).to(DEVICE)] = torch.from_numpy(owner).to(DEVICE)
    kept = keep[token]
    at, token = (torch.from_numpy(x[kept]).to(DEVICE) for x in (seat, token))
    for name, x in (("k", k_rot), ("v", v_rot)):
        arena[name].view(-1, *arena[name].shape[2:])[at] = x[token].to(arena[name].dtype)


def _kept(case, first, count, seq):
    """Which of the tokens at positions first .. first + count - 1 the window keeps."""
    pos = np.arange(first, first + count)
    return (pos >= seq - case["recent"]) | (pos < case["sink"] // case["page"] * case["page"])


def _world(case, seed):
    """The layer's state before the call and the call's inputs."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    host = np.random.RandomState(seed % (1 << 31))
    hq, hk, page = case["heads"], case["kv_heads"], case["page"]
    w = {"R_k": _rotation(2 * seed + 1), "R_v": _rotation(2 * seed + 2), "window": None}
    if case["kind"] == "write":
        n = case["tokens"]
        pages = n // page + 32
        slots = host.permutation(pages * page)[:n].astype(np.int64)
        slots[host.permutation(n)[:int(n * case["skipped"])]] = -1
    else:
        reqs = _requests(case)
        need = [-(-(n + h) // page) for n, h in reqs]
        pages = sum(need) + 3
        order = host.permutation(pages)
        table = np.zeros((len(reqs), max(need)), dtype=np.int32)
        at = 0
        for i, c in enumerate(need):
            table[i, :c] = order[at:at + c]
            at += c
    w["caches"] = [torch.zeros(pages, page, hk, case["slot"], dtype=torch.int8, device=DEVICE) if case["slot"] == D
                   else torch.zeros(pages, page, hk, case["slot"] // 2, dtype=torch.bfloat16, device=DEVICE)
                   for _ in range(2)]
    if case["kind"] == "write":
        w["k"], w["v"] = _kv(g, n, hk)
        w["slots"] = torch.from_numpy(slots).to(DEVICE)
        return w
    w["reqs"], w["table"] = reqs, table
    rows = _window_rows(case)
    if rows:
        w["window"] = {n: torch.zeros(rows, page, hk, D, device=DEVICE) for n in ("k", "v")}
        w["window"]["owner"] = torch.full((rows, page), -1, dtype=torch.int64, device=DEVICE)
    only = case["kind"] == "decode_only"
    rk, rv = w["R_k"].double(), w["R_v"].double()
    for (n, h), row in zip(reqs, table):
        h += n if only else 0
        if h == 0:
            continue
        k, v = _kv(g, h, hk)
        k_rot, v_rot = (k.double() @ rk).float(), (v.double() @ rv).float()
        slots = _slots(row, 0, h, page)
        _store(w["caches"], torch.from_numpy(slots).to(DEVICE), k_rot, v_rot, case)
        if rows:
            _claim(w["window"], case, slots, _kept(case, 0, h, h), k_rot, v_rot)
    new = sum(n for n, _ in reqs)
    w["q"] = _normal(g, new, hq, D).to(torch.bfloat16)
    w["starts"] = [0]
    for n, _ in reqs:
        w["starts"].append(w["starts"][-1] + n)
    w["seqs"] = [n + h for n, h in reqs]
    slots = np.concatenate([_slots(row, h, n, page) for (n, h), row in zip(reqs, table)])
    w["slots"] = torch.from_numpy(slots).to(DEVICE)
    w["k"], w["v"] = (None, None) if only else _kv(g, new, hk)
    return w


def _slots(row, first, count, page):
    pos = np.arange(first, first + count)
    return row[pos // page].astype(np.int64) * page + pos % page


# ------------------------------------------------------------------ the framework
def prepare(case, seed):
    from oscar_amd.backend import OscarAttentionBackendImpl
    from oscar_amd.kernels import staging

    w = _world(case, seed)
    impl = OscarAttentionBackendImpl.__new__(OscarAttentionBackendImpl)
    impl.head_size, impl.num_kv_heads, impl.num_heads = D, case["kv_heads"], case["heads"]
    impl.scale = D ** -0.5
    impl.key_cache = impl.value_cache = None
    impl._oscar_setup()
    impl._oscar_cfg = dataclasses.replace(
        impl._oscar, k_clip_ratio=case["clip_k"], v_clip_ratio=case["clip_v"], sink_tokens=case["sink"],
        recent_tokens=case["recent"], staging_tokens=case["staging"])
    layer = SimpleNamespace(layer_name="model.layers.3.self_attn.attn", _oscar_rots=(w["R_k"], w["R_v"]))
    # What the engine's worker hooks do once, when it allocates the caches.
    impl._set_caches(w["caches"])
    impl._layer_rots(layer, torch.device(DEVICE))
    if w["window"] is not None:
        impl._ensure_staging(layer, w["caches"])
        layer._oscar_stage_k.copy_(w["window"]["k"])
        layer._oscar_stage_v.copy_(w["window"]["v"])
        layer._oscar_slot_owner.copy_(w["window"]["owner"])
        for image, x in zip((layer._oscar_stage_kimg, layer._oscar_stage_vimg),
                            staging.stage_images(layer._oscar_stage_k, layer._oscar_stage_v)):
            image.copy_(x)
    state = {"kind": case["kind"], "impl": impl, "layer": layer, "caches": w["caches"], "slots": w["slots"],
             "k": w["k"], "v": w["v"]}
    if case["kind"] != "write":
        state["q"] = w["q"]
        state["output"] = torch.empty(w["q"].shape[0], case["heads"] * D, dtype=torch.bfloat16, device=DEVICE)
        state["metadata"] = SimpleNamespace(
            num_actual_tokens=w["q"].shape[0], slot_mapping=w["slots"],
            query_start_loc_cpu=torch.tensor(w["starts"], dtype=torch.int32), seq_lens_list=list(w["seqs"]),
            block_tables=torch.from_numpy(w["table"]).to(DEVICE),
            attn_state=SimpleNamespace(name="DecodeOnly" if case["kind"] == "decode_only" else "ChunkedPrefill"))
    return state


def run(state):
    impl, layer, caches = state["impl"], state["layer"], state["caches"]
    if state["kind"] == "write":
        impl.do_kv_cache_update(layer, state["k"], state["v"], caches, state["slots"])
        return {"k_cache": caches[0].view(torch.uint8), "v_cache": caches[1].view(torch.uint8)}
    output = impl.forward(layer, state["q"], state["k"], state["v"], caches, state["metadata"],
                          output=state["output"])
    if state["kind"] == "decode_only":
        return {"output": output}
    got = {"output": output, "k_cache": caches[0].view(torch.uint8), "v_cache": caches[1].view(torch.uint8)}
    if hasattr(layer, "_oscar_stage_k"):
        got.update(stage_k=layer._oscar_stage_k, stage_v=layer._oscar_stage_v, owner=layer._oscar_slot_owner)
    return got


def exact(case, seed):
    if case["kind"] == "write":
        return None                   # bytes only
    w = _world(case, seed)
    hq, hk, page = case["heads"], case["kv_heads"], case["page"]
    group = hq // hk
    only = case["kind"] == "decode_only"
    rk, rv = w["R_k"].double(), w["R_v"].double()
    q = w["q"].double() @ rk
    window = w["window"]
    if not only:
        k_new, v_new = w["k"].double() @ rk, w["v"].double() @ rv
        if window is not None:
            window = {n: x.double() if n != "owner" else x for n, x in window.items()}
            keep = np.concatenate([_kept(case, h, n, n + h) for n, h in w["reqs"]])
            _claim(window, case, w["slots"].cpu().numpy(), keep, k_new, v_new)
    out = torch.empty(q.shape[0], hq, D, dtype=torch.float64, device=DEVICE)
    for (n, h), row, a in zip(w["reqs"], w["table"], w["starts"]):
        h += n if only else 0
        slots = torch.from_numpy(_slots(row, 0, h, page)).to(DEVICE)
        keys, values = _load(w["caches"], slots)
        if window is not None:
            pages = slots // page
            seat = (pages % window["owner"].shape[0]) * page + slots % page
            mine = window["owner"].view(-1)[seat] == pages
            if only:
                mine = _window_segments(case, mine)
            keys[mine] = window["k"].view(-1, hk, D)[seat[mine]].double()
            values[mine] = window["v"].view(-1, hk, D)[seat[mine]].double()
        if not only:
            keys, values = torch.cat((keys, k_new[a:a + n])), torch.cat((values, v_new[a:a + n]))
        step = max(1, (1 << 26) // (group * max(1, h + n)))
        for t in range(0, n, step):
            m = min(step, n - t)
            seen = h if only else h + t + m
            position = torch.arange(seen, device=DEVICE)
            last = torch.arange(t, t + m, device=DEVICE).repeat_interleave(group) + (n if only else 1) + h - 1
            for c in range(hk):
                qs = q[a + t:a + t + m, c * group:(c + 1) * group].reshape(-1, D)
                s = (qs @ keys[:seen, c].t().contiguous()) * D ** -0.5
                s.masked_fill_(position > last[:, None], -math.inf)
                o = torch.softmax(s, -1) @ values[:seen, c].contiguous()
                out[a + t:a + t + m, c * group:(c + 1) * group] = o.view(m, group, D)
    got = {"output": (out @ rv.t().contiguous()).reshape(q.shape[0], hq * D)}
    if only:
        return got
    got.update(k_cache=None, v_cache=None)
    if window is not None:
        got.update(stage_k=window["k"], stage_v=window["v"], owner=None)
    return got


def _window_segments(case, mine):
    """The DecodeOnly read's window: the sink if all of it is staged, and the staged run up to the last position."""
    staged = mine.cpu().numpy()
    seq, sink = staged.size, case["sink"] // case["page"] * case["page"]
    head = sink if 0 < sink < seq and staged[:sink].all() else 0
    cut = seq
    while cut > max(seq - case["recent"], head) and staged[cut - 1]:
        cut -= 1
    keep = np.zeros(seq, dtype=bool)
    keep[:head] = True
    keep[cut:] = True
    return mine & torch.from_numpy(keep).to(DEVICE)
