"""The library's work as its users have it done, case by case, for timing.

A case is a dict of plain values; ``kind`` says which path of the library it takes:

``columns_step``   training step of the attention core on Sentinel's own matrices, fp32 ``[(head*d + dim), column]``, with
                   exact fp32 or 16-bit arithmetic (``HipFlashAttention``);
``native_step``    training step on contiguous ``[B, H, T, d]`` tensors, with or without the sparse mask;
``native_forward`` forward pass alone (prompt processing, evaluation);
``decode``         attention of one new token against a K/V cache (generation);
``dense_step``     masked softmax and its backward of the layer's dense path (flash attention switched off).

``listed()`` are representative shapes, ``draw()`` gives others of the same ranges.
"""
import math

import torch

from sentinel_amd import (HipFlashAttention, HipOps, decode_attention, flash_attention_backward, flash_attention_forward,
                          load_library)

_DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
_DTYPE_CODES = {"fp32": 0, "bf16": 1, "fp16": 2}


def _columns(name, q_heads, kv_heads, head_dim, seq_len, packs, compute, rope, keep):
    return dict(name=name, kind="columns_step", q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, seq_len=seq_len,
                packs=packs, compute=compute, rope=rope, keep=keep)


def _native(name, kind, batch, q_heads, kv_heads, seq_len, head_dim, dtype, sigma=1.0, window=0, global_tokens=0):
    return dict(name=name, kind=kind, batch=batch, q_heads=q_heads, kv_heads=kv_heads, seq_len=seq_len, head_dim=head_dim,
                dtype=dtype, sigma=sigma, window=window, global_tokens=global_tokens)


def _decode(name, q_heads, kv_heads, head_dim, length, capacity, window=0, global_tokens=0):
    return dict(name=name, kind="decode", q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, length=length,
                capacity=capacity, window=window, global_tokens=global_tokens)


def listed():
    return [
        # the quickstart language model: the smallest step there is, launches and host work decide
        _columns("quickstart_fp32_step", 4, 4, 16, 48, 4, "fp32", True, False),
        # a 768-wide 12-head layer at 256 tokens, packed to 4096 tokens a step, in the arithmetic a caller gets by default
        _columns("layer_fp32_step", 12, 12, 64, 256, 16, "fp32", True, False),
        # the shape Sentinel trains with: rotation fused, the forward's 16-bit operands kept for the backward
        _columns("gpt2_columns_step", 12, 12, 64, 1024, 8, "bf16", True, True),
        # grouped heads, a head dim between the kernels' tilings, sequences that end in mid-tile, nothing kept
        _columns("ragged_columns_step", 12, 4, 80, 333, 6, "fp16", True, False),
        # fine-tuning on short, odd-length sequences with 16-bit tensors
        _native("short_native_step", "native_step", 8, 16, 16, 509, 128, "bf16"),
        # the headline workload
        _native("target_native_step", "native_step", 4, 32, 32, 4096, 128, "bf16"),
        # prompt of one user through a grouped-query model
        _native("gqa_prefill", "native_forward", 1, 32, 8, 3001, 128, "bf16"),
        # long-context training, sharp scores
        _native("long_native_step", "native_step", 1, 16, 16, 16384, 64, "fp16", sigma=3.0),
        # sliding window with global tokens
        _native("window_native_step", "native_step", 4, 32, 32, 4096, 128, "bf16", window=512, global_tokens=64),
        # generation early in a small model's context: two launches and the host's work
        _decode("decode_small", 12, 12, 64, 1021, 2048),
        # generation deep in a large grouped-query model's context: the cache's bytes
        _decode("decode_long", 32, 8, 128, 32768, 32768),
        # the layer with flash attention off: score matrices of 12 heads x 16 packed sequences
        dict(name="dense_step", kind="dense_step", matrices=192, keys=256, queries=256, window=0, global_tokens=0),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("columns_fp32", "columns_16bit", "native_step", "native_forward", "window", "decode", "dense"))
    if kind == "columns_fp32":
        # the last number: lengths up to it stay within the time of the largest listed case
        q_heads, kv_heads, head_dim, longest = rng.choice(((4, 4, 16, 1024), (8, 8, 32, 768), (12, 12, 64, 384), (12, 4, 64, 192),
                                                           (6, 6, 40, 384), (8, 8, 128, 96)))
        seq_len = _log_int(rng, 16, longest)
        packs = max(1, min(32, rng.randint(1, max(1, 4096 // seq_len))))
        case = _columns("", q_heads, kv_heads, head_dim, seq_len, packs, "fp32", rng.random() < 0.5, False)
    elif kind == "columns_16bit":
        q_heads, kv_heads, head_dim = rng.choice(((12, 12, 64), (16, 16, 64), (12, 4, 64), (16, 8, 128), (12, 12, 96), (12, 4, 80)))
        seq_len = _log_int(rng, 64, 2048)
        packs = max(1, min(64, rng.randint(1, max(1, 16384 // seq_len))))
        case = _columns("", q_heads, kv_heads, head_dim, seq_len, packs, rng.choice(("bf16", "fp16")), rng.random() < 0.7,
                        rng.random() < 0.5)
    elif kind in ("native_step", "native_forward", "window"):
        q_heads, kv_heads, head_dim = rng.choice(((12, 12, 64), (16, 16, 64), (16, 4, 64), (32, 32, 128), (32, 8, 128), (16, 16, 128)))
        seq_len = _log_int(rng, 64 if kind != "window" else 512, 8192)
        # at most 16384 tokens, and no more work than the largest listed case has
        most = min(16384 // seq_len, (4 * 32 * 128 * 4096 ** 2) // (q_heads * head_dim * seq_len ** 2))
        batch = max(1, min(16, rng.randint(1, max(1, most))))
        window = global_tokens = 0
        if kind == "window":
            window = _log_int(rng, 64, seq_len // 2)
            global_tokens = rng.choice((0, 0, 1, 16, 64))
        case = _native("", "native_forward" if kind == "native_forward" else "native_step", batch, q_heads, kv_heads, seq_len,
                       head_dim, rng.choice(("bf16", "bf16", "fp16")), 1.0, window, global_tokens)
    elif kind == "decode":
        q_heads, kv_heads, head_dim = rng.choice(((12, 12, 64), (16, 16, 64), (32, 32, 128), (32, 8, 128), (16, 2, 128), (12, 6, 80)))
        length = _log_int(rng, 16, 32768 if kv_heads <= 8 else 16384)
        capacity = length + rng.randint(0, 255)
        if rng.random() < 0.75:  # caches are usually allocated in round sizes
            capacity = (capacity + 63) // 64 * 64
        window = _log_int(rng, 64, 4096) if rng.random() < 0.25 else 0
        case = _decode("", q_heads, kv_heads, head_dim, length, capacity, window, rng.choice((0, 16)) if window else 0)
    else:
        tokens = _log_int(rng, 16, 1024)
        matrices = max(1, min(512, rng.randint(1, max(1, (1 << 25) // (tokens * tokens)))))
        case = dict(kind="dense_step", matrices=matrices, keys=tokens, queries=tokens,
                    window=_log_int(rng, 8, 256) if rng.random() < 0.25 else 0, global_tokens=0)
    case.pop("name", None)
    return case


def _generator(seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(0x5E17 + seed)
    return gen


def _rope_tables(positions, head_dim):
    position = torch.arange(positions, device="cuda", dtype=torch.float32)[:, None]
    frequency = torch.pow(torch.tensor(10000.0, device="cuda"), -2.0 * torch.arange(head_dim // 2, device="cuda") / head_dim)[None, :]
    return torch.cos(position * frequency).contiguous(), torch.sin(position * frequency).contiguous()


def prepare(case, seed):
    gen = _generator(seed)
    state = {"case": case}

    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=gen)

    if case["kind"] == "columns_step":
        hq, hkv, d, t, packs = (case[k] for k in ("q_heads", "kv_heads", "head_dim", "seq_len", "packs"))
        columns = packs * t
        state["q"], state["g"] = normal(hq * d, columns), normal(hq * d, columns)
        state["k"], state["v"] = normal(hkv * d, columns), normal(hkv * d, columns)
        state["rope"] = _rope_tables(t, d) if case["rope"] else None
        # what the layer keeps from step to step: result matrices and the 16-bit workspace
        for name, like in (("out", "q"), ("dq", "q"), ("dk", "k"), ("dv", "v")):
            state[name] = torch.zeros_like(state[like])
        state["lse"] = torch.zeros(hq, columns, device="cuda")
        state["delta"] = torch.zeros(hq, columns, device="cuda")
        need = load_library().sentinel_hip_flash_workspace_bytes(0, _DTYPE_CODES[case["compute"]], 0, hq, hkv, d, t, packs, 1)
        state["workspace"] = torch.empty(need, dtype=torch.uint8, device="cuda") if need else None
    elif case["kind"] in ("native_step", "native_forward"):
        b, hq, hkv, t, d = (case[k] for k in ("batch", "q_heads", "kv_heads", "seq_len", "head_dim"))
        dtype = _DTYPES[case["dtype"]]
        state["q"] = (case["sigma"] * normal(b, hq, t, d)).to(dtype)
        state["k"] = (case["sigma"] * normal(b, hkv, t, d)).to(dtype)
        state["v"] = normal(b, hkv, t, d).to(dtype)
        state["out"] = torch.empty_like(state["q"])
        state["lse"] = torch.empty(b, hq, t, device="cuda")
        if case["kind"] == "native_step":
            state["g"] = normal(b, hq, t, d).to(dtype)
            for name, like in (("dq", "q"), ("dk", "k"), ("dv", "v")):
                state[name] = torch.empty_like(state[like])
            state["delta"] = torch.empty(hq, b * t, device="cuda")
    elif case["kind"] == "decode":
        hq, hkv, d = case["q_heads"], case["kv_heads"], case["head_dim"]
        state["q"] = normal(hq * d, 1)
        state["k"], state["v"] = normal(hkv * d, case["capacity"]), normal(hkv * d, case["capacity"])
        state["out"] = torch.empty(hq * d, 1, device="cuda")
        # a generation loop allocates its scratch once, for the longest context it will see
        need = load_library().sentinel_hip_decode_workspace_bytes(hq, d, case["capacity"])
        short = load_library().sentinel_hip_decode_workspace_bytes(hq, d, case["length"])
        state["workspace"] = torch.empty(max(need, short, 16), dtype=torch.uint8, device="cuda")
    else:
        shape = (case["matrices"], case["keys"], case["queries"])
        state["raw_scores"], state["raw_gradient"] = 8.0 * normal(*shape), normal(*shape)
        state["scores"], state["gradient"] = torch.empty(shape, device="cuda"), torch.empty(shape, device="cuda")
    return state


def _run_columns_step(s):
    c = s["case"]
    hq, hkv, d, t = c["q_heads"], c["kv_heads"], c["head_dim"], c["seq_len"]
    geometry = (hq, d, 1.0 / math.sqrt(d), True, 0, t, c["packs"])
    options = dict(kv_head_count=hkv)
    if c["compute"] != "fp32":
        options.update(compute=c["compute"], workspace=s["workspace"], rope=s["rope"])
    out, lse = HipFlashAttention.forward_multi_head(s["q"], s["k"], s["v"], s["out"], s["lse"], *geometry,
                                                    keep_for_backward=c["keep"], **options)
    dq, dk, dv, _ = HipFlashAttention.backward_multi_head(s["q"], s["k"], s["v"], out, lse, s["g"], s["dq"], s["dk"], s["dv"],
                                                          s["delta"], *geometry, reuse_forward_workspace=c["keep"], **options)
    if s["rope"] is not None and c["compute"] == "fp32":
        # exact arithmetic rotates in passes of its own; Q and K come rotated (where the projections wrote them), the
        # gradients are rotated back here
        HipOps.rotary_rotate_inverse_in_place(dq, hq, d, d // 2, *s["rope"], 0, t)
        HipOps.rotary_rotate_inverse_in_place(dk, hkv, d, d // 2, *s["rope"], 0, t)
    return out, lse, dq, dk, dv


def run(state):
    s, c = state, state["case"]
    if c["kind"] == "columns_step":
        return _run_columns_step(s)
    if c["kind"] in ("native_step", "native_forward"):
        mask = dict(window_size=c["window"], global_token_count=c["global_tokens"])
        out, lse = flash_attention_forward(s["q"], s["k"], s["v"], out=s["out"], lse=s["lse"], **mask)
        if c["kind"] == "native_forward":
            return out, lse
        dq, dk, dv = flash_attention_backward(s["q"], s["k"], s["v"], out, lse, s["g"], dq=s["dq"], dk=s["dk"], dv=s["dv"],
                                              delta=s["delta"], **mask)
        return out, lse, dq, dk, dv
    if c["kind"] == "decode":
        return decode_attention(s["q"], s["k"], s["v"], c["length"], c["q_heads"], c["head_dim"], kv_head_count=c["kv_heads"],
                                window_size=c["window"], global_token_count=c["global_tokens"], out=s["out"],
                                workspace=s["workspace"])
    # the copies stand for the matrix products that write the scores and their gradient, which the calls then overwrite
    s["scores"].copy_(s["raw_scores"])
    s["gradient"].copy_(s["raw_gradient"])
    scale = 1.0 / 8.0
    HipOps.masked_softmax_in_place(s["scores"], scale, c["window"], c["global_tokens"])
    HipOps.masked_softmax_backward_in_place(s["scores"], s["gradient"], scale, c["window"], c["global_tokens"])
    return s["scores"], s["gradient"]


def _visible_pairs(length, window, global_tokens):
    """(query, key) pairs of one causal sequence under the sparse mask."""
    if window <= 0 or window >= length:
        return length * (length + 1) // 2
    return sum(min(i + 1, window) + min(global_tokens, max(i + 1 - window, 0)) for i in range(length))


def work(case):
    c = case
    if c["kind"] == "decode":
        visible = c["length"]
        if 0 < c["window"] < c["length"]:
            visible = c["window"] + min(c["global_tokens"], c["length"] - c["window"])
        return {"bytes": 4.0 * (2 * c["kv_heads"] * c["head_dim"] * visible + 2 * c["q_heads"] * c["head_dim"]),
                "flops": 4.0 * c["q_heads"] * c["head_dim"] * visible}
    if c["kind"] == "dense_step":
        elements = float(c["matrices"]) * c["keys"] * c["queries"]
        return {"bytes": 16.0 * elements, "flops": 12.0 * elements}
    batch = c.get("batch", c.get("packs"))
    window, global_tokens = c.get("window", 0), c.get("global_tokens", 0)
    size = 4 if c["kind"] == "columns_step" or c["dtype"] == "fp32" else 2
    q_elements = float(batch) * c["q_heads"] * c["seq_len"] * c["head_dim"]
    kv_elements = float(batch) * c["kv_heads"] * c["seq_len"] * c["head_dim"]
    rows = float(batch) * c["q_heads"] * c["seq_len"]
    pairs = float(batch) * c["q_heads"] * _visible_pairs(c["seq_len"], window, global_tokens)
    if c["kind"] == "native_forward":  # Q, K, V in; O, LSE out; two products
        return {"bytes": size * (2 * q_elements + 2 * kv_elements) + 4 * rows, "flops": 4.0 * c["head_dim"] * pairs}
    # Q, K, V, dO in; O, LSE, dQ, dK, dV out; two products forward and five backward
    return {"bytes": size * (4 * q_elements + 4 * kv_elements) + 4 * rows, "flops": 14.0 * c["head_dim"] * pairs}


def tolerance(case):
    arithmetic = case.get("compute", case.get("dtype", "fp32"))
    # 32-bit sums; one rounding of operands, probabilities and results to 8 (bf16) or 11 (fp16) bits
    return {"rel": {"fp32": 1e-5, "bf16": 1e-2, "fp16": 3e-3}[arithmetic]}
