"""The calls whose time matters, as a program that serves diffusion transformers makes them.

Six kinds of work, all through the package's public names:

  attention  wrapper.run() over packed symbols (decode of the symbols and block-sparse attention)
  gemm_q     flashomni_gemm: the Q projection of the token blocks and heads that are not cached
  gemm_o     flashomni_gemm_reduction: the output projection, cache pass and final pass
  layer      one sparse step of a layer: GEMM-Q, wrapper.run(), GEMM-O's final pass
  update     one full step that renews what the sparse steps reuse: dense GEMM-Q, dense attention,
             new symbols from pooled scores, both passes of GEMM-O
  pack       segment_packbits of the two boolean maps that a mask policy produced

Heads are 128 wide and blocks 128 x 128.  Symbols are random where a policy chose them by score and
have the local windows of video models where "frame" is given; text tokens come first and their key
blocks are always kept.
"""
import math

import torch

import flashomni_amd as fo

BLOCK = 128
DIM = 128
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _attention(name, qo, kv, heads, kv_heads=None, dtype="bf16", p_cached=0.25, p_keep=0.5, text=512, frame=0,
               layout="NHD", lse=False, plan=False):
    return {"name": name, "kind": "attention", "qo": qo, "kv": kv, "heads": heads, "kv_heads": kv_heads or heads,
            "dtype": dtype, "p_cached": p_cached, "p_keep": p_keep, "text": text, "frame": frame, "layout": layout,
            "lse": lse, "plan": plan}


def _dense(name, kind, batch, tokens, heads, dtype="bf16", p_cached=0.25, p_keep=0.5, text=512, frame=0, fp8=False,
           skip_text=0):
    return {"name": name, "kind": kind, "batch": batch, "tokens": tokens, "heads": heads, "dtype": dtype,
            "p_cached": p_cached, "p_keep": p_keep, "text": text, "frame": frame, "fp8": fp8,
            "skip_text": skip_text}


def listed():
    return [
        # a first call, a unit test, a tiny model: nothing but latency
        _attention("attention_small", "384", "384", 2, text=128),
        # an image transformer's layer: 4096 image and 512 text tokens
        _attention("attention_flux", "4608", "4608", 24),
        # high-resolution image, fp16, no cached block and 80 % of the key blocks skipped
        _attention("attention_image_16k", "16896", "16896", 24, dtype="fp16", p_cached=0.0, p_keep=0.2, text=0),
        # video: eight frames of 64 x 64 latent patches, windows in space and time
        _attention("attention_video_33k", "33280", "33280", 24, p_cached=0.3, p_keep=0.05, frame=4096),
        # requests of uneven lengths, grouped-query heads, planned anew for each batch, with log-sum-exp
        _attention("attention_ragged_gqa", "1000,129,300,1", "1100,64,77,513", 8, kv_heads=2, dtype="fp16",
                   text=0, lse=True, plan=True),
        # the image stream's Q projection late in sampling: nine tiles of ten come from the cache
        _dense("gemm_q_image_16k", "gemm_q", 1, 16384, 24, p_cached=0.9, skip_text=512),
        # output projection of an image layer: what the cached heads give, then the rest added to it
        _dense("gemm_o_flux", "gemm_o", 1, 4608, 24),
        # a small model at low resolution, conditional and unconditional request in one batch
        _dense("layer_small_pair", "layer", 2, 1100, 8, text=128),
        # one sparse step of an image transformer's layer
        _dense("layer_flux", "layer", 1, 4608, 24),
        # one sparse step of a large video model's layer, q and k as two-term fp8
        _dense("layer_video_76k_fp8", "layer", 1, 76112, 40, p_cached=0.2, p_keep=0.02, frame=3600, fp8=True),
        # the full step of an image transformer's layer, every few sampling steps
        _dense("update_flux", "update", 1, 4608, 24),
        # masks of a video layer from a policy outside this package
        _dense("pack_video_33k", "pack", 1, 33280, 24, p_cached=0.3, p_keep=0.05, frame=4096),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["attention", "attention", "gemm_q", "gemm_o", "layer", "layer", "update", "pack"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    heads = rng.choice([2, 3, 4, 8, 12, 16, 24, 40])
    p_cached = round(rng.uniform(0.0, 0.9), 2)
    p_keep = round(math.exp(rng.uniform(math.log(0.02), math.log(0.8))), 3)
    if kind == "attention":
        count = rng.choice([1, 1, 1, 2, 3, 5])
        high = min(33280, 800000 // heads) // count
        qo = [_log_int(rng, 100, high) for _ in range(count)]
        ragged = rng.random() < 0.3
        kv = [_log_int(rng, 60, high) for _ in range(count)] if ragged else qo
        group = rng.choice([1, 1, 1, 2, 4]) if heads % 4 == 0 else 1
        return _drawn(_attention("", ",".join(map(str, qo)), ",".join(map(str, kv)), heads, heads // group, dtype,
                                 p_cached, p_keep, rng.choice([0, 128, 512]),
                                 rng.choice([0, 0, 1560, 3600, 4096]) if count == 1 and not ragged else 0,
                                 rng.choice(["NHD", "NHD", "NHD", "HND"]), rng.random() < 0.3, rng.random() < 0.3))
    batch = rng.choice([1, 1, 1, 2])
    tokens = _log_int(rng, 300, min(40000, (300000 if kind == "update" else 1000000) // heads) // batch)
    video = tokens > 16000
    return _drawn(_dense("", kind, batch, tokens, heads, dtype, p_cached, min(p_keep, 0.2) if video else p_keep,
                         rng.choice([t for t in (128, 256, 512) if 2 * t <= tokens]), rng.choice([1560, 3600, 4096]) if video else 0,
                         kind == "layer" and dtype == "bf16" and rng.random() < 0.3,
                         rng.choice([0, 512]) if kind == "gemm_q" else 0))


def _drawn(case):
    del case["name"]
    return case


# ---- symbols ----------------------------------------------------------------------------------------
def _blocks(n):
    return -(-n // BLOCK)


def _lens(case):
    """(q tokens, kv tokens) of every request."""
    if case["kind"] == "attention":
        return list(zip(map(int, case["qo"].split(",")), map(int, case["kv"].split(","))))
    return [(case["tokens"] + case["skip_text"],) * 2] * case["batch"]


def _group(case):
    return case["heads"] // case.get("kv_heads", case["heads"])


def _kept(case, q_len, kv_len, device):
    """[q blocks, kv blocks] True where a key block is kept whatever its score."""
    group = _group(case)
    # the token that a symbol row begins with (with grouped heads a row packs `group` heads of a token)
    q_tok = torch.arange(_blocks(q_len * group), device=device) * BLOCK // group
    k_tok = torch.arange(_blocks(kv_len), device=device) * BLOCK
    kept = (q_tok[:, None] // BLOCK) == (k_tok[None, :] // BLOCK)
    kept |= k_tok[None, :] < case["text"]
    if case["frame"]:
        q_vid, k_vid = q_tok - case["text"], k_tok - case["text"]
        df = (q_vid[:, None] // case["frame"] - k_vid[None, :] // case["frame"]).abs()
        dp = ((q_vid % case["frame"])[:, None] // BLOCK - (k_vid % case["frame"])[None, :] // BLOCK).abs()
        video = (q_vid[:, None] >= 0) & (k_vid[None, :] >= 0)
        kept |= video & ((df == 0) | ((df == 1) & (dp <= 2)))
    return kept


def _maps(case, gen):
    """The boolean maps of all requests, flat and one after the other, and where each request's begin."""
    heads = case["heads"] // _group(case)
    flags, keeps, flag_ip, keep_ip = [], [], [0], [0]
    for q_len, kv_len in _lens(case):
        kept = _kept(case, q_len, kv_len, gen.device)
        rows, cols = kept.shape
        flags.append((torch.rand(rows, heads, generator=gen, device=gen.device) >= case["p_cached"]).view(-1))
        keep = torch.rand(rows, heads, cols, generator=gen, device=gen.device) < case["p_keep"]
        keeps.append((keep | kept[:, None, :]).view(-1))
        flag_ip.append(flag_ip[-1] + flags[-1].numel())
        keep_ip.append(keep_ip[-1] + keeps[-1].numel())
    ip = lambda v: torch.tensor(v, dtype=torch.int32, device=gen.device)
    return torch.cat(flags), ip(flag_ip), torch.cat(keeps), ip(keep_ip)


def _symbols(case, gen):
    flags, flag_ip, keep, keep_ip = _maps(case, gen)
    info, info_ip = fo.segment_packbits(flags, flag_ip, "little")
    kv_info, kv_ip = fo.segment_packbits(keep, keep_ip, "little")
    return {"info": info, "info_ip": info_ip, "kv_info": kv_info, "kv_ip": kv_ip}


# ---- what is in hand, and one pass -------------------------------------------------------------------
def _plan(state, dtype):
    state["wrapper"].plan(state["qo_ip"], state["kv_ip_tokens"], state["heads"], state["kv_heads"], DIM,
                          q_data_type=dtype)


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    rand = lambda *shape, std=1.0: (torch.randn(*shape, generator=gen, device=dev) * std).to(dtype)
    kind, heads = case["kind"], case["heads"]
    state = {"case": case, "dtype": dtype, "heads": heads, "kv_heads": case.get("kv_heads", heads)}
    if kind == "pack":
        state["flags"], state["flag_ip"], state["keep"], state["keep_ip"] = _maps(case, gen)
        return state
    if kind != "update":
        state.update(_symbols(case, gen))
    if kind in ("attention", "layer", "update"):
        lens = _lens(case)
        ends = lambda v: torch.tensor([0] + v, dtype=torch.int32).cumsum(0).to(torch.int32)
        state["qo_ip"], state["kv_ip_tokens"] = ends([a for a, _ in lens]), ends([b for _, b in lens])
        workspace = torch.empty(128 << 20, dtype=torch.uint8, device=dev)
        state["wrapper"] = fo.BatchFlashOmniFAWithRaggedKVWrapper(workspace, case.get("layout", "NHD"))
        state["plan_dtype"] = torch.float8_e4m3fn if case.get("fp8") else dtype
        _plan(state, state["plan_dtype"])
        n_q, n_kv = int(state["qo_ip"][-1]), int(state["kv_ip_tokens"][-1])
        shape = (n_kv, state["kv_heads"], DIM)
        if case.get("layout") == "HND":
            shape = (shape[1], shape[0], DIM)
        state["k"], state["v"] = rand(*shape), rand(*shape)
        if kind == "attention":
            state["q"] = rand(n_q, heads, DIM)
            # kept between calls: rows of cached blocks stay as they are
            state["lse"] = torch.zeros(n_q, heads, device=dev) if case["lse"] else None
            return state
    hidden, batch, tokens = heads * DIM, case["batch"], case["tokens"]
    if kind in ("gemm_q", "layer", "update"):
        state["x"], state["w_q"], state["b_q"] = (rand(batch, tokens, hidden), rand(hidden, hidden, std=0.02),
                                                  rand(hidden, std=0.02))
    if kind in ("gemm_o", "layer", "update"):
        state["w_o"], state["b_o"] = rand(hidden, hidden, std=0.02), rand(hidden, std=0.02)
    if kind == "gemm_q":
        # the projection of the last step, whose cached tiles stay
        state["q"] = rand(batch, tokens, hidden)
    if kind == "gemm_o":
        state["a"] = rand(batch, tokens, hidden)
    if kind == "layer":
        # the cached heads' part of the output, as the last full step left it
        past = rand(batch, tokens, hidden, std=0.05)
        state["partial"] = fo.flashomni_gemm_reduction(past, state["w_o"], heads, state["info"], state["info_ip"], 0,
                                                       bias=state["b_o"], is_for_cache=True)
        if case["fp8"]:
            state["blocks"] = tuple(t.to(dev) for t in fo.token_blocks(state["kv_ip_tokens"]))
    if kind == "update":
        n = _blocks(tokens)
        state["pooled"] = torch.randn(batch, heads, n, n, generator=gen, device=dev) * 1.5
    return state


def run(state):
    s, case, heads = state, state["case"], state["heads"]
    kind = case["kind"]
    if kind == "attention":
        if case["plan"]:
            _plan(s, s["plan_dtype"])
        return s["wrapper"].run(s["q"], s["k"], s["v"], s["info"], s["kv_info"], s["info_ip"], s["kv_ip"],
                                lse=s["lse"], return_lse=case["lse"])
    if kind == "pack":
        return (fo.segment_packbits(s["flags"], s["flag_ip"], "little"),
                fo.segment_packbits(s["keep"], s["keep_ip"], "little"))
    if kind == "gemm_q":
        return fo.flashomni_gemm(s["x"], s["w_q"], heads, s["info"], s["info_ip"], case["skip_text"], s["b_q"],
                                 out=s["q"])
    if kind == "gemm_o":
        partial = fo.flashomni_gemm_reduction(s["a"], s["w_o"], heads, s["info"], s["info_ip"], 0, bias=s["b_o"],
                                              is_for_cache=True)
        return partial, fo.flashomni_gemm_reduction(s["a"], s["w_o"], heads, s["info"], s["info_ip"], 0,
                                                    bias=partial)
    if kind == "layer":
        symbols = (s["info"], s["kv_info"], s["info_ip"], s["kv_ip"])
        if case["fp8"]:
            k8, k_scale, k_lo = fo.quant_fp8_block(s["k"], s["kv_ip_tokens"], blocks=s["blocks"], residual=True)
            _, q8, q_scale, q_lo = fo.flashomni_gemm(s["x"], s["w_q"], heads, s["info"], s["info_ip"], 0, s["b_q"],
                                                     out=False, quant_out="residual")
            o = s["wrapper"].run(q8.view(-1, heads, DIM), k8, s["v"], *symbols, q_scale=q_scale, k_scale=k_scale,
                                 q_lo=q_lo.view(-1, heads, DIM), k_lo=k_lo)
        else:
            q = fo.flashomni_gemm(s["x"], s["w_q"], heads, s["info"], s["info_ip"], 0, s["b_q"])
            o = s["wrapper"].run(q.view(-1, heads, DIM), s["k"], s["v"], *symbols)
        return o, fo.flashomni_gemm_reduction(o.view(s["x"].shape), s["w_o"], heads, s["info"], s["info_ip"], 0,
                                              bias=s["partial"])
    q = fo.flashomni_gemm(s["x"], s["w_q"], heads, num_text_tokens=0, bias=s["b_q"], is_full=True)
    o = s["wrapper"].run(q.view(-1, heads, DIM), s["k"], s["v"], is_full=True)
    info, info_ip, kv_info, kv_ip = fo.sparse_symbols_from_scores(s["pooled"], _blocks(case["text"]), 0.2, 0.3)
    a = o.view(s["x"].shape)
    partial = fo.flashomni_gemm_reduction(a, s["w_o"], heads, info, info_ip, 0, bias=s["b_o"], is_for_cache=True)
    y = fo.flashomni_gemm_reduction(a, s["w_o"], heads, info, info_ip, 0, bias=partial)
    return o, y, partial, info, info_ip, kv_info, kv_ip


# ---- what a pass cannot do without --------------------------------------------------------------------
def work(case):
    """Expected over the random symbols: computed blocks, tiles and head slices only, every input that
    they need read once and every output written once."""
    kind, heads = case["kind"], case["heads"]
    active = 1.0 - case["p_cached"]
    group = _group(case)
    flag_bits = keep_bits = pairs = 0
    n_q = n_kv = 0
    for q_len, kv_len in _lens(case):
        kept = _kept(case, q_len, kv_len, "cpu").double()
        density = float((kept + (1 - kept) * case["p_keep"]).mean()) if kind != "update" else 1.0
        pairs += density * q_len * kv_len
        flag_bits += kept.shape[0] * heads // group
        keep_bits += kept.numel() * heads // group
        n_q, n_kv = n_q + q_len, n_kv + kv_len
    bits = (flag_bits + keep_bits) / 8
    if kind == "pack":
        return {"bytes": 9 * bits, "flops": 0}
    if kind == "attention":
        kv = 2 * 2 * n_kv * case["kv_heads"] * DIM
        return {"flops": 4 * DIM * heads * active * pairs,
                "bytes": 2 * (1 + active) * n_q * heads * DIM + kv + bits + (4 * n_q * heads if case["lse"] else 0)}
    rows, hidden = case["batch"] * case["tokens"], heads * DIM
    matrix, weight = 2 * rows * hidden, 2 * hidden * hidden
    product = 2 * rows * hidden * hidden
    if kind == "gemm_q":
        return {"flops": active * product, "bytes": (1 + active) * matrix + weight}
    if kind == "gemm_o":  # either pass reads its own heads' columns; the partial is written and read
        return {"flops": product, "bytes": 4 * matrix + weight}
    attention = 4 * DIM * heads * pairs
    if kind == "layer":   # x, k, v, partial in; o and y out
        return {"flops": active * (2 * product + attention), "bytes": 6 * matrix + 2 * weight + bits}
    scores = case["batch"] * heads * _blocks(case["tokens"]) ** 2
    return {"flops": 2 * product + attention, "bytes": 6 * matrix + 2 * weight + 4 * scores + bits}


def tolerance(case):
    """Bytes and indexes are the same.  Attention rounds its probabilities to the 16-bit type and every
    result once; a GEMM only its results."""
    if case["kind"] == "pack":
        return "exact"
    half = case["dtype"] == "fp16"
    if case["kind"] in ("gemm_q", "gemm_o"):
        return {"rel": 5e-4 if half else 4e-3}
    return {"rel": 2e-3 if half else 1e-2}
