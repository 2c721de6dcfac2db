"""The calls a serving program makes into this framework, as measurable cases.

A case names one pass through the Python entry points (`ggml_flash_attn_ext`, `kv_write`, `ggml_rope_ext`, `ggml_mul_mat`,
`FrontBatch`): an attention node of a decode step or of a prompt chunk, or a whole attention layer between the q / kv projections
and wo.  Shapes are DeepSeek-V2-Lite's (16 heads) and DeepSeek-V2's (128 heads, or what a tensor-parallel device holds of them),
rows of 576 latent + rotary values, pages of 128 tokens.

    decode    one query token per sequence; a block table over shuffled pages, or one contiguous cache (batch 1)
    shared    a decode batch over one cache without a block table: the f16 mask picks every token's cells
    prefill   a prompt chunk behind cached tokens under a causal f16 mask, paged (several sequences) or contiguous (one)
    layer     rope of q_pe, absorb product, rope of k_pe + cache write, attention, un-absorb product; decode or prompt chunk
"""
import math
import random

import torch

import jittorinfer_amd as J

SCALE = 1.0 / math.sqrt(192.0)
PAGE = 128
ROW = {"bf16": 1152, "f16": 1152, "q8_0": 612}
KV_TYPE = {"bf16": J.MLA_TYPE_BF16, "f16": J.MLA_TYPE_F16, "q8_0": J.MLA_TYPE_Q8_0}
DTYPE = {"bf16": torch.bfloat16, "f16": torch.float16}
ROPE = dict(n_dims=64, n_ctx_orig=4096, freq_scale=0.025, ext_factor=1.0, attn_factor=0.8)   # YaRN, as DeepSeek-V2 configures it


def _decode(name, batch, heads, lo, hi, kv, paged=True):
    return dict(name=name, kind="decode", batch=batch, heads=heads, lo=lo, hi=hi, kv=kv, paged=paged, new=1, lens_seed=7)


def _prefill(name, batch, heads, new, cached, kv, paged):
    return dict(name=name, kind="prefill", batch=batch, heads=heads, lo=cached, hi=cached, kv=kv, paged=paged, new=new, lens_seed=7)


def listed():
    return [
        # one user of the 16-head model, 1024 tokens in a contiguous cache of the default cache type: latency only
        _decode("decode_1x16_1k_f16", 1, 16, 1024, 1024, "f16", paged=False),
        # a small server of the 16-head model: 8 users, contexts of 512 to 4096 tokens
        _decode("decode_8x16_ragged_bf16", 8, 16, 512, 4096, "bf16"),
        # a full server of the 128-head model: 32 users at 8192 tokens
        _decode("decode_32x128_8k_bf16", 32, 128, 8192, 8192, "bf16"),
        # the same with a quantized cache, 64 users, ragged
        _decode("decode_64x128_ragged_q8", 64, 128, 2048, 8192, "q8_0"),
        # the 16-head model with a quantized cache, 64 users, ragged
        _decode("decode_64x16_ragged_q8", 64, 16, 2048, 8192, "q8_0"),
        # one user of the 128-head model deep in a long context
        _decode("decode_1x128_32k_bf16", 1, 128, 32768, 32768, "bf16"),
        # a decode batch as an unmodified graph builder presents it: one cache, the mask assigns cells to users
        dict(name="shared_32x16_8k_bf16", kind="shared", batch=32, heads=16, lo=8192, hi=8192, kv="bf16", paged=False, new=1, lens_seed=7),
        # chunked prefill, 4 users of the 16-head model: 512 new tokens behind 2048 cached ones
        _prefill("prefill_4x16_512_after_2048_bf16", 4, 16, 512, 2048, "bf16", True),
        # the first 512 tokens of a prompt, 128 heads, nothing cached yet
        _prefill("prefill_1x128_512_first_bf16", 1, 128, 512, 0, "bf16", False),
        # the ragged last chunk of a prompt, 128 heads, default cache type
        _prefill("prefill_1x128_333_after_4000_f16", 1, 128, 333, 4000, "f16", False),
        # one attention layer of a decode step, projections' output to wo's input: 32 users of the 128-head model
        dict(name="layer_32x128_8k_bf16", kind="layer", batch=32, heads=128, lo=8192, hi=8192, kv="bf16", paged=True, new=1, lens_seed=7),
        # one attention layer of a prompt of 2048 tokens, 16-head model
        dict(name="layer_1x16_2048_first_bf16", kind="layer", batch=1, heads=16, lo=0, hi=0, kv="bf16", paged=False, new=2048, lens_seed=7),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the same ranges; no dearer than the dearest listed one in bytes or in operations."""
    most = [work(c) for c in listed()]
    max_bytes, max_flops = max(w["bytes"] for w in most), max(w["flops"] for w in most)
    while True:
        kind = rng.choice(["decode"] * 4 + ["prefill"] * 3 + ["shared", "layer", "layer"])
        heads = rng.choice([16, 16, 32, 64, 128, 128])
        kv = rng.choice(["bf16", "bf16", "f16", "q8_0"])
        c = dict(kind=kind, heads=heads, kv=kv, lens_seed=rng.randrange(1 << 30), new=1, paged=True)
        if kind in ("decode", "shared"):
            c["batch"] = _log_int(rng, 1, 128) if kind == "decode" else _log_int(rng, 2, 64)
            c["hi"] = _log_int(rng, 128, 32768 if c["batch"] <= 4 else 8192)
            c["lo"] = c["hi"] if rng.random() < 0.3 else max(1, int(c["hi"] * rng.uniform(0.1, 0.9)))
            c["paged"] = kind == "decode" and not (c["batch"] == 1 and rng.random() < 0.5)
        elif kind == "prefill":
            c["batch"] = rng.choice([1, 1, 2, 3, 4])
            c["new"] = _log_int(rng, 16, 2048)
            c["lo"] = c["hi"] = rng.choice([0, _log_int(rng, 64, 8192)])
            c["paged"] = c["batch"] > 1
        else:
            c["kv"] = kv = rng.choice(["bf16", "f16"])
            if rng.random() < 0.6:
                c["batch"] = _log_int(rng, 1, 64)
                c["hi"] = _log_int(rng, 256, 8192)
                c["lo"] = max(1, int(c["hi"] * rng.uniform(0.1, 1.0)))
            else:
                c["batch"], c["new"], c["paged"] = 1, _log_int(rng, 32, 2048), False
                c["lo"] = c["hi"] = rng.choice([0, _log_int(rng, 64, 4096)])
        w = work(c)
        if w["bytes"] <= max_bytes and w["flops"] <= max_flops:
            return c


def _lens(case):
    """Keys every sequence's query tokens can see at most: cached tokens plus the new ones of a chunk (a decode step's length
    counts its own token)."""
    r = random.Random(case["lens_seed"])
    extra = case["new"] if case["new"] > 1 or case["kind"] == "prefill" else 0
    return [r.randint(case["lo"], case["hi"]) + extra for _ in range(case["batch"])]


def _causal(case):
    return case["kind"] == "prefill" or case["new"] > 1


def _cells(n):
    return (n + 31) // 32 * 32   # a contiguous cache ends on a multiple of 32 cells


def work(case):
    H, new, lens, row = case["heads"], case["new"], _lens(case), ROW[case["kv"]]
    n_q = case["batch"] * new
    if _causal(case):
        pairs = sum(new * (n - new) + new * (new + 1) // 2 for n in lens)
        mask = new * max(lens) * 2
    else:
        pairs, mask = sum(lens), 0
    if case["kind"] == "shared":
        mask = case["batch"] * sum(_cells(n) for n in lens) * 2
    flops = pairs * H * (2 * 576 + 2 * 512)
    nbytes = sum(lens) * row + mask
    if case["kind"] != "layer":
        return {"bytes": nbytes + n_q * H * (576 + 512) * 4, "flops": flops}
    weights = 2 * H * 512 * 128
    nbytes += weights * 2 + n_q * (H * (192 + 128) + 576) * 4 + n_q * row
    return {"bytes": nbytes, "flops": flops + 2 * n_q * weights}


def _q8_rows(x):
    """float32 [n, 576] -> Q8_0 rows [n, 612]: per block of 32 an f16 scale amax / 127 and 32 int8 values."""
    blocks = x.view(-1, 18, 32)
    d = (blocks.abs().amax(dim=2, keepdim=True) / 127.0)
    qs = torch.round(blocks / d.clamp_min(1e-20)).clamp_(-127, 127).to(torch.int8)
    out = torch.empty((x.shape[0], 18, 34), dtype=torch.uint8, device=x.device)
    out[:, :, :2] = d.to(torch.float16).view(torch.uint8).view(-1, 18, 2)
    out[:, :, 2:] = qs.view(torch.uint8)
    return out.view(-1, 612)


def _rows(g, n, kv, sigma):
    """n cache rows ~ N(0, sigma) in the storage type, made in pieces so that the float32 values never take much memory."""
    pieces = []
    for i in range(0, n, 65536):
        x = torch.randn((min(65536, n - i), 576), generator=g, device=g.device) * sigma
        pieces.append(_q8_rows(x) if kv == "q8_0" else x.to(DTYPE[kv]))
    return torch.cat(pieces)


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    B, H, new, kv = case["batch"], case["heads"], case["new"], case["kv"]
    lens = _lens(case)
    sigma = 0.5 if H == 128 else 1.0
    s = {"case": case, "mask": None, "block_table": None, "seq_lens": None}
    if case["paged"]:
        n_blocks = [(n + PAGE - 1) // PAGE for n in lens]
        perm = torch.randperm(sum(n_blocks), generator=g, device=dev).to(torch.int32)
        table = torch.zeros((B, max(n_blocks)), dtype=torch.int32, device=dev)
        at = 0
        for b, n in enumerate(n_blocks):
            table[b, :n] = perm[at:at + n]
            at += n
        s["block_table"], s["seq_lens"] = table, torch.tensor(lens, dtype=torch.int32, device=dev)
        s["cache"] = _rows(g, sum(n_blocks) * PAGE, kv, sigma)
    else:
        s["cache"] = _rows(g, sum(_cells(n) for n in lens), kv, sigma)
    if _causal(case):
        n = max(lens)
        width = n if case["paged"] else _cells(n)
        width = (width + 31) // 32 * 32
        key = torch.arange(width, device=dev)[None, :]
        s["mask"] = torch.where(key > (n - new) + torch.arange(new, device=dev)[:, None], float("-inf"), 0.0).to(torch.float16)
    elif case["kind"] == "shared":
        s["mask"] = torch.full(((B + 63) // 64 * 64, s["cache"].shape[0]), float("-inf"), dtype=torch.float16, device=dev)
        at = 0
        for b, n in enumerate(lens):
            s["mask"][b, at:at + n] = 0
            at += _cells(n)
    elif not case["paged"] and _cells(lens[0]) != lens[0]:
        # a contiguous cache that the sequence has not filled: the cells past its end are masked
        s["mask"] = torch.where(torch.arange(s["cache"].shape[0], device=dev)[None, :] >= lens[0], float("-inf"), 0.0).to(torch.float16)
    n_seq, n_tok = (1, B) if case["kind"] == "shared" else (B, new)
    s["out"] = torch.empty((n_seq, n_tok, H, 512), dtype=torch.float32, device=dev)
    if case["kind"] == "layer":
        T = B * new
        s["q_proj"] = torch.randn((T, H, 192), generator=g, device=dev)
        s["kv_new"] = torch.randn((T, 576), generator=g, device=dev) * sigma
        s["wkv_b"] = (torch.randn((2 * H * 512 * 128,), generator=g, device=dev) * 0.05).to(DTYPE[kv]).view(torch.int16)
        s["q"] = torch.empty((H, T, 576), dtype=torch.float32, device=dev)
        s["cur"] = torch.empty((T, H, 128), dtype=torch.float32, device=dev)
        if new == 1:
            s["pos"] = (s["seq_lens"] - 1).contiguous()
            s["seq_ids"] = torch.arange(B, dtype=torch.int32, device=dev)
        else:
            s["pos"] = torch.arange(lens[0] - new, lens[0], dtype=torch.int32, device=dev)
    else:
        s["q"] = torch.randn((n_seq, H, n_tok, 576), generator=g, device=dev)
    return s


def _attention(s, q):
    kv = s["case"]["kv"]
    cache = s["cache"] if s["case"]["paged"] else s["cache"].unsqueeze(0)
    return J.ggml_flash_attn_ext(q, cache, KV_TYPE[kv], dv=512, mask=s["mask"], scale=SCALE, block_table=s["block_table"],
                                 seq_lens=s["seq_lens"], out=s["out"])


def _layer(s):
    case = s["case"]
    H, kvt, decode = case["heads"], KV_TYPE[case["kv"]], case["new"] == 1
    q_proj, q, half = s["q_proj"], s["q"], H * 512 * 128
    where = dict(block_table=s["block_table"], seq_ids=s["seq_ids"], positions=s["pos"]) if decode else dict(row0=case["lo"])
    batch = J.FrontBatch()
    J.ggml_rope_ext(q_proj[:, :, 128:], s["pos"], out=q[:, :, 512:].permute(1, 0, 2), batch=batch, **ROPE)
    J.ggml_mul_mat(s["wkv_b"][:half].view(H, 512, 128), kvt, q_proj[:, :, :128].permute(1, 0, 2), out=q[:, :, :512], batch=batch)
    J.kv_write(s["kv_new"], s["cache"], kvt, k_pe=s["kv_new"][:, 512:], rope=dict(pos=s["pos"], **ROPE), batch=batch, **where)
    batch.launch()
    out = _attention(s, q.permute(1, 0, 2).unsqueeze(2) if decode else q.unsqueeze(0))
    rows = out[:, 0] if decode else out[0]
    J.ggml_mul_mat(s["wkv_b"][half:].view(H, 128, 512), kvt, rows.permute(1, 0, 2), out=s["cur"].permute(1, 0, 2))
    return s["cur"], s["cache"]


def run(s):
    return _layer(s) if s["case"]["kind"] == "layer" else _attention(s, s["q"])


def tolerance(case):
    # About four times what the paths show against the same operands in 64 bits (1.4e-4 to 2.5e-4 for 16-bit caches, whose
    # probabilities and split partials are 16-bit; 3e-4 to 5e-4 for Q8_0, where q * d of K, V and Q is rounded to a 16-bit operand).
    # The un-absorb product of a layer rounds the attention rows to bf16 first, and a row that differs in its last f32 bits may round
    # the other way there (7e-4).
    if case["kv"] == "q8_0":
        return {"rel": 2e-3, "max": 1.5e-2}
    if case["kind"] == "layer" and case["kv"] == "bf16":
        return {"rel": 3e-3, "max": 1.8e-2}
    return {"rel": 1e-3, "max": 6e-3}
