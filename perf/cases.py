"""The calls that the framework is timed on.

Each case is one thing a user's program does with this package, at sizes of
the Qwen3-32B projections and of the tests: from 16 decode tokens to a prefill of
8 x 1024, both GEMM arms (the tile-local Strassen product and its matched cubic),
the fused epilogues, FP32 inputs, the weight gradient, and one whole decoder
block. Weights are packed once, as a program that serves or trains with them
keeps them; activations and gradients arrive new in every pass and are packed
inside it.
"""

import math

import torch

import strassen_tpu_amd as smx
from strassen_tpu_amd import qwen3_block as qb

DEVICE = "cuda:0"
HEAD_DIM = 128
THETA, EPS = 1e6, 1e-6


def _gemm(name, algo, m, k, n, tile, epilogue):
    bm, bn, bk = tile
    return {"name": name, "kind": "gemm", "algo": algo, "m": m, "k": k, "n": n, "bm": bm, "bn": bn, "bk": bk,
            "epilogue": epilogue}


def listed():
    return [
        # One decode step of 16 sequences through an MLP's gate|up projection.
        _gemm("decode_16_gate_up", "strassen", 16, 5120, 51200, (16, 1024, 512), "swiglu"),
        # The cubic arm on 48 decode rows through an 8192-wide projection, one
        # of the smallest calls of a serving step.
        _gemm("decode_48_query_cubic", "cubic", 48, 5120, 8192, (16, 1024, 512), "none"),
        # A short prompt or a large decode batch on the down projection, whose
        # K is the longest of the model's.
        _gemm("short_256_down", "strassen", 256, 25600, 5120, (256, 1024, 512), "residual_add"),
        # The square product of the accuracy tests, at the default tile.
        _gemm("square_1024", "strassen", 1024, 1024, 1024, (1024, 1024, 512), "none"),
        # Two requests' prompt tokens, a ragged count padded only to 16 rows.
        _gemm("ragged_1808_attention_out", "strassen", 1808, 8192, 5120, (16, 1024, 512), "residual_add"),
        # The q and k projections of a 2048-token prefill chunk: one packed
        # activation, two GEMMs with the per-head norm and RoPE fused.
        {"name": "chunk_2048_qk", "kind": "qk", "algo": "strassen", "m": 2048, "k": 5120, "heads": 64, "kv_heads": 8,
         "bm": 1024, "bn": 1024, "bk": 512},
        # FP32 inputs at the highest dot precision (six bf16 passes).
        {"name": "fp32_highest_1024", "kind": "fp32", "m": 1024, "k": 2048, "n": 2048, "bm": 1024, "bn": 1024,
         "bk": 512, "precision": "highest"},
        # The row norm, scale and residual behind a projection back to the hidden size.
        {"name": "norm_residual_2048", "kind": "norm", "m": 2048, "k": 5120, "n": 5120, "bm": 256, "bn": 5120,
         "bk": 512},
        # The weight gradient of a projection over 4096 tokens: both operands
        # are new in every step and lie token-major, as the layers produce them.
        {"name": "weight_grad_4096", "kind": "wgrad", "m": 5120, "k": 4096, "n": 8192, "bm": 1024, "bn": 1024,
         "bk": 512},
        # The down projection of the 8 x 1024 prefill on the matched cubic.
        _gemm("prefill_8192_down_cubic", "cubic", 8192, 25600, 5120, (1024, 1024, 512), "residual_add"),
        # The gate|up projection of the 8 x 1024 prefill, the largest GEMM.
        _gemm("prefill_8192_gate_up", "strassen", 8192, 5120, 51200, (1024, 1024, 512), "swiglu"),
        # A whole Qwen3-32B decoder block, 8 sequences of 1024 tokens.
        {"name": "block_8x1024", "kind": "block", "algo": "strassen", "batch": 8, "seq": 1024, "bm": 1024, "bn": 1024,
         "bk": 512},
    ]


def _log(rng, low, high, step):
    """A multiple of step in low .. high, spread over the logarithm."""
    value = math.exp(rng.uniform(math.log(low), math.log(high)))
    return min(high, max(low, int(round(value / step)) * step))


def _row_tile(m):
    """The largest tile that the rows fill whole: 1024, 512 or 256, else 16."""
    return next((bm for bm in (1024, 512, 256) if m % bm == 0), 16)


def draw(rng):
    kind = rng.choice(("decode", "decode", "short", "prefill", "prefill", "ragged", "qk", "fp32", "norm", "wgrad",
                       "block"))
    bn = rng.choice((256, 512, 1024))
    if kind in ("decode", "short", "prefill", "ragged"):
        algo, k, n = "strassen", _log(rng, 512, 25600, 512), _log(rng, 1024, 51200, bn)
        if kind == "decode":
            m = _log(rng, 16, 256, 16)
            bm = rng.choice((16, m))
            if rng.random() < 0.25:
                algo, n = "cubic", 8192
        elif kind == "short":
            m = _log(rng, 256, 1024, 256)
            bm = _row_tile(m)
        elif kind == "ragged":
            m = _log(rng, 272, 2048, 16)
            bm = 16
        elif rng.random() < 0.35:
            # the cubic on whole prefill batches, its columns in whole or half rounds of the chip
            algo, m = "cubic", rng.choice((2048, 4096, 8192))
            bm = 1024
            step = 1024 * 8192 // m
            n = _log(rng, step, 51200 // step * step, step)
        else:
            m = _log(rng, 1024, 8192, 256)
            bm = _row_tile(m)
        step = n if algo == "cubic" else bn
        while m * k * n > 8192 * 5120 * 51200:
            if algo == "cubic":
                k = k // 2 // 512 * 512
            else:
                n = n // 2
        n = max(step, n // step * step)
        return _gemm("", algo, m, k, n, (bm, bn, 512),
                     rng.choice(("swiglu", "residual_add", "residual_add", "bias_add", "geglu", "none")))
    if kind == "qk":
        m = _log(rng, 256, 8192, 256)
        # whole column tiles of bn for both projections
        kv_heads = 8 * rng.randint(1, 2)
        return {"name": "", "kind": "qk", "algo": "strassen", "m": m,
                "k": _log(rng, 1024, 8192, 512), "heads": 8 * rng.randint(2, 8), "kv_heads": kv_heads,
                "bm": _row_tile(m), "bn": 1024, "bk": 512}
    if kind == "fp32":
        m = _log(rng, 256, 2048, 256)
        return {"name": "", "kind": "fp32", "m": m, "k": _log(rng, 512, 4096, 512), "n": _log(rng, 1024, 4096, 1024),
                "bm": _row_tile(m), "bn": bn, "bk": 512, "precision": rng.choice(("default", "high", "highest"))}
    if kind == "norm":
        m, n = _log(rng, 256, 8192, 256), _log(rng, 1024, 8192, 256)
        return {"name": "", "kind": "norm", "m": m, "k": _log(rng, 1024, 8192, 512), "n": n, "bm": 256, "bn": n,
                "bk": 512}
    if kind == "wgrad":
        m = _log(rng, 1024, 8192, 256)
        return {"name": "", "kind": "wgrad", "m": m, "k": _log(rng, 1024, 8192, 512),
                "n": _log(rng, 1024, 8192, 1024), "bm": _row_tile(m), "bn": bn, "bk": 512}
    batch, seq = rng.randint(1, 8), rng.choice((256, 512, 768, 1024))
    return {"name": "", "kind": "block", "algo": "strassen", "batch": batch, "seq": seq,
            "bm": _row_tile(batch * seq), "bn": 1024, "bk": 512}


# ---------------------------------------------------------------------------
# Inputs, from the seed alone
# ---------------------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _activation(g, rows, cols, dtype=torch.bfloat16):
    """A normalised hidden state: N(0, 1)."""
    return torch.randn(rows, cols, device=DEVICE, generator=g).to(dtype)


def _weight(g, k, n, dtype=torch.bfloat16):
    """A projection [K, N] ~ N(0, 0.02), a view of [N, K] storage as nn.Linear keeps it."""
    return (torch.randn(n, k, device=DEVICE, generator=g) * 0.02).to(dtype).t()


def _scale(g, n):
    return (1.0 + 0.1 * torch.randn(n, device=DEVICE, generator=g)).to(torch.bfloat16)


def _angles(rows):
    """RoPE angles [rows, 64] of sequences of 1024 tokens."""
    position = (torch.arange(rows, device=DEVICE) % 1024).float()[:, None]
    return position / THETA ** (torch.arange(0, HEAD_DIM, 2, device=DEVICE).float() / HEAD_DIM)[None, :]


def _inputs(case, seed):
    g, kind = _generator(seed), case["kind"]
    if kind == "block":
        return _activation(g, case["batch"] * case["seq"], qb.QWEN3_32B.hidden), qb.BlockWeights.random_init(
            qb.QWEN3_32B, DEVICE, seed=seed + 1)
    m, k = case["m"], case["k"]
    if kind == "qk":
        heads = (case["heads"], case["kv_heads"])
        cos, sin = (f(_angles(m)).to(torch.bfloat16) for f in (torch.cos, torch.sin))
        return (_activation(g, m, k), [_weight(g, k, h * HEAD_DIM) for h in heads],
                [_scale(g, HEAD_DIM) for _ in heads], cos, sin)
    n = case["n"]
    if kind == "wgrad":
        # activations and output gradients of k tokens, one row a token
        return _activation(g, k, m), (torch.randn(k, n, device=DEVICE, generator=g) * 1e-2).to(torch.bfloat16)
    if kind == "fp32":
        return _activation(g, m, k, torch.float32), _weight(g, k, n, torch.float32)
    if kind == "norm":
        return _activation(g, m, k), _weight(g, k, n), _activation(g, m, n), _scale(g, n)
    extra = None
    if case["epilogue"] == "residual_add":
        extra = _activation(g, m, n)
    elif case["epilogue"] == "bias_add":
        extra = _scale(g, n)
    return _activation(g, m, k), _weight(g, k, n), extra


def _pack(algo, w, case):
    layout = smx.strassen_weight_layout if algo == "strassen" else smx.cubic_weight_layout
    return layout(w, case["bn"], case["bk"])


def prepare(case, seed):
    inputs, kind = _inputs(case, seed), case["kind"]
    tile = {x: case[x] for x in ("bm", "bn", "bk")}
    state = {"case": case, "tile": tile, "x": inputs[0]}
    if kind == "block":
        state["block"] = qb.PreparedBlock(inputs[1], qb.QWEN3_32B, case["algo"], batch=case["batch"], seq=case["seq"],
                                          tile=tuple(tile.values()))
    elif kind == "qk":
        _, weights, scales, cos, sin = inputs
        bn = case["bn"]
        state["weights"] = [_pack(case["algo"], smx.rope_weight_layout(w, bn, HEAD_DIM), case) for w in weights]
        cos, sin = smx.rope_layout_tables(cos, sin, bn // 2, HEAD_DIM)
        state["options"] = [dict(epilogue="qk_norm_rope", rope_cos=cos, rope_sin=sin, rope_head_dim=HEAD_DIM,
                                 rope_eps=EPS, rope_scale=smx.rope_scale_layout(s, bn, HEAD_DIM)) for s in scales]
    elif kind == "wgrad":
        state["dy"] = inputs[1]
    elif kind == "fp32":
        state["w"] = smx.strassen_weight_layout(inputs[1], case["bn"], case["bk"], dot_precision=case["precision"])
    elif kind == "norm":
        state["w"], state["residual"], state["scale"] = _pack("strassen", inputs[1], case), inputs[2], inputs[3]
    else:
        w, epilogue = inputs[1], case["epilogue"]
        if epilogue in ("swiglu", "geglu"):
            w = smx.swiglu_weight_layout(w, case["bn"])
        state["w"] = _pack(case["algo"], w, case)
        options = state["options"] = {} if epilogue == "none" else {"epilogue": epilogue}
        if inputs[2] is not None:
            options["residual" if epilogue == "residual_add" else "bias"] = inputs[2]
    return state


def run(state):
    case, tile, x = state["case"], state["tile"], state["x"]
    kind = case["kind"]
    if kind == "block":
        return qb.block_forward(x, state["block"])
    if kind == "fp32":
        return smx.strassen_matmul(x, state["w"], dot_precision=case["precision"], **tile)
    if kind == "norm":
        return smx.strassen_matmul(x, state["w"], epilogue="norm_residual_add", residual=state["residual"],
                                   norm_scale=state["scale"], norm_eps=EPS, **tile)
    if kind == "wgrad":
        dy = smx.strassen_weight_layout(state["dy"], case["bn"], case["bk"])
        return smx.strassen_matmul_lhs_transposed(x, dy, **tile)
    matmul = smx.strassen_matmul if case["algo"] == "strassen" else smx.cubic_matmul
    if kind == "qk":
        shared = smx.pack_activation(x, 7 if case["algo"] == "strassen" else 8, case["bm"], case["bk"])
        return [matmul(shared, w, **options, **tile) for w, options in zip(state["weights"], state["options"])]
    return matmul(x, state["w"], **state["options"], **tile)


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how near two correct results lie
# ---------------------------------------------------------------------------


def _product(m, k, n, algo, size=2, out=None):
    """Bytes and operations of one product: operands once, the output once,
    seven of the cubic's eight quadrant products for Strassen."""
    out = n if out is None else out
    return size * (m * k + k * n + m * out), 2 * m * k * n * (7 / 8 if algo == "strassen" else 1)


def work(case):
    kind = case["kind"]
    if kind == "block":
        d, m = qb.QWEN3_32B, case["batch"] * case["seq"]
        q, kv = d.heads * d.head_dim, d.kv_heads * d.head_dim
        parts = [_product(m, d.hidden, q, case["algo"]), _product(m, d.hidden, kv, case["algo"]),
                 _product(m, d.hidden, kv, "cubic"), _product(m, q, d.hidden, case["algo"]),
                 _product(m, d.hidden, 2 * d.ffn, case["algo"]), _product(m, d.ffn, d.hidden, case["algo"])]
        weights = 2 * (2 * d.hidden * (q + kv) + 3 * d.hidden * d.ffn)
        # the block's input and output and its weights; causal attention is half of two products
        return {"bytes": weights + 4 * m * d.hidden,
                "flops": sum(f for _, f in parts) + 2 * m * case["seq"] * q}
    m, k = case["m"], case["k"]
    if kind == "qk":
        n = (case["heads"] + case["kv_heads"]) * HEAD_DIM
        moved, flops = _product(m, k, n, case["algo"])
        return {"bytes": moved + 4 * m * HEAD_DIM, "flops": flops}
    n = case["n"]
    if kind == "fp32":
        moved, flops = _product(m, k, n, "strassen", size=4)
        return {"bytes": moved, "flops": flops * {"default": 1, "high": 3, "highest": 6}[case["precision"]]}
    gated = case.get("epilogue") in ("swiglu", "geglu")
    moved, flops = _product(m, k, n, case.get("algo", "strassen"), out=n // 2 if gated else n)
    if kind == "norm" or case.get("epilogue") == "residual_add":
        moved += 2 * m * n
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """About three to four times the distance to the 64-bit result: 4.7e-3 for
    the Strassen product (its operand sums are rounded to bf16), 1.7e-3 for
    the cubic, 9e-3 for the block, whose layers follow one another."""
    kind = case["kind"]
    if kind == "fp32":
        # One bf16 pass of FP32 inputs rounds its operands to bf16; three and
        # six passes carry 16 and 24 bits of them.
        return {"rel": {"default": 1.5e-2, "high": 4e-5, "highest": 2e-6}[case["precision"]]}
    if kind == "block":
        return {"rel": 2e-2}
    return {"rel": 7e-3 if case.get("algo") == "cubic" else 1.5e-2}


# ---------------------------------------------------------------------------
# The same results in 64 bits, in plain torch
# ---------------------------------------------------------------------------


def _matmul64(a, b, chunk=8192):
    """a @ b in float64, a column range at a time."""
    a = a.double()
    return torch.cat([a @ b[:, i:i + chunk].double() for i in range(0, b.shape[1], chunk)], dim=1)


def _head_norm_rope(x, scale, cos, sin):
    """RMSNorm over each head of x [rows, heads, 128], scaled, then RoPE with tables [rows, 64]."""
    x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * scale.double()
    a, b = x[..., :64], x[..., 64:]
    cos, sin = cos.double()[:, None, :], sin.double()[:, None, :]
    return a * cos - b * sin, b * cos + a * sin


def _rms(x, scale):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * scale.double()


def _block64(case, x, w):
    d, batch, seq = qb.QWEN3_32B, case["batch"], case["seq"]
    x = x.double()
    h = _rms(x, w.attention_norm)
    cos, sin = (f(_angles(seq)).to(torch.bfloat16).repeat(batch, 1) for f in (torch.cos, torch.sin))
    q = torch.cat(_head_norm_rope(_matmul64(h, w.query).view(-1, d.heads, HEAD_DIM), w.query_norm, cos, sin), -1)
    k = torch.cat(_head_norm_rope(_matmul64(h, w.key).view(-1, d.kv_heads, HEAD_DIM), w.key_norm, cos, sin), -1)
    v = _matmul64(h, w.value).view(-1, d.kv_heads, HEAD_DIM)
    hidden = torch.full((seq, seq), -math.inf, dtype=torch.float64, device=DEVICE).triu(1)
    attended = torch.empty_like(q)
    for s in range(0, batch * seq, seq):
        for i in range(d.heads):
            j = i * d.kv_heads // d.heads
            scores = q[s:s + seq, i] @ k[s:s + seq, j].t().contiguous() / HEAD_DIM ** 0.5 + hidden
            attended[s:s + seq, i] = torch.softmax(scores, -1) @ v[s:s + seq, j].contiguous()
    x = x + _matmul64(attended.flatten(1), w.attention_output)
    gate, up = _matmul64(_rms(x, w.mlp_norm), w.gate_up).chunk(2, dim=-1)
    return x + _matmul64(torch.nn.functional.silu(gate) * up, w.mlp_down)


def exact(case, seed):
    inputs, kind = _inputs(case, seed), case["kind"]
    if kind == "block":
        return _block64(case, *inputs)
    if kind == "qk":
        x, weights, scales, cos, sin = inputs
        out = []
        for w, scale in zip(weights, scales):
            heads = _matmul64(x, w).view(case["m"], -1, HEAD_DIM)
            a, b = _head_norm_rope(heads, scale, cos, sin)
            # a column tile of bn holds bn/128 heads: their first halves, then their second
            a, b = (half.reshape(case["m"], -1, case["bn"] // 2) for half in (a, b))
            out.append(torch.stack((a, b), dim=2).reshape(case["m"], -1))
        return out
    if kind == "wgrad":
        return _matmul64(inputs[0].t().contiguous(), inputs[1])
    y = _matmul64(inputs[0], inputs[1])
    if kind == "fp32":
        return y
    if kind == "norm":
        return _rms(y, inputs[3]) + inputs[2].double()
    epilogue = case["epilogue"]
    if epilogue in ("swiglu", "geglu"):
        gate, up = y.chunk(2, dim=-1)
        gate = torch.nn.functional.silu(gate) if epilogue == "swiglu" else torch.nn.functional.gelu(
            gate, approximate="tanh")
        return gate * up
    return y if inputs[2] is None else y + inputs[2].double()
