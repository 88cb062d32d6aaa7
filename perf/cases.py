"""The work that programs built on this framework have it do, as measurable cases.

Five kinds of call, each through the entry point that a program uses:

* ``quant``: residual add + RMSNorm + group quantization of one layer's activations.  Without
  norm_out the functional form (which allocates its three outputs), with norm_out the
  reference-signature form into the caller's buffers.
* ``parts``: the same with x given as the partial sums of a tensor-parallel layer's ranks.
* ``gemm``: the fp8 linear layer that consumes the quantizer's codes and scales.
* ``dsa``: top-k selection of key/value blocks and their page-table entries.
* ``mla``: the MLA backward (dq and dc_kv), gradients into the caller's buffers.

``listed()`` names twelve of them; ``draw(rng)`` gives more over the same ranges: 1 to 16384 tokens,
hidden sizes 512 to 8192, weights up to 4608 x 8192, 1 to 1024 queries over 256 to 16384 blocks, and
sequences of 64 to 4096.
"""
import math

import torch

from __graft_entry__ import load_package

pkg = load_package()

DEV = "cuda"
FP8 = torch.float8_e4m3fn
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32, "fp8": FP8,
          "int8": torch.int8, "i32": torch.int32, "i64": torch.int64}
SIZE = {"bf16": 2, "f16": 2, "f32": 4, "ue8m0": 1}
QMAX = {"fp8": 448.0, "int8": 127.0}
EPS = 1e-6
EXACT_ROWS = 16          # rows of each head whose dq the MLA backward computes exactly
MOST_BYTES = 1.0e9       # a drawn case moves no more than this, and multiplies no more than
MOST_FLOPS = 9.0e11      # this (the largest listed cases: 1.09e9 bytes, 9.6e11 operations)


# ------------------------------------------------------------------------------------ the cases

def _quant(name, M, D, G=128, q="fp8", scale="f32", col=False, act="bf16", res="bf16", norm=False,
           rounding="rne"):
    return {"name": name, "kind": "quant", "M": M, "D": D, "G": G, "q": q, "scale": scale,
            "col": col, "act": act, "res": res, "norm": norm, "rounding": rounding}


def _parts(name, M, D, nparts, G=128, scale="f32", col=False):
    return {"name": name, "kind": "parts", "M": M, "D": D, "nparts": nparts, "G": G,
            "scale": scale, "col": col}


def _gemm(name, M, N, K, scale="f32", col=True):
    return {"name": name, "kind": "gemm", "M": M, "N": N, "K": K, "scale": scale, "col": col}


def _dsa(name, B, H, Q, NB, top_k, bs, dtype="f32", index="i32"):
    return {"name": name, "kind": "dsa", "B": B, "H": H, "Q": Q, "NB": NB, "top_k": top_k,
            "bs": bs, "dtype": dtype, "index": index}


def _mla(name, B, H, S, D, grad="bf16"):
    return {"name": name, "kind": "mla", "B": B, "H": H, "S": S, "D": D, "grad": grad}


def listed():
    return [
        # One decode step of four sequences: the smallest call, where the launch counts.
        _quant("quant_decode_4x8192", 4, 8192, q="int8"),
        # A chunk of ragged length in the reference's own output mode (norm_out, int8 by
        # truncation, row-major scales) with an fp32 residual stream.
        _quant("quant_ragged_777x5120", 777, 5120, q="int8", act="bf16", res="f32", norm=True,
               rounding="trunc"),
        # The benchmark's headline: one layer's prefill of 16384 tokens.
        _quant("quant_prefill_16384x7168", 16384, 7168, col=True),
        # One rank's rows after a reduction over eight ranks.
        _parts("parts8_2048x7168", 2048, 7168, 8),
        # The linear layer in a decode step of 32 sequences (weights read once).
        _gemm("gemm_decode_32x4096x7168", 32, 4096, 7168),
        # The fused q_a + kv_a projection of a ragged chunk, UE8M0 scales.
        _gemm("gemm_chunk_1000x2112x7168", 1000, 2112, 7168, scale="ue8m0"),
        # The gate + up projection of the headline prefill.
        _gemm("gemm_prefill_16384x4096x7168", 16384, 4096, 7168),
        # Block selection for a prefill of 512 queries, causal prefixes.
        _dsa("dsa_prefill_2x32x512x4096", 2, 32, 512, 4096, 128, 64),
        # A short ragged one: rows that are not 16-byte aligned, int64 positions.
        _dsa("dsa_ragged_1x8x129x1021", 1, 8, 129, 1021, 64, 128, index="i64"),
        # One decode step over long contexts, bf16 scores.
        _dsa("dsa_decode_16x16x1x16384", 16, 16, 1, 16384, 256, 16, dtype="bf16"),
        # The MLA backward of the reference's largest sequence, and of a short ragged one that
        # accumulates in fp32.
        _mla("mla_2x64x4096x512", 2, 64, 4096, 512),
        _mla("mla_short_1x64x300x512", 1, 64, 300, 512, grad="f32"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_once(rng):
    kind = rng.choice(("quant", "quant", "parts", "gemm", "gemm", "dsa", "dsa", "mla"))
    if kind == "quant":
        G = rng.choice((64, 128, 128, 256))
        act, res = rng.choice((("bf16", "bf16"), ("bf16", "bf16"), ("bf16", "f32"), ("f16", "f16"),
                               ("f16", "f32"), ("f32", "f32")))
        q = rng.choice(("fp8", "int8"))
        return _quant("", _log_int(rng, 1, 16384), G * _log_int(rng, 512 // G, 8192 // G), G, q,
                      rng.choice(("f32", "ue8m0")), rng.random() < 0.5, act, res,
                      rng.random() < 0.4, "trunc" if q == "int8" and rng.random() < 0.5 else "rne")
    if kind == "parts":
        return _parts("", _log_int(rng, 1, 4096), 128 * _log_int(rng, 8, 64), rng.randint(2, 8),
                      scale=rng.choice(("f32", "ue8m0")), col=rng.random() < 0.5)
    if kind == "gemm":
        return _gemm("", _log_int(rng, 1, 16384), 16 * _log_int(rng, 16, 288),
                     128 * _log_int(rng, 4, 64), rng.choice(("f32", "ue8m0")), rng.random() < 0.7)
    if kind == "dsa":
        NB = _log_int(rng, 256, 16384)
        top_k = rng.choice((32, 64, 128, 128, 256, 512, 1024))
        return _dsa("", rng.randint(1, 4), rng.choice((8, 16, 32)), _log_int(rng, 1, 1024),
                    NB if rng.random() < 0.4 else (NB + 7) // 8 * 8, min(top_k, NB // 2),
                    rng.choice((16, 64, 128)), rng.choice(("f32", "f32", "bf16")),
                    rng.choice(("i32", "i32", "i64")))
    return _mla("", rng.randint(1, 2), rng.choice((8, 16, 32, 64)), _log_int(rng, 64, 4096),
                rng.choice((512, 512, 64 * rng.randint(2, 10))), rng.choice(("bf16", "f32")))


def draw(rng):
    while True:
        case = _draw_once(rng)
        del case["name"]
        w = work(case)
        if w["bytes"] <= MOST_BYTES and w["flops"] <= MOST_FLOPS:
            return case


# ------------------------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _activations(g, M, D, dtype):
    """N(0, 1) with the outlier channels (1 %, times 50) that hidden states have in earnest."""
    x = _randn(g, M, D)
    channels = torch.randperm(D, generator=g, device=DEV)[:max(1, round(0.01 * D))]
    x[:, channels] *= 50.0
    return x.to(dtype)


def _norm_weight(g, D, dtype):
    return (1.0 + 0.1 * _randn(g, D)).to(dtype)


def _block_scale(absmax, scale):
    """(scale as stored, its value) of blocks with these largest magnitudes."""
    s = (absmax / 448.0).clamp_min(1e-12)
    if scale == "f32":
        return s, s
    e = torch.ceil(torch.log2(s)).clamp(-127, 127)
    return (e + 127).to(torch.uint8), torch.exp2(e)


def _quantized_rows(g, M, K, scale, col):
    """fp8 codes and 1 x 128 scales of M rows of activations."""
    x = _activations(g, M, K, torch.float32).view(M, K // 128, 128)
    stored, s = _block_scale(x.abs().amax(-1), scale)
    codes = (x / s[..., None]).clamp(-448.0, 448.0).to(FP8).view(M, K)
    return codes, stored.t().contiguous().t() if col else stored.contiguous()


def _quantized_weight(g, N, K, scale):
    """fp8 codes and 128 x 128 scales of an N x K weight."""
    nb, kb = -(-N // 128), K // 128
    w = torch.zeros(nb * 128, K, device=DEV)
    w[:N] = 0.02 * _randn(g, N, K)
    w = w.view(nb, 128, kb, 128)
    stored, s = _block_scale(w.abs().amax((1, 3)), scale)
    codes = (w / s[:, None, :, None]).clamp(-448.0, 448.0).to(FP8).view(nb * 128, K)
    return codes[:N].contiguous(), stored.contiguous()


def _kv_lens(case):
    """Context lengths (tokens) of the batches: the table's capacity less a few blocks each."""
    full = case["NB"] * case["bs"]
    return [max(1, full - 3 * b * case["bs"]) for b in range(case["B"])]


def _positions(case):
    """Query q of batch b sees a causal prefix; the last one sees all of the context."""
    Q = case["Q"]
    return [[(q + 1) * kv // Q - 1 for q in range(Q)] for kv in _kv_lens(case)]


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind in ("quant", "parts"):
        M, D = case["M"], case["D"]
        act = DTYPES[case.get("act", "bf16")]
        res = DTYPES[case.get("res", "bf16")]
        if kind == "parts":
            sd = case["nparts"] ** -0.5
            st = {"parts": [(sd * _activations(g, M, D, torch.float32)).to(act)
                            for _ in range(case["nparts"])]}
        else:
            st = {"x": _activations(g, M, D, act)}
        st["residual"] = _activations(g, M, D, res)
        st["weight"] = _norm_weight(g, D, act)
        if case.get("norm"):
            st["residual_out"] = torch.empty_like(st["residual"])
            st["norm_out"] = torch.empty_like(st["x"])
            st["q"] = torch.empty(M, D, dtype=DTYPES[case["q"]], device=DEV)
            st["scale"] = pkg.empty_scales(M, D // case["G"], ue8m0=case["scale"] == "ue8m0",
                                           col_major=case["col"], device=DEV)
    elif kind == "gemm":
        a_q, a_scale = _quantized_rows(g, case["M"], case["K"], case["scale"], case["col"])
        b_q, b_scale = _quantized_weight(g, case["N"], case["K"], case["scale"])
        st = {"a_q": a_q, "a_scale": a_scale, "b_q": b_q, "b_scale": b_scale}
    elif kind == "dsa":
        B, H, Q, NB, k = (case[n] for n in ("B", "H", "Q", "NB", "top_k"))
        index = DTYPES[case["index"]]
        st = {"scores": _randn(g, B, H, Q, NB).to(DTYPES[case["dtype"]]),
              "page_table": torch.stack([b * NB + torch.randperm(NB, generator=g, device=DEV)
                                         for b in range(B)]).to(torch.int32),
              "q_pos": torch.tensor(_positions(case), dtype=index, device=DEV),
              "kv_lens": torch.tensor(_kv_lens(case), dtype=index, device=DEV),
              "out_blocks": torch.empty(B, H, Q, k, dtype=torch.int32, device=DEV),
              "out_pages": torch.empty(B, H, Q, k, dtype=torch.int32, device=DEV)}
    else:
        B, H, S, D = (case[n] for n in ("B", "H", "S", "D"))
        grad = DTYPES[case["grad"]]
        q = _randn(g, B, H, S, D).to(torch.bfloat16)
        c = _randn(g, B, S, D).to(torch.bfloat16)
        do = _randn(g, B, H, S, D).to(torch.bfloat16)
        # out and lse of the causal forward for the rows that the backward reads; the others
        # only have to be there.
        out = (0.05 * _randn(g, B, H, S, D)).to(torch.bfloat16)
        lse = torch.log(torch.arange(1, S + 1, device=DEV, dtype=torch.float32))
        lse = lse.expand(B, H, S).contiguous()
        E = min(EXACT_ROWS, S)
        p, lse_e = _forward(q[:, :, :E].double(), c[:, :E].double(), D ** -0.5)
        lse[:, :, :E] = lse_e.float()
        out[:, :, :E] = torch.matmul(p, c[:, None, :E].double()).to(torch.bfloat16)
        st = {"q": q, "c_kv": c, "out": out, "do": do, "lse": lse,
              "dq": torch.empty(B, H, S, D, dtype=grad, device=DEV),
              "dc_kv": torch.empty(B, S, D, dtype=grad, device=DEV)}
    st["case"] = case
    return st


def _forward(q, c, scale):
    """(probabilities, lse) of causal attention with K = V = C, in 64 bits."""
    E = q.shape[2]
    logits = torch.matmul(q, c[:, None].transpose(-1, -2).contiguous()) * scale
    logits = logits.masked_fill(~torch.ones(E, E, dtype=torch.bool, device=DEV).tril(),
                                float("-inf"))
    return torch.softmax(logits, -1), torch.logsumexp(logits, -1)


# ------------------------------------------------------------------------------------ one pass

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "quant":
        if case["norm"]:
            return pkg.fused_add_rmsnorm_group_quant(
                state["x"], state["residual"], state["weight"], state["residual_out"],
                state["norm_out"], state["q"], state["scale"], EPS, case["G"],
                rounding=None if case["q"] == "fp8" else case["rounding"])
        return pkg.fused_add_rmsnorm_group_quant_fn(
            state["x"], state["residual"], state["weight"], EPS, case["G"], DTYPES[case["q"]],
            scale_col_major=case["col"], scale_ue8m0=case["scale"] == "ue8m0",
            rounding=case["rounding"])
    if kind == "parts":
        return pkg.fused_reduce_add_rmsnorm_group_quant(
            state["parts"], state["residual"], state["weight"], EPS, case["G"],
            scale_col_major=case["col"], scale_ue8m0=case["scale"] == "ue8m0")
    if kind == "gemm":
        return pkg.fp8_block_scaled_gemm(state["a_q"], state["a_scale"], state["b_q"],
                                         state["b_scale"])
    if kind == "dsa":
        return pkg.dsa_topk_page_table_transform(
            state["scores"], state["page_table"], state["q_pos"], state["kv_lens"],
            state["out_blocks"], state["out_pages"], case["bs"], case["top_k"])
    return pkg.mla_bwd_nope_dkdv(state["q"], state["c_kv"], state["out"], state["do"],
                                 state["lse"], state["dq"], state["dc_kv"], case["D"] ** -0.5)


# ------------------------------------------------------------------------------------ its work

def work(case):
    kind = case["kind"]
    if kind in ("quant", "parts"):
        M, D = case["M"], case["D"]
        ba, br = SIZE[case.get("act", "bf16")], SIZE[case.get("res", "bf16")]
        nx = case.get("nparts", 1)
        per = ba * nx + 2 * br + 1 + (ba if case.get("norm") else 0)
        return {"bytes": M * D * per + ba * D + M * (D // case["G"]) * SIZE[case["scale"]],
                "flops": M * D * (8 + nx)}
    if kind == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        sb = SIZE[case["scale"]]
        return {"bytes": M * K + N * K + 2 * M * N + sb * (K // 128) * (M + -(-N // 128)),
                "flops": 2 * M * N * K}
    if kind == "dsa":
        B, H, Q, NB, k = (case[n] for n in ("B", "H", "Q", "NB", "top_k"))
        valid = 0
        for kv, row in zip(_kv_lens(case), _positions(case)):
            blocks = min(-(-kv // case["bs"]), NB)
            valid += sum(min(p // case["bs"] + 1, blocks) for p in row if p >= 0) * H
        idx = 8 if case["index"] == "i64" else 4
        return {"bytes": valid * SIZE[case["dtype"]] + 8 * B * H * Q * k + 4 * B * NB
                + idx * (B * Q + B), "flops": 2 * valid}
    B, H, S, D = (case[n] for n in ("B", "H", "S", "D"))
    E, gb, n = min(EXACT_ROWS, S), SIZE[case["grad"]], B * H * S * D
    return {"bytes": (2 + gb) * n + gb * B * S * D + 4 * B * H * E * D + 2 * B * E * D
            + 4 * B * H * E, "flops": 2 * n + 6 * B * H * E * E * D}


def tolerance(case):
    kind = case["kind"]
    if kind in ("quant", "parts", "dsa"):
        # One definition down to the last bit: the sum of squares is in 64 bits and every other
        # step is rounded where the operator says; selections are whole numbers.
        return "exact"
    if kind == "gemm":
        # bf16 results of 32-bit sums: measured against 64 bits rel 1.7e-3, max 3.9e-3 (half a
        # step of bf16); a sum in another order moves a few results by one step.
        return {"rel": 7e-3, "max": 1.6e-2}
    # The rows with the exact gradient round probabilities and their gradients to bf16, so a
    # 32-bit sum in another order moves a rare one by a step of 2^-8: 32- against 64-bit sums
    # before those roundings measured rel 7e-6 and max 1.2e-2 (one element's step against the
    # much smaller rows around it) on 2 x 64 heads, and a short case with one such step reaches
    # about 5e-5.  bf16 gradients add their own rounding.
    return {"rel": 2e-4 if case["grad"] == "f32" else 7e-3, "max": 5e-2}


# ------------------------------------------------------------------------------------ in 64 bits

def _rows_exact(case, x, st):
    """r, n, codes and scales of RMSNorm and group quantization in 64 bits; codes and UE8M0
    scales that are whole numbers have no value between."""
    M, D, G = case["M"], case["D"], case["G"]
    r = x + st["residual"].double()
    inv = torch.rsqrt(r.square().mean(1, keepdim=True) + EPS)
    n = r * inv * st["weight"].double()
    qmax = QMAX[case.get("q", "fp8")]
    s = (n.view(M, D // G, G).abs().amax(-1) / qmax).clamp_min(1e-12)
    stored = s
    if case["scale"] == "ue8m0":
        # The step of the scale follows the 32-bit scale: a 64-bit one may fall on the other side.
        stored, s = None, None
    codes = None
    if s is not None and case.get("q", "fp8") == "fp8":
        codes = (n.view(M, D // G, G) / s[..., None]).view(M, D)
    return r, n, codes, stored


def exact(case, seed):
    kind = case["kind"]
    if kind == "dsa":
        return None
    st = prepare(case, seed)
    if kind in ("quant", "parts"):
        x = sum(p.double() for p in st["parts"]) if kind == "parts" else st["x"].double()
        r, n, codes, s = _rows_exact(case, x, st)
        return (r, n, codes, s) if case.get("norm") else (r, codes, s)
    if kind == "gemm":
        M, N, K = case["M"], case["N"], case["K"]

        def value(s):
            return s.double() if s.dtype == torch.float32 else torch.exp2(s.double() - 127.0)

        a = st["a_q"].to(torch.float32).double().view(M, K // 128, 128)
        a = (a * value(st["a_scale"])[..., None]).view(M, K)
        b = st["b_q"].to(torch.float32).double().view(N, K // 128, 128)
        b = (b * value(st["b_scale"]).repeat_interleave(128, 0)[:N, :, None]).view(N, K)
        return torch.matmul(a, b.t())
    # dq = sm_scale do, but for the first rows of each head, whose gradient is that of causal
    # attention; dc = the sum over the later rows of the heads' do / (i + 1).
    E, scale = min(EXACT_ROWS, case["S"]), case["D"] ** -0.5
    do = st["do"].double()
    dq = do * scale
    q, c = st["q"][:, :, :E].double(), st["c_kv"][:, :E].double()
    logits = torch.matmul(q, c[:, None].transpose(-1, -2).contiguous()) * scale
    p = torch.exp(logits - st["lse"][:, :, :E, None].double()).tril()
    delta = (st["out"][:, :, :E].double() * do[:, :, :E]).sum(-1, keepdim=True)
    dp = torch.matmul(do[:, :, :E].contiguous(), c[:, None].transpose(-1, -2).contiguous())
    dq[:, :, :E] = torch.matmul(p * (dp - delta) * scale, c[:, None])
    hs = do.sum(1) / torch.arange(1, case["S"] + 1, device=DEV, dtype=torch.float64)[None, :, None]
    return dq, hs.flip(1).cumsum(1).flip(1)
