"""The workloads that the library's speed is judged on: what a decoder's host program has the row ops do
around its GEMMs and its attention, through the `exl3r.ffi` wrappers on torch tensors.

Sizes are the repository's configurations: hidden 5120 with 64 / 8 heads of 128 and an intermediate size of
17408 or 25600 (the large dense model), hidden 1024 with 16 / 8 heads and 3072 (the small one), the
gated-attention and gated-delta-net layers of the hybrid model, vocabulary 151936.  `draw` spreads token
counts, widths, heads, dtypes and options over the ranges between and around them.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.getcwd(), "exllamav3-rs_amd"))

import exl3r  # noqa: E402
import exl3r.ffi as ffi  # noqa: E402

F16, BF16, F32 = torch.float16, torch.bfloat16, torch.float32
DT = {"f16": F16, "bf16": BF16, "f32": F32}
BYTES = {"f16": 2, "bf16": 2, "f32": 4}
EPS = 1e-6
PAGE = 256
HAD = 1.0 / math.sqrt(128.0)


def listed():
    return [
        # Single-stream decode, graph-captured as the reference's infer loop is: one token through the row ops of
        # 16 layers of the large model (embedding + norm, RoPE + paged append, norm, SiLU-mul per layer, final
        # norm, greedy pick over f32 logits).  The smallest calls: launches and latency are all there is.
        dict(name="decode_step_graph_b1", kind="step", bsz=1, layers=16, hidden=5120, hq=64, hk=8, inter=25600,
             vocab=151936),
        # Batched decode, eager: one layer's four row ops over 64 sequences of one token each.
        dict(name="decode_layer_64", kind="layer", bsz=64, seq=1, hidden=5120, hq=64, hk=8, hd=128, inter=17408,
             dtype="f16", res="f32"),
        # A short prompt through one layer of the small model, eager.
        dict(name="prefill_layer_512", kind="layer", bsz=1, seq=512, hidden=1024, hq=16, hk=8, hd=128, inter=3072,
             dtype="f16", res="f32"),
        # The row ops of a long bf16 prefill without quantised projections: residual norm and SiLU-mul.
        dict(name="prefill_rows_8192", kind="rows", rows=8192, hidden=5120, inter=17408, act="silu", dtype="bf16",
             res="bf16"),
        # The embedding of a long prefill: bf16 table to the f32 residual stream, Zipf-distributed ids.
        dict(name="embed_16384", kind="embed", n=16384, vocab=151936, hidden=5120, table="bf16", out="f32", norm=False),
        # EXL3 prefill, attention input: the previous projection's output rotation, the residual norm and the
        # input rotations of q, k and v.
        dict(name="norm_had_4096", kind="norm_had", rows=4096, hidden=5120, n_out=3, rotate=True, res="f32"),
        # EXL3 prefill, MLP: the gate and up output rotations, SiLU-mul and down_proj's input rotation.
        dict(name="mlp_had_4096", kind="mlp_had", rows=4096, inter=25600, act="silu", rotate=True),
        # EXL3 prefill, attention: q / k / v output rotations, head norm, RoPE and the paged append.
        dict(name="attn_had_4096", kind="attn_had", bsz=1, seq=4096, hq=64, hk=8, mode="neox"),
        # The hybrid model's gated attention, ragged prefill: q | g heads of 256 with a quarter of them rotary,
        # head norm with bias 1, and the output gate read in place.
        dict(name="gated_attn_4639", kind="gated_attn", tokens=4639, hq=16, hk=2, hd=256, rot=64, dtype="bf16"),
        # Multimodal prefill: RoPE with a table of precomputed angles.
        dict(name="mrope_4096", kind="mrope", bsz=1, seq=4096, hq=32, hk=8, hd=128, dtype="f16", norm=True),
        # The hybrid model's gated-delta-net output: gated norm over the heads and o_proj's input rotation.
        dict(name="gdn_out_4096", kind="gdn", tokens=4096, heads=32, hd=128, had=True),
        # Sampling for 64 sequences from the head's f32 logits.
        dict(name="sample_64", kind="sample", rows=64, vocab=151936, dtype="f32", gumbel=True),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _heads(rng):
    return rng.choice([(16, 8), (32, 8), (64, 8), (32, 4), (40, 8), (24, 4)])


def draw(rng):
    kind = rng.choice(["step", "layer", "layer", "rows", "embed", "norm_had", "mlp_had", "attn_had", "gated_attn",
                       "mrope", "gdn", "sample", "sample"])
    hidden = 128 * _log(rng, 8, 40)
    if kind == "step":
        hq, hk = _heads(rng)
        return dict(kind=kind, bsz=rng.randint(1, 8), layers=rng.randint(2, 16), hidden=hidden, hq=hq, hk=hk,
                    inter=128 * _log(rng, 24, 200), vocab=rng.choice([151936, rng.randint(32000, 152000)]))
    if kind == "layer":
        hq, hk = _heads(rng)
        bsz, seq = (_log(rng, 1, 256), 1) if rng.random() < 0.5 else (rng.randint(1, 3), _log(rng, 5, 700))
        dtype = rng.choice(["f16", "bf16"])
        return dict(kind=kind, bsz=bsz, seq=seq, hidden=hidden, hq=hq, hk=hk, hd=rng.choice([128, 128, 64]),
                    inter=128 * _log(rng, 24, 136), dtype=dtype, res=rng.choice(["f32", dtype]))
    if kind == "rows":
        dtype = rng.choice(["f16", "bf16", "bf16"])
        return dict(kind=kind, rows=_log(rng, 512, 8192), hidden=hidden, inter=128 * _log(rng, 24, 136),
                    act=rng.choice(["silu", "gelu"]), dtype=dtype, res=rng.choice(["f32", dtype]))
    if kind == "embed":
        norm = rng.random() < 0.4
        return dict(kind=kind, n=_log(rng, 64, 16384), vocab=rng.randint(32000, 151936), hidden=hidden,
                    table=rng.choice(["bf16", "f16"]), out="f32", norm=norm)
    if kind == "norm_had":
        return dict(kind=kind, rows=_log(rng, 64, 4096), hidden=hidden, n_out=rng.choice([2, 3]),
                    rotate=rng.random() < 0.7, res="f32")
    if kind == "mlp_had":
        return dict(kind=kind, rows=_log(rng, 64, 4096), inter=128 * _log(rng, 24, 200), act=rng.choice(["silu", "gelu"]),
                    rotate=rng.random() < 0.7)
    if kind == "attn_had":
        hq, hk = _heads(rng)
        bsz = rng.choice([1, 1, 2, 3, 16])
        return dict(kind=kind, bsz=bsz, seq=_log(rng, 1, 4096 // bsz), hq=hq, hk=hk,
                    mode=rng.choice(["neox", "neox", "neox", "gptj"]))
    if kind == "gated_attn":
        hq, hk, hd, rot = rng.choice([(16, 2, 256, 64), (32, 4, 128, 128), (24, 4, 256, 64), (8, 2, 256, 64)])
        return dict(kind=kind, tokens=_log(rng, 33, 4639 * 16 * 256 // (hq * hd) * 9 // 10), hq=hq, hk=hk, hd=hd, rot=rot,
                    dtype=rng.choice(["f16", "bf16"]))
    if kind == "mrope":
        hq, hk, hd = rng.choice([(32, 8, 128), (16, 8, 128), (28, 4, 128), (16, 16, 64), (16, 16, 72)])
        bsz = rng.randint(1, 3)
        return dict(kind=kind, bsz=bsz, seq=_log(rng, 16, 4096 // bsz), hq=hq, hk=hk, hd=hd,
                    dtype=rng.choice(["f16", "bf16"]), norm=hd == 128)
    if kind == "gdn":
        return dict(kind=kind, tokens=_log(rng, 1, 4096), heads=rng.choice([16, 32]), hd=128, had=rng.random() < 0.6)
    gumbel = rng.random() < 0.6
    return dict(kind="sample", rows=_log(rng, 1, 64), vocab=rng.choice([151936, 128256, rng.randint(32000, 152000)]),
                dtype=rng.choice(["f32", "f32", "f16", "bf16"]), gumbel=gumbel)


class _Maker:
    """Seeded tensors: normal values rounded to their dtype, signs of the rotations' diagonals, ints."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))
        self.rng = np.random.default_rng(int(seed))

    def normal(self, shape, mean, std, dtype):
        v = torch.empty(shape, device="cuda", dtype=F32).normal_(mean, std, generator=self.g)
        return v.to(dtype)

    def signs(self, n):
        v = torch.randint(0, 2, (n,), device="cuda", generator=self.g)
        return (v * 2 - 1).to(F16)

    def zipf(self, n, vocab):
        p = np.arange(1, vocab + 1, dtype=np.float64) ** -1.1
        c = np.cumsum(p)
        ids = np.minimum(np.searchsorted(c, self.rng.random(n) * c[-1]), vocab - 1).astype(np.int64)
        return torch.from_numpy(ids).cuda()

    def ragged(self, tokens):
        """Per-token positions of sequences of 64 to 512 tokens that start anywhere below 32768."""
        out, n = [], 0
        while n < tokens:
            m = min(tokens - n, int(self.rng.integers(64, 513)))
            out.append(int(self.rng.integers(0, 32768)) + np.arange(m))
            n += m
        return torch.from_numpy(np.concatenate(out).astype(np.int32)).cuda()


def _inv_freq(rot):
    return torch.from_numpy((1.0 / 1e6 ** (np.arange(0, rot, 2, dtype=np.float64) / rot)).astype(np.float32)).cuda()


def _paged(m, bsz, seq, hk, hd, dtype, past=2000):
    """Zeroed caches, a shuffled block table and cache lengths with room for seq more tokens."""
    blocks = (past + seq) // PAGE + 1
    pages = bsz * blocks + 1
    table = torch.from_numpy(m.rng.permutation(pages)[:bsz * blocks].reshape(bsz, blocks).astype(np.int32)).cuda()
    lens = torch.from_numpy(m.rng.integers(0, past, bsz).astype(np.int32)).cuda()
    kc = torch.zeros((pages, PAGE, hk, hd), device="cuda", dtype=dtype)
    return dict(kc=kc, vc=torch.zeros_like(kc), table=table, lens=lens)


def prepare(case, seed):
    m, kind = _Maker(seed), case["kind"]
    s = dict(case)
    if kind == "step":
        return _prepare_step(s, m)
    if kind == "layer":
        T, H, dt = s["bsz"] * s["seq"], s["hidden"], DT[s["dtype"]]
        s.update(x1=m.normal((T, H), 0, 1, dt), x2=m.normal((T, H), 0, 1, dt), r=m.normal((T, H), 0, 4, DT[s["res"]]),
                 w1=m.normal((H,), 1, 0.1, dt), w2=m.normal((H,), 1, 0.1, dt),
                 y1=torch.empty((T, H), device="cuda", dtype=dt), y2=torch.empty((T, H), device="cuda", dtype=dt),
                 gate=m.normal((T, s["inter"]), 0, 1, dt), up=m.normal((T, s["inter"]), 0, 1, dt),
                 z=torch.empty((T, s["inter"]), device="cuda", dtype=dt), **_attention(s, m, dt))
    elif kind == "rows":
        T, H, dt = s["rows"], s["hidden"], DT[s["dtype"]]
        s.update(x=m.normal((T, H), 0, 1, dt), r=m.normal((T, H), 0, 4, DT[s["res"]]), w=m.normal((H,), 1, 0.1, dt),
                 y=torch.empty((T, H), device="cuda", dtype=dt), gate=m.normal((T, s["inter"]), 0, 1, dt),
                 up=m.normal((T, s["inter"]), 0, 1, dt), z=torch.empty((T, s["inter"]), device="cuda", dtype=dt))
    elif kind == "embed":
        H = s["hidden"]
        s.update(rows=m.normal((s["vocab"], H), 0, 0.02, DT[s["table"]]), ids=m.zipf(s["n"], s["vocab"]),
                 h=torch.empty((s["n"], H), device="cuda", dtype=DT[s["out"]]))
        if s["norm"]:
            s.update(w=m.normal((H,), 1, 0.1, F16), y=torch.empty((s["n"], H), device="cuda", dtype=F16))
    elif kind == "norm_had":
        T, H = s["rows"], s["hidden"]
        s.update(x=m.normal((T, H), 0, 1, F16), r=m.normal((T, H), 0, 4, DT[s["res"]]), w=m.normal((H,), 1, 0.1, F16),
                 post=m.signs(H) if s["rotate"] else None, pre=[m.signs(H) for _ in range(s["n_out"])],
                 outs=[torch.empty((T, H), device="cuda", dtype=F16) for _ in range(s["n_out"])])
    elif kind == "mlp_had":
        T, n = s["rows"], s["inter"]
        s.update(gate=m.normal((T, n), 0, 1, F16), up=m.normal((T, n), 0, 1, F16), pre=m.signs(n),
                 gp=m.signs(n) if s["rotate"] else None, upp=m.signs(n) if s["rotate"] else None,
                 out=torch.empty((T, n), device="cuda", dtype=F16))
    elif kind == "attn_had":
        s.update(hd=128, **_attention(dict(s, hd=128), m, F16))
        s.update(sq=m.signs(s["hq"] * 128), sk=m.signs(s["hk"] * 128), sv=m.signs(s["hk"] * 128))
    elif kind == "gated_attn":
        T, hq, hk, hd, dt = s["tokens"], s["hq"], s["hk"], s["hd"], DT[s["dtype"]]
        s.update(qg=m.normal((1, T, hq, 2 * hd), 0, 1, dt), k=m.normal((1, T, hk, hd), 0, 1, dt),
                 q=torch.empty((1, T, hq, hd), device="cuda", dtype=dt), o=m.normal((T * hq, hd), 0, 1, dt),
                 z=torch.empty((T * hq, hd), device="cuda", dtype=dt), qn=m.normal((hd,), 0, 0.1, dt),
                 kn=m.normal((hd,), 0, 0.1, dt), inv=_inv_freq(s["rot"]), pos=m.ragged(T).view(1, T))
    elif kind == "mrope":
        B, S, hd, dt = s["bsz"], s["seq"], s["hd"], DT[s["dtype"]]
        # angles of positions in the text / image grid, a table per sequence when there are several
        grid = torch.from_numpy(np.sort(m.rng.integers(0, S + 1, (B, S, 1)), axis=1).astype(np.float32)).cuda()
        table = grid * _inv_freq(hd)
        s.update(q=m.normal((B, S, s["hq"], hd), 0, 1, dt), k=m.normal((B, S, s["hk"], hd), 0, 1, dt),
                 qn=m.normal((hd,), 1, 0.1, dt) if s["norm"] else None, kn=m.normal((hd,), 1, 0.1, dt) if s["norm"] else None,
                 angles=(table[0] if B == 1 else table).contiguous())
    elif kind == "gdn":
        n, hd = s["tokens"] * s["heads"], s["hd"]
        s.update(x=m.normal((n, hd), 0, 1, BF16), g=m.normal((n, hd), 0, 2, F32), w=m.normal((hd,), 1, 0.1, F32),
                 pre=m.signs(s["heads"] * hd), out=torch.empty((n, hd), device="cuda", dtype=F16))
    else:
        s.update(logits=m.normal((s["rows"], s["vocab"]), 0, 3, DT[s["dtype"]]),
                 ids=torch.zeros(s["rows"], dtype=torch.int64, device="cuda"), random=int(m.rng.integers(0, 2 ** 32)))
    return s


def _attention(s, m, dt):
    B, S, hd = s["bsz"], s["seq"], s["hd"]
    q = m.normal((B, S, s["hq"], hd), 0, 1, dt)
    return dict(q=q, qo=torch.empty_like(q), k=m.normal((B, S, s["hk"], hd), 0, 1, dt),
                v=m.normal((B, S, s["hk"], hd), 0, 1, dt), qn=m.normal((hd,), 1, 0.1, dt), kn=m.normal((hd,), 1, 0.1, dt),
                inv=_inv_freq(hd), **_paged(m, B, S, s["hk"], hd, dt))


def _prepare_step(s, m):
    B, H = s["bsz"], s["hidden"]
    s.update(emb=m.normal((s["vocab"], H), 0, 0.02, BF16), ids=m.zipf(B, s["vocab"]),
             h=torch.empty((B, H), device="cuda", dtype=F32), y=torch.empty((B, H), device="cuda", dtype=F16),
             wf=m.normal((H,), 1, 0.1, F16), logits=m.normal((B, s["vocab"]), 0, 3, F32),
             next=torch.zeros(B, dtype=torch.int64, device="cuda"), blocks=[])
    for _ in range(s["layers"]):
        s["blocks"].append(dict(
            w1=m.normal((H,), 1, 0.1, F16), w2=m.normal((H,), 1, 0.1, F16), y1=torch.empty((B, H), device="cuda", dtype=F16),
            y2=torch.empty((B, H), device="cuda", dtype=F16), a_out=m.normal((B, H), 0, 1, F16),
            m_out=m.normal((B, H), 0, 1, F16), gate=m.normal((B, s["inter"]), 0, 1, F16),
            up=m.normal((B, s["inter"]), 0, 1, F16), z=torch.empty((B, s["inter"]), device="cuda", dtype=F16),
            **_attention(dict(s, seq=1, hd=128), m, F16)))
    _step(s)
    torch.cuda.synchronize()
    s["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s["graph"]):
        _step(s)
    return s


def _step(s):
    pending = None
    for b in s["blocks"]:
        if pending is None:
            ffi.embedding_rms_norm(s["emb"], s["ids"], s["h"], b["w1"], b["y1"], EPS)
        else:
            ffi.rms_norm_res_in(pending, b["w1"], b["y1"], s["h"], EPS)
        _paged_rope(b)
        ffi.rms_norm_res_in(b["a_out"], b["w2"], b["y2"], s["h"], EPS)
        ffi.silu_mul(b["gate"], b["up"], b["z"])
        pending = b["m_out"]
    ffi.rms_norm_res_in(pending, s["wf"], s["y"], s["h"], EPS)
    ffi.argmax_sample(s["logits"], s["next"])


def _paged_rope(b):
    ffi.rope_paged_kv(b["q"], b["qo"], b["k"], None, b["v"], b["inv"], 0, b["lens"], b["qn"], b["kn"], EPS, 0.0,
                      exl3r.ROPE_NEOX, 1.0, b["kc"], b["vc"], b["table"], b["lens"])


def run(s):
    kind = s["kind"]
    if kind == "step":
        s["graph"].replay()
        return [s["h"], s["y"], s["next"]] + [b[n] for b in s["blocks"][-4:] for n in ("y1", "y2", "z", "qo", "kc", "vc")]
    if kind == "layer":
        ffi.rms_norm_res_in(s["x1"], s["w1"], s["y1"], s["r"], EPS)
        _paged_rope(s)
        ffi.rms_norm_res_in(s["x2"], s["w2"], s["y2"], s["r"], EPS)
        ffi.silu_mul(s["gate"], s["up"], s["z"])
        return [s[n] for n in ("y1", "y2", "r", "z", "qo", "kc", "vc")]
    if kind == "rows":
        ffi.rms_norm_res_in(s["x"], s["w"], s["y"], s["r"], EPS)
        (ffi.silu_mul if s["act"] == "silu" else ffi.gelu_mul)(s["gate"], s["up"], s["z"])
        return [s["y"], s["r"], s["z"]]
    if kind == "embed":
        if s["norm"]:
            ffi.embedding_rms_norm(s["rows"], s["ids"], s["h"], s["w"], s["y"], EPS)
            return [s["h"], s["y"]]
        ffi.embedding(s["rows"], s["ids"], s["h"])
        return [s["h"]]
    if kind == "norm_had":
        ffi.rms_norm_had(s["x"], s["w"], s["outs"], s["pre"], EPS, r=s["r"], rotate_x=s["rotate"], x_post_scale=s["post"])
        return s["outs"] + [s["r"]]
    if kind == "mlp_had":
        ffi.act_mul_had(s["act"], s["gate"], s["up"], s["out"], s["pre"], rotate_x=s["rotate"], rotate_y=s["rotate"],
                        x_post_scale=s["gp"], y_post_scale=s["upp"])
        return [s["out"]]
    if kind == "attn_had":
        mode = exl3r.ROPE_NEOX if s["mode"] == "neox" else exl3r.ROPE_GPTJ
        ffi.rope_paged_kv_had(s["q"], s["q"], s["k"], None, s["v"], s["inv"], 0, s["lens"], s["qn"], s["kn"], EPS, 0.0,
                              mode, 1.0, s["kc"], s["vc"], s["table"], s["lens"], q_post_scale=s["sq"],
                              k_post_scale=s["sk"], v_post_scale=s["sv"])
        return [s["q"], s["kc"], s["vc"]]
    if kind == "gated_attn":
        ffi.rope_qg(s["qg"], s["q"], s["k"], s["k"], s["inv"], 0, None, s["qn"], s["kn"], EPS, 1.0, exl3r.ROPE_NEOX, 1.0,
                    position_ids=s["pos"])
        hd = s["hd"]
        ffi.mul_sigmoid(s["o"], s["qg"].view(-1, 2 * hd)[:, hd:], s["z"])
        return [s["q"], s["k"], s["z"]]
    if kind == "mrope":
        ffi.rope(s["q"], s["q"], s["k"], s["k"], s["angles"], 0, None, s["qn"], s["kn"], EPS, 0.0, exl3r.ROPE_NEOX, 1.0)
        return [s["q"], s["k"]]
    if kind == "gdn":
        if s["had"]:
            ffi.gated_rms_norm_had(s["x"], s["w"], s["g"], s["out"], EPS, s["pre"], pre_rows=s["heads"])
        else:
            ffi.gated_rms_norm(s["x"], s["w"], s["out"], s["g"], EPS)
        return [s["out"]]
    if s["gumbel"]:
        ffi.gumbel_sample(s["logits"], s["ids"], random=s["random"])
    else:
        ffi.argmax_sample(s["logits"], s["ids"])
    return [s["ids"]]


def work(case):
    c, kind = case, case["kind"]
    if kind == "step":
        B, H = c["bsz"], c["hidden"]
        norm = B * H * (2 + 4 + 4 + 2) + H * 2
        rope = B * 128 * 2 * (2 * c["hq"] + 4 * c["hk"]) + 2 * 128 * 2 + 256
        layer = 2 * norm + rope + 3 * B * c["inter"] * 2
        return dict(bytes=c["layers"] * layer + norm + B * c["vocab"] * 4, flops=c["layers"] * B * (20 * H + 6 * c["inter"]))
    if kind == "layer":
        T, H, hd, e = c["bsz"] * c["seq"], c["hidden"], c["hd"], 2
        norm = T * H * (2 * e + 2 * BYTES[c["res"]]) + H * e
        rope = T * hd * e * (2 * c["hq"] + 4 * c["hk"]) + 2 * hd * e
        return dict(bytes=2 * norm + rope + 3 * T * c["inter"] * e, flops=T * (10 * H + 10 * hd * (c["hq"] + c["hk"]) + 6 * c["inter"]))
    if kind == "rows":
        T, H = c["rows"], c["hidden"]
        return dict(bytes=T * H * (4 + 2 * BYTES[c["res"]]) + H * 2 + 3 * T * c["inter"] * 2, flops=T * (5 * H + 6 * c["inter"]))
    if kind == "embed":
        # the table rows that Zipf ids name at least once
        p = np.arange(1, c["vocab"] + 1, dtype=np.float64) ** -1.1
        distinct = float(np.sum(-np.expm1(c["n"] * np.log1p(-np.minimum(p / p.sum(), 0.999999)))))
        return dict(bytes=(distinct * 2 + c["n"] * (BYTES[c["out"]] + (2 if c["norm"] else 0))) * c["hidden"] + c["n"] * 8,
                    flops=c["n"] * c["hidden"] * (4 if c["norm"] else 0))
    if kind == "norm_had":
        n = c["rows"] * c["hidden"]
        return dict(bytes=n * (2 + 2 * BYTES[c["res"]] + 2 * c["n_out"]) + c["hidden"] * 2 * (2 + c["n_out"]),
                    flops=n * (5 + 8 * (c["n_out"] + int(c["rotate"]))))
    if kind == "mlp_had":
        n = c["rows"] * c["inter"]
        return dict(bytes=6 * n + c["inter"] * 2 * 3, flops=n * (6 + 8 * (1 + 2 * int(c["rotate"]))))
    if kind == "attn_had":
        T = c["bsz"] * c["seq"]
        return dict(bytes=T * 128 * 2 * (2 * c["hq"] + 4 * c["hk"]) + (c["hq"] + 2 * c["hk"]) * 256,
                    flops=T * 128 * 18 * (c["hq"] + 2 * c["hk"]))
    if kind == "gated_attn":
        T, n = c["tokens"], c["tokens"] * c["hq"] * c["hd"]
        return dict(bytes=n * 2 * 5 + T * c["hk"] * c["hd"] * 4 + T * 4, flops=n * 14)
    if kind == "mrope":
        T = c["bsz"] * c["seq"]
        return dict(bytes=T * (c["hq"] + c["hk"]) * c["hd"] * 4 + T * (c["hd"] // 2) * 4, flops=T * (c["hq"] + c["hk"]) * c["hd"] * 10)
    if kind == "gdn":
        n = c["tokens"] * c["heads"] * c["hd"]
        return dict(bytes=n * 8 + c["hd"] * 4 + c["heads"] * c["hd"] * 2, flops=n * (10 + 8 * int(c["had"])))
    n = c["rows"] * c["vocab"]
    return dict(bytes=n * BYTES[c["dtype"]] + c["rows"] * 8, flops=n * (12 if c["gumbel"] else 1))


# About four times the distance from 64-bit results: the rounding of the outputs' own type, where a head norm or
# a rotation's scale comes in between twice.  The paged caches are mostly empty here, so the largest difference,
# measured against a whole cache's root mean square, is far larger for them.
_F16 = {"rel": 1.6e-3, "max": 1.2e-2, "differ": 0}
_BF16 = {"rel": 1.2e-2, "max": 5e-2, "differ": 0}
_CACHES = {"f16": 0.2, "bf16": 0.9}


def tolerance(case):
    kind = case["kind"]
    if kind == "sample" or (kind == "embed" and not case["norm"]):
        return "exact"
    t = dict(_BF16 if case.get("dtype") == "bf16" else _F16)
    if kind in ("step", "layer", "attn_had"):
        t["max"] = _CACHES[case.get("dtype", "f16")]
    return t


# ------------------------------------------------------------------------------------------------
# The same results in 64 bits, in plain torch.

def _d(t):
    return t.double()


def _norm(x, w, bias=0.0):
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS)
    return y if w is None else y * (_d(w) + bias)


def _had(x, pre=None, post=None):
    """The 128-point transform of every block of 128 columns, in the natural (Sylvester) order."""
    shape = x.shape
    if pre is not None:
        x = x * _d(pre)
    h = torch.ones((1, 1), device=x.device, dtype=torch.float64)
    for _ in range(7):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    x = (x.reshape(-1, 128) @ h * HAD).reshape(shape)
    return x if post is None else x * _d(post)


def _rotate(x, angles, mode="neox"):
    """x [B, S, heads, hd], angles [B, S, R / 2]."""
    a = angles[:, :, None, :]
    c, sn, h = a.cos(), a.sin(), angles.shape[-1]
    y = x.clone()
    if mode == "neox":
        p, q = x[..., :h], x[..., h:2 * h]
        y[..., :h], y[..., h:2 * h] = p * c - q * sn, q * c + p * sn
    else:
        p, q = x[..., 0:2 * h:2], x[..., 1:2 * h:2]
        y[..., 0:2 * h:2], y[..., 1:2 * h:2] = p * c - q * sn, q * c + p * sn
    return y


def _angles(inv, pos):
    return (inv * pos.float().unsqueeze(-1)).double()   # the angle is a 32-bit product by definition


def _exact_attention(b, q, k, v, mode="neox"):
    B, S = q.shape[:2]
    pos = b["lens"].view(B, 1) + torch.arange(S, device="cuda", dtype=torch.int32).view(1, S)
    a = _angles(b["inv"], pos)
    q, k = (_rotate(_norm(t, w), a, mode) for t, w in ((q, b["qn"]), (k, b["kn"])))
    kc, vc = _d(b["kc"]), _d(b["vc"])
    page = torch.gather(b["table"].long(), 1, (pos // PAGE).long())
    kc[page, (pos % PAGE).long()], vc[page, (pos % PAGE).long()] = k, v
    return q, kc, vc


def _silu(x):
    return x * torch.sigmoid(x)


def _act(act, x, u):
    return (_silu(x) if act == "silu" else torch.nn.functional.gelu(x, approximate="tanh")) * u


def _exact_step(s):
    r, outs, pending = _d(s["emb"][s["ids"]]), [], None
    for b in s["blocks"]:
        r = r if pending is None else r + _d(pending)
        y1 = _norm(r, b["w1"])
        r = r + _d(b["a_out"])
        q, kc, vc = _exact_attention(b, _d(b["q"]), _d(b["k"]), _d(b["v"]))
        outs.append([y1, _norm(r, b["w2"]), _act("silu", _d(b["gate"]), _d(b["up"])), q, kc, vc])
        pending = b["m_out"]
    r = r + _d(pending)
    return [r, _norm(r, s["wf"]), None] + [t for o in outs[-4:] for t in o]


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return None
    s = prepare(case, seed)
    if kind == "step":
        return _exact_step(s)
    if kind == "layer":
        r1 = _d(s["r"]) + _d(s["x1"])
        r2 = r1 + _d(s["x2"])
        q, kc, vc = _exact_attention(s, _d(s["q"]), _d(s["k"]), _d(s["v"]))
        return [_norm(r1, s["w1"]), _norm(r2, s["w2"]), r2, _act("silu", _d(s["gate"]), _d(s["up"])), q, kc, vc]
    if kind == "rows":
        r = _d(s["r"]) + _d(s["x"])
        return [_norm(r, s["w"]), r, _act(s["act"], _d(s["gate"]), _d(s["up"]))]
    if kind == "embed":
        h = _d(s["rows"][s["ids"]])
        return [h, _norm(h, s["w"])] if s["norm"] else [h]
    if kind == "norm_had":
        x = _had(_d(s["x"]), post=s["post"]) if s["rotate"] else _d(s["x"])
        r = _d(s["r"]) + x
        y = _norm(r, s["w"])
        return [_had(y, p) for p in s["pre"]] + [r]
    if kind == "mlp_had":
        g, u = _d(s["gate"]), _d(s["up"])
        if s["rotate"]:
            g, u = _had(g, post=s["gp"]), _had(u, post=s["upp"])
        return [_had(_act(s["act"], g, u), s["pre"])]
    if kind == "attn_had":
        q, k, v = (_had(_d(s[n]).flatten(2), post=s["s" + n]).view_as(s[n]) for n in "qkv")
        return list(_exact_attention(s, q, k, v, s["mode"]))
    if kind == "gated_attn":
        hd = s["hd"]
        a = _angles(s["inv"], s["pos"])
        q = _rotate(_norm(_d(s["qg"][..., :hd]), s["qn"], 1.0), a)
        k = _rotate(_norm(_d(s["k"]), s["kn"], 1.0), a)
        return [q, k, _d(s["o"]) * torch.sigmoid(_d(s["qg"][..., hd:]).reshape(-1, hd))]
    if kind == "mrope":
        a = _d(s["angles"]).view(-1, s["seq"], s["angles"].shape[-1])
        q, k = _d(s["q"]), _d(s["k"])
        if s["norm"]:
            q, k = _norm(q, s["qn"]), _norm(k, s["kn"])
        return [_rotate(q, a), _rotate(k, a)]
    y = _norm(_d(s["x"]), s["w"]) * _silu(_d(s["g"]))
    return [_had(y.view(-1, s["heads"] * s["hd"]), s["pre"]).view_as(y) if s["had"] else y]
