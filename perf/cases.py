"""The work this engine does for its users, as timed cases: single layers through the kernel ABI (include/sn_kernels.h)
and whole steps through sn_step (include/sn.h), at the sizes of the repository's own configurations (the 4B dense model,
the 30B mixture of experts, the 4096 x 4096 matmul, prompt steps of 512 rows) and ragged ones between them.

  linear   RMSNorm + Q8_0 operand + one Q4_0 or Q8_0 matmul (a projection)
  mlp      RMSNorm + operand, gate|up with SwiGLU, operand, down
  attn     a whole attention layer: norm + operand, q|k|v, QK-norm + RoPE + cache write, paged attention, operand, o
  head     norm + Q8_K operand, Q6_K LM head, greedy argmax
  moe      router, top-k and grouping, gathered operand, grouped gate|up expert matmul
  engine   sn_step of a model (a few layers of the 4B shape) with logits of the rows that asked for them

A row's result is the oracle's arithmetic (Q8_0 / Q8_K activations, integer block sums, fp16 cache); exact() gives the
same in 64-bit torch, the quantizations being part of what is computed.
"""
import ctypes as C
import math
import os
import struct
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "sonic-llm_amd"))
import sllm_next as S  # noqa: E402

EPS = 1e-6
ROPE_BASE = 1e6
F64 = torch.float64

# (E, H, KVH, F) of the repository's models: the 4B dense, the 30B-A3B's attention and dense width, the 0.6B fixture
DENSE_4B = dict(E=2560, H=32, KVH=8, F=9728)
MOE_30B = dict(E=2048, H=32, KVH=4, F=6144)
SMALL = dict(E=1024, H=16, KVH=8, F=3072)
ENGINE = dict(layers=6, V=32000, **DENSE_4B)


def listed():
    return [
        # the o projection of one chat's decode row: the smallest call there is
        dict(name="linear_q4_1", kind="linear", M=1, N=2560, K=4096, wt=2),
        # the single-matmul configuration: 8 rows, 4096 x 4096
        dict(name="linear_q4_8", kind="linear", M=8, N=4096, K=4096, wt=2),
        # q|k|v of a Q8_0 model over a mixed step of 100 rows (chats, drafts under check and a prompt's tail)
        dict(name="linear_q8_100", kind="linear", M=100, N=6144, K=2560, wt=8),
        # a decode step's MLP, 32 sequences
        dict(name="mlp_32", kind="mlp", M=32, E=2560, F=9728),
        # a short prompt of odd length
        dict(name="mlp_333", kind="mlp", M=333, E=2560, F=9728),
        # a large prompt chunk: the largest call
        dict(name="mlp_2048", kind="mlp", M=2048, E=2560, F=9728),
        # a decode step's attention layer: 32 sequences, contexts spread over 256..4096, 64-cell pages
        dict(name="attn_decode_32", kind="attn", n_seq=32, rows=1, lo=256, hi=4096, page=64, E=2560, H=32, KVH=8),
        # a prompt step's attention layer: 512 rows of one prompt behind 1536 cells
        dict(name="attn_prompt_512", kind="attn", n_seq=1, rows=512, lo=1536, hi=1536, page=64, E=2560, H=32, KVH=8),
        # the LM head of the published files (Q6_K) for 32 sampled rows
        dict(name="head_q6k_32", kind="head", M=32, N=151936, K=2560),
        # a decode step's routing and gate|up experts, 32 rows, 8 of 128 experts
        dict(name="moe_32", kind="moe", R=32, E=2048, N=1536, NE=128, k=8),
        # a decode step of 32 chats at 2048 cells; two of them sample from their logits
        dict(name="step_decode_32", kind="engine", n_seq=32, rows=1, ctx=2048, n_logits=2),
        # a 512-row prompt step, the prompt's second chunk, its last row sampled from its logits
        dict(name="step_prompt_512", kind="engine", n_seq=1, rows=512, ctx=512, n_logits=1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "mlp", "mlp", "attn_d", "attn_d", "attn_p", "attn_p", "head", "moe",
                       "engine_d", "engine_p"])
    model = rng.choice([DENSE_4B, DENSE_4B, MOE_30B, SMALL])
    att = {k: model[k] for k in ("E", "H", "KVH")}
    if kind == "linear":
        return dict(kind="linear", M=_log(rng, 1, 1024), N=_log(rng, 1000, 12000), K=32 * _log(rng, 32, 300),
                    wt=rng.choice([2, 2, 8]))
    if kind == "mlp":
        return dict(kind="mlp", M=_log(rng, 1, 2000), E=model["E"], F=model["F"])
    if kind == "attn_d":  # decode rows, or a few draft rows a sequence under check
        lo = _log(rng, 16, 3000)
        return dict(kind="attn", n_seq=_log(rng, 1, 48), rows=rng.choice([1, 1, 1, 2, 4, 5]), lo=lo,
                    hi=_log(rng, lo, 4096), page=rng.choice([32, 64, 64]), **att)
    if kind == "attn_p":  # prompts
        n = rng.choice([1, 1, 1, 2, 4])
        lo = rng.choice([0, _log(rng, 16, 3000)])
        return dict(kind="attn", n_seq=n, rows=max(8, _log(rng, 32, 1024) // n), lo=lo, hi=lo, page=64, **att)
    if kind == "head":
        return dict(kind="head", M=_log(rng, 1, 64), N=rng.choice([151936, 32000, 100003]), K=rng.choice([1024, 2048, 2560]))
    if kind == "moe":
        return dict(kind="moe", R=_log(rng, 1, 512), E=2048, N=1536, NE=128, k=8)
    if kind == "engine_d":
        return dict(kind="engine", n_seq=_log(rng, 1, 40), rows=rng.choice([1, 1, 4]), ctx=_log(rng, 64, 2048), n_logits=1)
    return dict(kind="engine", n_seq=1, rows=_log(rng, 48, 512), ctx=rng.choice([0, 64, 512, 1024]), n_logits=1)


def _contexts(c):
    """The sequences' cells before this step, spread evenly over lo..hi."""
    n = c["n_seq"]
    return [c["lo"] + (c["hi"] - c["lo"]) * i // max(1, n - 1) for i in range(n)]


def work(c):
    kind = c["kind"]
    if kind == "linear":
        M, N, K = c["M"], c["N"], c["K"]
        return {"bytes": N * K * (18 if c["wt"] == 2 else 34) / 32 + 4 * M * (N + K), "flops": 2.0 * M * N * K}
    if kind == "mlp":
        M, E, F = c["M"], c["E"], c["F"]
        return {"bytes": 3 * E * F * 18 / 32 + 8 * M * E, "flops": 6.0 * M * E * F}
    if kind == "attn":
        M, E, H, KVH = c["n_seq"] * c["rows"], c["E"], c["H"], c["KVH"]
        w = (2 * H + 2 * KVH) * 128 * E
        cells = sum(x + c["rows"] for x in _contexts(c))
        pairs = sum(c["rows"] * x + c["rows"] * (c["rows"] + 1) / 2 for x in _contexts(c))
        return {"bytes": w * 18 / 32 + 8 * M * E + cells * KVH * 128 * 4, "flops": 2.0 * M * w + pairs * H * 128 * 4}
    if kind == "head":
        M, N, K = c["M"], c["N"], c["K"]
        return {"bytes": N * K * 210 / 256 + 4 * M * (N + K), "flops": 2.0 * M * N * K}
    if kind == "moe":
        R, E, N, NE, k = c["R"], c["E"], c["N"], c["NE"], c["k"]
        used = NE * (1 - (1 - k / NE) ** R)  # experts that R rows of k choices reach
        return {"bytes": used * N * E * 18 / 32 + 4 * NE * E + 4 * R * E + 4 * R * k * N, "flops": 2.0 * R * k * N * E}
    m = ENGINE
    M, E, H, KVH, F = c["n_seq"] * c["rows"], m["E"], m["H"], m["KVH"], m["F"]
    w = (2 * H + 2 * KVH) * 128 * E + 3 * E * F
    out = c["n_seq"]
    pairs = c["n_seq"] * (c["rows"] * c["ctx"] + c["rows"] * (c["rows"] + 1) / 2)
    return {"bytes": m["layers"] * (w * 18 / 32 + c["n_seq"] * (c["ctx"] + c["rows"]) * KVH * 128 * 4) +
                     m["V"] * E * 18 / 32 + 4 * out * m["V"],
            "flops": m["layers"] * (2.0 * M * w + pairs * H * 128 * 4) + 2.0 * out * m["V"] * E}


def tolerance(c):
    # about four times what another correct path shows. linear, head, moe: 32-bit sums of exact integer block sums, at
    # most one quantization flip of a normed value between rsqrt roundings. mlp, attn: a second quantization sits
    # inside, whose flips (one step of 1/127 of a block's largest value) follow from the last bits of the first sums.
    # engine: those flips through six layers of a random model (the 64-bit path, with the same quantizations, is
    # 0.03 off a prompt step's logits and 0.003 off a decode step's).
    return {"linear": {"rel": 4e-4, "max": 0.1}, "head": {"rel": 4e-4, "max": 0.1, "differ": 0.01},
            "moe": {"rel": 4e-4, "max": 0.1}, "mlp": {"rel": 2e-3, "max": 0.2},
            "attn": {"rel": 2e-3, "max": 0.2}, "engine": {"rel": 3e-2, "max": 0.5}}[c["kind"]]


# ---- inputs ---------------------------------------------------------------------------------------------------------
def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000003 + salt)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _q4_blocks(g, N, K, std=0.02):
    """GGUF Q4_0 rows (18-byte blocks: fp16 d, 16 bytes of nibbles) of N x K normal weights."""
    x = _randn(g, N, K // 32, 32) * std
    m = torch.gather(x, 2, x.abs().argmax(2, keepdim=True))
    d = m / -8
    q = torch.clamp(torch.floor(x * torch.where(d != 0, 1 / d, 0) + 8.5), 0, 15).to(torch.uint8)
    out = torch.empty(N, K // 32, 18, dtype=torch.uint8, device="cuda")
    out[:, :, :2] = d.half().view(torch.uint8).view(N, K // 32, 2)
    out[:, :, 2:] = q[:, :, :16] | (q[:, :, 16:] << 4)
    return out


def _q8_blocks(g, N, K, std=0.02):
    """GGUF Q8_0 rows (34-byte blocks: fp16 d, 32 int8)."""
    x = _randn(g, N, K // 32, 32) * std
    d = x.abs().amax(2, keepdim=True) / 127
    q = torch.round(x / d).to(torch.int8)
    out = torch.empty(N, K // 32, 34, dtype=torch.uint8, device="cuda")
    out[:, :, :2] = d.half().view(torch.uint8).view(N, K // 32, 2)
    out[:, :, 2:] = q.view(torch.uint8)
    return out


def _q6k_blocks(g, N, K):
    """GGUF Q6_K rows (210-byte blocks: ql[128], qh[64], int8 scales[16], fp16 d)."""
    out = torch.randint(0, 256, (N, K // 256, 210), generator=g, device="cuda", dtype=torch.uint8)
    sc = torch.randint(-15, 16, (N, K // 256, 16), generator=g, device="cuda", dtype=torch.int8)
    d = (_randn(g, N, K // 256, 1).abs() * 5e-5 + 2e-5).half()
    out[:, :, 192:208] = sc.view(torch.uint8)
    out[:, :, 208:] = d.view(torch.uint8).view(N, K // 256, 2)
    return out


def _inputs(c, seed):
    """The host-visible inputs of a case (raw GGUF weights, rows, cache), from the seed alone."""
    g, kind = _gen(seed, 1), c["kind"]
    blocks = _q8_blocks if c.get("wt") == 8 else _q4_blocks
    if kind == "linear":
        return dict(w=blocks(g, c["N"], c["K"]), x=_randn(g, c["M"], c["K"]), nw=1 + 0.1 * _randn(g, c["K"]))
    if kind == "mlp":
        return dict(gu=_q4_blocks(g, 2 * c["F"], c["E"]), dn=_q4_blocks(g, c["E"], c["F"]),
                    x=_randn(g, c["M"], c["E"]), nw=1 + 0.1 * _randn(g, c["E"]))
    if kind == "head":
        return dict(w=_q6k_blocks(g, c["N"], c["K"]), x=_randn(g, c["M"], c["K"]), nw=1 + 0.1 * _randn(g, c["K"]))
    if kind == "moe":
        return dict(w=_q4_blocks(g, c["NE"] * c["N"], c["E"]), x=_randn(g, c["R"], c["E"]),
                    router=_randn(g, c["NE"], c["E"]) / math.sqrt(c["E"]))
    if kind == "attn":
        H, KVH, E, pc, rows = c["H"], c["KVH"], c["E"], c["page"], c["rows"]
        r = np.random.default_rng(seed)
        ctx = r.permutation(_contexts(c)).astype(np.int32)
        need = [(int(x) + rows + pc - 1) // pc for x in ctx]
        n_pages = sum(need) + 3
        perm, at = r.permutation(n_pages).astype(np.int32), 0
        pt = np.full((c["n_seq"], max(need)), -1, np.int32)
        for s, n in enumerate(need):
            pt[s, :n] = perm[at:at + n]
            at += n
        pool = torch.Generator(device="cuda")
        pool.manual_seed(seed * 7919 + 5)
        shape = (n_pages, KVH, pc * 128)
        return dict(wqkv=_q4_blocks(g, (H + 2 * KVH) * 128, E), wo=_q4_blocks(g, E, H * 128),
                    x=_randn(g, c["n_seq"] * rows, E), nw=1 + 0.1 * _randn(g, E), qw=1 + 0.1 * _randn(g, 128),
                    kw=1 + 0.1 * _randn(g, 128), ctx=ctx, pt=pt,
                    seq=np.repeat(np.arange(c["n_seq"], dtype=np.int32), rows),
                    pos=(ctx[:, None] + np.arange(rows, dtype=np.int32)).reshape(-1).astype(np.int32),
                    k=torch.randn(shape, generator=pool, device="cuda", dtype=torch.float16),
                    v=torch.randn(shape, generator=pool, device="cuda", dtype=torch.float16))
    n, rows, ctx, m = c["n_seq"], c["rows"], c["ctx"], ENGINE
    r = np.random.default_rng(seed)
    # sn_kv_load's layout: per layer K then V, each [cells][KVH * 128] fp16
    kv = None
    if ctx:
        kv = torch.randn(n, m["layers"], 2, ctx, m["KVH"] * 128, generator=g, device="cuda", dtype=torch.float16)
    return dict(tok=r.integers(0, m["V"], n * rows).astype(np.int32),
                seq=np.repeat(np.arange(n, dtype=np.int32), rows),
                pos=np.tile(ctx + np.arange(rows, dtype=np.int32), n).astype(np.int32),
                out=(np.arange(1, n + 1, dtype=np.int32) * rows - 1).astype(np.int32),
                logit_rows=np.sort(r.permutation(n)[:min(n, c["n_logits"])]).astype(np.int32), kv=kv)


def _model():
    """The engine cases' model file, written once a machine (random weights, as the benchmark's)."""
    m = ENGINE
    path = os.path.join(tempfile.gettempdir(), "sn_cases_%dL_%d_%d_%d.gguf" % (m["layers"], m["E"], m["V"], os.getuid()))
    if not os.path.exists(path):
        part = "%s.%d" % (path, os.getpid())
        S.write_model(part, S.model_cfg(m["layers"], m["E"], m["H"], m["KVH"], m["F"], m["V"], rope_base=ROPE_BASE, eps=EPS), 42)
        os.replace(part, path)
    return path


# ---- what a program keeps: weights in the library's layout, work lists, workspaces, an open engine -------------------
class _Handle:
    """A library handle given back when its state is dropped."""

    def __init__(self, h, free):
        self.h, self.free = h, free

    def __del__(self):
        if self.h:
            self.free(self.h)
            self.h = None


def _p(t):
    return t.data_ptr() if t is not None else None


def _st():
    return torch.cuda.current_stream().cuda_stream


def _buf(n):
    return torch.zeros(max(int(n), 256), dtype=torch.uint8, device="cuda")


def _ok(rc):
    if rc != 0:
        raise RuntimeError("the library returned %d" % rc)


def _q4_tiles(blocks, N, K):
    L = S.lib()
    t = _buf(L.snk_q4_stripes_bytes(N, K))
    _ok(L.snk_q4_repack(_p(blocks), N, K, _p(t), _st()))
    return t


def prepare(c, seed):
    L, kind, i = S.lib(), c["kind"], _inputs(c, seed)
    f32 = dict(dtype=torch.float32, device="cuda")
    s = dict(kind=kind, c=c, x=i.get("x"), nw=i.get("nw"))
    if kind == "linear":
        M, N, K = c["M"], c["N"], c["K"]
        if c["wt"] == 2:
            s["w"], s["ws"] = _q4_tiles(i["w"], N, K), _buf(L.snk_q4_workspace_bytes(M, N, K))
        else:
            s["w"], s["ws"] = _buf(L.snk_q8_tiles_bytes(N, K)), _buf(L.snk_q8_workspace_bytes(M, N, K))
            _ok(L.snk_q8_repack(_p(i["w"]), N, K, _p(s["w"]), _st()))
        s["xa"], s["y"] = _buf(L.snk_xa_bytes(M, K)), torch.empty(M, N, **f32)
    elif kind == "mlp":
        M, E, F = c["M"], c["E"], c["F"]
        s["gu"], s["dn"] = _q4_tiles(i["gu"], 2 * F, E), _q4_tiles(i["dn"], E, F)
        s["xa"], s["xh"] = _buf(L.snk_xa_bytes(M, E)), _buf(L.snk_xa_bytes(M, F))
        s["h"], s["y"] = torch.empty(M, F, **f32), torch.empty(M, E, **f32)
        s["ws"] = _buf(max(L.snk_q4_workspace_bytes(M, 2 * F, E), L.snk_q4_workspace_bytes(M, E, F)))
    elif kind == "head":
        M, N, K = c["M"], c["N"], c["K"]
        s["w"], s["xk"] = _buf(L.snk_q6k_tiles_bytes(N, K)), _buf(L.snk_xk_bytes(M, K))
        _ok(L.snk_q6k_repack(_p(i["w"]), N, K, _p(s["w"]), _st()))
        s["y"], s["tok"] = torch.empty(M, N, **f32), torch.empty(M, dtype=torch.int32, device="cuda")
        s["ws"] = _buf(L.snk_argmax_workspace_bytes(M, N))
    elif kind == "moe":
        R, E, N, NE, k = c["R"], c["E"], c["N"], c["NE"], c["k"]
        P = L.snk_moe_tile_rows(R, NE, k)
        i32 = dict(dtype=torch.int32, device="cuda")
        s.update(P=P, router=i["router"], w=_q4_tiles(i["w"], NE * N, E), stride=L.snk_q4_stripes_bytes(N, E),
                 lg=torch.empty(R, NE, **f32), ids=torch.empty(R, k, **i32), pw=torch.empty(R, k, **f32),
                 prow=torch.empty(R, k, **i32), rsrc=torch.full((P,), -1, **i32), items=torch.zeros(P // 16, 2, **i32),
                 count=torch.zeros(1, **i32), xa=_buf(L.snk_xa_bytes(P, E)), part=torch.zeros(P, N, **f32))
    elif kind == "attn":
        M, E, H, KVH = c["n_seq"] * c["rows"], c["E"], c["H"], c["KVH"]
        N = (H + 2 * KVH) * 128
        err = C.create_string_buffer(512)
        h = L.snk_attn_new(M, S._p(i["seq"]), S._p(i["pos"]), H, KVH, i["pt"].shape[1], c["page"], err, 512)
        if not h:
            raise RuntimeError(err.value.decode())
        s.update(plan=_Handle(h, L.snk_attn_free), wqkv=_q4_tiles(i["wqkv"], N, E), wo=_q4_tiles(i["wo"], E, H * 128),
                 qw=i["qw"], kw=i["kw"], k=i["k"], v=i["v"], max_pages=i["pt"].shape[1],
                 pt=torch.from_numpy(i["pt"]).cuda(), seq=torch.from_numpy(i["seq"]).cuda(),
                 pos=torch.from_numpy(i["pos"]).cuda(), xa=_buf(L.snk_xa_bytes(M, E)), xo=_buf(L.snk_xa_bytes(M, H * 128)),
                 qkv=torch.empty(M, N, **f32), ao=torch.empty(M, H * 128, **f32), y=torch.empty(M, E, **f32),
                 ws=_buf(max(L.snk_q4_workspace_bytes(M, N, E), L.snk_q4_workspace_bytes(M, E, H * 128))),
                 theta=float(np.float32(np.power(np.float32(ROPE_BASE), np.float32(-2.0 / 128)))))
    else:
        n, rows, ctx = c["n_seq"], c["rows"], c["ctx"]
        eng = S.Engine(_model(), slots=n, ctx=(ctx + rows + 63) // 64 * 64, max_rows=max(n * rows, 16))
        s.update(eng=eng, keep=_Handle(eng, lambda e: e.close()), tok=i["tok"], seq=i["seq"], pos=i["pos"], out=i["out"],
                 logit_rows=i["logit_rows"], n_write=n * rows if rows <= 5 else 0)
        if i["kv"] is not None:
            for q in range(n):
                eng.kv_load(q, ctx, i["kv"][q].cpu().numpy().view(np.uint16))
    torch.cuda.synchronize()
    return s


def run(s):
    L, c, kind, st = S.lib(), s["c"], s["kind"], _st()
    if kind == "linear":
        M, N, K = c["M"], c["N"], c["K"]
        _ok(L.snk_quant_act(_p(s["x"]), M, K, K, _p(s["nw"]), EPS, _p(s["xa"]), st))
        gemm = L.snk_q4_gemm if c["wt"] == 2 else L.snk_q8_gemm
        _ok(gemm(_p(s["w"]), _p(s["xa"]), M, N, K, _p(s["y"]), N, 0, _p(s["ws"]), s["ws"].numel(), st))
        return s["y"]
    if kind == "mlp":
        M, E, F = c["M"], c["E"], c["F"]
        _ok(L.snk_quant_act(_p(s["x"]), M, E, E, _p(s["nw"]), EPS, _p(s["xa"]), st))
        # prompt rows take the matmul whose epilogue writes the next one's operand; it answers 1 where it does not apply
        rc = L.snk_q4_gemm_swiglu(_p(s["gu"]), _p(s["xa"]), M, 2 * F, E, _p(s["h"]), _p(s["xh"]), st)
        if rc == 1:
            _ok(L.snk_q4_gemm(_p(s["gu"]), _p(s["xa"]), M, 2 * F, E, _p(s["h"]), F, 2, _p(s["ws"]), s["ws"].numel(), st))
            _ok(L.snk_quant_act(_p(s["h"]), M, F, F, None, EPS, _p(s["xh"]), st))
        else:
            _ok(rc)
        _ok(L.snk_q4_gemm(_p(s["dn"]), _p(s["xh"]), M, E, F, _p(s["y"]), E, 0, _p(s["ws"]), s["ws"].numel(), st))
        return {"h": s["h"], "y": s["y"]}
    if kind == "head":
        M, N, K = c["M"], c["N"], c["K"]
        _ok(L.snk_quant_q8k(_p(s["x"]), M, K, K, _p(s["nw"]), EPS, _p(s["xk"]), st))
        _ok(L.snk_q6k_gemm(_p(s["w"]), _p(s["xk"]), M, N, K, _p(s["y"]), N, st))
        _ok(L.snk_argmax(_p(s["y"]), N, M, None, 0, None, _p(s["tok"]), None, _p(s["ws"]), s["ws"].numel(), st))
        return {"logits": s["y"], "tokens": s["tok"]}
    if kind == "moe":
        R, E, N, NE, k, P = c["R"], c["E"], c["N"], c["NE"], c["k"], s["P"]
        _ok(L.snk_moe_router(_p(s["x"]), R, E, _p(s["router"]), NE, _p(s["lg"]), st))
        _ok(L.snk_moe_select(_p(s["lg"]), R, NE, k, _p(s["ids"]), _p(s["pw"]), _p(s["prow"]), _p(s["rsrc"]),
                             _p(s["items"]), _p(s["count"]), st))
        rows = s["x"].index_select(0, s["rsrc"].clamp_min(0))
        _ok(L.snk_quant_act(_p(rows), P, E, E, None, EPS, _p(s["xa"]), st))
        _ok(L.snk_gemm_grouped(2, _p(s["w"]), s["stride"], _p(s["items"]), _p(s["count"]), P // 16, _p(s["xa"]), P, N, E,
                               _p(s["part"]), s["part"].numel() * 4, _p(s["rsrc"]), st))
        return {"ids": s["ids"], "weights": s["pw"], "rows": s["part"]}
    if kind == "attn":
        M, E, H, KVH, plan = c["n_seq"] * c["rows"], c["E"], c["H"], c["KVH"], s["plan"].h
        N, QD = (H + 2 * KVH) * 128, H * 128
        _ok(L.snk_quant_act(_p(s["x"]), M, E, E, _p(s["nw"]), EPS, _p(s["xa"]), st))
        _ok(L.snk_q4_gemm(_p(s["wqkv"]), _p(s["xa"]), M, N, E, _p(s["qkv"]), N, 0, _p(s["ws"]), s["ws"].numel(), st))
        _ok(L.snk_qk_rope(_p(s["qkv"]), N, M, H, KVH, _p(s["qw"]), _p(s["kw"]), EPS, s["theta"], _p(s["seq"]),
                          _p(s["pos"]), _p(s["pt"]), s["max_pages"], c["page"], _p(s["k"]), _p(s["v"]), st))
        _ok(L.snk_attn_run(plan, _p(s["qkv"]), N, _p(s["k"]), _p(s["v"]), _p(s["pt"]), 1 / math.sqrt(128), _p(s["ao"]),
                           QD, st))
        _ok(L.snk_quant_act(_p(s["ao"]), M, QD, QD, None, EPS, _p(s["xo"]), st))
        _ok(L.snk_q4_gemm(_p(s["wo"]), _p(s["xo"]), M, E, QD, _p(s["y"]), E, 0, _p(s["ws"]), s["ws"].numel(), st))
        return {"attention": s["ao"], "y": s["y"], "k": s["k"], "v": s["v"]}
    tok = s["eng"].step(s["tok"], s["seq"], s["pos"], s["out"], n_write=s["n_write"])
    return {"logits": s["eng"].logits(s["logit_rows"]), "tokens": tok}


# ---- the same in 64 bits --------------------------------------------------------------------------------------------
def _w4(b):
    """Q4_0 blocks [..., K / 32, 18] as 64-bit weights [..., K]."""
    d = b[..., :2].contiguous().view(torch.float16).to(F64)
    q = torch.cat([b[..., 2:] & 15, b[..., 2:] >> 4], -1).to(F64) - 8
    return (q * d).flatten(-2)


def _w8(b):
    d = b[..., :2].contiguous().view(torch.float16).to(F64)
    return (b[..., 2:].contiguous().view(torch.int8).to(F64) * d).flatten(-2)


def _w6k(b):
    """Q6_K blocks: element e = 128 h + 32 c + l has its low 4 bits in ql[64 h + 32 (c % 2) + l] (nibble c / 2), its
    high 2 at bit 2 c of qh[32 h + l], and the scale of its 16-element group."""
    lead = b.shape[:-1]
    ql, qh = b[..., :128].reshape(*lead, 2, 2, 32), b[..., 128:192].reshape(*lead, 2, 1, 32)
    low = torch.stack([ql[..., 0, :] & 15, ql[..., 1, :] & 15, ql[..., 0, :] >> 4, ql[..., 1, :] >> 4], -2)
    sh = torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.uint8)[:, None]
    q = (low | (((qh >> sh) & 3) << 4)).reshape(*lead, 16, 16).to(F64) - 32
    sc = b[..., 192:208].contiguous().view(torch.int8).to(F64)
    d = b[..., 208:].contiguous().view(torch.float16).to(F64)
    return (q * (sc * d)[..., None]).flatten(-3)


def _norm(x, w):
    x = x.to(F64)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.to(F64)


def _q8_0(x):
    """Rows rounded to Q8_0: per 32 values q = round(127 x / amax), d = amax / 127 in fp16."""
    b = x.to(F64).reshape(*x.shape[:-1], -1, 32)
    a = b.abs().amax(-1, keepdim=True)
    return (torch.round(b * torch.where(a > 0, 127 / a, 0)) * (a / 127).float().half().to(F64)).reshape(x.shape)


def _q8_k(x):
    """Rows rounded to Q8_K: per 256 values q = min(127, round(x * -127 / max)), d = max / -127, max the value of
    largest magnitude (the first on ties)."""
    b = x.to(F64).reshape(*x.shape[:-1], -1, 256)
    m = torch.gather(b, -1, b.abs().argmax(-1, keepdim=True))
    q = torch.clamp_max(torch.round(b * torch.where(m != 0, -127 / m, 0)), 127)
    return (q * (m / -127)).reshape(x.shape)


def _swiglu(g, u):
    return g * torch.sigmoid(g) * u


def _rope(x, w, pos):
    """Heads [M][n][128] normed by w and rotated (pairs i, i + 64); the angles by successive 32-bit multiplies, as the
    model's rotation is defined."""
    x = _norm(x, w)
    th = pos.to(torch.float32)
    scale = torch.tensor(float(np.float32(np.power(np.float32(ROPE_BASE), np.float32(-2.0 / 128)))), device=x.device, dtype=torch.float32)
    ths = []
    for _ in range(64):
        ths.append(th)
        th = th * scale
    t = torch.stack(ths, -1).to(F64)[:, None, :]
    a, b = x[..., :64], x[..., 64:]
    return torch.cat([a * t.cos() - b * t.sin(), a * t.sin() + b * t.cos()], -1)


def _attend(q, k, v, first):
    """q [R][H][128] at positions first.., k and v [cells][KVH][128]."""
    R, H, _ = q.shape
    KVH = k.shape[1]
    out = torch.empty_like(q)
    cells = torch.arange(k.shape[0], device=q.device)
    mask = cells[None, :] > (first + torch.arange(R, device=q.device))[:, None]
    for h in range(H):
        s = (q[:, h] @ k[:, h * KVH // H].T) / math.sqrt(128)
        out[:, h] = torch.softmax(s.masked_fill(mask, -math.inf), -1) @ v[:, h * KVH // H]
    return out


def _exact_engine(c, i):
    m, n, rows, ctx = ENGINE, c["n_seq"], c["rows"], c["ctx"]
    E, H, KVH = m["E"], m["H"], m["KVH"]
    raw = np.memmap(_model(), np.uint8, mode="r")
    at = [24]

    def num(fmt):
        v = struct.unpack_from("<" + fmt, raw, at[0])[0]
        at[0] += struct.calcsize(fmt)
        return v

    def text():
        k = num("Q")
        at[0] += k
        return bytes(raw[at[0] - k:at[0]]).decode()

    n_t, n_kv = struct.unpack_from("<QQ", raw, 8)
    size = {0: 1, 1: 1, 2: 2, 3: 2, 4: 4, 5: 4, 6: 4, 7: 1, 10: 8, 11: 8, 12: 8}
    for _ in range(n_kv):
        text()
        t = num("I")
        if t == 8:
            text()
        elif t == 9:
            it, k = num("I"), num("Q")
            for _ in range(k):
                text() if it == 8 else at.__setitem__(0, at[0] + size[it])
        else:
            at[0] += size[t]
    table = {}
    for _ in range(n_t):
        name, dims = text(), num("I")
        ne = [num("Q") for _ in range(dims)]
        table[name] = (ne, num("I"), num("Q"))
    data = (at[0] + 31) // 32 * 32

    def w(name):
        ne, t, off = table[name]
        r = int(np.prod(ne[1:])) if len(ne) > 1 else 1
        nb = {0: 4 * ne[0], 2: ne[0] // 32 * 18}[t]
        b = torch.from_numpy(np.array(raw[data + off:data + off + r * nb])).cuda()
        return b.view(torch.float32).reshape(r, ne[0]).squeeze(0) if t == 0 else _w4(b.reshape(r, -1, 18))

    pos = torch.from_numpy(i["pos"]).cuda()
    x = w("token_embd.weight")[torch.from_numpy(i["tok"]).long().cuda()].to(F64)
    for l in range(m["layers"]):
        p = "blk.%d." % l
        a = _q8_0(_norm(x, w(p + "attn_norm.weight")))
        q = _rope((a @ w(p + "attn_q.weight").T).reshape(-1, H, 128), w(p + "attn_q_norm.weight"), pos)
        k = _rope((a @ w(p + "attn_k.weight").T).reshape(-1, KVH, 128), w(p + "attn_k_norm.weight"), pos).half().to(F64)
        v = (a @ w(p + "attn_v.weight").T).reshape(-1, KVH, 128).half().to(F64)
        o = torch.empty_like(q)
        for s in range(n):
            r = slice(s * rows, (s + 1) * rows)
            ks, vs = k[r], v[r]
            if ctx:
                old = i["kv"][s, l].to(F64).reshape(2, ctx, KVH, 128)
                ks, vs = torch.cat([old[0], ks]), torch.cat([old[1], vs])
            o[r] = _attend(q[r], ks, vs, ctx)
        x = x + _q8_0(o.reshape(-1, H * 128)) @ w(p + "attn_output.weight").T
        a = _q8_0(_norm(x, w(p + "ffn_norm.weight")))
        x = x + _q8_0(_swiglu(a @ w(p + "ffn_gate.weight").T, a @ w(p + "ffn_up.weight").T)) @ w(p + "ffn_down.weight").T
    rows_out = torch.from_numpy(i["out"][i["logit_rows"]]).long().cuda()
    return {"logits": _q8_0(_norm(x[rows_out], w("output_norm.weight"))) @ w("output.weight").T, "tokens": None}


def exact(c, seed):
    kind, i = c["kind"], _inputs(c, seed)
    if kind == "linear":
        return _q8_0(_norm(i["x"], i["nw"])) @ (_w4 if c["wt"] == 2 else _w8)(i["w"]).T
    if kind == "mlp":
        a = _q8_0(_norm(i["x"], i["nw"])) @ _w4(i["gu"]).T
        a = a.reshape(c["M"], -1, 2, 16)  # 16 gate columns, then their 16 up columns
        h = _swiglu(a[:, :, 0], a[:, :, 1]).reshape(c["M"], c["F"])
        return {"h": h, "y": _q8_0(h) @ _w4(i["dn"]).T}
    if kind == "head":
        y = _q8_k(_norm(i["x"], i["nw"])) @ _w6k(i["w"]).T
        return {"logits": y, "tokens": None}
    if kind == "moe":
        R, N, NE, k = c["R"], c["N"], c["NE"], c["k"]
        x = i["x"].to(F64)
        lg = x @ i["router"].to(F64).T
        ids = torch.sort(lg, dim=-1, descending=True, stable=True).indices[:, :k]
        wt = torch.gather(torch.softmax(lg, -1), 1, ids)
        part = torch.zeros(S.lib().snk_moe_tile_rows(R, NE, k), N, device="cuda", dtype=F64)
        a, w, at = _q8_0(x), i["w"].reshape(NE, N, -1, 18), 0
        for e in range(NE):  # an expert's rows in order, from a new 16-row tile
            r = (ids == e).any(1).nonzero()[:, 0]
            if len(r):
                part[at:at + len(r)] = a[r] @ _w4(w[e]).T
                at += (len(r) + 15) // 16 * 16
        return {"ids": None, "weights": wt / wt.sum(-1, keepdim=True), "rows": part}
    if kind == "attn":
        M, H, KVH, pc, rows = c["n_seq"] * c["rows"], c["H"], c["KVH"], c["page"], c["rows"]
        qkv = (_q8_0(_norm(i["x"], i["nw"])) @ _w4(i["wqkv"]).T).reshape(M, H + 2 * KVH, 128)
        pos, seq = torch.from_numpy(i["pos"]).cuda(), torch.from_numpy(i["seq"]).cuda().long()
        pt = torch.from_numpy(i["pt"]).cuda().long()
        q = _rope(qkv[:, :H], i["qw"], pos)
        # a K region is chunk-major (16 chunks of 8 dims, each of every cell), a V region cell-major
        kp = i["k"].to(F64).reshape(-1, KVH, 16, pc, 8).permute(0, 3, 1, 2, 4).reshape(-1, pc, KVH, 128).contiguous()
        vp = i["v"].to(F64).reshape(-1, KVH, pc, 128).permute(0, 2, 1, 3).contiguous()
        page, cell = pt[seq, pos.long() // pc], pos.long() % pc
        kp[page, cell] = _rope(qkv[:, H:H + KVH], i["kw"], pos).half().to(F64)
        vp[page, cell] = qkv[:, H + KVH:].half().to(F64)
        o = torch.empty_like(q)
        for s in range(c["n_seq"]):
            n, r = int(i["ctx"][s]) + rows, slice(s * rows, (s + 1) * rows)
            pages = pt[s, :(n + pc - 1) // pc]
            o[r] = _attend(q[r], kp[pages].reshape(-1, KVH, 128)[:n], vp[pages].reshape(-1, KVH, 128)[:n], int(i["ctx"][s]))
        o = o.reshape(M, H * 128)
        kp = kp.reshape(-1, pc, KVH, 16, 8).permute(0, 2, 3, 1, 4).reshape(i["k"].shape)
        vp = vp.permute(0, 2, 1, 3).reshape(i["v"].shape)
        return {"attention": o, "y": _q8_0(o) @ _w4(i["wo"]).T, "k": kp, "v": vp}
    return _exact_engine(c, i)
