"""The work that a program using this library has it do, as measurable cases: the blocks of one
transformer layer through the public calls of hipster_amd.qmm, in the order an engine issues them.

ops
  moe_decode    MoE block of a decode step, T = 1..8 tokens: norm -> q8, router GEMV, routing + experts
  ffn_decode    gated MLP of a decode or draft-verification step, M = 1..16 tokens: norm -> q8, gate|up
                GEMV, silu * up -> q8, down GEMV
  gemv_f32      one f32-activation Q4_K GEMV, 1..8 columns
  proj_prefill  attention projections of a prompt chunk: norm -> bf16, q, k, v and o GEMMs
  ffn_prefill   gated MLP of a prompt chunk: norm -> bf16, gate and up GEMMs, silu * up -> bf16, down GEMM
  moe_prefill   MoE block of a prompt chunk on bf16 activations: routing, device sort, grouped gate/up
                and down GEMMs, combine (Q4_K experts: gate, up and silu in one call; other expert
                formats: the separate calls)
  moe_q8        the reference engine's own prefill call: moe_gemm with q8 activations and host tile
                counts (gate, up, silu -> q8, down, combine)

Sizes are those of hipster_amd.synth (a dense 5120 / 17408 model, a 512-expert 2048 / 512 MoE, Zipf
routed prompts) and of the reference engine's MoE (2560 / 640, Q5_K gate and up, Q5_1 down).  Weights
are random GGUF blocks with the distributions of hipster_amd.synth, scaled so that a layer's outputs are
of order 1.
"""
import numpy as np
import torch

from hipster_amd import qmm, synth

Q4_K, Q5_K, IQ4_XS, Q6_K, Q8_0, Q5_1 = (synth.Q4_K, synth.Q5_K, synth.IQ4_XS, synth.Q6_K_SOA, synth.Q8_0_SOA, synth.Q5_1_SOA)
FMT = {"Q4_K": Q4_K, "Q5_K": Q5_K, "IQ4_XS": IQ4_XS, "Q6_K": Q6_K, "Q8_0": Q8_0, "Q5_1": Q5_1}
BITS = {"Q4_K": 4.5, "Q5_K": 5.5, "IQ4_XS": 4.25, "Q6_K": 6.5625, "Q8_0": 8.5, "Q5_1": 6.0}    # stored bits per weight
EPS = 1e-6
DEV = "cuda"


def listed():
    return [
        # one user's decode step through the MoE block: the smallest call, latency and launches count
        dict(name="moe_decode_t1", op="moe_decode", T=1, H=2048, F=512, E=512, topk=10),
        # a verification step of eight drafted tokens (or eight users)
        dict(name="moe_decode_t8", op="moe_decode", T=8, H=2048, F=512, E=512, topk=10),
        # one user's decode step through the dense MLP of a Q4_K_M file (Q4_K gate and up, Q6_K down)
        dict(name="ffn_decode_m1", op="ffn_decode", M=1, H=5120, F=17408, fmt="Q4_K", dfmt="Q6_K"),
        # the same MLP verifying a draft of six tokens
        dict(name="ffn_decode_m6", op="ffn_decode", M=6, H=5120, F=17408, fmt="Q4_K", dfmt="Q6_K"),
        # f32 activations kept in f32 (the call for inputs that q8 would hurt), a four-token step
        dict(name="gemv_f32_m4", op="gemv_f32", M=4, N=17408, K=5120),
        # the attention projections of a short question
        dict(name="proj_prefill_m40", op="proj_prefill", M=40, H=5120, NQ=6144, NKV=1024, fmt="Q4_K"),
        # a prompt of ordinary, ragged length through the dense MLP
        dict(name="ffn_prefill_m300", op="ffn_prefill", M=300, H=5120, F=17408, fmt="Q4_K", dfmt="Q6_K"),
        # a full prompt chunk through the dense MLP: the largest call
        dict(name="ffn_prefill_m2048", op="ffn_prefill", M=2048, H=5120, F=17408, fmt="Q4_K", dfmt="Q6_K"),
        # a full prompt chunk through the 512-expert MoE
        dict(name="moe_prefill_t2048", op="moe_prefill", T=2048, H=2048, F=512, E=512, topk=10, quant="q4"),
        # a short question through it: almost every expert has a handful of rows
        dict(name="moe_prefill_t96", op="moe_prefill", T=96, H=2048, F=512, E=512, topk=10, quant="q4"),
        # the reference engine's expert sizes and formats, a prompt of ordinary length
        dict(name="moe_prefill_q5_t600", op="moe_prefill", T=600, H=2560, F=640, E=512, topk=10, quant="q5"),
        # the unchanged engine's own prefill calls, 16-column tiles (its default)
        dict(name="moe_q8_t512", op="moe_q8", T=512, H=2048, F=512, E=512, topk=10, ct=1),
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], its logarithm uniform."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    op = rng.choice(["moe_decode", "ffn_decode", "ffn_decode", "gemv_f32", "proj_prefill", "proj_prefill", "ffn_prefill",
                     "ffn_prefill", "moe_prefill", "moe_prefill", "moe_q8"])
    if op == "moe_decode":
        return dict(op=op, T=rng.randint(1, 8), H=256 * rng.randint(6, 12), F=256 * rng.randint(1, 4),
                    E=rng.choice([64, 128, 160, 256, 384, 512]), topk=rng.choice([4, 6, 8, 10]))
    if op == "ffn_decode":
        return dict(op=op, M=rng.randint(1, 16), H=512 * rng.randint(4, 10), F=512 * rng.randint(10, 34),
                    fmt=rng.choice(["Q4_K", "Q4_K", "Q5_K", "IQ4_XS", "Q8_0"]), dfmt=rng.choice(["Q6_K", "Q6_K", "Q4_K", "Q8_0", "Q5_1"]))
    if op == "gemv_f32":
        return dict(op=op, M=rng.randint(1, 8), N=_spread(rng, 1000, 17408), K=256 * rng.randint(6, 24))
    if op == "proj_prefill":
        return dict(op=op, M=_spread(rng, 17, 2048), H=512 * rng.randint(4, 10), NQ=512 * rng.randint(4, 12),
                    NKV=rng.choice([256, 512, 1000, 1024]), fmt=rng.choice(["Q4_K", "Q4_K", "Q6_K", "Q5_K", "Q8_0"]))
    if op == "ffn_prefill":
        return dict(op=op, M=_spread(rng, 17, 2048), H=512 * rng.randint(4, 10), F=512 * rng.randint(10, 34),
                    fmt=rng.choice(["Q4_K", "Q4_K", "Q5_K", "IQ4_XS", "Q8_0"]), dfmt=rng.choice(["Q6_K", "Q6_K", "Q4_K", "Q8_0", "Q5_1"]))
    E, topk = rng.choice([(64, 6), (128, 8), (256, 8), (512, 10)])
    if op == "moe_q8":
        return dict(op=op, T=_spread(rng, 16, 1024), H=256 * rng.randint(6, 10), F=256 * rng.randint(1, 3), E=E, topk=topk, ct=rng.choice([1, 2, 3]))
    quant = rng.choice(["q4", "q4", "q5"])
    F = 128 * rng.randint(4, 6) if quant == "q5" else 256 * rng.randint(2, 3)
    return dict(op=op, T=_spread(rng, 16, 2048), H=256 * rng.randint(6, 10), F=F, E=E, topk=topk, quant=quant)


# ---- inputs ----
def _bytes(g, n, nb):
    """n blocks of nb uniform random bytes."""
    words = -(-n * nb // 8)
    return torch.randint(-(1 << 63), (1 << 63) - 1, (words,), dtype=torch.int64, device=DEV, generator=g).view(torch.uint8)[: n * nb].view(n, nb)


# root mean square of a weight whose block scales are |N(0, 1)| and whose other bytes are uniform
_RMS = {Q4_K: 306.0, Q5_K: 611.0, IQ4_XS: 1205.0, Q6_K: 1290.0, Q8_0: 74.7, Q5_1: 17.9}


def _halves(g, n, sigma, signed=False):
    v = torch.randn(n, device=DEV, generator=g) * sigma
    return (v if signed else v.abs()).half().view(torch.uint8).view(n, 2)


def _weights(g, fmt, N, K):
    """A [N][K] matrix in format fmt, uint8 [N, row bytes], distributed as hipster_amd.synth.blocks with the
    scales brought to a trained model's: weights of root mean square 1 / sqrt(K)."""
    sig = 1.0 / (_RMS[fmt] * K ** 0.5)
    if fmt in (Q4_K, Q5_K, IQ4_XS):
        n, nb = N * (K // 256), synth.BLOCK[fmt][1]
        b = _bytes(g, n, nb)
        b[:, 0:2] = _halves(g, n, sig)
        if fmt != IQ4_XS:
            b[:, 2:4] = _halves(g, n, sig)
        return b.reshape(N, -1)
    if fmt == Q6_K:      # per row: ql K/2, qh K/4, scales K/16, d K/128
        return torch.cat([_bytes(g, N, K // 2 + K // 4 + K // 16), _halves(g, N * (K // 256), sig).view(N, -1)], 1)
    if fmt == Q8_0:      # per row: q K, d K/16
        return torch.cat([_bytes(g, N, K), _halves(g, N * (K // 32), sig).view(N, -1)], 1)
    return torch.cat([_bytes(g, N, K // 2 + K // 8), _halves(g, N * (K // 32), sig).view(N, -1),      # Q5_1: qs, qh, d, m
                      _halves(g, N * (K // 32), sig, signed=True).view(N, -1)], 1)


def _logits(g, T, E, zipf):
    """[T][E + 1]: N(0, 1), for prompts with the Zipf(1.1) bias of hipster_amd.synth.router_logits."""
    lg = torch.randn((T, E + 1), device=DEV, generator=g)
    if zipf:
        ranks = torch.randperm(E, device=DEV, generator=g) + 1
        lg[:, :E] -= 1.1 * torch.log(ranks.float())
    return lg


def _moe_fmts(c):
    return (Q5_K, Q5_1) if c.get("quant") == "q5" else (Q4_K, Q4_K)


def prepare(c, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    f32 = lambda *shape: torch.zeros(shape, dtype=torch.float32, device=DEV)      # noqa: E731
    i32 = lambda *shape: torch.zeros(shape, dtype=torch.int32, device=DEV)        # noqa: E731
    rand = lambda *shape: torch.randn(shape, device=DEV, generator=g)             # noqa: E731
    norm = lambda n: 1 + 0.1 * rand(n)                                            # noqa: E731
    op, s = c["op"], dict(c=c)
    if op == "gemv_f32":
        s.update(W=_weights(g, Q4_K, c["N"], c["K"]), x=rand(c["M"], c["K"]), y=f32(c["M"], c["N"]))
        return s
    H = c["H"]
    if op in ("ffn_decode", "ffn_prefill"):
        M, F = c["M"], c["F"]
        fmt, dfmt = FMT[c["fmt"]], FMT[c["dfmt"]]
        s.update(Wg=_weights(g, fmt, F, H), Wu=_weights(g, fmt, F, H), Wd=_weights(g, dfmt, H, F), x=rand(M, H), wn=norm(H),
                 gate=f32(M, F), up=f32(M, F), y=f32(M, H))
        if op == "ffn_decode":
            s.update(xn=f32(M, H), xq=qmm.XQ8Buf(M, H), hq=qmm.XQ8Buf(M, F))
        else:
            s.update(xb=torch.zeros((M, H), dtype=torch.bfloat16, device=DEV), h=torch.zeros((M, F), dtype=torch.bfloat16, device=DEV))
        return s
    if op == "proj_prefill":
        M, NQ, NKV, fmt = c["M"], c["NQ"], c["NKV"], FMT[c["fmt"]]
        s.update(Wq=_weights(g, fmt, NQ, H), Wk=_weights(g, fmt, NKV, H), Wv=_weights(g, fmt, NKV, H), Wo=_weights(g, fmt, H, NQ),
                 x=rand(M, H), wn=norm(H), att=rand(M, NQ), q=f32(M, NQ), k=f32(M, NKV), v=f32(M, NKV), y=f32(M, H),
                 xb=torch.zeros((M, H), dtype=torch.bfloat16, device=DEV), ab=torch.zeros((M, NQ), dtype=torch.bfloat16, device=DEV))
        return s
    T, F, E, topk = c["T"], c["F"], c["E"], c["topk"]
    NS = T * (topk + 1)
    fmt, dfmt = _moe_fmts(c)
    s.update(Wg=_weights(g, fmt, E * F, H), Wu=_weights(g, fmt, E * F, H), Wd=_weights(g, dfmt, E * H, F),
             Sg=_weights(g, fmt, F, H), Su=_weights(g, fmt, F, H), Sd=_weights(g, dfmt, H, F),
             ids=i32(T, topk + 1), w=f32(T, topk + 1), y=f32(T, H), x=rand(T, H))
    s.update(ebg=s["Wg"].numel() // E, ebd=s["Wd"].numel() // E)
    if op == "moe_decode":
        s.update(wn=norm(H), xn=f32(T, H), xq=qmm.XQ8Buf(T, H), Wr=rand(E + 1, H) * H ** -0.5, logits=f32(T, E + 1),
                 ws=torch.zeros(qmm.moe_decode_ws_bytes(T, topk, F), dtype=torch.uint8, device=DEV))
        return s
    s.update(logits=_logits(g, T, E, True), kpos=i32(NS), rowtok=i32(NS), counts=i32(2), dn=f32(NS, H))
    if op == "moe_prefill":
        cap = qmm.moe_tiles_capacity(T, topk + 1, E)
        s.update(cap=cap, tiles=i32(cap, 3), xb=s["x"].bfloat16(), h=torch.zeros((NS, F), dtype=torch.bfloat16, device=DEV))
        if c["quant"] != "q4":
            s.update(gate=f32(NS, F), up=f32(NS, F))
        return s
    # moe_q8: the engine sorts on the host between the routing and the expert GEMMs, so the tile lists and
    # their counts are at hand before the calls
    tiles = i32(qmm.moe_tiles_capacity(T, topk + 1, E, 16 * c["ct"]), 3)
    qmm.moe_route_n(s["logits"], s["ids"], s["w"], T, E, E + 1, topk)
    qmm.moe_sort(s["ids"], T, topk + 1, E, 16 * c["ct"], s["kpos"], s["rowtok"], tiles, s["counts"])
    nt, nst = [int(v) for v in s["counts"].cpu()]
    s.update(tiles=tiles[:nt].contiguous(), stiles=tiles[nt:nt + nst].contiguous(), nt=nt, nst=nst, xq=qmm.XQ8Buf(T, H),
             hq=qmm.XQ8Buf(NS, F), gate=f32(NS, F), up=f32(NS, F))
    return s


# ---- one pass ----
def run(s):
    c = s["c"]
    op = c["op"]
    if op == "gemv_f32":
        qmm.gemv_q4_K_f32(s["W"], s["x"], s["y"], c["N"], c["K"], c["M"])
        return {"y": s["y"]}
    H = c["H"]
    if op == "ffn_decode":
        M, F, fmt, dfmt = c["M"], c["F"], FMT[c["fmt"]], FMT[c["dfmt"]]
        qmm.add_rmsnorm_quant(s["x"], None, s["wn"], s["xn"], s["xq"], M, H, EPS)
        qmm.gemv_multi([(fmt, s["Wg"], s["gate"], F, H), (fmt, s["Wu"], s["up"], F, H)], s["xq"], M)
        qmm.silu_mul_quant(s["gate"], s["up"], s["hq"], M * F)
        qmm.gemv_multi([(dfmt, s["Wd"], s["y"], H, F)], s["hq"], M)
        return {"gate": s["gate"], "up": s["up"], "y": s["y"]}
    if op == "ffn_prefill":
        M, F, fmt, dfmt = c["M"], c["F"], FMT[c["fmt"]], FMT[c["dfmt"]]
        qmm.add_rmsnorm_bf16(s["x"], None, s["wn"], s["xb"], M, H, EPS)
        qmm.gemm_wq(fmt, s["Wg"], s["xb"], s["gate"], M, F, H)
        qmm.gemm_wq(fmt, s["Wu"], s["xb"], s["up"], M, F, H)
        qmm.silu_mul_bf16(s["gate"], s["up"], s["h"], M * F)
        qmm.gemm_wq(dfmt, s["Wd"], s["h"], s["y"], M, H, F)
        return {"gate": s["gate"], "up": s["up"], "y": s["y"]}
    if op == "proj_prefill":
        M, NQ, NKV, fmt = c["M"], c["NQ"], c["NKV"], FMT[c["fmt"]]
        qmm.add_rmsnorm_bf16(s["x"], None, s["wn"], s["xb"], M, H, EPS)
        qmm.gemm_wq(fmt, s["Wq"], s["xb"], s["q"], M, NQ, H)
        qmm.gemm_wq(fmt, s["Wk"], s["xb"], s["k"], M, NKV, H)
        qmm.gemm_wq(fmt, s["Wv"], s["xb"], s["v"], M, NKV, H)
        qmm.f32_to_bf16(s["att"], s["ab"], M * NQ)
        qmm.gemm_wq(fmt, s["Wo"], s["ab"], s["y"], M, H, NQ)
        return {"q": s["q"], "k": s["k"], "v": s["v"], "y": s["y"]}
    T, F, E, topk = c["T"], c["F"], c["E"], c["topk"]
    NS, fmt, dfmt = T * (topk + 1), *_moe_fmts(c)
    if op == "moe_decode":
        qmm.add_rmsnorm_quant(s["x"], None, s["wn"], s["xn"], s["xq"], T, H, EPS)
        qmm.f32_gemv(s["Wr"], s["xn"], s["logits"], E + 1, H, T)
        qmm.moe_decode(fmt, s["Wg"], s["Wu"], s["Wd"], s["ebg"], s["ebd"], s["Sg"], s["Su"], s["Sd"], s["logits"], E + 1, E, topk,
                       s["xq"], T, H, F, s["ids"], s["w"], s["ws"], s["y"])
        return {"logits": s["logits"], "ids": s["ids"], "w": s["w"], "y": s["y"]}
    if op == "moe_prefill":
        qmm.moe_route_n(s["logits"], s["ids"], s["w"], T, E, E + 1, topk)
        qmm.moe_sort(s["ids"], T, topk + 1, E, qmm.MOE_TILE_ROWS, s["kpos"], s["rowtok"], s["tiles"], s["counts"])
        if c["quant"] == "q4":
            qmm.moe_gemm_gate_up_bf16(fmt, fmt, s["Wg"], s["Sg"], s["Wu"], s["Su"], s["ebg"], s["tiles"], s["counts"], s["cap"],
                                      s["rowtok"], s["xb"], s["h"], F, H)
        else:
            qmm.moe_gemm_bf16(fmt, fmt, s["Wg"], s["Sg"], s["ebg"], s["tiles"], s["counts"], s["cap"], s["rowtok"], s["xb"], s["gate"], F, H)
            qmm.moe_gemm_bf16(fmt, fmt, s["Wu"], s["Su"], s["ebg"], s["tiles"], s["counts"], s["cap"], s["rowtok"], s["xb"], s["up"], F, H)
            qmm.moe_silu_bf16(s["gate"], s["up"], s["h"], NS * F)
        qmm.moe_gemm_bf16(dfmt, dfmt, s["Wd"], s["Sd"], s["ebd"], s["tiles"], s["counts"], s["cap"], None, s["h"], s["dn"], H, F)
    else:
        qmm.quantize_x_q8(s["x"], s["xq"], T, H)
        qmm.moe_gemm(fmt, fmt, s["Wg"], s["Sg"], s["ebg"], s["tiles"], s["nt"], s["stiles"], s["nst"], c["ct"], s["rowtok"], s["xq"], s["gate"], F, H)
        qmm.moe_gemm(fmt, fmt, s["Wu"], s["Su"], s["ebg"], s["tiles"], s["nt"], s["stiles"], s["nst"], c["ct"], s["rowtok"], s["xq"], s["up"], F, H)
        qmm.moe_silu_quant(s["gate"], s["up"], s["hq"], NS, F)
        qmm.moe_gemm(dfmt, dfmt, s["Wd"], s["Sd"], s["ebd"], s["tiles"], s["nt"], s["stiles"], s["nst"], c["ct"], None, s["hq"], s["dn"], H, F)
    qmm.moe_combine_sorted(s["dn"], s["w"], s["kpos"], s["y"], T, topk + 1, H)
    return {"ids": s["ids"], "w": s["w"], "y": s["y"]}


# ---- what a pass cannot do without ----
def work(c):
    """Weights, activations in and results out once each; two flops per multiply-add."""
    op = c["op"]
    if op == "gemv_f32":
        M, N, K = c["M"], c["N"], c["K"]
        return {"bytes": N * K * BITS["Q4_K"] / 8 + 4 * M * (N + K), "flops": 2 * M * N * K}
    H = c["H"]
    if op in ("ffn_decode", "ffn_prefill"):
        M, F = c["M"], c["F"]
        return {"bytes": H * F * (2 * BITS[c["fmt"]] + BITS[c["dfmt"]]) / 8 + 4 * M * (2 * H + 2 * F), "flops": 6 * M * H * F}
    if op == "proj_prefill":
        M, NQ, NKV = c["M"], c["NQ"], c["NKV"]
        return {"bytes": H * (2 * NQ + 2 * NKV) * BITS[c["fmt"]] / 8 + 4 * M * (2 * H + 2 * NQ + 2 * NKV), "flops": 4 * M * H * (NQ + NKV)}
    # MoE: the distinct experts that T tokens reach (a sample of the routing) and the shared one
    T, F, E, topk = c["T"], c["F"], c["E"], c["topk"]
    g = np.random.default_rng(0)
    lg = g.standard_normal((T, E))
    if op != "moe_decode":
        lg -= 1.1 * np.log(1.0 + np.arange(E))[None, :]
    distinct = len(np.unique(np.argpartition(-lg, topk - 1, axis=1)[:, :topk])) + 1
    bits = 2 * BITS["Q5_K"] + BITS["Q5_1"] if c.get("quant") == "q5" else 3 * BITS["Q4_K"]
    router = 4 * H * (E + 1) if op == "moe_decode" else 0
    return {"bytes": distinct * H * F * bits / 8 + router + T * (8 * H + 4 * (E + 1)), "flops": 6 * T * (topk + 1) * H * F}


def tolerance(c):
    """About four times the distance of each op from the 64-bit result.  f32 sums alone are 1e-7 off; an f32
    sum in another order also moves a few activations of the next stage to the neighbouring q8 or bf16 value
    (4e-5 in the q8 MLP; 1.2e-4 in the bf16 MLP, 1e-5 after one rounding, 4e-6 in the MoE's last sum)."""
    return {"rel": {"gemv_f32": 1e-6, "moe_decode": 2e-4, "ffn_decode": 2e-4, "moe_q8": 2e-4, "proj_prefill": 4e-5,
                    "ffn_prefill": 5e-4, "moe_prefill": 4e-5}[c["op"]]}


# ---- the same in 64 bits ----
def _f16(b):
    """float64 of the f16 at the last dimension's byte pairs."""
    return b.contiguous().view(torch.float16).double()


_IQ4 = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]      # the levels of the format (ggml's kvalues_iq4nl)


def _scales_k(s):
    """Q4_K / Q5_K: 12 packed bytes [n, 12] -> scales and mins [n, 8]."""
    lo, mid, hi = s[:, 0:4], s[:, 4:8], s[:, 8:12]
    sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1)
    mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1)
    return sc.double(), mn.double()


def _dequant(fmt, W, N, K):
    """float64 [N][K] of the GGUF weights."""
    W = W.reshape(N, -1)
    if fmt in (Q4_K, Q5_K):
        b = W.reshape(N * (K // 256), -1)
        sc, mn = _scales_k(b[:, 4:16])
        d, m = _f16(b[:, 0:2]) * sc, _f16(b[:, 2:4]) * mn
        qs = b[:, -128:].reshape(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
        if fmt == Q5_K:
            bit = torch.arange(8, dtype=torch.uint8, device=W.device).view(1, 8, 1)
            q = q | (((b[:, 16:48].unsqueeze(1) >> bit) & 1) << 4)
        return (d.unsqueeze(2) * q.double() - m.unsqueeze(2)).reshape(N, K)
    if fmt == IQ4_XS:
        b = W.reshape(N * (K // 256), -1)
        ib = torch.arange(8, device=W.device)
        sl = (b[:, 4:8].repeat_interleave(2, 1) >> (4 * (ib & 1)).to(torch.uint8)) & 15
        sh = (b[:, 2:4].contiguous().view(torch.int16).int() >> (2 * ib).int()) & 3
        ls = (sl.int() | (sh << 4)).double() - 32
        qs = b[:, 8:136].reshape(-1, 8, 16)
        q = torch.tensor(_IQ4, dtype=torch.float64, device=W.device)[torch.cat([qs & 15, qs >> 4], 2).long()]
        return ((_f16(b[:, 0:2]) * ls).unsqueeze(2) * q).reshape(N, K)
    if fmt == Q6_K:
        nb = K // 256
        ql = W[:, : K // 2].reshape(N, nb, 2, 2, 32)                       # half, ql run, byte
        qh = W[:, K // 2: K // 2 + K // 4].reshape(N, nb, 2, 32)
        sc = W[:, 3 * K // 4: 3 * K // 4 + K // 16].contiguous().view(torch.int8).double().reshape(N, nb, 16)
        d = _f16(W[:, -(K // 128):]).reshape(N, nb, 1)
        quarter = [(ql[:, :, :, g & 1] & 15 if g < 2 else ql[:, :, :, g & 1] >> 4) | (((qh >> (2 * g)) & 3) << 4) for g in range(4)]
        q = torch.stack(quarter, 3).double() - 32                          # [N][nb][half][quarter][32]
        return ((d * sc).unsqueeze(3) * q.reshape(N, nb, 16, 16)).reshape(N, K)
    if fmt == Q8_0:
        q = W[:, :K].contiguous().view(torch.int8).double().reshape(N, K // 32, 32)
        return (_f16(W[:, K:]).unsqueeze(2) * q).reshape(N, K)
    n32 = K // 32
    qs = W[:, : K // 2].reshape(N, n32, 16)
    qh = W[:, K // 2: K // 2 + K // 8].contiguous().view(torch.int32).reshape(N, n32, 1)
    bit = torch.arange(32, dtype=torch.int32, device=W.device)
    q = torch.cat([qs & 15, qs >> 4], 2).double() + 16 * ((qh >> bit) & 1).double()
    d = _f16(W[:, K // 2 + K // 8: K // 2 + K // 8 + 2 * n32])
    m = _f16(W[:, K // 2 + K // 8 + 2 * n32:])
    return (d.unsqueeze(2) * q + m.unsqueeze(2)).reshape(N, K)


def _bf16(v):
    return v.float().bfloat16().double()


def _q8(v):
    """q8 per 32, the activations' own rounding: the values it stands for."""
    b = v.reshape(-1, 32)
    amax = b.abs().amax(1, keepdim=True)
    q = torch.round(b * torch.where(amax > 0, 127.0 / amax, torch.zeros_like(amax)))
    return (q * (amax / 127.0)).reshape(v.shape)


def _norm(x, w):
    x = x.double()
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * w.double()


def _silu(g, u):
    return g / (1.0 + torch.exp(-g)) * u


def exact(c, seed):
    s = prepare(c, seed)
    op = c["op"]
    if op == "gemv_f32":
        return {"y": s["x"].double() @ _dequant(Q4_K, s["W"], c["N"], c["K"]).t()}
    H = c["H"]
    if op in ("ffn_decode", "ffn_prefill"):
        F, fmt, dfmt = c["F"], FMT[c["fmt"]], FMT[c["dfmt"]]
        act, wt = (_q8, lambda w: w) if op == "ffn_decode" else (_bf16, _bf16)
        x = act(_norm(s["x"], s["wn"]))
        gate = x @ wt(_dequant(fmt, s["Wg"], F, H)).t()
        up = x @ wt(_dequant(fmt, s["Wu"], F, H)).t()
        return {"gate": gate, "up": up, "y": act(_silu(gate, up)) @ wt(_dequant(dfmt, s["Wd"], H, F)).t()}
    if op == "proj_prefill":
        fmt, x = FMT[c["fmt"]], _bf16(_norm(s["x"], s["wn"]))
        out = {n: x @ _bf16(_dequant(fmt, s["W" + n], s[n].shape[1], H)).t() for n in "qkv"}
        out["y"] = _bf16(s["att"].double()) @ _bf16(_dequant(fmt, s["Wo"], H, c["NQ"])).t()
        return out
    T, F, E, topk = c["T"], c["F"], c["E"], c["topk"]
    fmt, dfmt = _moe_fmts(c)
    act, wt = (_bf16, _bf16) if op == "moe_prefill" else (_q8, lambda w: w)
    if op == "moe_decode":
        xn = _norm(s["x"], s["wn"])
        logits, x = xn @ s["Wr"].double().t(), act(xn)
    else:
        logits, x = s["logits"].double(), act(s["x"].double())
    p, ids = torch.softmax(logits[:, :E], 1).topk(topk, 1)
    w = torch.cat([p / p.sum(1, keepdim=True), torch.sigmoid(logits[:, E:E + 1])], 1)
    rows_of = lambda e: (ids == e).nonzero(as_tuple=True) if e >= 0 else (torch.arange(T, device=DEV), torch.full((T,), topk, device=DEV))  # noqa: E731
    down = torch.zeros((T, topk + 1, H), dtype=torch.float64, device=DEV)
    Wg, Wu, Wd = (s[n].view(E, -1) for n in ("Wg", "Wu", "Wd"))
    for e in [-1] + torch.unique(ids).tolist():
        t, slot = rows_of(e)
        gate = x[t] @ wt(_dequant(fmt, s["Sg"] if e < 0 else Wg[e], F, H)).t()
        up = x[t] @ wt(_dequant(fmt, s["Su"] if e < 0 else Wu[e], F, H)).t()
        down[t, slot] = act(_silu(gate, up)) @ wt(_dequant(dfmt, s["Sd"] if e < 0 else Wd[e], H, F)).t()
    out = {"ids": None, "w": w, "y": (w.unsqueeze(2) * down).sum(1)}
    return dict(out, logits=logits) if op == "moe_decode" else out
