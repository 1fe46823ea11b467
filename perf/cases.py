"""What the attention hot path is timed on: the calls an xDiT-style DiT pipeline makes in one block
on one GPU, through the package's public entry points.

A case is a dict of plain values.  `kind` says which entry point it goes through:

  usp     usp.USP: self-attention, or joint attention (image queries beside `Sj` text tokens handed
          over as joint tensors), or cross-attention (`Sk` != `Sq`); `backend` "mi355" or "mi355_fp8"
          (16-bit tensors in, quantised inside the call); BHSD-contiguous tensors, or the BSHD
          projection outputs viewed as BHSD (`layout`)
  fwd     ops.attn_fwd, the registry form that returns the log-sum-exp beside the output
  ring    the ring schedule of one rank over `chunks` K/V chunks: ring.xdit_ring_flash_attn_func on
          BSHD tensors ("mi355", every step folded by the attention kernel), or usp.USP on BHSD
          tensors ("mi355_fp8", a call and a merge per step)
  flux    prologue.flux_joint_qkv: RMSNorm of Q and K, [text; image] concatenation, rotary
          embedding and re-layout of an MMDiT block's six projection outputs
  rope    prologue.norm_rope on one projection output: norm over head_dim or over the whole token,
          rotary embedding, BSHD -> BHSD

Sizes are those of the model shapes that bench.py and the tests use (image models at 512 and 1024
pixels, video shards at 480p and 720p, a Ulysses-8 rank's share of the heads) and, in `draw`, the
ranges between and around them.
"""
import math

import torch

from xdit_amd import attention_backend, ops, prologue, ring, usp

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}
_BACKENDS = {"mi355": attention_backend.AttentionBackendType.MI355, "mi355_fp8": attention_backend.AttentionBackendType.MI355_FP8}


def _attn(kind, name, B, H, Sq, Sk, D, dtype="bf16", Sj=0, layout="bhsd", backend="mi355", chunks=1):
    return {"name": name, "kind": kind, "B": B, "H": H, "Sq": Sq, "Sk": Sk, "Sj": Sj, "D": D, "dtype": dtype,
            "layout": layout, "backend": backend, "chunks": chunks}


def listed():
    return [
        # the smallest call: a Ulysses-8 rank's 3 of 24 heads of a 512-pixel MMDiT block (1024 image + 512 text tokens)
        _attn("usp", "flux512_3heads", 1, 3, 1024, 1024, 128, Sj=512),
        # text cross-attention of a 1024-pixel DiT, head_dim 72, 120 text keys, straight from the projections (BSHD memory)
        _attn("usp", "pixart1024_cross", 2, 16, 4096, 120, 72, layout="bshd"),
        # fp32 self-attention at 512 pixels, head_dim 72
        _attn("usp", "pixart512_fp32", 1, 16, 1024, 1024, 72, dtype="fp32"),
        # joint attention of a 1024-pixel MMDiT block: the headline workload, text keys as a second segment
        _attn("usp", "flux1024_joint", 1, 24, 4096, 4096, 128, Sj=512),
        # the same block on the fp8 backend: bf16 tensors in, quantisation inside the call
        _attn("usp", "flux1024_fp8", 1, 24, 4608, 4608, 128, backend="mi355_fp8"),
        # classifier-free-guidance batch of a head_dim-64 model, ragged sequence (4096 image + 154 text tokens), output and log-sum-exp
        _attn("fwd", "sd3_1024", 2, 24, 4250, 4250, 64, dtype="fp16"),
        # 480p video self-to-text cross-attention: many query rows, 512 keys
        _attn("usp", "wan480p_cross", 1, 40, 32760, 512, 128),
        # one rank's ring of 4 over a 1024-pixel MMDiT block
        _attn("ring", "flux1024_ring4", 1, 24, 4608, 4608, 128, layout="bshd", chunks=4),
        # 720p video, one rank's 3 of 24 heads, output and log-sum-exp: the longest sequence
        _attn("fwd", "hunyuan720p_3heads", 1, 3, 119056, 119056, 128),
        # 720p video, one rank's 5 of 40 heads on the fp8 backend
        _attn("usp", "wan720p_5heads_fp8", 1, 5, 75600, 75600, 128, backend="mi355_fp8"),
        # pre-attention step of a 1024-pixel MMDiT block
        {"name": "flux1024_prologue", "kind": "flux", "B": 1, "H": 24, "S": 4096, "Sj": 512, "D": 128, "dtype": "bf16", "norm": "head", "rope": "interleaved"},
        # pre-attention step of Q of a 480p video block: norm over all heads of a token
        {"name": "wan480p_prologue_q", "kind": "rope", "B": 1, "H": 40, "S": 32760, "Sj": 0, "D": 128, "dtype": "bf16", "norm": "token", "rope": "wan"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# no drawn attention call does more than this many multiply-adds times two (the largest listed one: 21.8e12)
_MOST_FLOPS = {"bf16": 8e12, "fp16": 8e12, "fp32": 4e11}


def draw(rng):
    kind = rng.choice(["self", "self", "self", "joint", "joint", "cross", "cross", "fp8", "fp8", "ring", "flux", "rope"])
    if kind == "flux":
        return {"kind": "flux", "B": rng.choice([1, 1, 2]), "H": rng.randint(3, 32), "S": _log_int(rng, 256, 16384), "Sj": rng.choice([77, 154, 256, 333, 512]),
                "D": rng.choice([64, 128]), "dtype": rng.choice(["bf16", "bf16", "fp16"]), "norm": "head", "rope": "interleaved"}
    if kind == "rope":
        norm = rng.choice(["head", "token"])
        return {"kind": "rope", "B": rng.choice([1, 1, 2]), "H": rng.randint(3, 40), "S": _log_int(rng, 1024, 60000), "Sj": 0, "D": rng.choice([64, 128]),
                "dtype": rng.choice(["bf16", "bf16", "fp16"]), "norm": norm, "rope": "wan" if norm == "token" else rng.choice(["interleaved", "split_half"])}
    B = rng.choice([1, 1, 2])
    H = rng.choice([1, 2, 3, 5, 6, 10, 12, 16, 20, 24, 30, 40, 48])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    D = rng.choice([128, 128, 128, 64, 64, 72, 88, 96])
    layout = rng.choice(["bhsd", "bhsd", "bshd"])
    backend, Sj, chunks = "mi355", 0, 1
    if kind == "cross":
        Sq, Sk = _log_int(rng, 1024, 80000), rng.choice([77, 120, 226, 256, 300, 512])
    else:
        Sq = Sk = _log_int(rng, 512, 100000)
    if kind == "self" and rng.random() < 0.2:
        dtype = "fp32"
    elif kind == "joint":
        Sj = rng.choice([77, 154, 226, 256, 512])
    elif kind == "fp8":
        backend, D = "mi355_fp8", rng.choice([128, 128, 64])
        Sj = rng.choice([0, 0, 226, 512])
    elif kind == "ring":
        chunks = rng.choice([2, 4, 8])
        D = rng.choice([128, 128, 64])
        backend = rng.choice(["mi355", "mi355", "mi355_fp8"])
        layout = "bshd" if backend == "mi355" else "bhsd"
        H = max(3, H)
        Sq = Sk = _log_int(rng, 2048, 40000) // chunks * chunks
    while 4.0 * B * H * (Sq + Sj) * (Sk + Sj) * D > _MOST_FLOPS[dtype]:
        if H > 1:
            H = (H + 1) // 2
        else:
            Sq = Sk = int(Sq * 0.7)
    c = _attn("ring" if kind == "ring" else "usp" if rng.random() < 0.7 or backend == "mi355_fp8" or Sj else "fwd", "", B, H, Sq, Sk, D, dtype, Sj, layout, backend, chunks)
    del c["name"]
    return c


class _State:
    pass


def _rms(x, g):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * g


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    dt = _DTYPES[case["dtype"]]
    s = _State()
    s.case = case

    def normal(*shape):
        return torch.randn(shape, generator=gen, device=dev, dtype=torch.float32)

    def gain(n):
        return (0.8 + 0.4 * torch.rand(n, generator=gen, device=dev)).to(dt)

    B, H, D = case["B"], case["H"], case["D"]
    if case["kind"] in ("flux", "rope"):
        S, Sj = case["S"], case["Sj"]
        ang = torch.rand((S + Sj, D // 2), generator=gen, device=dev) * (2 * math.pi)
        ang = ang.repeat_interleave(2, dim=1) if case["rope"] != "split_half" else torch.cat([ang, ang], 1)
        s.rotary = (ang.cos().contiguous(), ang.sin().contiguous())
        if case["kind"] == "flux":
            s.img = [normal(B, S, H * D).to(dt) for _ in range(3)]
            s.txt = [normal(B, Sj, H * D).to(dt) for _ in range(3)]
            s.gains = [gain(D) for _ in range(4)]
        else:
            s.x = normal(B, S, H, D).to(dt)
            s.gains = [gain(H * D if case["norm"] == "token" else D)]
        return s

    # q and k as a block's norm_q / norm_k leave them (per-head RMSNorm with a gain near 1), v as projected
    gq, gk = gain(D).float(), gain(D).float()

    def tensor(S, g=None):
        shape = (B, S, H, D) if case["layout"] == "bshd" else (B, H, S, D)
        x = normal(*shape)
        x = (x if g is None else _rms(x, g)).to(dt)
        return x.transpose(1, 2) if case["layout"] == "bshd" and case["kind"] != "ring" else x

    s.q, s.k, s.v = tensor(case["Sq"], gq), tensor(case["Sk"], gk), tensor(case["Sk"])
    s.joint = [tensor(case["Sj"], gq), tensor(case["Sj"], gk), tensor(case["Sj"])] if case["Sj"] else None
    s.backend = _BACKENDS[case["backend"]]
    s.group = ring.LocalRing(case["chunks"]) if case["kind"] == "ring" else None
    return s


def run(s):
    c = s.case
    kind = c["kind"]
    if kind == "flux":
        return prologue.flux_joint_qkv(*s.img, *s.txt, c["H"], *s.gains, s.rotary)
    if kind == "rope":
        return prologue.norm_rope(s.x, weight=s.gains[0], freqs_cis=s.rotary, sequence_dim=1, norm=c["norm"], rope=c["rope"])
    if kind == "fwd":
        return ops.attn_fwd(s.q, s.k, s.v)
    if kind == "ring" and c["backend"] == "mi355":
        out, lse, _ = ring.xdit_ring_flash_attn_func(s.q, s.k, s.v, group=s.group, return_attn_probs=True)
        return out, lse
    if s.joint is not None:
        jq, jk, jv = s.joint
        return usp.USP(s.q, s.k, s.v, joint_query=jq, joint_key=jk, joint_value=jv, joint_strategy="front", backend=s.backend)
    return usp.USP(s.q, s.k, s.v, backend=s.backend, ring_chunks=c["chunks"])


def work(case):
    b = _BYTES[case["dtype"]]
    B, H, D = case["B"], case["H"], case["D"]
    if case["kind"] in ("flux", "rope"):
        rows = B * (case["S"] + case["Sj"])
        tensors = 3 if case["kind"] == "flux" else 1
        rotated = 2 if case["kind"] == "flux" else 1
        # each element read and written once, the cos and sin tables read once
        return {"bytes": 2.0 * b * tensors * rows * H * D + 8.0 * (case["S"] + case["Sj"]) * D, "flops": 10.0 * rotated * rows * H * D}
    Sq, Sk = case["Sq"] + case["Sj"], case["Sk"] + case["Sj"]
    return {"bytes": float(B * H * D * b) * (2 * Sq + 2 * Sk) + (4.0 * B * H * Sq if case["kind"] != "usp" else 0.0),
            "flops": 4.0 * B * H * Sq * Sk * D}


def tolerance(case):
    if case["kind"] in ("flux", "rope"):
        # a rounding of the norm's statistic flips the last place of a few elements in a thousand
        return {"rel": 1e-3}
    if case["backend"] == "mi355_fp8":
        # probabilities carry the four significant bits of e4m3: another split of the keys, so another
        # reference maximum for part of the rows, moves the output by 2e-2
        return {"rel": 3e-2}
    # against float64: 2.9e-3 (bf16), 3.0e-4 (fp16), 5.2e-7 (fp32); bf16 with the keys split in another way: 3.5e-3
    return {"rel": {"bf16": 1e-2, "fp16": 1.2e-3, "fp32": 4e-6}[case["dtype"]]}
