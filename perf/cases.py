"""Timing cases of the DiT block runner: what a caller of libhexanima_hip.so has it do, through the public C-ABI.

Seven kinds of call, from one linear to a whole denoise:

  linear   hxa_linear                       the plain fp16 / W8A16 / W4A16 linear
  attn     hxa_attention                    self, cross and masked joint attention over heads of 128
  norm     hxa_norm_mod                     the modulated LayerNorm / RMSNorm
  block    hxa_block_run                    a run of DiT blocks on resident weight packs: Anima structure (kind 0), MOSS
                                            structure (1), MOSS with the rapid-moss LoRA (2)
  mega     hxa_anima_modulation, mega_block the reference's block interface as its runner drives it, on host buffers
  denoise  hxa_dit_*                        a whole few-step denoise, latent in and latent out

Device operands are torch tensors; every kernel call goes to torch's current stream. The weights are what the
quantiser of a real exporter leaves: N(0, 0.02) rounded to fp16, or to int8 / int4 groups of 32 with fp16 scales.
"""
import ctypes as C
import math

import numpy as np
import torch

from hexanima_amd import hip

DEV = "cuda"
HALF, F64 = torch.float16, torch.float64
FMT = {"f16": hip.W_F16, "q8": hip.W_Q8, "q4": hip.W_Q4}
WBYTES = {"f16": 2.0, "q8": 1.0 + 2.0 / 32, "q4": 0.5 + 2.0 / 32}  # bytes a weight, its share of the group scale in it


def listed():
    return [
        # the square projection of a small picture (256 x 256 pixels) or of 256 text tokens: the smallest linear
        dict(name="linear_q8_proj_256", kind="linear", M=256, K=2048, N=2048, fmt="q8", tiled=True, mins=False),
        # the long-K MLP-down with int4 weights and their mins, rows that fill no tile
        dict(name="linear_q4_down_1000", kind="linear", M=1000, K=8192, N=2048, fmt="q4", tiled=True, mins=True),
        # the fused qkv of a 1024 x 1024 picture, fp16 weights as a framework stores them ([N][K]): many full tiles
        dict(name="linear_f16_qkv_4096", kind="linear", M=4096, K=2048, N=6144, fmt="f16", tiled=False, mins=False),
        # self-attention of a low-res first step (a quarter of 1536 tokens)
        dict(name="attn_self_384", kind="attn", T=384, NKV=384, nvalid=384, H=16, batch=1),
        # joint image + text attention at the reference's own token count, 1562 valid of 1568
        dict(name="attn_joint_1562", kind="attn", T=1568, NKV=1568, nvalid=1562, H=24, batch=1),
        # joint attention of a 1-megapixel picture: 6144 image + 512 text tokens
        dict(name="attn_joint_6656", kind="attn", T=6656, NKV=6656, nvalid=6656, H=24, batch=1),
        # the adaLN norm in front of every site of a block
        dict(name="norm_ln_1536", kind="norm", T=1536, D=2048, rms=False),
        # Anima blocks on a small picture, fp16 weights, where launches and idle CUs count
        dict(name="block_anima_f16_512", kind="block", structure=0, D=2048, F=8192, T=512, batch=1, nvalid=512, C=256,
             attn="f16", mlp="f16", depth=4),
        # the 2.9B-class block at its benchmark size, int8 weights
        dict(name="block_anima_q8_1536", kind="block", structure=0, D=2560, F=10240, T=1536, batch=1, nvalid=1536,
             C=256, attn="q8", mlp="q8", depth=4),
        # MOSS blocks as they ship (int8, the rapid-moss LoRA in every projection) at the reference's token count
        dict(name="block_moss_lora_1562", kind="block", structure=2, D=3072, F=8192, T=1568, batch=1, nvalid=1562, C=0,
             attn="q8", mlp="q8", depth=4),
        # 28 q8 blocks through the reference's boundary: modulation, then mega_block block by block, x in and out of a
        # host blob (512 x 512 pixels, the 512 context tokens of the reference's runner)
        dict(name="mega_q8_1024", kind="mega", fmt="q8", gh=32, gw=32, nctx=512, blocks=28),
        # the 2B picture: four Euler steps at 512 x 768 pixels, the first one low-res
        dict(name="denoise_f16_1536", kind="denoise", D=2048, F=8192, fmt="f16", lat_h=96, lat_w=64, C=256, blocks=28,
             batch=1, low=1, steps=4),
    ]


def _log(rng, lo, hi, multiple=1):
    return max(multiple, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / multiple)) * multiple)


def draw(rng):
    kind = rng.choice(["linear", "linear", "attn", "attn", "norm", "block", "block", "block", "mega", "denoise"])
    if kind == "linear":
        fmt = rng.choice(["f16", "q8", "q4"])
        return dict(kind=kind, M=_log(rng, 16, 6656), K=_log(rng, 512, 12288, 32), N=_log(rng, 512, 16384, 8), fmt=fmt,
                    tiled=rng.random() < 0.6, mins=fmt == "q4" and rng.random() < 0.5)
    if kind == "attn":
        T, H = _log(rng, 48, 6656), rng.choice([8, 16, 20, 24])
        if rng.random() < 0.3:  # cross attention over text keys
            NKV = 32 * rng.randint(1, 16)
            return dict(kind=kind, T=T, NKV=NKV, nvalid=NKV, H=H, batch=1)
        NKV = (T + 31) // 32 * 32
        return dict(kind=kind, T=NKV, NKV=NKV, nvalid=rng.choice([T, NKV]), H=H, batch=rng.choice([1, 1, 2]) if T < 3000 else 1)
    if kind == "norm":
        return dict(kind=kind, T=_log(rng, 32, 6656), D=rng.choice([1024, 2048, 2560, 3072]), rms=rng.random() < 0.5)
    if kind == "block":
        structure = rng.choice([0, 0, 1, 2])
        top = 2048 if structure == 2 else 4096
        T = _log(rng, 64, top, 32)
        if structure == 0:
            D = rng.choice([1024, 2048, 2560])
            fmt = rng.choice(["f16", "q8", "q4"])
            return dict(kind=kind, structure=0, D=D, F=4 * D, T=T, batch=rng.choice([1, 1, 2]) if T <= 1024 else 1, nvalid=T,
                        C=32 * rng.randint(1, 16), attn=fmt, mlp=fmt, depth=2)
        if structure == 1:
            fa, fm = rng.choice([("q8", "q4"), ("q8", "q8"), ("f16", "f16")])
            return dict(kind=kind, structure=1, D=3072, F=12288, T=T, batch=1, nvalid=T - rng.randint(0, 31), C=0, attn=fa,
                        mlp=fm, depth=2)
        return dict(kind=kind, structure=2, D=3072, F=8192, T=T, batch=1, nvalid=T - rng.randint(0, 31), C=0, attn="q8",
                    mlp="q8", depth=2)
    if kind == "mega":
        gh = 8 * rng.randint(2, 5)
        return dict(kind=kind, fmt=rng.choice(["q8", "q8", "f16"]), gh=gh, gw=4 * rng.randint(4, 10), nctx=rng.choice([128, 256, 512]),
                    blocks=rng.choice([8, 16, 28]))
    low = rng.choice([0, 1])
    return dict(kind=kind, D=rng.choice([1024, 2048]), F=8192, fmt=rng.choice(["f16", "q8"]), lat_h=16 * rng.randint(2, 4 + low),
                lat_w=32 * rng.randint(1, 2), C=32 * rng.randint(2, 8), blocks=rng.choice([8, 28]), batch=1, low=low,
                steps=rng.choice([2, 4]))


# ---------------------------------------------------------------------------------------------------------------- inputs
class State:
    pass


def _gen(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1000003 + salt)
    return g


def _randn(g, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32) * std).to(dtype)


def _weight(g, N, K, fmt, tiled=True, mins=False, std=0.02):
    """-> (weight bytes, fp16 scales [K/32][N] or None, fp16 mins or None, the values W [N][K] fp16)"""
    w = _randn(g, N, K, std=std)
    if fmt == "f16":
        W = w.half()
        raw = W.view(N, K // 32, 32)
        raw = raw.permute(1, 0, 2) if tiled else raw
        return raw.contiguous().view(-1).view(torch.uint8), None, None, W
    w = w.view(N, K // 32, 32)
    z = None
    if fmt == "q8":
        s = (w.abs().amax(-1) / 127).clamp_min(6.2e-5).half()
        q = torch.round(w / s[..., None].float()).clamp(-127, 127)
        W = (q * s[..., None].float()).half()
        raw = q.to(torch.int8)
    else:
        if mins:
            lo, hi = w.amin(-1), w.amax(-1)
            s = ((hi - lo) / 15).clamp_min(6.2e-5).half()
            z = lo.half()
            nib = torch.round((w - z[..., None].float()) / s[..., None].float()).clamp(0, 15)
            W = (nib.double() * s[..., None].double() + z[..., None].double()).half()
        else:
            s = (w.abs().amax(-1) / 7).clamp_min(6.2e-5).half()
            nib = torch.round(w / s[..., None].float()).clamp(-8, 7) + 8
            W = ((nib - 8) * s[..., None].float()).half()
        # a 32-bit word holds 8 k values: k0 + 2 j at bits 4 j, k0 + 2 j + 1 at bits 16 + 4 j
        n = nib.to(torch.int64).view(N, K // 32, 4, 4, 2)
        shift = torch.arange(4, device=DEV).view(4, 1) * 4 + torch.arange(2, device=DEV).view(1, 2) * 16
        word = (n << shift).sum((-1, -2))
        word = torch.where(word >= 1 << 31, word - (1 << 32), word).to(torch.int32)
        raw = word.contiguous().view(torch.uint8).view(N, K // 32, 16)
    raw = raw.permute(1, 0, 2) if tiled else raw
    return (raw.contiguous().view(-1).view(torch.uint8), s.t().contiguous(), None if z is None else z.t().contiguous(),
            W.reshape(N, K))


def _rope_anima(gh, gw):
    """the 3-axis split-half table over 128: 22 zero angles, 21 along h, 21 along w"""
    fh = 10000.0 ** (-2.0 * np.arange(21) / 42.0)
    hh, ww = np.divmod(np.arange(gh * gw), gw)
    ang = np.concatenate([np.zeros((gh * gw, 22)), hh[:, None] * fh, ww[:, None] * fh], 1)
    return np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)


def _rope_tokens(T):
    """a table for T tokens of no particular grid: 64 frequencies of one position"""
    ang = np.arange(T)[:, None] * 10000.0 ** (-np.arange(64) / 64.0)[None, :]
    return np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)


def _gains(g, n):
    """q / k norm gains around 1, the q ones with 1 / sqrt(128) folded in"""
    v = 1.0 + _randn(g, n, 128, std=0.1)
    v[0::2] *= 128 ** -0.5
    return v


def _pack(g, c):
    """one block's weights -> (pack bytes on the GPU, matrices W as fp16, vector section)"""
    kind, D, F = c["structure"], c["D"], c["F"]
    DC = 1024 if kind == 0 else 0
    fa, fm = FMT[c["attn"]], FMT[c["mlp"]]
    total, offs, voff = hip.pack_layout(kind, D, F, DC, fa, fm)
    buf = torch.zeros(total, dtype=torch.uint8, device=DEV)
    name = {v: k for k, v in FMT.items()}
    mats = []
    for i, ((N, K), fmt, (wo, so)) in enumerate(zip(hip.pack_shapes(kind, D, F, DC), hip.pack_fmts(kind, fa, fm), offs)):
        raw, s, _, W = _weight(g, N, K, name[fmt])
        if kind == 2 and i == 0:  # q, k, v rows each use their own 128 LoRA columns, the others are zero
            keep = torch.ones(N, K, dtype=torch.bool, device=DEV)
            for p in range(3):
                for r in range(3):
                    if r != p:
                        keep[p * D:(p + 1) * D, D + 128 * r:D + 128 * (r + 1)] = False
            W = W * keep
            unit = raw.numel() // (N * K)
            tiles = raw.view(K // 32, N, 32 * unit)
            raw = (tiles * keep.view(N, K // 32, 32).permute(1, 0, 2)[..., :1].to(torch.uint8)).reshape(-1)
        buf[wo:wo + raw.numel()] = raw
        if s is not None:
            buf[so:so + 2 * s.numel()] = s.view(-1).view(torch.uint8)
        mats.append(W)
    if kind == 0:
        vec = _gains(g, 4).reshape(-1)
    else:
        vec = torch.cat([_gains(g, 2).reshape(-1), 1.0 + _randn(g, 2 * D, std=0.1)])
    buf[voff:voff + 4 * vec.numel()] = vec.contiguous().view(torch.uint8)
    return buf, mats, vec


def _block_inputs(c, seed, weights):
    """weights(pack, matrices, vectors) is called with each block in turn"""
    g = _gen(seed, 1)
    kind, D, T, B = c["structure"], c["D"], c["T"], c["batch"]
    x = _randn(g, B * T, D)
    ctx = _randn(g, B * c["C"], 1024, dtype=HALF) if kind == 0 else None
    cos, sin = _rope_tokens(T)
    rows = 9 if kind == 0 else 6
    mods = []
    for k in range(c["depth"]):
        mod = _randn(g, rows, D, std=0.2)
        if kind == 0:  # the cross-attention site carries the identity modulation
            mod[3:5] = 0.0
            mod[5] = 1.0
        mods.append(mod)
        weights(*_pack(g, c))
    return x, ctx, torch.from_numpy(cos).to(DEV), torch.from_numpy(sin).to(DEV), mods


# the blkNN.bin layout: ten matrices one after another, the gains, then per site the modulation's A [256][2048], B [6144][256]
ANIMA_D, ANIMA_F, ANIMA_DC = 2048, 8192, 1024
ANIMA_MATS = [(2048, 2048)] * 5 + [(2048, 1024)] * 2 + [(2048, 2048), (8192, 2048), (2048, 8192)]  # [N][K]: sq sk sv so cq ck cv co m1 m2


def _blk_file(g, fmt):
    """-> (file bytes as numpy, offsets of the matrices and the gains, matrices, gains, [(A, B)] per site)"""
    parts, offs, mats, at = [], [], [], 0
    for N, K in ANIMA_MATS:
        raw, s, _, W = _weight(g, N, K, fmt, tiled=False)
        if fmt == "f16":
            rec = W.view(N // 32, 32, K // 32, 16, 2).permute(0, 2, 3, 1, 4).contiguous().view(-1).view(torch.uint8)
        else:
            u = (raw.view(torch.int8).to(torch.int16) + 128).to(torch.uint8)
            u = u.view(N // 32, 32, K // 32, 16, 2).permute(0, 2, 3, 1, 4).reshape(N // 32, K // 32, 1024)
            sc = s.view(K // 32, N // 32, 32).permute(1, 0, 2)[..., None].expand(-1, -1, -1, 2).contiguous()
            rec = torch.cat([sc.view(N // 32, K // 32, 64).view(torch.uint8), u], -1).reshape(-1)
        offs.append(at)
        at += rec.numel()
        parts.append(rec)
        mats.append(W)
    gains = _gains(g, 4).reshape(-1)
    offs.append(at)
    parts.append(gains.contiguous().view(torch.uint8))
    parts.append(torch.zeros(4096 - 2048, dtype=torch.uint8, device=DEV))
    modw = [(_randn(g, 256, 2048, std=0.02, dtype=HALF), _randn(g, 6144, 256, std=0.02, dtype=HALF)) for _ in range(3)]
    for a, b in modw:
        parts += [a.view(-1).view(torch.uint8), b.view(-1).view(torch.uint8)]
    return torch.cat(parts).cpu().numpy(), offs, mats, gains, modw


def _x32(x):
    """rows [R][C] -> 32 x 32 tiles"""
    R, Cc = x.shape
    return x.reshape(R // 32, 32, Cc // 32, 32).transpose(0, 2, 1, 3)


def _mega_inputs(c, seed):
    rng = np.random.default_rng(seed)
    T = c["gh"] * c["gw"]
    x = rng.standard_normal((T, ANIMA_D), dtype=np.float32)
    ctx = rng.standard_normal((c["nctx"], ANIMA_DC), dtype=np.float32).astype(np.float16)
    emb = rng.standard_normal(ANIMA_D, dtype=np.float32)
    lora = rng.standard_normal(6144, dtype=np.float32) * np.float32(0.1)
    cos, sin = _rope_anima(c["gh"], c["gw"])
    return x, ctx, emb, lora, cos, sin


def _denoise_inputs(c, seed):
    rng = np.random.default_rng(seed)
    lat = rng.standard_normal((c["batch"], 16, c["lat_h"], c["lat_w"]), dtype=np.float32)
    ctx = rng.standard_normal((c["batch"], c["C"], 1024), dtype=np.float32)
    return lat, ctx


# --------------------------------------------------------------------------------------------------------------- prepare
class Mega(State):
    def __del__(self):
        if getattr(self, "h", None) is not None:
            hip.lib().mega_close(self.h)


class Denoise(State):
    def __del__(self):
        if getattr(self, "dit", None):
            hip.lib().hxa_dit_destroy(self.dit)


def prepare(case, seed):
    hip.init(0)
    L, c = hip.lib(), dict(case)
    kind = c["kind"]
    if kind == "linear":
        s = State()
        g = _gen(seed)
        s.A = _randn(g, c["M"], c["K"], dtype=HALF)
        s.w, s.s, s.z, _ = _weight(g, c["N"], c["K"], c["fmt"], c["tiled"], c["mins"])
        s.fmt = FMT[c["fmt"]] | (hip.W_KTILED if c["tiled"] else 0)
        s.out = torch.empty(c["M"], c["N"], dtype=HALF, device=DEV)
        s.ws_bytes = L.hxa_linear_ws_bytes(c["M"], c["N"], c["K"], s.fmt)
        s.ws = torch.empty(max(s.ws_bytes, 16), dtype=torch.uint8, device=DEV)
    elif kind == "attn":
        s = State()
        g = _gen(seed)
        n, B, D = c["NKV"], c["batch"], c["H"] * 128
        # q and k come RMS-normalised per head, q with 1 / sqrt(128) in its gain; V transposed, images side by side
        s.q = _randn(g, B * c["T"], D, std=128 ** -0.5, dtype=HALF)
        s.k = _randn(g, B * n, D, dtype=HALF)
        s.vt = _randn(g, D, B * n, dtype=HALF)
        s.o = torch.empty(B * c["T"], D, dtype=HALF, device=DEV)
    elif kind == "norm":
        s = State()
        g = _gen(seed)
        D = c["D"]
        s.x = _randn(g, c["T"], D, std=2.0)
        s.shift, s.scale = _randn(g, D, std=0.2), _randn(g, D, std=0.2)
        s.w = 1.0 + _randn(g, D, std=0.1) if c["rms"] else None
        s.h = torch.empty(c["T"], D, dtype=HALF, device=DEV)
    elif kind == "block":
        s = State()
        s.packs = []
        s.x0, s.ctx, s.cos, s.sin, s.mods = _block_inputs(c, seed, lambda pack, mats, vec: s.packs.append(pack))
        s.x = torch.empty_like(s.x0)
        s.d = hip.BlockDims(c["structure"], c["D"], c["D"] // 128, c["F"], c["C"], 1024 if c["structure"] == 0 else 0, c["T"],
                            c["batch"], c["nvalid"], FMT[c["attn"]], FMT[c["mlp"]], 1, 0)
        s.ws = torch.zeros(L.hxa_block_ws_bytes(C.byref(s.d)), dtype=torch.uint8, device=DEV)
    elif kind == "mega":
        s = Mega()
        s.h = None
        g = _gen(seed, 2)
        x, ctx, s.emb, s.lora, cos, sin = _mega_inputs(c, seed)
        T = x.shape[0]
        two = [_blk_file(g, c["fmt"]) for _ in range(2)]  # the blocks take turns on two files' bytes, each registered by itself
        s.files = [f[0] for f in two]
        s.x = np.ascontiguousarray(_x32(x)).reshape(-1)
        c16 = ctx.reshape(c["nctx"] // 32, 16, 2, 32, 32).transpose(0, 3, 1, 4, 2)  # 32 x 32 tiles, row pairs interleaved
        rope = [np.ascontiguousarray(_x32(t)).reshape(-1) for t in (cos, sin)]
        parts = [s.x, np.ascontiguousarray(c16).reshape(-1)] + rope
        s.blob = np.concatenate([p.view(np.uint8) for p in parts])
        at = np.cumsum([0] + [p.nbytes for p in parts])
        offs = two[0][1]
        # meta[]: blob offsets of x, ctx, mod, gain, cos, sin; weight offsets; stage buffers (none); tokens, context, flags
        meta = [int(at[0]), int(at[1]), 0, offs[10], int(at[2]), int(at[3])] + offs[:10] + [-1] * 9 + [T, c["nctx"], 0, 4, 0, 0, int(c["fmt"] == "q8")]
        s.meta = []
        for k in range(c["blocks"]):
            m = list(meta)
            m[29], m[30] = int(k == c["blocks"] - 1), int(k == 0)  # release after the last block, first on the first
            s.meta.append((C.c_int * len(m))(*m))
        s.fds = np.arange(100, 100 + c["blocks"], dtype=np.int32)
        s.mod = np.zeros((c["blocks"], 9, ANIMA_D), np.float32)
        h = C.c_uint64()
        hip.check(L.mega_open(b"", C.byref(h)), "mega_open")
        s.h = h
        for k, fd in enumerate(s.fds):
            f = s.files[k % 2]
            hip.check(L.hxa_register(h, int(fd), f.ctypes.data, f.nbytes, hip.KIND_WEIGHTS_ANIMA), "register")
        hip.check(L.hxa_register(h, 1, s.blob.ctypes.data, s.blob.nbytes, hip.KIND_BLOB), "register")
    else:
        s = Denoise()
        s.dit = None
        s.lat, s.ctx = _denoise_inputs(c, seed)
        f = FMT[c["fmt"]]
        bd = hip.BlockDims(0, c["D"], c["D"] // 128, c["F"], c["C"], 1024, 0, c["batch"], 0, f, f, 1)
        cfg = hip.DitCfg(bd, c["blocks"], 16, c["lat_h"], c["lat_w"], 256, 0)
        dit = C.c_void_p()
        hip.check(L.hxa_dit_create(C.byref(cfg), int(seed) + 1, C.byref(dit)), "dit_create")
        s.dit = dit
        s.sigmas = [1.0 - i / c["steps"] for i in range(c["steps"] + 1)]
    s.case = c
    return s


# ------------------------------------------------------------------------------------------------------------------- run
def _p(t):
    return None if t is None else t.data_ptr()


def run(s):
    L, c = hip.lib(), s.case
    kind = c["kind"]
    st = torch.cuda.current_stream().cuda_stream
    if kind == "linear":
        hip.check(L.hxa_linear(_p(s.A), c["K"], c["M"], s.fmt, _p(s.w), _p(s.s), _p(s.z), c["N"], c["K"], _p(s.out), c["N"],
                               _p(s.ws), s.ws_bytes, st), "linear")
        return s.out
    if kind == "attn":
        T, n, D, B = c["T"], c["NKV"], c["H"] * 128, c["batch"]
        hip.check(L.hxa_attention(_p(s.q), D, _p(s.k), D, _p(s.vt), B * n, _p(s.o), D, T, n, c["nvalid"], c["H"], B, T * D, n * D,
                                  n, T * D, st), "attention")
        return s.o
    if kind == "norm":
        hip.check(L.hxa_norm_mod(_p(s.x), c["D"], c["T"], c["D"], _p(s.shift), _p(s.scale), _p(s.w), 1e-6, _p(s.h), c["D"], st),
                  "norm_mod")
        return s.h
    if kind == "block":
        s.x.copy_(s.x0)  # the residual stream that reaches these blocks
        for pack, mod in zip(s.packs, s.mods):
            hip.check(L.hxa_block_run(C.byref(s.d), _p(pack), _p(s.x), _p(s.ctx), _p(mod), _p(s.cos), _p(s.sin), _p(s.ws), 0, None,
                                      0, st), "block_run")
        return s.x
    if kind == "mega":
        n = s.x.nbytes
        s.blob[:n].view(np.float32)[:] = s.x  # the caller lays its tokens into the blob
        hip.check(L.hxa_anima_modulation(s.h, s.fds.ctypes.data, c["blocks"], s.emb.ctypes.data, s.lora.ctypes.data,
                                         s.mod.ctypes.data), "modulation")
        rc = C.c_int()
        for k, meta in enumerate(s.meta):
            hip.check(L.mega_block(s.h, meta, len(meta), int(s.fds[k]), 1, s.mod[k].ctypes.data, s.mod[k].nbytes, None, 0,
                                   C.byref(rc)), "mega_block")
            hip.check(rc.value, "mega_block")
        return s.blob[:n].view(np.float32).copy()
    hip.check(L.hxa_dit_set_inputs(s.dit, s.lat.ctypes.data, s.ctx.ctypes.data), "set_inputs")
    for i in range(c["steps"]):
        if i < c["low"]:
            hip.check(L.hxa_dit_step_lowres(s.dit, s.sigmas[i], s.sigmas[i + 1], 2, 1), "step_lowres")
        else:
            hip.check(L.hxa_dit_step(s.dit, s.sigmas[i], s.sigmas[i + 1], 1), "step")
    out = np.empty_like(s.lat)
    hip.check(L.hxa_dit_get_latent(s.dit, out.ctypes.data), "get_latent")
    return out


# ------------------------------------------------------------------------------------------------------------------ work
def _block_work(structure, D, F, T, B, nvalid, Cn, fa, fm):
    """(bytes, flops) of one block: every weight once, x in and out"""
    R = 128
    if structure == 0:
        attn, mlp = [(3 * D, D), (D, D), (D, D), (D, D)], [(F, D), (D, F)]
        fl = sum(2.0 * B * T * n * k for n, k in attn + mlp) + 2.0 * B * Cn * 2 * D * 1024
        fl += 4.0 * B * T * D * (T + Cn)
        attn = attn + [(2 * D, 1024)]
    else:
        attn, mlp = [(3 * D, D), (D, D)], [(2 * F, D), (D, F)]
        if structure == 2:  # the A matrices, and 128 more columns of every projection
            attn += [(3 * R, D), (R, D), (3 * D, R), (D, R)]
            mlp += [(R, D), (R, F), (2 * F, R), (D, R)]
        fl = sum(2.0 * B * T * n * k for n, k in attn + mlp) + 4.0 * B * T * D * nvalid
    by = sum(n * k for n, k in attn) * WBYTES[fa] + sum(n * k for n, k in mlp) * WBYTES[fm]
    return by + 8.0 * B * T * D, fl


def work(case):
    c = dict(case)
    kind = c["kind"]
    if kind == "linear":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": 2.0 * M * K + WBYTES[c["fmt"]] * N * K + 2.0 * M * N, "flops": 2.0 * M * N * K}
    if kind == "attn":
        T, n, D, B = c["T"], c["nvalid"], c["H"] * 128, c["batch"]
        return {"bytes": 2.0 * B * D * (2 * T + 2 * n), "flops": 4.0 * B * T * n * D}
    if kind == "norm":
        return {"bytes": 6.0 * c["T"] * c["D"], "flops": 8.0 * c["T"] * c["D"]}
    if kind == "block":
        by, fl = _block_work(c["structure"], c["D"], c["F"], c["T"], c["batch"], c["nvalid"], c["C"], c["attn"], c["mlp"])
        return {"bytes": by * c["depth"], "flops": fl * c["depth"]}
    if kind == "mega":
        T = c["gh"] * c["gw"]
        by, fl = _block_work(0, ANIMA_D, ANIMA_F, T, 1, T, c["nctx"], c["fmt"], c["fmt"])
        mod = 3.0 * (256 * 2048 + 6144 * 256)
        return {"bytes": (by + 2 * mod) * c["blocks"], "flops": (fl + 2 * mod) * c["blocks"]}
    T = c["lat_h"] * c["lat_w"] // 4
    by = fl = 0.0
    for i in range(c["steps"]):
        t = T // 4 if i < c["low"] and (T // 4) % 32 == 0 and c["lat_h"] % 4 == 0 and c["lat_w"] % 4 == 0 else T
        b, f = _block_work(0, c["D"], c["F"], t, c["batch"], t, c["C"], c["fmt"], c["fmt"])
        by += (b + 12.0 * c["D"] * c["D"]) * c["blocks"]
        fl += (f + 12.0 * c["D"] * c["D"]) * c["blocks"]
    return {"bytes": by, "flops": fl}


def tolerance(case):
    """About four times the error measured against 64-bit values (2.1e-4 for what is rounded to fp16 once, 2.8e-4 after an
    attention, 2.0e-4 to 3.4e-4 over four blocks, 5.3e-4 over a denoise); two roundings of the same value apart by their sum."""
    return {"linear": {"rel": 1e-3, "max": 4e-3}, "attn": {"rel": 1.2e-3, "max": 2e-2}, "norm": {"rel": 1e-3, "max": 4e-3},
            "block": {"rel": 1.5e-3, "max": 4e-2}, "mega": {"rel": 1.5e-3, "max": 4e-2},
            "denoise": {"rel": 2.5e-3, "max": 5e-2}}[case["kind"]]


# ----------------------------------------------------------------------------------------------------------------- exact
def _norm(x, rms, w, shift, scale):
    if not rms:
        x = x - x.mean(-1, keepdim=True)
    x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6)
    return x * (1.0 + scale) * (1.0 if w is None else w) + shift


def _heads(x, gain, cos=None, sin=None):
    """per-head RMSNorm * gain, then RoPE on the pairs (d, d + 64)"""
    n, D = x.shape
    x = x.view(n, D // 128, 128)
    x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * gain
    if cos is not None:
        a, b = x[..., :64], x[..., 64:]
        cc, ss = cos[:, None], sin[:, None]
        x = torch.cat([a * cc - b * ss, a * ss + b * cc], -1)
    return x.reshape(n, D)


def _attend(q, k, v, nvalid):
    o = torch.empty_like(q)
    for h in range(q.shape[1] // 128):
        i = slice(128 * h, 128 * h + 128)
        for t in range(0, q.shape[0], 2048):
            p = torch.softmax(q[t:t + 2048, i] @ k[:nvalid, i].t().contiguous(), -1)
            o[t:t + 2048, i] = p @ v[:nvalid, i].contiguous()
    return o


def _gelu(t, tanh):
    if tanh:
        return 0.5 * t * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (t + 0.044715 * t ** 3)))
    return 0.5 * t * torch.special.erfc(-t / math.sqrt(2.0))


def _mm(x, W):
    return x @ W.to(F64).t().contiguous()


def _anima_block(x, ctx, mod, cos, sin, W, vec, tanh):
    """one image; W = qkv, o, cq, ckv, co, w1, w2"""
    D = x.shape[1]
    g, mod = vec.to(F64).view(4, 128), mod.to(F64)
    h = _norm(x, False, None, mod[0], mod[1])
    qkv = _mm(h, W[0])
    q, k = _heads(qkv[:, :D], g[0], cos, sin), _heads(qkv[:, D:2 * D], g[1], cos, sin)
    x = x + mod[2] * _mm(_attend(q, k, qkv[:, 2 * D:], len(x)), W[1])
    h = _norm(x, False, None, mod[3], mod[4])
    ckv = _mm(ctx, W[3])
    q, k = _heads(_mm(h, W[2]), g[2]), _heads(ckv[:, :D], g[3])
    x = x + mod[5] * _mm(_attend(q, k, ckv[:, D:], len(ctx)), W[4])
    h = _norm(x, False, None, mod[6], mod[7])
    return x + mod[8] * _mm(_gelu(_mm(h, W[5]), tanh), W[6])


def _moss_block(x, mod, cos, sin, W, vec, nvalid):
    """one image; W = qkv, o, up_gate, down and, with the LoRA, its A matrices, whose products extend the rows"""
    D = x.shape[1]
    mod, vec = mod.to(F64), vec.to(F64)

    def proj(a, i):
        return _mm(torch.cat([a, _mm(a, W[4 + i])], 1) if len(W) > 4 else a, W[i])

    h = _norm(x, True, vec[256:256 + D], mod[0], mod[1])
    qkv = proj(h, 0)
    q, k = _heads(qkv[:, :D], vec[:128], cos, sin), _heads(qkv[:, D:2 * D], vec[128:256], cos, sin)
    x = x + mod[2] * proj(_attend(q, k, qkv[:, 2 * D:], nvalid), 1)
    h = _norm(x, True, vec[256 + D:], mod[3], mod[4])
    ug = proj(h, 2)
    ug = ug.view(len(x), -1, 2, 32)
    u, gt = ug[:, :, 0].reshape(len(x), -1), ug[:, :, 1].reshape(len(x), -1)
    return x + mod[5] * proj(25.0 * torch.tanh(u / 25.0) * 4.0 * torch.tanh(gt / 4.0) * torch.sigmoid(gt), 3)


def exact(case, seed):
    c = dict(case)
    kind = c["kind"]
    if kind == "linear":
        g = _gen(seed)
        A = _randn(g, c["M"], c["K"], dtype=HALF)
        W = _weight(g, c["N"], c["K"], c["fmt"], c["tiled"], c["mins"])[3]
        return _mm(A.to(F64), W)
    if kind == "attn":
        g = _gen(seed)
        T, n, B, D = c["T"], c["NKV"], c["batch"], c["H"] * 128
        q = _randn(g, B * T, D, std=128 ** -0.5, dtype=HALF).to(F64)
        k = _randn(g, B * n, D, dtype=HALF).to(F64)
        v = _randn(g, D, B * n, dtype=HALF).to(F64).t().contiguous()
        return torch.cat([_attend(q[b * T:(b + 1) * T], k[b * n:(b + 1) * n], v[b * n:(b + 1) * n], c["nvalid"]) for b in range(B)])
    if kind == "norm":
        g = _gen(seed)
        D = c["D"]
        x, shift, scale = _randn(g, c["T"], D, std=2.0), _randn(g, D, std=0.2), _randn(g, D, std=0.2)
        w = (1.0 + _randn(g, D, std=0.1)).to(F64) if c["rms"] else None
        return _norm(x.to(F64), c["rms"], w, shift.to(F64), scale.to(F64))
    if kind == "block":
        blocks = []
        x, ctx, cos, sin, mods = _block_inputs(c, seed, lambda pack, mats, vec: blocks.append((mats, vec)))
        T, x, cos, sin = c["T"], x.to(F64), cos.to(F64), sin.to(F64)
        for b in range(c["batch"]):
            xi = x[b * T:(b + 1) * T]
            for (mats, vec), mod in zip(blocks, mods):
                if c["structure"] == 0:
                    xi = _anima_block(xi, ctx[b * c["C"]:(b + 1) * c["C"]].to(F64), mod, cos, sin, mats, vec, True)
                else:
                    xi = _moss_block(xi, mod, cos, sin, mats, vec, c["nvalid"])
            x[b * T:(b + 1) * T] = xi
        return x
    if kind == "mega":
        g = _gen(seed, 2)
        x, ctx, emb, lora, cos, sin = (torch.from_numpy(a).to(DEV).to(F64) for a in _mega_inputs(c, seed))
        two = [_blk_file(g, c["fmt"]) for _ in range(2)]
        mods = []
        for _, _, _, _, modw in two:
            silu = (emb * torch.sigmoid(emb))[None]
            mods.append(torch.cat([(lora + _mm(_mm(silu, a), b)[0]).view(3, ANIMA_D) for a, b in modw]))
        for k in range(c["blocks"]):
            _, _, m, gains, _ = two[k % 2]
            W = [torch.cat(m[:3]), m[3], m[4], torch.cat(m[5:7]), m[7], m[8], m[9]]
            x = _anima_block(x, ctx, mods[k % 2], cos, sin, W, gains, False)
        return np.ascontiguousarray(_x32(x.cpu().numpy())).reshape(-1)
    return None  # the denoise runs on weights that the runner draws itself
