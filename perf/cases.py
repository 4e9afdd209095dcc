"""The workloads this package is timed on, and what they compute in 64 bits.

Each case is a dict of plain values.  ``prepare`` makes what a user's program
holds before the call, ``run`` is one pass through the package's public entry
points, ``exact`` the same outputs from plain torch in float64.
"""

import math
from functools import partial

import torch
import torch.nn.functional as F

from imfvideo_amd import ops
from imfvideo_amd.imf_dit_video import TransformerBlock, precompute_axial_rope_3d
from imfvideo_amd.mla_video_sparse_jvp import tile_permutation
from imfvideo_amd.sla2_attention import SLA2AttentionImpl
from imfvideo_amd.sla2_cube_qat import SLA2CubeQATAttentionImpl, sla2_cube_qat_jvp_fused
from imfvideo_amd.sla2_mla_jvp import sla2_mla_jvp
from imfvideo_amd.sla2_vendor import SLA2

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
E = 64
LOG2E = 1.4426950408889634
EPS_L = 1e-5
# widths of the DiT block of the repository's training benchmark
D_MODEL, N_HEADS, DQ, DC, DN, DR, DV, MLP_RATIO = 512, 8, 256, 128, 32, 32, 64, 4


def listed():
    return [
        # A unit-test sized call (the reference's test geometry: 4 video tiles and
        # an 18-token prefix): launches and host work decide.
        dict(name="jvp_tiny", kind="jvp", dtype="bf16", B=1, H=4, Np=4, P=18, topk=0.5, proj=True),
        # A short clip: 4,096 tokens, 4 heads, 10 % of the tiles.
        dict(name="jvp_4k", kind="jvp", dtype="bf16", B=1, H=4, Np=64, P=0, topk=0.1, proj=False),
        # The du/dt pass of a training step in the module's default setting: top 3 %
        # of the tiles, learned router projections, a text prefix, fp16, batch 2.
        dict(name="jvp_prefix_14k", kind="jvp", dtype="fp16", B=2, H=8, Np=216, P=77, topk=0.03,
             proj=True),
        # The headline workload: forward and JVP at 29,952 tokens (12 x 48 x 52).
        dict(name="jvp_30k", kind="jvp", dtype="bf16", B=1, H=8, Np=468, P=0, topk=0.1, proj=False),
        # The same op without tangents (the sampler's forward).
        dict(name="primal_30k", kind="primal", dtype="bf16", B=1, H=8, Np=468, P=0, topk=0.1,
             proj=False),
        # The 1-D variant with dense-ish routing (top 25 %) on a ragged length.
        dict(name="jvp1d_29k", kind="jvp1d", dtype="fp16", B=1, H=4, L=29138, bq=128, topk=0.25),
        # One attention training step (forward and backward) of the module at full
        # video length, batch 2, sequence kept tile-major.
        dict(name="train_30k", kind="cube_train", dtype="fp16", B=2, H=8, gt=12, gh=48, gw=52, P=0,
             topk=0.1, tile_major=True),
        # A training step on a small clip in model order, with a prefix.
        dict(name="train_1k", kind="cube_train", dtype="bf16", B=1, H=4, gt=4, gh=16, gw=16, P=18,
             topk=0.1, tile_major=False),
        # The guidance branch: the module without gradients, model order, prefix.
        dict(name="guide_8k", kind="cube_guide", dtype="bf16", B=1, H=8, gt=8, gh=32, gw=32, P=77,
             topk=0.1, tile_major=False),
        # Inference of the 1-D SLA2 module with INT8 scores, ragged length.
        dict(name="infer1d_14k", kind="sla2_infer", dtype="bf16", B=1, H=8, L=13901, bq=128,
             topk=0.1, int8=True),
        # A training step of the 1-D attention module (16-bit scores).
        dict(name="train1d_4k", kind="sla2_train", dtype="fp16", B=1, H=8, L=4159, topk=0.1),
        # A whole DiT block, forward and backward under bf16 autocast, batch 2.
        dict(name="block_8k", kind="block_train", dtype="bf16", B=2, H=8, gt=8, gh=32, gw=32, P=0,
             topk=0.1, tile_major=True),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    most = work(next(c for c in listed() if c["name"] == "train_30k"))["flops"]
    while True:
        kind = rng.choice(["jvp", "jvp", "primal", "jvp1d", "cube_train", "cube_guide",
                           "sla2_infer", "sla2_train", "block_train"])
        c = dict(kind=kind, dtype=rng.choice(["bf16", "fp16"]), B=rng.choice([1, 1, 2]),
                 H=rng.choice([1, 2, 3, 4, 6, 8]),
                 topk=rng.choice([0.03, 0.1, 0.25, round(rng.uniform(0.02, 0.4), 3)]))
        if kind in ("jvp", "primal"):
            c.update(Np=_logint(rng, 4, 468), P=rng.choice([0, _logint(rng, 1, 200)]),
                     proj=rng.random() < 0.5)
        elif kind in ("jvp1d", "sla2_infer", "sla2_train"):
            c.update(L=_logint(rng, 274, 29952))
            if kind == "sla2_train":
                c.update(dtype="fp16")
            else:
                c.update(bq=rng.choice([64, 128, 256]))
            if kind == "sla2_infer":
                c.update(int8=rng.random() < 0.7)
        else:
            c.update(gt=4 * rng.randint(1, 3), gh=4 * _logint(rng, 1, 13), gw=4 * _logint(rng, 2, 13),
                     P=rng.choice([0, _logint(rng, 1, 200)]), tile_major=rng.random() < 0.5)
            if kind == "block_train":
                c.update(dtype="bf16", H=N_HEADS, P=0, tile_major=True)
        if work(c)["flops"] <= most:
            return c


# ---------------------------------------------------------------------------
# Sizes of a case
# ---------------------------------------------------------------------------
def _geometry(c):
    """(L, Np, P, bq) of a case; the 1-D cases have every 64-row block routable."""
    if "L" in c:
        return c["L"], -(-c["L"] // E), 0, c.get("bq", 128)
    Np = c["Np"] if "Np" in c else (c["gt"] // 4) * (c["gh"] // 4) * (c["gw"] // 4)
    return Np * E + c["P"], Np, c["P"], E


def _topk(c, Np):
    return max(1, min(Np, int(c["topk"] * Np)))


def work(c):
    """Bytes: inputs and outputs once.  flops: two per multiply-add of the routed
    64 x 64 x 64 tile products and of the linear branch's states and products."""
    L, Np, P, _ = _geometry(c)
    B, H, nb = c["B"], c["H"], -(-L // E)
    T = _topk(c, Np) + (nb - Np)
    kind, pairs, gemm, t = c["kind"], B * H * nb * T, 2 * E ** 3, B * H * L * E
    fwd = {"jvp": 6, "jvp1d": 6}.get(kind, 2)
    lin = {"jvp": 6, "jvp1d": 6}.get(kind, 2)
    bwd = kind in ("cube_train", "sla2_train", "block_train")
    flops = pairs * gemm * (fwd + (7 if bwd else 0)) + B * H * nb * gemm * (lin + (6 if bwd else 0))
    if kind in ("jvp", "jvp1d"):
        nbytes = 6 * t * 2 + 2 * t * 4
    elif kind == "primal":
        nbytes = 3 * t * 2 + t * 4
    elif bwd:
        nbytes = 8 * t * 2
    else:
        nbytes = 4 * t * 2
    if kind == "block_train":
        macs = (D_MODEL * (DQ + DC + DR) + DQ * H * (DN + DR) + DC * H * (DN + DV)
                + 2 * D_MODEL * H * DV + 3 * D_MODEL * D_MODEL * MLP_RATIO)
        flops += 3 * 2 * B * L * macs
        nbytes = 4 * B * L * D_MODEL * 4 + 2 * macs * 4
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------------------
# Inputs and passes
# ---------------------------------------------------------------------------
def _rms(x):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6)


def _tensors(c, seed, n):
    """q, k (per-token RMS-normalised, as behind a qk-norm), v and n - 3 more, all
    (B, H, L, 64) in the case's dtype: N(0, 1) tokens on a component that the
    tokens of a tile share and that varies slowly from tile to tile."""
    L, _, _, _ = _geometry(c)
    B, H, nb = c["B"], c["H"], -(-L // E)
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    out = []
    for i in range(n):
        x = rnd(B, H, L, E)
        if i < 3:
            walk = rnd(B, H, nb + 7, E).cumsum(2)
            tile = (F.pad(walk, (0, 0, 1, 0))[:, :, 8:] - F.pad(walk, (0, 0, 1, 0))[:, :, :nb]) / 8 ** 0.5
            x += 0.5 * tile.repeat_interleave(E, dim=2)[:, :, :L]
        if i < 2:
            x = _rms(x)
        out.append(x)
    return out, g


def _alpha_logits(g, H, M):
    return 2.2 + 0.3 * torch.randn(H, M, generator=g, device=DEV)


def prepare(c, seed):
    L, Np, P, bq = _geometry(c)
    B, H, kind, dt = c["B"], c["H"], c["kind"], DTYPES[c["dtype"]]
    s = {"case": c}
    if kind == "block_train":
        return _prepare_block(c, seed)
    n = 6 if kind in ("jvp", "jvp1d") else 4
    x, g = _tensors(c, seed, n)
    if n == 6:
        x[3:] = [0.1 * t for t in x[3:]]
    x = [t.to(dt) for t in x]
    M = -(-L // bq)
    logits = _alpha_logits(g, H, M)
    proj = [torch.eye(E, device=DEV) + 0.1 * torch.randn(E, E, generator=g, device=DEV)
            for _ in range(2)]
    if kind in ("jvp", "primal"):
        s.update(x=x, alpha=torch.sigmoid(logits), proj=proj if c["proj"] else [None, None])
    elif kind == "jvp1d":
        s.update(x=x, alpha=torch.sigmoid(logits))
    elif kind in ("cube_train", "cube_guide"):
        impl = SLA2CubeQATAttentionImpl(E, L, H, (c["gt"], c["gh"], c["gw"]), topk=c["topk"],
                                        pre_permuted=c["tile_major"]).to(DEV)
        with torch.no_grad():
            impl.alpha_logit.copy_(logits)
            impl.proj_q.copy_(proj[0])
            impl.proj_k.copy_(proj[1])
        if not c["tile_major"]:  # model order: the prefix first
            x = [t[:, :, impl.inv] for t in x]
        x = [t.permute(0, 2, 1, 3).contiguous() for t in x]  # (B, L, H, 64)
        if kind == "cube_train":
            x = [t.requires_grad_() for t in x[:3]] + x[3:]
        s.update(x=x, impl=impl)
    elif kind == "sla2_train":
        impl = SLA2AttentionImpl(E, L, H, topk=c["topk"]).to(DEV)
        with torch.no_grad():
            impl.sla2.alpha_logit.copy_(logits)
        x = [t.permute(0, 2, 1, 3).contiguous() for t in x]
        s.update(x=[t.requires_grad_() for t in x[:3]] + x[3:], impl=impl)
    else:
        impl = SLA2(E, topk=c["topk"], bq=bq, use_bf16=c["dtype"] == "bf16",
                    use_int8=c["int8"]).to(DEV)
        impl.alpha_logit = torch.nn.Parameter(logits)
        s.update(x=x, impl=impl)
    return s


def _prepare_block(c, seed):
    L, Np, P, _ = _geometry(c)
    grid = (c["gt"], c["gh"], c["gw"])
    g = torch.Generator(device=DEV).manual_seed(seed)
    impl = partial(SLA2CubeQATAttentionImpl, seq_len=L, num_heads=c["H"], grid=grid,
                   topk=c["topk"], pre_permuted=True)
    block = TransformerBlock(D_MODEL, c["H"], DQ, DC, DN, DR, DV, mlp_ratio=MLP_RATIO,
                             weight_init_constant=0.5, attn_impl=impl).to(DEV)
    with torch.no_grad():
        for p in block.parameters():
            if p.dim() == 2 and p.shape[0] != p.shape[1] or p.shape == (D_MODEL, D_MODEL):
                p.copy_(torch.randn(p.shape, generator=g, device=DEV) * 0.5 / p.shape[1] ** 0.5)
        block.attn.attn_impl.alpha_logit.copy_(_alpha_logits(g, c["H"], -(-L // E)))
        block.attn_scale.fill_(0.1)
        block.mlp_scale.fill_(0.1)
    perm, _, _ = tile_permutation(grid, (4, 4, 4), 0, torch.device("cpu"))
    cos, sin = (t[perm].to(DEV) for t in precompute_axial_rope_3d(DR, grid, 0, axis_dims=(8, 12, 12)))
    x = torch.randn(c["B"], L, D_MODEL, generator=g, device=DEV)
    x = x + 0.5 * torch.randn(c["B"], -(-L // E), D_MODEL, generator=g, device=DEV).repeat_interleave(
        E, dim=1)[:, :L]
    dy = torch.randn(c["B"], L, D_MODEL, generator=g, device=DEV)
    names = [n for n, p in block.named_parameters() if ".proj_" not in n]
    params = dict(block.named_parameters())
    return {"case": c, "x": x.requires_grad_(), "dy": dy, "block": block, "cos": cos, "sin": sin,
            "names": names, "wrt": [params[n] for n in names]}


def run(s):
    c = s["case"]
    L, Np, P, bq = _geometry(c)
    kind = c["kind"]
    if kind == "jvp":
        return sla2_cube_qat_jvp_fused(*s["x"], s["alpha"], c["topk"], Np, E, P, *s["proj"])
    if kind == "primal":
        o, _ = ops.cube_jvp(*s["x"][:3], None, None, None, s["alpha"], c["topk"], Np, P, *s["proj"])
        return o
    if kind == "jvp1d":
        return sla2_mla_jvp(*s["x"], s["alpha"], c["topk"], bq, E)
    if kind == "cube_train":
        q, k, v, do = s["x"]
        o = s["impl"](q, k, v)
        grads = torch.autograd.grad(o, [q, k, v, s["impl"].alpha_logit], do)
        return [o.detach(), *grads, s["impl"].logit_max_log2]
    if kind == "sla2_train":
        q, k, v, do = s["x"]
        o = s["impl"](q, k, v)
        return [o.detach(), *torch.autograd.grad(o, [q, k, v, s["impl"].sla2.alpha_logit], do)]
    if kind == "block_train":
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = s["block"](s["x"], s["cos"], s["sin"])
        grads = torch.autograd.grad(y, [s["x"], *s["wrt"]], s["dy"])
        return {"y": y.detach(), "dx": grads[0], **dict(zip(s["names"], grads[1:])),
                "logit_max_log2": s["block"].attn.attn_impl.logit_max_log2}
    with torch.no_grad():
        return s["impl"](*s["x"][:3])


# About four times the largest relative error against `exact` that 70 listed and drawn
# cases showed on one MI355X, by kind and 16-bit type.  In the whole block another
# rounding of q or k routes another tile now and then (0.3 % of the routed tiles against
# float64), which moves the attention weights' gradients by 5-14 %.
TOLERANCE = {
    "jvp": {"bf16": 8e-3, "fp16": 1e-3}, "primal": {"bf16": 1.4e-3, "fp16": 2.5e-4},
    "jvp1d": {"bf16": 6e-3, "fp16": 1e-3}, "cube_train": {"bf16": 7e-3, "fp16": 2.3e-3},
    "cube_guide": {"bf16": 7e-3, "fp16": 1.6e-3}, "sla2_infer": {"bf16": 9e-3, "fp16": 2e-3},
    "sla2_train": {"fp16": 2.3e-3}, "block_train": {"bf16": 0.3},
}


def tolerance(c):
    return {"rel": TOLERANCE[c["kind"]][c["dtype"]]}


# ---------------------------------------------------------------------------
# The same outputs in float64
# ---------------------------------------------------------------------------
def _tiles(x, nb):
    """(B, H, L, 64) -> (B * H, nb, 64, 64), zero rows past L."""
    B, H, L, D = x.shape
    return F.pad(x, (0, 0, 0, nb * E - L)).reshape(B * H, nb, E, D)


def _quant(x, nb, rows, trunc):
    """INT8 values (float64 tiles) and per-row scales of (B, H, L, 64) 16-bit values:
    symmetric over blocks of `rows` rows, in the fp32 arithmetic that defines
    the integers (round half away from zero; `trunc`: fl(x/s + 0.5) truncated)."""
    B, H, L, D = x.shape
    n = -(-nb * E // rows)
    xb = F.pad(x.float(), (0, 0, 0, n * rows - L)).reshape(B * H, n, rows, D)
    s = xb.abs().amax((-2, -1), keepdim=True) / torch.full((), 127.0, device=x.device) + 1e-12
    y = xb / s
    if trunc:
        q = torch.trunc(y + torch.where(xb >= 0, 0.5, -0.5))
    else:
        q = torch.sign(y) * torch.floor(y.abs().double() + 0.5).float()
    q = q.reshape(B * H, n * rows, D)[:, :nb * E].reshape(B * H, nb, E, D)
    s = s.reshape(B * H, n, 1).expand(B * H, n, rows).reshape(B * H, n * rows)[:, :nb * E]
    return q.double(), s.double().reshape(B * H, nb, E)


def _pool(x, rows):
    B, H, L, D = x.shape
    n = -(-L // rows)
    xb = F.pad(x.double(), (0, 0, 0, n * rows - L)).reshape(B * H, n, rows, D)
    cnt = torch.clamp(L - rows * torch.arange(n, device=x.device), max=rows)
    return xb.sum(2) / cnt[:, None]


def _lut(q, k, T, Np, bq, proj, nb):
    """Routed tile ids per 64-row query block, best first, prefix blocks last."""
    qp, kp = _pool(q, bq), _pool(k, E)[:, :Np]
    if proj is not None and proj[0] is not None:
        qp, kp = qp @ proj[0].double().T, kp @ proj[1].double().T
    lut = torch.topk(qp @ kp.transpose(-1, -2), T, dim=-1).indices
    lut = lut.repeat_interleave(bq // E, dim=1)[:, :nb]
    tail = torch.arange(Np, nb, device=q.device).expand(lut.shape[0], nb, nb - Np)
    return torch.cat([lut, tail], -1)


def _col(x, lut, j):
    """Tile lut[:, :, j] of x (G, N, ...) for every query block."""
    return x[torch.arange(x.shape[0], device=x.device)[:, None], lut[..., j]]


def _mm(a, b):
    return torch.matmul(a, b)


def _sparse(qt, qscale, kt, kscale, vt, lut, L, tan=None, p8=False, vscale=None):
    """Softmax attention over the routed tiles -> (o, do, lse in log2).  tan: tiles
    (q, k, dq, dk, dv) of the unquantised tangent.  p8: the INT8 P of the
    training and inference kernels, against the running maximum."""
    G, N = kt.shape[:2]
    valid = (torch.arange(N * E, device=qt.device) < L).reshape(1, N, E).expand(G, N, E)
    m = torch.full(qt.shape[:3], -math.inf, device=qt.device, dtype=torch.float64)
    l = torch.zeros_like(m)
    mu = torch.zeros_like(m)
    o = torch.zeros_like(qt)
    do = torch.zeros_like(qt)
    for j in range(lut.shape[-1]):
        s = _mm(qt, _col(kt, lut, j).transpose(-1, -2).contiguous())
        s = s * (qscale[..., None] * _col(kscale, lut, j)[:, :, None, :] * (E ** -0.5 * LOG2E))
        s = s.masked_fill(~_col(valid, lut, j)[:, :, None, :], -math.inf)
        new = torch.maximum(m, s.amax(-1))
        al, p = torch.exp2(m - new), torch.exp2(s - new[..., None])
        l, m = l * al + p.sum(-1), new
        vj = _col(vt, lut, j)
        pv = p
        if p8:
            pv = torch.trunc(127.0 * p + 0.5) / 127.0 * _col(vscale, lut, j)[:, :, None, :]
        o = o * al[..., None] + _mm(pv, vj)
        if tan is not None:
            q, k, dq, dk, dv = tan
            ds = _mm(dq, _col(k, lut, j).transpose(-1, -2).contiguous())
            ds = (ds + _mm(q, _col(dk, lut, j).transpose(-1, -2).contiguous())) * E ** -0.5
            t = p * ds
            mu = mu * al + t.sum(-1)
            do = do * al[..., None] + _mm(t, vj) + _mm(p, _col(dv, lut, j))
    o = o / l[..., None]
    do = do / l[..., None] - (mu / l)[..., None] * o
    return o, do, m + torch.log2(l)


def _phi(x, dx=None):
    p = torch.softmax(x.double(), -1)
    if dx is None:
        return p, None
    return p, p * (dx - (p * dx).sum(-1, keepdim=True))


def _unselected(lut, N):
    """(G, M, N) float64: 1 where query block m does not attend tile n exactly."""
    G, M, _ = lut.shape
    return torch.ones(G, M, N, device=lut.device, dtype=torch.float64).scatter_(2, lut, 0.0)


def _linear(qt, kt, vt, keep, L, tan=None, signed=True):
    """Linear attention over the tiles that `keep` marks -> (o, do, H, z, den)."""
    G, N = kt.shape[:2]
    M = qt.shape[1]
    valid = (torch.arange(N * E, device=qt.device) < L).reshape(1, N, E, 1)
    dk = None if tan is None else tan[3]
    kphi, dkphi = _phi(kt, dk)
    kphi = kphi * valid
    qphi, dqphi = _phi(qt, None if tan is None else tan[2])
    comp = lambda st: _mm(keep, st.reshape(G, N, -1)).reshape(G, M, *st.shape[2:])
    kT = kphi.transpose(-1, -2).contiguous()
    Hc, zc = comp(_mm(kT, vt)), comp(kphi.sum(2))
    num, den = _mm(qphi, Hc), _mm(qphi, zc[..., None])[..., 0]
    den = den + (torch.where(den >= 0, EPS_L, -EPS_L) if signed else EPS_L)
    o, do = num / den[..., None], None
    if tan is not None:
        dkphi = dkphi * valid
        dHc = comp(_mm(dkphi.transpose(-1, -2).contiguous(), vt) + _mm(kT, tan[4]))
        dzc = comp(dkphi.sum(2))
        dnum = _mm(dqphi, Hc) + _mm(qphi, dHc)
        dden = _mm(dqphi, zc[..., None])[..., 0] + _mm(qphi, dzc[..., None])[..., 0]
        do = (dnum - o * dden[..., None]) / den[..., None]
    return o, do, Hc, zc, den


def _rows(x, B, H, L):
    return x.reshape(B, H, -1, x.shape[-1])[:, :, :L]


def _forward(q, k, v, a, lut, L, int8, trunc=False, qrows=E, p8=False, tan=None, signed=True):
    """The op on (B, H, L, 64) values -> (o, do, saved).  a: (H, nb) per 64-row block."""
    B, H = q.shape[:2]
    nb = -(-L // E)
    qt, kt, vt = (_tiles(t.double(), nb) for t in (q, k, v))
    one = torch.ones(B * H, nb, E, device=q.device, dtype=torch.float64)
    tant = None
    if tan is not None:
        tant = (qt, kt, *(_tiles(t.double(), nb) for t in tan))
    if int8:
        (q8, qs), (k8, ks) = _quant(q, nb, qrows, trunc), _quant(k, nb, E, trunc)
        v8, vs = _quant(v, nb, E, trunc) if p8 else (vt, None)
        o_s, do_s, lse = _sparse(q8, qs, k8, ks, v8, lut, L, tant, p8, vs)
    else:
        o_s, do_s, lse = _sparse(qt, one, kt, one, vt, lut, L, tant)
    keep = _unselected(lut, nb)
    o_l, do_l, Hc, zc, den = _linear(qt, kt, vt, keep, L, tant, signed)
    ar = a.double().expand(B, H, nb).reshape(B * H, nb, 1, 1)
    o = ar * o_s + (1 - ar) * o_l
    do = None if tan is None else ar * do_s + (1 - ar) * do_l
    return o, do, (qt, kt, vt, o_s, o_l, lse, den, Hc, zc, keep, ar)


def _backward(saved, lut, do, B, H, L):
    """Straight-through backward: the sparse branch re-differentiated at the
    unquantised q, k, v with the forward's lse."""
    qt, kt, vt, o_s, o_l, lse, den, Hc, zc, keep, a = saved
    G, nb = qt.shape[:2]
    dot = _tiles(do.double(), nb)
    do_s, do_l = a * dot, (1 - a) * dot
    seg = (dot * (o_s - o_l)).sum((2, 3)).reshape(B, H, nb).sum(0)
    delta = (o_s * do_s).sum(-1)
    valid = (torch.arange(nb * E, device=qt.device) < L).reshape(1, nb, E).expand(G, nb, E)
    dq, dk, dv = torch.zeros_like(qt), torch.zeros_like(kt), torch.zeros_like(vt)
    rowv = valid[..., None].double()
    for j in range(lut.shape[-1]):
        kj, vj = _col(kt, lut, j), _col(vt, lut, j)
        x = _mm(qt, kj.transpose(-1, -2).contiguous()) * (E ** -0.5 * LOG2E) - lse[..., None]
        p = torch.exp2(torch.clamp(x, max=4.0))
        p = p * _col(valid, lut, j)[:, :, None, :] * rowv
        ds = p * (_mm(do_s, vj.transpose(-1, -2).contiguous()) - delta[..., None]) * E ** -0.5
        dq += _mm(ds, kj)
        ix = lut[..., j, None, None].expand(G, nb, E, E)
        dk.scatter_add_(1, ix, _mm(ds.transpose(-1, -2).contiguous(), qt))
        dv.scatter_add_(1, ix, _mm(p.transpose(-1, -2).contiguous(), do_s))
    qphi, kphi = _phi(qt)[0], _phi(kt)[0]
    g = do_l / den[..., None] * rowv
    s = (do_l * o_l).sum(-1) / den * rowv[..., 0]
    dqphi = _mm(g, Hc.transpose(-1, -2).contiguous()) - s[..., None] * zc[:, :, None, :]
    qT = qphi.transpose(-1, -2).contiguous()
    back = lambda st: _mm(keep.transpose(-1, -2).contiguous(), st.reshape(G, nb, -1)).reshape(st.shape)
    dh, dz = back(_mm(qT, g)), -back(_mm(qT, s[..., None])[..., 0])
    dkphi = _mm(vt, dh.transpose(-1, -2).contiguous()) + dz[:, :, None, :]
    dv += _mm(kphi, dh)
    chain = lambda f, df: f * (df - (f * df).sum(-1, keepdim=True))
    dq, dk = dq + chain(qphi, dqphi), dk + chain(kphi, dkphi)
    ab = a.reshape(B, H, nb)[0]
    return [_rows(t, B, H, L) for t in (dq, dk, dv)], seg, ab * (1 - ab)


class _ExactCube(torch.autograd.Function):
    """The cube module's training op on (B, H, L, 64) float64 values."""

    @staticmethod
    def forward(ctx, q, k, v, logit, lut):
        B, H, L, _ = q.shape
        o, _, saved = _forward(q, k, v, torch.sigmoid(logit), lut, L, True, True, E, True)
        ctx.saved, ctx.lut, ctx.shape = saved, lut, (B, H, L)
        ctx.mark_non_differentiable(lse := saved[5].reshape(B, H, -1)[:, :, :L].amax((0, 2)))
        return _rows(o, B, H, L).clone(), lse

    @staticmethod
    def backward(ctx, do, _):
        (dq, dk, dv), seg, da = _backward(ctx.saved, ctx.lut, do, *ctx.shape)
        return dq, dk, dv, seg * da, None


def exact(c, seed):
    s = prepare(c, seed)
    L, Np, P, bq = _geometry(c)
    B, H, kind = c["B"], c["H"], c["kind"]
    nb, T = -(-L // E), _topk(c, Np)
    if kind == "block_train":
        return _exact_block(s)
    x = [t.detach() for t in s["x"]]
    if kind in ("jvp", "primal", "jvp1d"):
        proj = s.get("proj")
        lut = _lut(x[0], x[1], T, Np, bq, proj, nb)
        a = s["alpha"].repeat_interleave(bq // E, dim=1)[:, :nb]
        tan = None if kind == "primal" else x[3:]
        o, do, _ = _forward(*x[:3], a, lut, L, kind != "jvp1d", tan=tan)
        o = _rows(o, B, H, L)
        return o if tan is None else (o, _rows(do, B, H, L))
    impl = s["impl"]
    if kind in ("cube_train", "cube_guide"):
        x = [t.permute(0, 2, 1, 3) for t in x]
        if not c["tile_major"]:
            x = [t[:, :, impl.perm] for t in x]
        x = [t.half() for t in x[:3]] + x[3:]
        logit = impl.alpha_logit.detach()
        lut = _lut(x[0], x[1], T, Np, E, (impl.proj_q.detach(), impl.proj_k.detach()), nb)
        out = lambda t: (t if c["tile_major"] else t[:, :, impl.inv]).permute(0, 2, 1, 3)
        o, _, saved = _forward(*x[:3], torch.sigmoid(logit), lut, L, True, True, E, True)
        o = out(_rows(o, B, H, L))
        if kind == "cube_guide":
            return o
        grads, seg, da = _backward(saved, lut, x[3], B, H, L)
        lse = saved[5].reshape(B, H, -1)[:, :, :L].amax((0, 2))
        return [o, *(out(t) for t in grads), seg * da, lse]
    if kind == "sla2_train":
        x = [t.permute(0, 2, 1, 3) for t in x]
        logit = impl.sla2.alpha_logit.detach()
        a = torch.sigmoid(logit).repeat_interleave(bq // E, dim=1)[:, :nb]
        lut = _lut(x[0], x[1], T, Np, bq, None, nb)
        o, _, saved = _forward(*x[:3], a, lut, L, False)
        grads, seg, da = _backward(saved, lut, x[3], B, H, L)
        seg = F.pad(seg, (0, -nb % (bq // E))).reshape(H, -1, bq // E).sum(-1)
        a = torch.sigmoid(logit.double())
        out = lambda t: t.permute(0, 2, 1, 3)
        return [out(_rows(o, B, H, L)), *(out(t) for t in grads), seg * a * (1 - a)]
    a = torch.sigmoid(impl.alpha_logit.detach()).repeat_interleave(bq // E, dim=1)[:, :nb]
    lut = _lut(x[0], x[1], T, Np, bq, None, nb)
    o, _, _ = _forward(*x[:3], a, lut, L, c["int8"], False, bq, c["int8"])
    return _rows(o, B, H, L)


def _exact_block(s):
    """The DiT block in float64: pre-norm MLA attention with the cube op, SwiGLU MLP,
    vector-gated residuals; gradients of x and the parameters for s["dy"]."""
    c = s["case"]
    B, (L, Np, _, _) = c["B"], _geometry(c)
    H, nb = c["H"], -(-L // E)
    p = {n: t.detach().double().requires_grad_() for n, t in zip(s["names"], s["wrt"])}
    w = lambda n: p[n + ".weight"]
    x0 = s["x"].detach().double().requires_grad_()
    rms = lambda t, wt: t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + 1e-6) * wt
    cos, sin = (t.double()[None, :, None, :] for t in (s["cos"], s["sin"]))

    def rope(t):
        re, im = t[..., 0::2], t[..., 1::2]
        return torch.stack([re * cos - im * sin, re * sin + im * cos], -1).flatten(-2)

    n1 = rms(x0, w("norm1"))
    q = (rms(n1 @ w("attn.q_a_proj").T, w("attn.q_a_layernorm")) @ w("attn.q_b_proj").T).view(
        B, L, H, DN + DR)
    kva = n1 @ w("attn.kv_a_proj").T
    kv = (rms(kva[..., :DC], w("attn.kv_a_layernorm")) @ w("attn.kv_b_proj").T).view(B, L, H, DN + DV)
    q = torch.cat([rms(q[..., :DN], w("attn.q_norm")), rope(q[..., DN:])], -1)
    kr = rope(kva[..., DC:].unsqueeze(2)).expand(B, L, H, DR)
    k = torch.cat([rms(kv[..., :DN], w("attn.k_norm")), kr], -1)
    q, k, v = (t.permute(0, 2, 1, 3) for t in (q, k, kv[..., DN:]))
    impl = s["block"].attn.attn_impl
    lut = _lut(q.detach(), k.detach(), _topk(c, Np), Np, E,
               (impl.proj_q.detach(), impl.proj_k.detach()), nb)
    o, lse = _ExactCube.apply(q, k, v, p["attn.attn_impl.alpha_logit"], lut)
    o = o.permute(0, 2, 1, 3).reshape(B, L, H * DV) * torch.sigmoid(n1 @ w("attn.g_proj").T)
    x1 = x0 + (o @ w("attn.out_proj").T) * p["attn_scale"]
    n2 = rms(x1, w("norm2"))
    gate, up = n2 @ w("mlp.w1").T, n2 @ w("mlp.w3").T
    act = 4.0 * torch.tanh(gate / 4.0) * torch.sigmoid(gate) * 25.0 * torch.tanh(up / 25.0)
    y = x1 + (act @ w("mlp.w2").T) * p["mlp_scale"]
    grads = torch.autograd.grad(y, [x0, *(p[n] for n in s["names"])], s["dy"].double())
    return {"y": y.detach(), "dx": grads[0], **dict(zip(s["names"], grads[1:])),
            "logit_max_log2": lse}
