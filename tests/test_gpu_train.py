"""GPU parity of the training forward (semantics of _CubeQATFunction.forward,
models/sla2_cube_qat.py:703-752) against the CPU oracle's train_fwd (marked gpu).

Quantised operands and scales bit-exact; 16-bit outputs (o, o_s, o_l, qphi)
within max-abs 2e-2 and rel-L2 1e-2; lse (log2 domain) within 1e-3 absolute;
den and htot relative 1e-3.
"""
import numpy as np
import pytest
import torch

from oracle import sla2_oracle as O
from tests.helpers import make_inputs, max_abs, rel_l2
from tests.test_gpu_parity import TOL_MAX, TOL_REL, config_inputs, cuda, golden, say

pytestmark = pytest.mark.gpu


def expected_v8f(v8, L):
    """V8 (B,H,L,64) -> (B,H,Nb,4096) with [ct][lane=16g+r][s=4kb+i] = V8[16kb+4g+i][16ct+r]."""
    B, H = v8.shape[:2]
    nb = -(-L // 64)
    x = torch.zeros(B, H, nb * 64, 64, dtype=torch.int8)
    x[:, :, :L] = torch.as_tensor(v8)
    x = x.view(B, H, nb, 4, 4, 4, 4, 16)        # [kb][g][i][ct][r]
    return x.permute(0, 1, 2, 6, 4, 7, 3, 5).reshape(B, H, nb, 4096)


def check_quant(qz, f, L):
    for n in ("q", "k", "v"):
        x8, xs = O.quantize_blocks_trunc(f[n])
        assert np.array_equal(qz[n + "s"].cpu().numpy(), xs), n
        if n == "v":
            assert torch.equal(qz["v8f"].cpu(), expected_v8f(x8, L))
        else:
            assert np.array_equal(qz[n + "8"].cpu().numpy(), x8), n


def compare(out, ref, tag=""):
    for n in ("o", "o_s", "o_l", "qphi"):
        got = out[n].cpu().float()
        print(f"  {tag}{n} max {max_abs(got, ref[n]):.2e} rel {rel_l2(got, ref[n]):.2e}", flush=True)
        assert max_abs(got, ref[n]) < TOL_MAX and rel_l2(got, ref[n]) < TOL_REL, n
    lse = out["lse"].cpu()
    print(f"  {tag}lse max {max_abs(lse, ref['lse']):.2e}", flush=True)
    assert max_abs(lse, ref["lse"]) < 1e-3
    assert rel_l2(out["den"].cpu(), ref["den"]) < 1e-3
    assert rel_l2(out["htot"].cpu(), ref["htot"]) < 1e-3
    assert rel_l2(out["ztot"].cpu(), ref["ztot"]) < 1e-5


def run_train(ins, alpha, lut, Np):
    from imfvideo_amd import ops
    g = {n: cuda(ins[n]) for n in ("q", "k", "v")}
    out = ops.train_fwd(g["q"], g["k"], g["v"], cuda(alpha), cuda(torch.as_tensor(lut)), Np)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("name", ["ref_geom_bf16", "tiny_f16", "two_tails_bf16"])
def test_train_fwd_golden(name):
    say("train_fwd golden", name)
    z, dt, ins = golden(name)
    Np, P = int(z["Np"]), int(z["P"])
    alpha = torch.from_numpy(z["alpha"])
    out = run_train(ins, alpha, z["lut"], Np)
    f = {n: t.float() for n, t in ins.items()}
    check_quant(out, f, f["q"].shape[2])
    ref = O.train_fwd(f["q"], f["k"], f["v"], alpha, z["lut"], Np, P, t16=dt)
    compare(out, ref)


def test_train_fwd_config1_and_determinism():
    say("train_fwd config1 (1,4,4096)")
    ins, Np, P = config_inputs(1)
    f = {n: t.float() for n, t in ins.items()}
    lut, T, _, _ = O.route(f["q"], f["k"], 0.1, Np, P)
    g = torch.Generator().manual_seed(5)
    alpha = torch.rand(4, Np, generator=g) * 0.8 + 0.1
    out = run_train(ins, alpha, lut, Np)
    check_quant(out, f, 4096)
    compare(out, O.train_fwd(f["q"], f["k"], f["v"], alpha, lut, Np, P))
    again = run_train(ins, alpha, lut, Np)
    for n in ("o", "lse", "den"):
        assert torch.equal(out[n], again[n]), n


def test_train_fwd_ragged_fp16_and_alpha_endpoints():
    say("train_fwd ragged prefix fp16, alpha 0 / 1")
    B, H, Np, P = 2, 2, 5, 37
    L = Np * 64 + P
    q, k, v = make_inputs(31, B, H, L, dtype=torch.float16, tangent=False)
    ins = dict(q=q, k=k, v=v)
    f = {n: t.float() for n, t in ins.items()}
    lut, T, _, _ = O.route(f["q"], f["k"], 0.4, Np, P)
    for a in (0.0, 1.0, 0.3):
        alpha = torch.full((H, Np + 1), a)
        out = run_train(ins, alpha, lut, Np)
        ref = O.train_fwd(f["q"], f["k"], f["v"], alpha, lut, Np, P, t16=torch.float16)
        compare(out, ref, f"a={a} ")
        if a == 1.0:
            assert torch.equal(out["o"], out["o_s"])
        if a == 0.0:
            assert torch.equal(out["o"], out["o_l"])


@pytest.mark.parametrize("dt,T", [(torch.bfloat16, 3), (torch.float16, 2), (torch.bfloat16, 4)])
def test_train_fwd_score_form(dt, T):
    """Augmented LUTs of at most 4 columns run the score form of the linear branch
    (kernel_linear.py:260-272), wider ones the state form, as the reference
    selects (models/sla2_cube_qat.py:739).  Where the two forms round at
    different points, the GPU result is the nearer to the form it claims."""
    from imfvideo_amd import ops
    say("train_fwd score form", dt, "T", T)
    B, H, Np, P = 2, 2, 6, 29
    L = Np * 64 + P
    q, k, v = make_inputs(41 + T, B, H, L, dtype=dt, tangent=False)
    ins = dict(q=q, k=k, v=v)
    f = {n: t.float() for n, t in ins.items()}
    g = torch.Generator().manual_seed(T)
    lut = np.stack([np.stack([np.stack([torch.randperm(Np, generator=g)[:T].numpy()
                                        for _ in range(Np + 1)]) for _ in range(H)])
                    for _ in range(B)]).astype(np.int32)
    alpha = torch.rand(H, Np + 1, generator=g) * 0.8 + 0.1
    out = run_train(ins, alpha, lut, Np)
    score = T + 1 <= ops.SCORE_FORM_MAX_J
    ref = O.train_fwd(f["q"], f["k"], f["v"], alpha, lut, Np, P, t16=dt)
    compare(out, ref)
    other = O.train_fwd(f["q"], f["k"], f["v"], alpha, lut, Np, P, t16=dt, score_form=not score)
    got = out["o_l"].cpu().float()
    near, far = rel_l2(got, ref["o_l"]), rel_l2(got, other["o_l"])
    print(f"  o_l rel to its form {near:.2e}, to the other form {far:.2e}", flush=True)
    assert near < 0.5 * far


def test_train_fwd_1d_score_form():
    """1-D module forward (bq = 128, 16-bit scores) with a 2-column LUT: the score
    form of _complement_linear_attention (kernel_linear.py:357)."""
    from imfvideo_amd import ops
    say("train_fwd_1d score form bq=128 T=2")
    B, H, L, bq = 1, 2, 777, 128
    q, k, v = make_inputs(47, B, H, L, dtype=torch.float16, tangent=False)
    nb, mq = -(-L // 64), -(-L // bq)
    g = torch.Generator().manual_seed(3)
    lut = torch.stack([torch.randperm(nb, generator=g)[:2] for _ in range(B * H * mq)])
    lut = lut.view(B, H, mq, 2).int()
    alpha = torch.rand(H, mq, generator=g) * 0.8 + 0.1
    out = ops.train_fwd_1d(cuda(q), cuda(k), cuda(v), cuda(alpha), cuda(lut), bq)
    torch.cuda.synchronize()
    ref = O.train_fwd(q.float(), k.float(), v.float(), alpha, lut.numpy(), nb, 0,
                      t16=torch.float16, int8=False, bq=bq)
    for n in ("o", "o_s", "o_l", "qphi"):
        got = out[n].cpu().float()
        print(f"  {n} max {max_abs(got, ref[n]):.2e} rel {rel_l2(got, ref[n]):.2e}", flush=True)
        assert max_abs(got, ref[n]) < TOL_MAX and rel_l2(got, ref[n]) < TOL_REL, n
    assert rel_l2(out["den"].cpu(), ref["den"]) < 1e-3


def test_train_fwd_all_tiles_routed_and_zero_tiles():
    say("train_fwd T = Np, zero tiles")
    B, H, Np, P = 1, 2, 3, 10
    L = Np * 64 + P
    q, k, v = make_inputs(21, B, H, L, tangent=False)
    q[:, :, 64:128] = 0
    k[:, 1, :64] = 0
    ins = dict(q=q, k=k, v=v)
    lut = np.broadcast_to(np.arange(Np, dtype=np.int32), (B, H, 4, Np)).copy()
    alpha = torch.full((H, 4), 0.5)
    out = run_train(ins, alpha, lut, Np)
    f = {n: t.float() for n, t in ins.items()}
    check_quant(out, f, L)
    ref = O.train_fwd(f["q"], f["k"], f["v"], alpha, lut, Np, P)
    # the complement is empty: o_l = qphi . 0 / (+-eps) -> the 16-bit rounding of
    # (htot16 - htot) / eps; compare the sparse side and the finite output only
    for n in ("o_s", "qphi"):
        assert max_abs(out[n].cpu().float(), ref[n]) < TOL_MAX, n
    assert max_abs(out["lse"].cpu(), ref["lse"]) < 1e-3
    assert torch.isfinite(out["o"].float()).all()


def test_train_fwd_config3_full_size():
    say("train_fwd config3 full size (1,8,29952,64)")
    ins, Np, P = config_inputs(3)
    f = {n: t.float() for n, t in ins.items() if n in ("q", "k", "v")}
    lut, T, _, _ = O.route(f["q"], f["k"], 0.1, Np, P)
    alpha = torch.full((8, Np), 0.9)
    out = run_train(ins, alpha, lut, Np)
    assert torch.isfinite(out["o"].float()).all() and torch.isfinite(out["lse"]).all()
    check_quant(out, f, 29952)
    for h in range(8):  # every head
        sl = slice(h, h + 1)
        ref = O.train_fwd(f["q"][:, sl], f["k"][:, sl], f["v"][:, sl], alpha[sl], lut[:, sl],
                          Np, P)
        compare({n: (t[:, sl] if torch.is_tensor(t) and t.dim() >= 3 and t.shape[1] == 8 else t)
                 for n, t in out.items()}, ref, f"h{h} ")


# ---------------------------------------------------------------------------
# Backward (straight-through estimator) against O.train_bwd, fed the GPU
# forward's saved tensors.  16-bit gradients: rel-L2 1e-2, max-abs 2e-2 of
# max(1, max|ref|); d_alpha (fp32, atomics over b): rel-L2 1e-3.
# ---------------------------------------------------------------------------
def run_bwd(ins, alpha, lut, Np, P, seed=7, dscale=1.0):
    from imfvideo_amd import ops
    dt = ins["q"].dtype
    out = run_train(ins, alpha, lut, Np)
    g = torch.Generator().manual_seed(seed)
    do = (torch.randn(ins["q"].shape, generator=g) * dscale).to(dt)
    gq = {n: cuda(ins[n]) for n in ("q", "k", "v")}
    dq, dk, dv, da = ops.train_bwd(gq["q"], gq["k"], gq["v"], cuda(alpha), out, cuda(do))
    torch.cuda.synchronize()
    f = {n: ins[n].float() for n in ("q", "k", "v")}
    fwd = {n: out[n].cpu().float() for n in ("o_s", "o_l", "lse", "den", "qphi", "htot", "ztot")}
    ref = O.train_bwd(f["q"], f["k"], f["v"], alpha, lut, Np, P, fwd, do.float(), t16=dt)
    return dict(dq=dq.cpu().float(), dk=dk.cpu().float(), dv=dv.cpu().float(),
                d_alpha=da.cpu()), ref


def compare_bwd(got, ref, tag="", sl=slice(None)):
    for n in ("dq", "dk", "dv"):
        a, b = got[n][:, sl], ref[n]
        bound = TOL_MAX * max(1.0, b.abs().max().item())
        print(f"  {tag}{n} max {max_abs(a, b):.2e} (bound {bound:.2e}) rel {rel_l2(a, b):.2e}",
              flush=True)
        assert max_abs(a, b) < bound and rel_l2(a, b) < TOL_REL, n
    da = got["d_alpha"][sl]
    print(f"  {tag}d_alpha rel {rel_l2(da, ref['d_alpha']):.2e}", flush=True)
    assert rel_l2(da, ref["d_alpha"]) < 1e-3


@pytest.mark.parametrize("name", ["ref_geom_bf16", "tiny_f16", "two_tails_bf16"])
def test_train_bwd_golden(name):
    say("train_bwd golden", name)
    z, dt, ins = golden(name)
    Np, P = int(z["Np"]), int(z["P"])
    got, ref = run_bwd(ins, torch.from_numpy(z["alpha"]), z["lut"], Np, P)
    compare_bwd(got, ref)


def test_train_bwd_config1_ragged_fp16():
    say("train_bwd config1 and a ragged fp16 case")
    ins, Np, P = config_inputs(1)
    f = {n: t.float() for n, t in ins.items()}
    lut, T, _, _ = O.route(f["q"], f["k"], 0.1, Np, P)
    g = torch.Generator().manual_seed(5)
    alpha = torch.rand(4, Np, generator=g) * 0.8 + 0.1
    ins = {n: ins[n] for n in ("q", "k", "v")}
    got, ref = run_bwd(ins, alpha, lut, Np, P)
    compare_bwd(got, ref, "c1 ")
    B, H, Np, P = 2, 2, 5, 37
    L = Np * 64 + P
    q, k, v = make_inputs(31, B, H, L, dtype=torch.float16, tangent=False)
    ins = dict(q=q, k=k, v=v)
    f = {n: t.float() for n, t in ins.items()}
    lut, T, _, _ = O.route(f["q"], f["k"], 0.4, Np, P)
    alpha = torch.full((H, Np + 1), 0.3)
    got, ref = run_bwd(ins, alpha, lut, Np, P, dscale=0.5)
    compare_bwd(got, ref, "ragged ")


def test_train_bwd_config3_full_size():
    say("train_bwd config3 full size (1,8,29952,64)")
    ins, Np, P = config_inputs(3)
    ins = {n: ins[n] for n in ("q", "k", "v")}
    f = {n: t.float() for n, t in ins.items()}
    lut, T, _, _ = O.route(f["q"], f["k"], 0.1, Np, P)
    alpha = torch.full((8, Np), 0.9)
    from imfvideo_amd import ops
    out = run_train(ins, alpha, lut, Np)
    g = torch.Generator().manual_seed(7)
    do = torch.randn(ins["q"].shape, generator=g).to(torch.bfloat16)
    gq = {n: cuda(ins[n]) for n in ("q", "k", "v")}
    dq, dk, dv, da = ops.train_bwd(gq["q"], gq["k"], gq["v"], cuda(alpha), out, cuda(do))
    torch.cuda.synchronize()
    got = dict(dq=dq.cpu().float(), dk=dk.cpu().float(), dv=dv.cpu().float(), d_alpha=da.cpu())
    for n in ("dq", "dk", "dv"):
        assert torch.isfinite(got[n]).all(), n
    for h in range(8):  # every head
        sl = slice(h, h + 1)
        fwd = {n: out[n][:, sl].cpu().float() for n in ("o_s", "o_l", "lse", "den", "qphi", "htot", "ztot")}
        ref = O.train_bwd(f["q"][:, sl], f["k"][:, sl], f["v"][:, sl], alpha[sl], lut[:, sl], Np, P,
                          fwd, do[:, sl].float())
        compare_bwd(got, ref, f"h{h} ", sl)


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_bwd_prep_gradient_split_rounds_as_the_reference(dt):
    """do_s = (do * a).to(16-bit) as the reference's split kernel rounds it: the
    fp32 product first, then the 16-bit value.  A fused multiply-convert rounds
    once and differs wherever the fp32 product lands on a 16-bit rounding
    midpoint, which 16-bit do values times one fixed a hit for a few percent of
    the entries (fp16 with a = 0.9: about 4 %).  Bit for bit against the CPU's
    fp32 product, through the C ABI on bwd_prep's own output."""
    from imfvideo_amd import _lib, ops
    say("bwd_prep gradient split rounding", dt)
    B, H, L, D = 1, 2, 256, 64
    nb = L // 64
    g = torch.Generator().manual_seed(11)
    do = torch.randn(B, H, L, D, generator=g).to(dt)
    alpha = torch.tensor([[0.9, 0.3, 0.7, 0.55], [0.123, 0.999, 0.5, 0.8]], dtype=torch.float32)
    o_s = torch.randn(B, H, L, D, generator=g).to(dt)
    o_l = torch.randn(B, H, L, D, generator=g).to(dt)
    qphi = torch.softmax(torch.randn(B, H, L, D, generator=g), -1).to(dt)
    den = torch.rand(B, H, L, generator=g) + 1.0
    dv = lambda t: cuda(t).contiguous()
    gdo, gos, gol, gqp, gden, gal = (dv(t) for t in (do, o_s, o_l, qphi, den, alpha))
    dos, g16 = torch.empty_like(gdo), torch.empty_like(gdo)
    delta = torch.empty(B, H, L, device=gdo.device)
    srow = torch.empty_like(delta)
    seg = torch.zeros(H, nb, device=gdo.device)
    P = torch.empty(B, H, nb, D, D, device=gdo.device)
    Pz = torch.empty(B, H, nb, D, device=gdo.device)
    lib = _lib.load()
    _lib.check(lib.sla2h_bwd_prep(
        gdo.data_ptr(), gos.data_ptr(), gol.data_ptr(), gden.data_ptr(), gqp.data_ptr(),
        gal.data_ptr(), gal.stride(0), ops._dtype_code(gdo), B, H, L, D, 64, dos.data_ptr(),
        delta.data_ptr(), g16.data_ptr(), srow.data_ptr(), seg.data_ptr(), P.data_ptr(),
        Pz.data_ptr(), ops._stream(gdo.device)), "sla2h_bwd_prep")
    torch.cuda.synchronize()
    a_rows = alpha[:, torch.arange(L) // 64].view(1, H, L, 1)
    ref = (do.float() * a_rows).to(dt)  # fp32 product, then 16-bit (RNE)
    got = dos.cpu()
    assert torch.equal(got.view(torch.int16), ref.view(torch.int16))
    if dt == torch.float16:
        # the data reaches the midpoint cases the check is about: one rounding of
        # the exact product (numpy's float64 -> float16) differs from ref there
        exact = torch.from_numpy((do.double() * a_rows.double()).numpy().astype(np.float16))
        assert (exact.view(torch.int16) != ref.view(torch.int16)).float().mean() > 0.005


# ---------------------------------------------------------------------------
# 1-D SLA2 JVP (sla2_mla_jvp): bit-exact routing, outputs against O.jvp_1d
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("L,bq,dt", [(512, 128, torch.float16), (583, 128, torch.float16),
                                      (640, 64, torch.bfloat16), (583, 256, torch.bfloat16)])
def test_sla2_mla_jvp_small(L, bq, dt):
    say("sla2_mla_jvp", L, bq, dt)
    from imfvideo_amd.sla2_mla_jvp import route_blocks, sla2_mla_jvp
    B, H = 2, 2
    g = torch.Generator().manual_seed(L + bq)
    x = [torch.randn(B, H, L, 64, generator=g).to(dt) for _ in range(3)]
    d = [(torch.randn(B, H, L, 64, generator=g) * 0.1).to(dt) for _ in range(3)]
    pq = torch.eye(64) + 0.05 * torch.randn(64, 64, generator=g)
    lut, T = route_blocks(cuda(x[0]), cuda(x[1]), 0.3, bq, 64, proj_q=cuda(pq))
    elut, eT = O.route_1d(x[0].float(), x[1].float(), 0.3, bq, proj_q=pq)
    assert T == eT and np.array_equal(lut.cpu().numpy(), elut)
    mq = -(-L // bq)
    alpha = torch.rand(H, mq, generator=g) * 0.8 + 0.1
    o, do = sla2_mla_jvp(*(cuda(t) for t in x + d), cuda(alpha), 0.3, bq, 64, lut=lut, T=T)
    eo, edo = O.jvp_1d(*(t.float() for t in x + d), alpha, elut, bq, t16=dt)
    o, do = o.cpu(), do.cpu()
    print(f"  o max {max_abs(o, eo):.2e} rel {rel_l2(o, eo):.2e}  do max {max_abs(do, edo):.2e} "
          f"rel {rel_l2(do, edo):.2e}", flush=True)
    assert max_abs(o, eo) < TOL_MAX and rel_l2(o, eo) < TOL_REL
    assert max_abs(do, edo) < TOL_MAX and rel_l2(do, edo) < TOL_REL


def test_sla2_mla_jvp_config4_shape():
    say("sla2_mla_jvp (1,8,29952,64) bq=128")
    from imfvideo_amd.sla2_mla_jvp import sla2_mla_jvp
    ins, Np, P = config_inputs(3)
    x = [ins[n].half() for n in ("q", "k", "v", "dq", "dk", "dv")]
    o, do = sla2_mla_jvp(*(cuda(t) for t in x), 0.9, 0.1, 128, 64)
    o, do = o.cpu(), do.cpu()
    assert torch.isfinite(o).all() and torch.isfinite(do).all()
    for h in range(8):  # every head
        sl = slice(h, h + 1)
        xs = [t[:, sl].float() for t in x]
        lut, T = O.route_1d(xs[0], xs[1], 0.1, 128)
        eo, edo = O.jvp_1d(*xs, torch.full((1, 234), 0.9), lut, 128)
        print(f"  h{h} o rel {rel_l2(o[:, sl], eo):.2e} do rel {rel_l2(do[:, sl], edo):.2e}", flush=True)
        assert max_abs(o[:, sl], eo) < TOL_MAX and rel_l2(o[:, sl], eo) < TOL_REL
        assert max_abs(do[:, sl], edo) < TOL_MAX and rel_l2(do[:, sl], edo) < TOL_REL


# ---------------------------------------------------------------------------
# 1-D SLA2 module (SLA2AttentionImpl: fp16, no INT8, bq = 128, bk = 64)
# ---------------------------------------------------------------------------
def _tm16(t):
    return t.permute(0, 2, 1, 3).half().float()


def test_sla2_attention_impl_forward_and_gradients():
    say("SLA2AttentionImpl forward + backward (b=2, L=583, H=2)")
    from imfvideo_amd.sla2_attention import SLA2AttentionImpl
    torch.manual_seed(2)
    L, H = 583, 2
    mod = SLA2AttentionImpl(64, L, H, topk=0.3).cuda()
    with torch.no_grad():
        mod.sla2.alpha_logit.add_(torch.linspace(-1, 1, mod.sla2.alpha_logit.numel(),
                                                 device="cuda").view_as(mod.sla2.alpha_logit))
    g = torch.Generator().manual_seed(13)
    x = [torch.randn(2, L, H, 64, generator=g) for _ in range(4)]
    with torch.no_grad():  # inference path (sparse_attention + complement_linear_states)
        out0 = mod(*(cuda(t) for t in x[:3])).cpu()
    xs = [cuda(t).requires_grad_() for t in x[:3]]
    out = mod(*xs)         # training path
    (out * cuda(x[3])).sum().backward()
    grads = [t.grad.cpu() for t in xs] + [mod.sla2.alpha_logit.grad.cpu()]
    qh, kh, vh, doh = (_tm16(t) for t in x)
    # the router pools the fp32 inputs as given (reference core.py:88)
    lut, T = O.route_1d(x[0].permute(0, 2, 1, 3), x[1].permute(0, 2, 1, 3), 0.3, 128)
    nb = -(-L // 64)
    a = torch.sigmoid(mod.sla2.alpha_logit.detach().cpu())
    fwd = O.train_fwd(qh, kh, vh, a, lut, nb, 0, t16=torch.float16, int8=False, bq=128)
    eo = fwd["o"].permute(0, 2, 1, 3)
    ot = out.detach().cpu()
    print(f"  o (training) max {max_abs(ot, eo):.2e} rel {rel_l2(ot, eo):.2e}", flush=True)
    assert max_abs(ot, eo) < TOL_MAX and rel_l2(ot, eo) < TOL_REL
    ei = O.infer_1d(qh, kh, vh, a, lut, 128, int8=False)["o"].permute(0, 2, 1, 3)
    print(f"  o (inference) max {max_abs(out0, ei):.2e} rel {rel_l2(out0, ei):.2e}", flush=True)
    assert max_abs(out0, ei) < TOL_MAX and rel_l2(out0, ei) < TOL_REL
    ref = O.train_bwd(qh, kh, vh, a, lut, nb, 0, fwd, doh, t16=torch.float16, bq=128,
                      variant="1d")
    for got, name in zip(grads[:3], ("dq", "dk", "dv")):
        want = ref[name].permute(0, 2, 1, 3)
        print(f"  {name} max {max_abs(got, want):.2e} rel {rel_l2(got, want):.2e}", flush=True)
        assert rel_l2(got, want) < TOL_REL and max_abs(got, want) < TOL_MAX * max(1, want.abs().max())
    print(f"  d_alpha rel {rel_l2(grads[3], ref['d_alpha']):.2e}", flush=True)
    assert rel_l2(grads[3], ref["d_alpha"]) < 1e-2


def test_sla2_train_1d_config_shape():
    say("1-D training forward + backward (1,8,29952,64) bq=128")
    from imfvideo_amd import ops
    ins, Np, P = config_inputs(3)
    x = {n: ins[n].half() for n in ("q", "k", "v")}
    g = {n: cuda(t) for n, t in x.items()}
    lut, T = ops.route_1d(g["q"], g["k"], 0.1, 128)
    alpha = torch.full((8, 234), 0.9)
    out = ops.train_fwd_1d(g["q"], g["k"], g["v"], cuda(alpha), lut, 128)
    gen = torch.Generator().manual_seed(17)
    do = torch.randn(1, 8, 29952, 64, generator=gen).half()
    dq, dk, dv, da = ops.train_bwd(g["q"], g["k"], g["v"], cuda(alpha), out, cuda(do), bq=128)
    torch.cuda.synchronize()
    lut = lut.cpu().numpy()
    for h in range(8):  # every head
        sl = slice(h, h + 1)
        f = {n: t[:, sl].float() for n, t in x.items()}
        elut, eT = O.route_1d(f["q"], f["k"], 0.1, 128)
        assert np.array_equal(lut[:, sl], elut)
        ref = O.train_fwd(f["q"], f["k"], f["v"], alpha[sl], elut, 468, 0, t16=torch.float16,
                          int8=False, bq=128)
        got = {n: out[n][:, sl].cpu().float() for n in ("o", "o_s", "o_l", "qphi")}
        for n in got:
            print(f"  h{h} {n} rel {rel_l2(got[n], ref[n]):.2e}", flush=True)
            assert max_abs(got[n], ref[n]) < TOL_MAX and rel_l2(got[n], ref[n]) < TOL_REL
        fwd = {n: out[n][:, sl].cpu().float() for n in ("o_s", "o_l", "lse", "den", "qphi",
                                                        "htot", "ztot")}
        rb = O.train_bwd(f["q"], f["k"], f["v"], alpha[sl], elut, 468, 0, fwd, do[:, sl].float(),
                         t16=torch.float16, bq=128, variant="1d")
        for t_, n in ((dq, "dq"), (dk, "dk"), (dv, "dv")):
            a_ = t_[:, sl].cpu().float()
            print(f"  h{h} {n} rel {rel_l2(a_, rb[n]):.2e}", flush=True)
            assert rel_l2(a_, rb[n]) < TOL_REL and max_abs(a_, rb[n]) < TOL_MAX * max(1, rb[n].abs().max())
        assert rel_l2(da[sl].cpu(), rb["d_alpha"]) < 1e-2


@pytest.mark.parametrize("H,nb,T", [(9, 3, 1), (2, 33, 4), (1, 97, 2), (3, 130, 12), (1, 64, 16),
                                    (1, 520, 3), (5, 513, 6)])
def test_state_sums_beside_the_complement(H, nb, T):
    """The whole call takes the sums of the states over the tiles from the
    complement GEMM (masks inside it or not, one and two groups of query blocks,
    zall for the score form; states before and, from 2,561 tiles, behind the sparse
    kernel), the stages from their own kernel, in the same fp32 order: outputs and gradients equal to the bit."""
    from imfvideo_amd import ops
    print("[case] state sums", H, nb, T, flush=True)
    g = torch.Generator().manual_seed(nb + T)
    L = nb * 64
    q, k, v, do = (torch.randn(1, H, L, 64, generator=g).half().cuda() for _ in range(4))
    lut = torch.stack([torch.randperm(nb, generator=g)[:T] for _ in range(H * nb)])
    lut = lut.view(1, H, nb, T).to(torch.int32).cuda()
    logit = torch.randn(H, nb, generator=g).cuda()
    o, saved = ops.train_op_fwd(q, k, v, logit, lut, nb)
    a = torch.sigmoid(logit)
    ref = ops.train_fwd(q, k, v, a, lut, nb)
    assert torch.equal(o, ref["o"])
    got = ops.train_op_bwd(q, k, v, do, saved, nb, T)
    want = ops.train_bwd(q, k, v, a, ref, do)
    assert all(torch.equal(x, y) for x, y in zip(got[:3], want[:3]))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,L,Np,bq,T", [(1, 1, 64, 1, 64, 1), (2, 3, 274, 4, 64, 2),
                                           (1, 2, 700, 8, 64, 5), (2, 2, 583, 10, 128, 3),
                                           (1, 3, 1000, 16, 256, 6), (1, 2, 640, 10, 64, 10),
                                           (2, 1, 700, 11, 64, 5)])
@pytest.mark.parametrize("int8", [True, False])
def test_native_calls_match_the_stages(dt, B, H, L, Np, bq, T, int8):
    """The whole calls (one native entry each) against the same stages called one by
    one: prefix tails of none, one and several blocks, score- and state-form
    linear branch, every query block length.  Same kernels on the same values,
    so outputs are equal to the bit; the alpha gradient sums the batches in
    another order (fp32), and lse's per-head maximum is exact."""
    from imfvideo_amd import ops
    print("[case] native calls", dt, B, H, L, Np, bq, T, int8, flush=True)
    g = torch.Generator().manual_seed(L + T)
    x = [torch.randn(B, H, L, 64, generator=g).to(dt).cuda() for _ in range(6)]
    q, k, v, do, dk, dv = x
    nb, mq = -(-L // 64), -(-L // bq)
    lut = torch.stack([torch.randperm(Np, generator=g)[:T] for _ in range(B * H * mq)])
    lut = lut.view(B, H, mq, T).to(torch.int32).cuda()
    logit = torch.randn(H, mq, generator=g).cuda()
    a = torch.sigmoid(logit)
    stats = torch.zeros(H, device="cuda")
    o, saved = ops.train_op_fwd(q, k, v, logit, lut, Np, bq, int8, stats)
    if Np <= L // 64 and bq == 64:
        ref = ops.train_fwd(q, k, v, a, lut, Np, int8=int8)
    else:  # 1-D: every block routable, the last one possibly partial
        ref = ops.train_fwd_1d(q, k, v, a, lut, bq, int8=int8)
    assert torch.equal(o, ref["o"])
    assert torch.equal(stats, ref["lse"].amax(dim=(0, 2)))
    got = ops.train_op_bwd(q, k, v, do, saved, Np, T, bq)
    want = ops.train_bwd(q, k, v, a, ref, do, bq=bq)
    for n, gg, ww in zip(("dq", "dk", "dv"), got, want):
        assert torch.equal(gg, ww), n
    assert (got[3] - want[3]).abs().max() <= 1e-5 * want[3].abs().max()
    again = ops.train_op_bwd(q, k, v, do, saved, Np, T, bq)
    assert all(torch.equal(p, r) for p, r in zip(got, again))
    if Np == nb:
        f1 = ops.jvp_1d(q, k, v, do, dk, dv, a, lut, bq)
        f2 = ops.jvp_1d(q, k, v, do, dk, dv, a, lut, bq, return_aux=True)
        assert torch.equal(f1[0], f2[0]) and torch.equal(f1[1], f2[1])
        assert torch.equal(ops.sla2_infer(q, k, v, a, lut, bq, use_int8=int8),
                           ops.sla2_infer(q, k, v, a, lut, bq, use_int8=int8, return_parts=True)[0])
    if bq == 64 and Np <= L // 64:
        P = L - Np * 64
        for tan in ((do, dk, dv), (None, None, None)):
            for lut_ in (lut, None):
                f1 = ops.cube_jvp(q, k, v, *tan, a, T / Np, Np, P, lut=lut_)
                f2 = ops.cube_jvp(q, k, v, *tan, a, T / Np, Np, P, lut=lut_, return_aux=True)
                assert torch.equal(f1[0], f2[0])
                assert (f1[1] is None) == (tan[0] is None)
                assert f1[1] is None or torch.equal(f1[1], f2[1])


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,L,H,Np", [(1, 64, 1, 1), (2, 274, 3, 4), (1, 1000, 2, 15), (1, 577, 5, 8)])
@pytest.mark.parametrize("order", ["permuted", "tile_major"])
def test_train_in_matches_the_separate_passes(dt, B, L, H, Np, order):
    """The one-pass operands (fp16 rows, truncating INT8 values and scales, pooled
    and projected tiles) against rows_in, quant_train and pool_qk: equal to the
    bit, with a permutation and without, ragged and prefix blocks, zeros and
    values up to the fp16 maximum."""
    from imfvideo_amd import ops
    print("[case] train_in", dt, B, L, H, Np, order, flush=True)
    g = torch.Generator().manual_seed(L)
    xs = [(torch.randn(B, L, H, 64, generator=g) * s).to(dt) for s in (1.0, 50.0, 0.01)]
    xs[0][:, :64] = 0
    xs[1][0, -1, 0, 3] = 65504.0
    xs = [x.cuda() for x in xs]
    idx = torch.randperm(L, generator=g).cuda() if order == "permuted" else None
    pq, pk = (torch.randn(64, 64, generator=g).cuda() for _ in range(2))
    rows, ws, qpool, kpool_t = ops.train_in(xs, idx, Np, pq, pk)
    want = ops.rows_in(xs, idx)
    for a, b in zip(rows, want):
        assert torch.equal(a, b)
    qz = ops.quant_train(*want)
    off = 0
    for name in ("q8", "k8", "v8f", "qs", "ks", "vs"):
        t = qz[name]
        n = t.numel() * t.element_size()
        assert torch.equal(ws[off:off + n].view(t.dtype).view(t.shape), t), name
        off += -(-n // 256) * 256
    wq, wk = ops.pool_qk(want[0], want[1], 64, Np, pq, pk)
    assert torch.equal(qpool, wq) and torch.equal(kpool_t, wk)
    if order == "tile_major":
        views = [x.permute(0, 2, 1, 3) for x in want]
        none, ws2, qp2, kp2 = ops.train_in(views, None, Np, pq, pk, rows=False)
        # (the alignment gaps between the buffers are not written)
        n = L * B * H * 64
        assert none is None and torch.equal(ws2[:n], ws[:n])
        assert torch.equal(qp2, qpool) and torch.equal(kp2, kpool_t)


@pytest.mark.parametrize("T,int8", [(1, True), (6, True), (1, False), (6, False)])
def test_lse_maxima_replace_the_buffer_as_a_whole(T, int8):
    """The caller's buffer of lse maxima only ever receives a finished call's values:
    a call that is refused half-way (a prefix tail over the sparse kernel's 1,024
    tiles, after the setup ran) leaves it as it was, a good one replaces it and
    counts as an in-place change."""
    from imfvideo_amd import ops
    print("[case] lse maxima", T, int8, flush=True)
    g = torch.Generator().manual_seed(T)
    H = 2
    stats = torch.full((H,), 123.0, device="cuda")
    q, k, v = (torch.randn(1, H, 64 * 1060, 64, generator=g).half().cuda() for _ in range(3))
    logit = torch.zeros(H, 1060, device="cuda")
    lut = torch.arange(T, dtype=torch.int32).expand(1, H, 1060, T).contiguous().cuda()
    with pytest.raises(RuntimeError):
        ops.train_op_fwd(q, k, v, logit, lut, T, 64, int8, stats)
    torch.cuda.synchronize()
    assert stats.tolist() == [123.0] * H
    n, nb = 64 * 12, 12
    q, k, v = (t[:, :, :n].contiguous() for t in (q, k, v))
    lut, logit, version = lut[:, :, :nb].contiguous(), logit[:, :nb], stats._version
    ops.train_op_fwd(q, k, v, logit, lut, nb, 64, int8, stats)
    ref = ops.train_fwd(q, k, v, torch.sigmoid(logit), lut, nb, int8=int8)
    assert torch.equal(stats, ref["lse"].amax(dim=(0, 2))) and stats._version > version


@pytest.mark.parametrize("pre_permuted", [False, True])
def test_no_gradients_for_the_forward_workspace(pre_permuted, monkeypatch):
    """The forward's workspace and pooled tiles take no gradient: autograd makes no
    zero-filled tensors of their sizes (hundreds of MB at full length) for the
    backward of the module's operands."""
    from imfvideo_amd import sla2_cube_qat as M
    print("[case] workspace gradients", pre_permuted, flush=True)
    seen, backward = [], M._TrainIn.backward

    def spy(ctx, *ds):
        seen.append([d is None for d in ds])
        return backward(ctx, *ds)

    monkeypatch.setattr(M._TrainIn, "backward", staticmethod(spy))
    mod = M.SLA2CubeQATAttentionImpl(64, 274, 2, (4, 8, 8), topk=0.5, pre_permuted=pre_permuted).cuda()
    xs = [torch.randn(1, 274, 2, 64, device="cuda").requires_grad_() for _ in range(3)]
    grads = torch.autograd.grad(mod(*xs).float().pow(2).sum(), xs)
    assert seen == [[False] * 3 + [True] * 3]
    assert all(g.abs().sum() > 0 for g in grads)
