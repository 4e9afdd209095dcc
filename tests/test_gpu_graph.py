"""The fused cube fwd+JVP op (quantisation, routing, states, complement,
attention) captured in one HIP graph, stage by stage and as the whole calls that
users make: every replay, with eager calls of the op and synchronisations
between the replays, equals the eager result bit for bit (the op records no
memset and no host synchronisation, so a serving loop can capture it).  Config
1's shape (B=1, H=4, N=4,096)."""
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu


def test_cube_jvp_graph_replays_match_eager():
    from imfvideo_amd import ops
    print("[case] graph capture of the fused op, Config 1 shape", flush=True)
    sys.stdout.flush()
    g = torch.Generator().manual_seed(11)
    B, H, N, Np = 1, 4, 4096, 64
    dev = torch.device("cuda:0")
    q, k, v = (torch.randn(B, H, N, 64, generator=g).to(torch.bfloat16).to(dev) for _ in range(3))
    dq, dk, dv = ((0.1 * torch.randn(B, H, N, 64, generator=g)).to(torch.bfloat16).to(dev)
                  for _ in range(3))
    alpha = torch.full((H, Np), 0.9, device=dev)
    T = ops.topk_count(0.1, Np)

    def step():
        q8, qs, k8, ks, qpool, kpool_t, kb = ops.quant_pool_qk(q, k, Np, with_kb=True)
        lut = ops.route_topk(qpool, kpool_t, T, 0.125)
        st = ops.linear_states(k, v, Np, dk, dv, with_sums=False)
        comp = ops.complement(st, lut, Np, check_ids=False)
        return ops.fwd_jvp(q, q8, k8, qs, ks, st, comp, alpha, lut, Np, dq, kb=kb,
                           check_ids=False)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    torch.cuda.synchronize()
    for _ in range(4):
        graph.replay()
        torch.cuda.synchronize()
        eo, edo = step()
        torch.cuda.synchronize()
        assert torch.equal(out[0], eo) and torch.equal(out[1], edo)


def _check_replays(step, inputs):
    """step() captured once; four replays, each on refilled inputs and against an
    eager call on the same values."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    torch.cuda.synchronize()
    for _ in range(4):
        for x in inputs:
            x.copy_(torch.randn(x.shape, device="cuda") * 0.5)
        graph.replay()
        torch.cuda.synchronize()
        want = step()
        torch.cuda.synchronize()
        for a, b in zip(out, want):
            assert torch.equal(a, b)


@pytest.mark.parametrize("call", ["cube_jvp", "primal", "jvp_1d", "infer", "guide", "train"])
def test_whole_calls_graph_replays_match_eager(call):
    """The whole calls (native entries over one workspace) captured: the cube JVP and
    primal, the 1-D JVP, the INT8 1-D inference, the cube module without gradients
    and the training op forward and backward."""
    from imfvideo_amd import ops
    from imfvideo_amd.sla2_cube_qat import SLA2CubeQATAttentionImpl, sla2_cube_qat_jvp_fused
    from imfvideo_amd.sla2_mla_jvp import sla2_mla_jvp
    from imfvideo_amd.sla2_vendor import SLA2
    print("[case] graph capture of a whole call", call, flush=True)
    torch.manual_seed(12)
    H, L, Np, P = 4, 1042, 16, 18
    shape = (1, L, H, 64) if call == "guide" else (1, H, L, 64)
    x = [torch.randn(shape, device="cuda").to(torch.bfloat16) for _ in range(6)]
    alpha = torch.full((H, 17), 0.9, device="cuda")
    if call == "cube_jvp":
        step = lambda: sla2_cube_qat_jvp_fused(*x, alpha, 0.25, Np, 64, P)
    elif call == "primal":
        step = lambda: ops.cube_jvp(*x[:3], None, None, None, alpha, 0.25, Np, P)[:1]
    elif call == "jvp_1d":
        step = lambda: sla2_mla_jvp(*x, alpha[:, :9].contiguous(), 0.25, 128, 64)
    elif call == "infer":
        m = SLA2(64, topk=0.25, use_bf16=True).cuda().requires_grad_(False)
        step = lambda: [m(*x[:3])]
    elif call == "guide":
        m = SLA2CubeQATAttentionImpl(64, L, H, (4, 16, 16), topk=0.25).cuda().requires_grad_(False)
        step = lambda: [m(*x[:3])]
    else:
        q, k, v, do = x[:4]
        logit = torch.full((H, 17), 2.0, device="cuda")
        stats = torch.zeros(H, device="cuda")

        def step():
            qpool, kpool_t = ops.pool_qk(q, k, 64, Np)
            lut = ops.route_topk(qpool, kpool_t, 6, 0.125)
            o, saved = ops.train_op_fwd(q, k, v, logit, lut, Np, stats=stats)
            return [o, stats.clone(), *ops.train_op_bwd(q, k, v, do, saved, Np, 6)]

    with torch.no_grad():
        _check_replays(step, x)
