"""GPU parity of every HIP op against the CPU oracle (float64 oracle, float32 kernels).

Tolerances: relative 2e-5 plus an absolute floor scaled by the magnitude of the
quantity (float32 accumulation over up to a few hundred terms).
"""

import math

import pytest
import torch

from oracle import ops as O
from tests.helpers import assert_close, random_csr_graph, unit_vectors

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _ops():
    from flashcart_amd.o3 import _ops
    return _ops


def _close(got, want, what, rel=2e-5):
    """float32 GPU result against a float64 reference, relative to the reference's largest entry."""
    want = want.detach().double().cpu()
    assert_close(got, want, rel, rel * max(float(want.abs().max()) if want.numel() else 0.0, 1e-30), what)


@pytest.mark.parametrize("l_max", [0, 1, 2, 3])
def test_irreps_fwd_bwd(l_max):
    ops = _ops()
    x64 = unit_vectors(1000, seed=l_max).float().double().requires_grad_(True)
    ref = O.irreps(x64, l_max)
    g = torch.randn_like(ref)
    if l_max == 0:  # the expansion is the constant 1
        ref_gx = torch.zeros_like(x64)
    else:
        (ref_gx,) = torch.autograd.grad(ref, x64, g)
    x = x64.detach().float().to(DEV).requires_grad_(True)
    out = ops.irreps_fwd(x, l_max)
    (gx,) = torch.autograd.grad(out, x, g.float().to(DEV))
    assert_close(out, ref, 1e-5, 1e-6, "irreps fwd")
    assert_close(gx, ref_gx, 1e-5, 1e-5, "irreps bwd")


@pytest.mark.parametrize("kind", ["cheb_cos", "cheb_aff", "bessel", "cutoff"])
def test_radial_fwd_bwd(kind):
    ops = _ops()
    from flashcart_amd import _lib
    torch.manual_seed(1)
    d64 = torch.empty(4096).uniform_(0.0, 6.0).double().requires_grad_(True)
    if kind == "cheb_cos":
        ref, args = O.chebyshev(d64, 8, 5.0, 0.0, "cosine"), (_lib.BASIS_CHEBYSHEV_COSINE, 8, 0.0, 5.0, 0)
    elif kind == "cheb_aff":
        ref, args = O.chebyshev(d64, 8, 5.0, 0.5, "affine"), (_lib.BASIS_CHEBYSHEV_AFFINE, 8, 0.5, 5.0, 0)
    elif kind == "bessel":
        ref, args = O.bessel(d64, 8, 5.0), (_lib.BASIS_BESSEL, 8, 0.0, 5.0, 0)
    else:
        ref, args = O.cutoff(d64, 5.0, 6), (_lib.BASIS_NONE, 1, 0.0, 5.0, 6)
    g = torch.randn_like(ref)
    (ref_gd,) = torch.autograd.grad(ref, d64, g)
    d = d64.detach().float().to(DEV).requires_grad_(True)
    feats, env = ops.radial_fwd(d, *args)
    out = env if kind == "cutoff" else feats
    (gd,) = torch.autograd.grad(out, d, g.float().to(DEV))
    assert_close(out, ref, 2e-5, 2e-5, f"{kind} fwd")
    assert_close(gd, ref_gd, 1e-4, 1e-4, f"{kind} bwd")


def _tp_case(l1, l2, lo, f1, f2, sym=False, shared=False, reduced=False, conv=True, seed=0,
             degrees=(0, 1, 5, 26), n=37):
    ops = _ops()
    torch.manual_seed(seed)
    C = max(f1, f2)
    from oracle.cartesian import enumerate_paths
    P = len(enumerate_paths(l1, l2, lo, sym))
    if conv:
        ei = random_csr_graph(n, degrees, seed=seed)
        E = ei.shape[1]
        in1 = torch.randn(n, (l1 + 1) ** 2 * f1, dtype=torch.float64)
        in2 = torch.randn(E, (l2 + 1) ** 2 * f2, dtype=torch.float64)
        items = E
    else:
        ei = None
        in1 = torch.randn(n, (l1 + 1) ** 2 * f1, dtype=torch.float64)
        in2 = in1.clone() if sym else torch.randn(n, (l2 + 1) ** 2 * f2, dtype=torch.float64)
        items = n
    w = torch.randn(P * C, dtype=torch.float64) if shared else torch.randn(items, P * C, dtype=torch.float64)
    leaves64 = [t.clone().requires_grad_(True) for t in (in1, in2, w)]
    a1, a2, aw = leaves64
    ref = O.tensor_product(a1, a1 if sym else a2, aw, ei[0] if conv else None, ei[1] if conv else None,
                           l1, l2, lo, f1, f2, sym, shared, reduced)
    g = torch.randn_like(ref)
    ref_grads = torch.autograd.grad(ref, [a1, a2, aw] if not sym else [a1, aw], g)
    leaves = [t.detach().float().to(DEV).requires_grad_(True) for t in (in1, in2, w)]
    b1, b2, bw = leaves
    meta = ops.tp_meta(l1, l2, lo, f1, f2, sym, reduced)
    out = ops.tp_fwd(b1, b1 if sym else b2, bw, ei[0].to(DEV) if conv else None, ei[1].to(DEV) if conv else None,
                     l1, l2, lo, f1, f2, sym, shared, *meta, reduced)
    grads = torch.autograd.grad(out, [b1, b2, bw] if not sym else [b1, bw], g.float().to(DEV))
    scale = float(ref.abs().max()) + 1.0
    assert_close(out, ref, 2e-5, 2e-5 * scale, "tp fwd")
    for k, (gg, rr) in enumerate(zip(grads, ref_grads)):
        s = float(rr.abs().max()) + 1.0
        assert_close(gg, rr, 2e-5, 2e-5 * s, f"tp grad {k}")


CONV_CASES = [
    (0, 3, 3, 16, 1), (2, 3, 3, 16, 1), (1, 2, 2, 8, 1), (2, 2, 2, 8, 1), (3, 3, 3, 4, 1), (0, 2, 2, 64, 1),
    (2, 3, 3, 128, 1), (1, 1, 2, 8, 8), (2, 1, 1, 1, 8),
    # 64 channels with at most 40 output rows: the backward in sender order
    (2, 2, 2, 32, 1), (2, 2, 2, 64, 1), (1, 2, 2, 64, 1), (2, 1, 2, 64, 1),
]


@pytest.mark.parametrize("case", CONV_CASES, ids=lambda c: "x".join(map(str, c)))
def test_tp_conv(case):
    _tp_case(*case, conv=True)


@pytest.mark.parametrize("case", [(2, 3, 3, 128, 1), (2, 2, 2, 64, 1), (1, 2, 2, 64, 1), (2, 2, 2, 32, 1)],
                         ids=lambda c: "x".join(map(str, c)))
def test_tp_conv_chunk_boundaries(case):
    """Receiver and sender edge counts around the backward kernels' 16-edge chunks and their
    paired edge loop (odd last edges, a last edge on a chunk's first slot, one to three chunks),
    for one edge group (128 channels) and several (32 and 64): the staged indices and the
    operand waits keep every edge's result."""
    _tp_case(*case, conv=True, seed=5, degrees=(1, 15, 16, 17, 31, 32, 33, 47), n=48)


@pytest.mark.parametrize("need", [(True, True, False), (True, False, True), (False, True, True)])
def test_tp_conv_bwd_gradient_subsets(need):
    """The interaction-layer backward asked for a subset of its gradients (the second derivative
    asks for (in1, in2) without the weights): the general kernel that then runs forms each requested
    gradient exactly as the specialised all-gradients kernel does, bit for bit."""
    ops = _ops()
    g = torch.Generator().manual_seed(7)
    l1, l2, lo, C = 2, 3, 3, 128
    ei = random_csr_graph(40, (3, 9, 17), seed=4)
    E = ei.shape[1]
    from oracle.cartesian import enumerate_paths
    P = len(enumerate_paths(l1, l2, lo, False))
    in1 = torch.randn(40, 9 * C, generator=g).to(DEV)
    in2 = torch.randn(E, 16, generator=g).to(DEV)
    w = torch.randn(E, P * C, generator=g).to(DEV)
    meta = ops.tp_meta(l1, l2, lo, C, 1, False, False)
    go = torch.randn(40, ops._tp_out_dim(l1, l2, lo, C, 1, False, False), generator=g).to(DEV)
    args = (go, in1, in2, w, ei[0].to(DEV), ei[1].to(DEV), l1, l2, lo, C, 1, False, False, *meta, False)
    full = ops.tp_bwd(*args, True, True, True)
    part = ops.tp_bwd(*args, *need)
    for k in range(3):
        if need[k]:
            assert torch.equal(part[k], full[k]), f"gradient {k}"
        else:
            assert part[k].numel() == 0


def test_tp_conv_reduced_shared():
    _tp_case(2, 2, 2, 8, 1, shared=True, reduced=True, conv=True, seed=3)


@pytest.mark.parametrize("f1", [64, 128])
def test_tp_conv_shared_weights_full_width(f1):
    """Shared weights at the interaction layer's channel counts: the per-edge-weight backward
    specialisation does not apply (it reads one weight row per edge)."""
    _tp_case(2, 3, 3, f1, 1, shared=True, conv=True, seed=5)


ROW_CASES = [
    dict(l1=3, l2=3, lo=3, f1=8, f2=8, shared=True), dict(l1=3, l2=3, lo=2, f1=8, f2=8, shared=True),
    dict(l1=3, l2=3, lo=0, f1=8, f2=8, shared=True), dict(l1=3, l2=0, lo=3, f1=8, f2=1, shared=True),
    dict(l1=3, l2=3, lo=0, f1=8, f2=8, sym=True, shared=True), dict(l1=2, l2=2, lo=0, f1=16, f2=16, sym=True,
                                                                   shared=True),
    dict(l1=2, l2=2, lo=2, f1=1, f2=8), dict(l1=2, l2=2, lo=2, f1=8, f2=8, reduced=True),
    dict(l1=3, l2=3, lo=3, f1=128, f2=128, shared=True),
]


@pytest.mark.parametrize("case", ROW_CASES, ids=lambda c: "-".join(f"{k}{v}" for k, v in c.items()))
def test_tp_rows(case):
    _tp_case(conv=False, n=300, **case)


@pytest.mark.parametrize("l1,l2,lo,comps1,shared", [(3, 3, 3, 9, True), (3, 3, 2, 16, True), (2, 2, 2, 4, False),
                                                    (3, 3, 0, 1, True)])
def test_tp_rows_accumulate(l1, l2, lo, comps1, shared):
    """fc_tp_bwd_rows_acc: input gradients of the node-wise product plus residual gradients
    (res1 over the leading comps1 components of in1, res2 over all of in2, accumulated in
    place), against the float64 oracle's vector-Jacobian product plus the residuals."""
    ops = _ops()
    torch.manual_seed(l1 + 3 * lo + comps1)
    n, C = 300, 32
    from oracle.cartesian import enumerate_paths
    P = len(enumerate_paths(l1, l2, lo, False))
    in1 = torch.randn(n, (l1 + 1) ** 2 * C, dtype=torch.float64, requires_grad=True)
    in2 = torch.randn(n, (l2 + 1) ** 2 * C, dtype=torch.float64, requires_grad=True)
    w = torch.randn(P * C, dtype=torch.float64) if shared else torch.randn(n, P * C, dtype=torch.float64)
    ref = O.tensor_product(in1, in2, w, None, None, l1, l2, lo, C, C, False, shared, False)
    g = torch.randn_like(ref)
    q1, q2 = torch.autograd.grad(ref, [in1, in2], g)
    r1, r2 = q1, q2
    res1 = torch.randn(n, comps1 * C, dtype=torch.float64)
    res2 = torch.randn(n, (l2 + 1) ** 2 * C, dtype=torch.float64)
    r1 = r1.clone()
    r1[:, : comps1 * C] += res1
    r2 = r2 + res2
    d = [t.detach().float().to(DEV) for t in (in1, in2, w, g, res1, res2)]
    res1_dev = d[4].clone()
    g1, g2 = ops.tp_bwd_rows_acc(d[3], d[0], d[1], d[2], l1, l2, lo, C, shared, res1=d[4], res2=d[5],
                                 inplace2=True)
    assert g2.data_ptr() == d[5].data_ptr(), "full-width residual must be accumulated in place"
    assert torch.equal(d[4], res1_dev), "res1 must not be modified"
    assert_close(g1, r1, 2e-5, 2e-5 * (float(r1.abs().max()) + 1.0), "rows acc grad in1")
    assert_close(g2, r2, 2e-5, 2e-5 * (float(r2.abs().max()) + 1.0), "rows acc grad in2")
    # no residuals: plain input gradients
    h1, h2 = ops.tp_bwd_rows_acc(d[3], d[0], d[1], d[2], l1, l2, lo, C, shared)
    assert_close(h1, q1, 2e-5, 2e-5 * (float(q1.abs().max()) + 1.0), "rows grad in1")
    assert_close(h2, q2, 2e-5, 2e-5 * (float(q2.abs().max()) + 1.0), "rows grad in2")


@pytest.mark.parametrize("cfg", [(0, 0, 16, 16, None), (2, 2, 32, 16, None), (3, 3, 128, 128, [3, 5, 5, 4]),
                                 (2, 3, 64, 64, None), (3, 1, 8, 24, [1, 2, 3, 1])])
def test_linear(cfg):
    ops = _ops()
    lin, lout, fin, fout, paths = cfg
    paths = paths or [1] * (lin + 1)
    torch.manual_seed(5)
    n = 333
    in_dim = sum((2 * l + 1) * fin * paths[l] for l in range(lin + 1))
    x64 = torch.randn(n, in_dim, dtype=torch.float64, requires_grad=True)
    ws64 = [torch.randn(fout, fin * paths[l], dtype=torch.float64, requires_grad=True)
            for l in range(min(lin, lout) + 1)]
    ref = O.linear(x64, ws64, lin, lout, fin, fout, paths)
    g = torch.randn_like(ref)
    ref_g = torch.autograd.grad(ref, [x64] + ws64, g)
    x = x64.detach().float().to(DEV).requires_grad_(True)
    ws = [w.detach().float().to(DEV).requires_grad_(True) for w in ws64]
    scale = [float(fin * paths[l]) ** -0.5 for l in range(min(lin, lout) + 1)]
    out = ops.linear_fwd(x, ws, lin, lout, fin, fout, paths, scale, 1.0)
    got_g = torch.autograd.grad(out, [x] + ws, g.float().to(DEV))
    assert_close(out, ref, 1e-5, 1e-4, "linear fwd")
    for k, (a, b) in enumerate(zip(got_g, ref_g)):
        assert_close(a, b, 1e-5, 1e-4 * (float(b.abs().max()) + 1), f"linear grad {k}")


@pytest.mark.parametrize("shape", [(1000, 8, 64, 1, True), (777, 64, 2176, 0, True), (500, 64, 1, 0, True),
                                   (300, 256, 64, 1, True),
                                   # no bias, K = 64: the wide-output kernel (full and partial row blocks,
                                   # and a width that is not a multiple of 64)
                                   (1000, 64, 512, 0, False), (777, 64, 2176, 0, False), (129, 64, 300, 0, False)])
def test_dense(shape):
    ops = _ops()
    n, k, m, act, with_bias = shape
    torch.manual_seed(7)
    x64 = torch.randn(n, k, dtype=torch.float64, requires_grad=True)
    w64 = torch.randn(m, k, dtype=torch.float64, requires_grad=True)
    b64 = torch.randn(m, dtype=torch.float64, requires_grad=True) if with_bias else None
    ref = O.dense(x64, w64, b64)
    if act:
        ref = O.silu(ref)
    g = torch.randn_like(ref)
    leaves64 = [x64, w64] + ([b64] if with_bias else [])
    ref_g = torch.autograd.grad(ref, leaves64, g)
    leaves = [t.detach().float().to(DEV).requires_grad_(True) for t in leaves64]
    out, _ = ops.dense_fwd(leaves[0], leaves[1], leaves[2] if with_bias else None, float(k) ** -0.5, act)
    got = torch.autograd.grad(out, leaves, g.float().to(DEV))
    assert_close(out, ref, 1e-5, 1e-4, "dense fwd")
    for i, (a, r) in enumerate(zip(got, ref_g)):
        assert_close(a, r, 1e-5, 1e-4 * (float(r.abs().max()) + 1), f"dense grad {i}")


@pytest.mark.parametrize("n,n_in,m", [(1000, 8, 512), (300, 8, 2176), (257, 40, 200), (128, 64, 256), (5, 8, 64)])
def test_radial_mlp_fused(n, n_in, m):
    """The one-pass radial MLP (8 -> 64 -> 64 -> m, rescaled SiLU) and its input gradient
    against the float64 layer-by-layer chain: partial row blocks, an output width that is
    not a multiple of 64, more inputs than one MFMA column block."""
    ops = _ops()
    gen = torch.Generator().manual_seed(n + m)
    x64 = torch.randn(n, n_in, generator=gen, dtype=torch.float64, requires_grad=True)
    w0 = torch.randn(64, n_in, generator=gen, dtype=torch.float64)
    w1 = torch.randn(64, 64, generator=gen, dtype=torch.float64)
    w2 = torch.randn(m, 64, generator=gen, dtype=torch.float64)
    ref = O.dense(O.silu(O.dense(O.silu(O.dense(x64, w0)), w1)), w2)
    g = torch.randn(ref.shape, generator=gen, dtype=torch.float64)
    (ref_gx,) = torch.autograd.grad(ref, x64, g)
    x = x64.detach().float().to(DEV)
    w0f, w1f, w2f = (t.float().to(DEV) for t in (w0, w1, w2))
    s0, s1, s2 = float(n_in) ** -0.5, 0.125, 0.125
    with torch.no_grad():
        out = ops.radial_mlp_fwd(x, w0f, s0, w1f, s1, w2f, s2)
        gh2 = ops.dense_bwd(g.float().to(DEV), x.new_empty(0), w2f, s2, 0)
        gx = ops.radial_mlp_bwd(gh2, x, w0f, s0, w1f, s1)
    assert_close(out, ref, 1e-5, 2e-5 * float(ref.abs().max()), "radial mlp fwd")
    assert_close(gx, ref_gx, 1e-5, 2e-5 * float(ref_gx.abs().max()), "radial mlp input grad")


@pytest.mark.parametrize("n,degrees", [(64, (3, 7, 12)), (300, (1, 90, 200))])
def test_edge_geometry_positions_grad(n, degrees):
    """Edge geometry forward (rows staged through LDS per 256 edges, a partial last block) and
    the position gradient's segmented sums (one wave per node; segments above 64 edges)."""
    ops = _ops()
    from flashcart_amd import _lib
    from flashcart_amd.o3._graph import build_graph
    torch.manual_seed(11)
    pos64 = (torch.rand(n, 3) * 8.0).double().requires_grad_(True)
    ei = random_csr_graph(n, degrees, seed=2)
    E = ei.shape[1]
    shift = torch.randint(-1, 2, (E, 3)).double() * 8.0
    v = pos64[ei[1]] - pos64[ei[0]] + shift
    d = v.norm(dim=-1)
    r = v / d.clamp_min(O.MIN_EDGE_LENGTH).unsqueeze(-1)
    attrs = O.irreps(r, 3)
    feats = O.chebyshev(d, 8, 5.0, 0.0, "cosine")
    env = O.cutoff(d, 5.0, 6)
    ga, gf, ge = torch.randn_like(attrs), torch.randn_like(feats), torch.randn_like(env)
    loss = (attrs * ga).sum() + (feats * gf).sum() + (env * ge).sum()
    (ref_gpos,) = torch.autograd.grad(loss, pos64)
    pos = pos64.detach().float().to(DEV).requires_grad_(True)
    g = build_graph(ei.to(DEV), n)
    a2, f2, e2 = ops.edge_geometry(pos, shift.float().to(DEV), g.idx_i, g.idx_j, None, g.rowptr, g.sender_perm,
                                   g.sender_ptr, 3, _lib.BASIS_CHEBYSHEV_COSINE, 8, 0.0, 5.0, 6)
    assert_close(a2, attrs, 1e-5, 1e-5, "edge attrs")
    assert_close(f2, feats, 1e-5, 5e-5, "edge feats")
    assert_close(e2, env, 1e-5, 1e-6, "edge env")
    loss2 = (a2 * ga.float().to(DEV)).sum() + (f2 * gf.float().to(DEV)).sum() + (e2 * ge.float().to(DEV)).sum()
    (gpos,) = torch.autograd.grad(loss2, pos)
    assert_close(gpos, ref_gpos, 1e-4, 1e-4 * (float(ref_gpos.abs().max()) + 1), "edge grad positions")


def test_segment_sum():
    ops = _ops()
    torch.manual_seed(3)
    counts = torch.tensor([0, 5, 1, 17, 0, 3])
    ptr = torch.cat([torch.zeros(1, dtype=torch.long), counts.cumsum(0)])
    index = torch.repeat_interleave(torch.arange(len(counts)), counts)
    src = torch.randn(int(counts.sum()), dtype=torch.float64)
    ref = O.scatter_sum(src, index, len(counts))
    out = ops.segment_sum(src.float().to(DEV), ptr.to(DEV), index.to(DEV))
    assert_close(out, ref, 1e-6, 1e-6, "segment sum")


@pytest.mark.parametrize("l_max,C", [(0, 128), (1, 16), (2, 128), (3, 128), (3, 40)])
def test_rms_norm(l_max, C):
    """Fused RMS norm (forward, input and gain gradients) against the oracle's
    RMSLayerNorm restatement in float64."""
    ops = _ops()
    from oracle.model import rms_norm as ref_norm
    torch.manual_seed(l_max * 7 + C)
    n = 300
    x64 = (torch.randn(n, (l_max + 1) ** 2 * C, dtype=torch.float64) * torch.rand(n, 1, dtype=torch.float64) * 3)
    x64.requires_grad_(True)
    g64 = [(1.0 + 0.3 * torch.randn(C, dtype=torch.float64)).requires_grad_(True) for _ in range(l_max + 1)]
    sd = {f"ln.weights.{l}": g64[l] for l in range(l_max + 1)}
    ref = ref_norm(sd, "ln", x64, l_max, C)
    go = torch.randn_like(ref)
    ref_g = torch.autograd.grad(ref, [x64] + g64, go)
    x = x64.detach().float().to(DEV).requires_grad_(True)
    w = torch.stack([g.detach() for g in g64]).float().to(DEV).requires_grad_(True)
    out, _ = ops.rms_norm(x, w, l_max, 1e-6)
    gx, gw = torch.autograd.grad(out, [x, w], go.float().to(DEV))
    assert_close(out, ref, 2e-5, 2e-5 * float(ref.abs().max()), "rms fwd")
    assert_close(gx, ref_g[0], 1e-4, 1e-4 * float(ref_g[0].abs().max()), "rms grad x")
    assert_close(gw, torch.stack(ref_g[1:]), 1e-4, 1e-4 * float(torch.stack(ref_g[1:]).abs().max()), "rms grad g")


@pytest.mark.parametrize("lin,lout", [(3, 3), (2, 3), (3, 1)])
def test_linear_residual(lin, lout):
    """linear_fwd / linear_bwd with a residual added in the GEMM epilogue (ranks the map
    does not produce take the residual's values); gradients pass through to the residual."""
    ops = _ops()
    torch.manual_seed(9)
    n, fin, fout = 211, 16, 16
    in_dim = (lin + 1) ** 2 * fin
    out_dim = (lout + 1) ** 2 * fout
    x64 = torch.randn(n, in_dim, dtype=torch.float64, requires_grad=True)
    r64 = torch.randn(n, out_dim, dtype=torch.float64, requires_grad=True)
    ws64 = [torch.randn(fout, fin, dtype=torch.float64) for _ in range(min(lin, lout) + 1)]
    ref = O.linear(x64, ws64, lin, lout, fin, fout) + r64
    g = torch.randn_like(ref)
    ref_g = torch.autograd.grad(ref, [x64, r64], g)
    x = x64.detach().float().to(DEV).requires_grad_(True)
    r = r64.detach().float().to(DEV).requires_grad_(True)
    ws = [w.float().to(DEV) for w in ws64]
    scale = [fin ** -0.5] * len(ws)
    out = ops.linear_fwd(x, ws, lin, lout, fin, fout, [1] * (lin + 1), scale, 1.0, r)
    got = torch.autograd.grad(out, [x, r], g.float().to(DEV))
    assert_close(out, ref, 1e-5, 1e-4, "linear+residual fwd")
    assert_close(got[0], ref_g[0], 1e-5, 1e-4 * (float(ref_g[0].abs().max()) + 1), "linear+residual grad x")
    # pass-through: exactly the float32 upstream gradient
    assert_close(got[1], g.float().double(), 0.0, 0.0, "linear+residual grad residual")
    # dgrad with an accumulated gradient: gx = go @ W * s + acc
    acc = torch.randn(n, in_dim, device=DEV)
    gx = ops.linear_bwd(g.float().to(DEV), ws, lin, lout, fin, fout, [1] * (lin + 1), scale, 1.0, acc)
    plain = ops.linear_bwd(g.float().to(DEV), ws, lin, lout, fin, fout, [1] * (lin + 1), scale, 1.0)
    assert_close(gx, plain.double() + acc.double(), 1e-6, 1e-5, "dgrad + residual")


@pytest.mark.parametrize("l_max,act", [(3, 1), (2, 0), (0, 1)])
def test_gate(l_max, act):
    """Fused rank-wise gate against the reference formula (rescaled sigmoid, index_select,
    product) in float64, with both gradients."""
    ops = _ops()
    torch.manual_seed(l_max + 10 * act)
    n, C = 257, 64
    v64 = torch.randn(n, (l_max + 1) ** 2 * C, dtype=torch.float64, requires_grad=True)
    p64 = torch.randn(n, (l_max + 1) * C, dtype=torch.float64, requires_grad=True)
    gates = 1.8462285453386054 * torch.sigmoid(p64) if act == 1 else p64
    rank = torch.cat([torch.full((2 * l + 1,), l) for l in range(l_max + 1)])
    ref = (v64.view(n, -1, C) * gates.view(n, l_max + 1, C)[:, rank]).view(n, -1)
    g = torch.randn_like(ref)
    ref_g = torch.autograd.grad(ref, [v64, p64], g)
    v = v64.detach().float().to(DEV).requires_grad_(True)
    p = p64.detach().float().to(DEV).requires_grad_(True)
    out = ops.gate(v, p, l_max, act)
    got = torch.autograd.grad(out, [v, p], g.float().to(DEV))
    assert_close(out, ref, 1e-5, 1e-6, "gate fwd")
    assert_close(got[0], ref_g[0], 1e-5, 1e-6, "gate grad values")
    assert_close(got[1], ref_g[1], 1e-5, 1e-5 * float(ref_g[1].abs().max()), "gate grad pre")


@pytest.mark.parametrize("lin,lout,fin,fout,paths,n", [
    (3, 3, 128, 128, [1, 1, 1, 1], 3000),   # several row splits per rank, 128 x 128 tiles
    (2, 2, 16, 8, [1, 3, 2], 77),           # one split, 64 x 64 tiles, partial tiles
    (3, 1, 6, 10, [1, 1, 1, 1], 150),       # widths not multiples of 4: scalar loads
    (1, 2, 64, 200, [2, 1], 1200),
])
def test_linear_wgrad(lin, lout, fin, fout, paths, n):
    """Split-K MFMA weight gradients of the equivariant map against float64 sums of
    grad_out_l^T x_l, one rank per block of (2l+1) rows per node."""
    ops = _ops()
    g = torch.Generator().manual_seed(n + fin)
    common = min(lin, lout)
    in_dim = sum((2 * l + 1) * fin * paths[l] for l in range(lin + 1))
    out_dim = sum((2 * l + 1) * fout for l in range(lout + 1))
    x = torch.randn(n, in_dim, generator=g, dtype=torch.float64)
    go = torch.randn(n, out_dim, generator=g, dtype=torch.float64)
    ws = [torch.randn(fout, fin * paths[l], generator=g).to(DEV) for l in range(common + 1)]
    scale = [0.5 + l for l in range(common + 1)]
    with torch.no_grad():
        got = ops.linear_wgrad(go.float().to(DEV), x.float().to(DEV), ws, lin, lout, fin, fout, paths, scale, 0.75,
                               [True] * (common + 1))
    io = oo = 0
    for l in range(common + 1):
        k, m = fin * paths[l], 2 * l + 1
        xl = x[:, io:io + m * k].reshape(n * m, k)
        gl = go[:, oo:oo + m * fout].reshape(n * m, fout)
        want = gl.t() @ xl * (0.75 * scale[l])
        assert_close(got[l], want, 0.0, 2e-5 * float(want.abs().max()), f"wgrad rank {l}")
        io += m * k
        oo += m * fout
    with torch.no_grad():  # a subset of ranks
        part = ops.linear_wgrad(go.float().to(DEV), x.float().to(DEV), ws, lin, lout, fin, fout, paths, scale, 0.75,
                                [l == common for l in range(common + 1)])
    assert all(p is None for p in part[:common])
    assert_close(part[common], got[common].double(), 0.0, 0.0, "subset of ranks")


@pytest.mark.parametrize("n,k,m,act,bias", [(20000, 64, 2176, 0, False), (5000, 64, 64, 1, True),
                                            (333, 8, 64, 1, True), (90, 30, 17, 0, True)])
def test_dense_wgrad(n, k, m, act, bias):
    """Dense weight (and bias) gradients with the SiLU derivative applied to grad_out
    inside the kernel, against float64."""
    ops = _ops()
    g = torch.Generator().manual_seed(n + m)
    x = torch.randn(n, k, generator=g, dtype=torch.float64)
    go = torch.randn(n, m, generator=g, dtype=torch.float64)
    pre = torch.randn(n, m, generator=g, dtype=torch.float64)
    with torch.no_grad():
        gw, gb = ops.dense_wgrad(go.float().to(DEV), pre.float().to(DEV), act, x.float().to(DEV), 0.125, True, bias)
    h = go
    if act:
        s = torch.sigmoid(pre)
        h = go * 1.6765324703310907 * s * (1 + pre * (1 - s))
    want = h.t() @ x * 0.125
    assert_close(gw, want, 0.0, 2e-5 * float(want.abs().max()), "dense wgrad")
    if bias:
        wb = h.sum(0)
        assert_close(gb, wb, 0.0, 2e-5 * float(wb.abs().max()), "dense bias grad")
    else:
        assert gb is None


@pytest.mark.parametrize("lin,lout,fin,fout,in_paths", [(3, 3, 16, 16, [3, 5, 5, 4]), (3, 1, 8, 12, None),
                                                        (1, 3, 8, 8, None), (2, 0, 4, 8, [2, 3, 1])])
def test_reference_linear_ops(lin, lout, fin, fout, in_paths):
    """torch.ops.flashcart.linear_fwd / linear_bwd / linear_dbwd called with the reference's
    arguments (metadata, scale tensor and lists of o3.LinearLayer, as its triton_linear passes
    them, src/flashcart/o3/_linear.py:860-897) against the oracle: outputs, both gradients of
    linear_bwd, and the second derivatives reached through the registered autograd chain."""
    from flashcart_amd import o3
    import flashcart_amd.o3._second_order  # noqa: F401

    torch.manual_seed(3)
    lay = o3.LinearLayer(lin, lout, fin, fout, in_paths=in_paths).to(DEV)
    n = 37
    x = torch.randn(n, lay.in_dim, device=DEV, dtype=torch.float32)
    ws = [w.detach().clone() for w in lay.weight]
    args = (lay.meta, lay.out_dim, False, "ieee", *lay.meta_lists, lay.scale)
    out = torch.ops.flashcart.linear_fwd(x, ws, *args)
    xd = x.double().cpu().requires_grad_()
    wd = [w.double().cpu().requires_grad_() for w in ws]
    ref = O.linear(xd, wd, lin, lout, fin, fout, in_paths)
    _close(out, ref, "linear_fwd")
    go = torch.randn(n, lay.out_dim, device=DEV)
    gx, gws = torch.ops.flashcart.linear_bwd(go, x, ws, True, True, False, "ieee", *lay.meta_lists, lay.scale)
    rgx, *rgw = torch.autograd.grad(ref, [xd] + wd, go.double().cpu(), create_graph=True)
    _close(gx, rgx, "linear_bwd grad_x")
    for l, (a, b) in enumerate(zip(gws, rgw)):
        _close(a, b, f"linear_bwd grad_weight[{l}]")
    # second order through the registered autograd (linear_fwd -> linear_bwd -> linear_dbwd)
    xa = x.clone().requires_grad_()
    wa = [w.clone().requires_grad_() for w in ws]
    goa = go.clone().requires_grad_()
    o = torch.ops.flashcart.linear_fwd(xa, wa, *args)
    g1 = torch.autograd.grad(o, [xa] + wa, goa, create_graph=True)
    cots = [torch.randn_like(t) for t in g1]
    s2 = sum((a * c).sum() for a, c in zip(g1, cots))
    got2 = torch.autograd.grad(s2, [goa, xa] + wa, allow_unused=True)
    god = go.double().cpu().requires_grad_()
    rg1 = torch.autograd.grad(O.linear(xd, wd, lin, lout, fin, fout, in_paths), [xd] + wd, god, create_graph=True)
    rs2 = sum((a * c.double().cpu()).sum() for a, c in zip(rg1, cots))
    want2 = torch.autograd.grad(rs2, [god, xd] + wd, allow_unused=True)
    for k, (a, b) in enumerate(zip(got2, want2)):
        b = torch.zeros_like(a).double().cpu() if b is None else b
        _close(torch.zeros_like(b) if a is None else a, b, f"linear_dbwd input {k}")
    with pytest.raises(ValueError, match="dot_input_precision"):
        torch.ops.flashcart.linear_fwd(x, ws, lay.meta, lay.out_dim, False, "bf16", *lay.meta_lists, lay.scale)


def test_irreps_dbwd_op():
    """torch.ops.flashcart.irreps_dbwd (the Eq. (1) expansion's second derivative on the GPU)
    against double autograd of the oracle's expansion, l_max 0..3."""
    from tests.helpers import unit_vectors
    import flashcart_amd.o3._second_order  # noqa: F401

    for l_max in range(4):
        u = unit_vectors(300, seed=l_max)
        g = torch.randn(300, (l_max + 1) ** 2, dtype=torch.float64)
        v = torch.randn(300, 3, dtype=torch.float64)
        d_g, d_x = torch.ops.flashcart.irreps_dbwd(g.float().to(DEV), u.float().to(DEV), v.float().to(DEV), l_max)
        if l_max == 0:  # the expansion is the constant 1: both derivatives vanish
            assert float(d_g.abs().max()) == 0.0 and float(d_x.abs().max()) == 0.0
            continue
        ud = u.clone().requires_grad_()
        gd = g.clone().requires_grad_()
        (gx,) = torch.autograd.grad(O.irreps(ud, l_max), ud, gd, create_graph=True)
        want_g, want_x = torch.autograd.grad((gx * v).sum(), [gd, ud], allow_unused=True)
        _close(d_g, want_g, f"irreps_dbwd d_grad_output l={l_max}")
        _close(d_x, torch.zeros_like(ud) if want_x is None else want_x, f"irreps_dbwd d_x l={l_max}")


def test_shift_vectors_kernel():
    """fc_shift_vectors against the tensor-op sums it replaces, bit for bit: one cell and several
    cells; the translation of -S is the exact negation of that of S; a structure index out of range
    gives NaN rows; a differentiated cell keeps the tensor ops (and its gradient)."""
    from flashcart_amd.o3 import _ops
    from flashcart_amd.utils.geometry import shift_vectors

    def torch_sums(cell, shifts, idx_i, batch):
        s = shifts.to(cell.dtype)
        c = cell[0].unsqueeze(0) if cell.shape[0] == 1 else cell[batch[idx_i]]
        return s[:, 0:1] * c[:, 0] + s[:, 1:2] * c[:, 1] + s[:, 2:3] * c[:, 2]

    g = torch.Generator().manual_seed(11)
    n_nodes, n_edges = 300, 5000
    shifts = torch.randint(-3, 4, (n_edges, 3), generator=g)
    idx_i = torch.randint(0, n_nodes, (n_edges,), generator=g)
    batch = torch.sort(torch.randint(0, 4, (n_nodes,), generator=g)).values
    for n_cells in (1, 4):
        cell = (torch.randn(n_cells, 3, 3, generator=g) * 4.0 + 7.0 * torch.eye(3)).to(DEV)
        args = (shifts.to(DEV), idx_i.to(DEV), batch.to(DEV))
        print(f"shift vectors: {n_cells} cells, {n_edges} edges", flush=True)
        got = _ops.shift_vectors(cell, args[0], args[1], args[2])
        assert torch.equal(got, torch_sums(cell, *args))
        assert torch.equal(shift_vectors(cell, args[0], args[1], args[2], antisymmetric=True), got)
        assert torch.equal(_ops.shift_vectors(cell, -args[0], args[1], args[2]), -got)
    bad = batch.clone()
    bad[int(idx_i[7])] = 9
    got = _ops.shift_vectors(cell, shifts.to(DEV), idx_i.to(DEV), bad.to(DEV))
    rows = (bad[idx_i] == 9).to(DEV)
    assert torch.isnan(got[rows]).all() and not torch.isnan(got[~rows]).any()
    assert _ops.shift_vectors(cell[:1], shifts[:0].to(DEV), None, None).shape == (0, 3)
    # a differentiated cell: tensor ops, with the cell gradient
    cg = cell.clone().requires_grad_(True)
    sv = shift_vectors(cg, shifts.to(DEV), idx_i.to(DEV), batch.to(DEV), antisymmetric=True)
    assert sv.grad_fn is not None and torch.equal(sv.detach(), torch_sums(cell, shifts.to(DEV), idx_i.to(DEV),
                                                                          batch.to(DEV)))


def _map_bound(x, w, k):
    """Largest error of a float32 map of K terms: every product to 2^-23 (the parts of the split that are
    left out, below 2^-24, and its own rounding) and K / 16 roundings of the running sum, each at most
    2^-24 of the sum of magnitudes, with a factor of two for the order inside a matrix instruction."""
    return (k / 16 + 8) * 2.0 ** -23 * (x.abs() @ w.abs().t())


@pytest.mark.parametrize("n,lin,lout,fin,fout,paths", [
    # little work: 16 x 16 blocks, K below, at and above the 16 k chunks and the waves' shares of them
    (1, 0, 0, 4, 4, [1]), (17, 2, 2, 12, 20, [1, 2, 1]), (33, 3, 1, 36, 33, [1, 1, 1, 1]),
    (5, 1, 3, 128, 128, [7, 3]), (64, 0, 0, 512, 16, [1]), (43, 1, 2, 68, 36, [1, 2]),
    # 64-column tiles
    (50001, 0, 0, 32, 4, [1]), (6001, 1, 1, 32, 33, [1, 2]), (2203, 2, 1, 64, 63, [1, 1, 2]),
    (8129, 0, 0, 96, 65, [1]), (2033, 3, 3, 32, 100, [5, 1, 2, 3]), (1128, 1, 2, 160, 128, [1, 1]),
    # enough tiles for 128-column tiles: two column tiles, the second and the last row tile partial
    (40001, 0, 0, 32, 200, [1]), (8201, 3, 3, 32, 132, [1, 2, 1, 1]),
    # the same in the input gradient (K = 96, 64): columns in two tiles, and in one that is partial
    (40001, 0, 0, 140, 96, [1]), (8201, 3, 3, 36, 64, [1, 2, 1, 3]),
    # ranks of different K on both sides of the line between the 16 x 16 blocks and the tiles
    (199, 3, 3, 64, 64, [5, 3, 1, 2]), (301, 3, 3, 64, 64, [5, 3, 1, 2])])
def test_linear_tiles(n, lin, lout, fin, fout, paths):
    """The linear maps' kernels at the edges of their tiles (rows, columns, K steps), forward with a residual and
    input gradient, against float64 with an element-wise bound."""
    ops = _ops()
    g = torch.Generator(device=DEV).manual_seed(n + fout)
    common = min(lin, lout)
    x = torch.randn(n, sum((2 * l + 1) * fin * paths[l] for l in range(lin + 1)), device=DEV, generator=g)
    go = torch.randn(n, (lout + 1) ** 2 * fout, device=DEV, generator=g)
    ws = [torch.randn(fout, fin * paths[l], device=DEV, generator=g) for l in range(common + 1)]
    scale = [0.25 * (l + 1) for l in range(common + 1)]
    with torch.no_grad():
        out = ops.linear_fwd(x, ws, lin, lout, fin, fout, paths, scale, 1.0, go)
        gx = ops.linear_bwd(go, ws, lin, lout, fin, fout, paths, scale, 1.0)
    io = oo = 0
    for l in range(max(lin, lout) + 1):
        m = 2 * l + 1
        k = fin * paths[l] if l <= lin else 0
        gl = go[:, oo:oo + m * fout].reshape(n * m, fout).double() if l <= lout else None
        if l <= common:
            xl, w = x[:, io:io + m * k].reshape(n * m, k).double(), ws[l].double()
            for got, want, bound in (
                    (out[:, oo:oo + m * fout].reshape(n * m, fout), gl + scale[l] * (xl @ w.t()),
                     scale[l] * _map_bound(xl, w, k) + 2.0 ** -22 * (gl.abs() + 1)),
                    (gx[:, io:io + m * k].reshape(n * m, k), scale[l] * (gl @ w),
                     scale[l] * _map_bound(gl, w.t(), fout))):
                err = (got.double() - want).abs()
                assert bool((err <= bound).all()), f"rank {l}: {float((err / bound).max()):.2f} of the bound"
        elif l <= lout:  # ranks the map does not produce: the residual
            assert torch.equal(out[:, oo:oo + m * fout], go[:, oo:oo + m * fout])
        io += m * k
        oo += m * fout if l <= lout else 0


@pytest.mark.parametrize("n,fout", [(70, 40), (20000, 40), (40000, 136)])
def test_linear_special_values(n, fout):
    """Infinities and NaN propagate through the linear maps as IEEE sums (also where a weight is zero), and
    operands at both ends of float32's range keep its precision."""
    ops = _ops()
    k = 64
    g = torch.Generator(device=DEV).manual_seed(3)
    x = torch.randn(n, k, device=DEV, generator=g)
    w = torch.randn(fout, k, device=DEV, generator=g)
    w[5, 7] = 0.0
    x[1, 7] = float("inf")
    x[33, 9] = float("nan")
    x[34, 3] = float("-inf")
    x[40] *= 1e-36
    x[41] = 0.0
    x[42] *= 1e36
    x[43, 0] = 3.4e38  # rounds to infinity in 16 bits
    w[6] *= 1e-30
    with torch.no_grad():
        out = ops.linear_fwd(x, [w], 0, 0, k, fout, [1], [1e-3], 1.0)
        gx = ops.linear_bwd(out, [w], 0, 0, k, fout, [1], [1.0], 1.0)
    for a, b, s, got in ((x, w.t(), 1e-3, out), (out, w, 1.0, gx)):
        want = s * (a.double() @ b.double())
        assert torch.equal(got.isnan(), want.isnan())
        finite = want.abs() / s < 3e38  # the unscaled sum overflows float32 past that
        assert torch.equal(got[want.isinf()], want[want.isinf()].float())
        rows = torch.isfinite(a).all(1)
        bound = s * _map_bound(a[rows].double(), b.t().double(), a.shape[1]) + 2.0 ** -126
        err = (got[rows].double() - want[rows]).abs()
        assert bool((err <= bound)[finite[rows]].all())
    assert bool((out[41] == 0).all())


@pytest.mark.parametrize("n,k,fout", [
    (20000, 64, 64), (20011, 72, 96),     # 64-column tiles, the second with a partial one
    (40000, 136, 160), (40065, 200, 32)])  # 128-column tiles
def test_linear_gradient_special_values(n, k, fout):
    """Infinities, NaN and operands at both ends of float32's range in the gradient that the map's input gradient
    contracts (rows of tiles, the last one too): IEEE sums, full precision elsewhere, also in the tiles that hold them."""
    ops = _ops()
    g = torch.Generator(device=DEV).manual_seed(k)
    go = torch.randn(n, fout, device=DEV, generator=g)
    w = torch.randn(fout, k, device=DEV, generator=g)
    w[7, 5] = 0.0
    w[9, k - 1] = float("inf")
    w[0, k - 1] = 0.0  # (3.4e38 below times a weight above 1 is infinite in float32 alone)
    w[11] *= 1e-30
    go[1, 7] = float("inf")
    go[33, 9] = float("nan")
    go[n - 1, 3] = float("-inf")
    go[n - 2, 9] = 0.0  # 0 x inf
    go[40] *= 1e-36
    go[41] = 0.0
    go[42] *= 1e30
    go[43, 0] = 3.4e38  # rounds to infinity in 16 bits
    with torch.no_grad():
        got = ops.linear_bwd(go, [w], 0, 0, k, fout, [1], [1e-3], 1.0)
    unscaled = go.double() @ w.double()
    assert torch.equal(got.isnan(), unscaled.isnan())
    assert torch.equal(got[unscaled.isinf()], unscaled[unscaled.isinf()].float())
    rows, cols = torch.isfinite(go).all(1), torch.isfinite(w).all(0)
    a, b = go[rows].double(), w[:, cols].double()
    err = (got[rows][:, cols].double() - 1e-3 * (a @ b)).abs()
    fits = (a.abs() @ b.abs()) < 3e38  # no partial sum overflows
    assert bool((err <= 1e-3 * _map_bound(a, b.t(), fout) + 2.0 ** -126)[fits].all()) and float(fits.double().mean()) > 0.99
    assert bool((got[41][cols] == 0).all())


def test_split_operands_bottom_of_range():
    """Operands in the last normal binades and subnormal ones keep all their bits in the kernels that split them: map,
    input gradient (of 64 and 128 columns), weight gradient and wide output, with the small operand on either side,
    against float64. The results are normal numbers."""
    ops = _ops()
    n = 40001
    g = torch.Generator(device=DEV).manual_seed(5)

    def small(rows, cols):  # rows of 2^-120 to 2^-146
        e = torch.arange(rows, device=DEV) % 27 + 120
        return (torch.randn(rows, cols, device=DEV, generator=g).double() * torch.exp2(-e.double())[:, None]).float()

    def large(rows, cols):
        return torch.randn(rows, cols, device=DEV, generator=g) * 2.0 ** 60

    def check(got, a, b, k, what):
        a, b = a.double(), b.double()
        assert bool(((got.double() - a @ b.t()).abs() <= _map_bound(a, b, k)).all()), what

    for left, right in ((small, large), (large, small)):
        for k, m in ((64, 64), (96, 160)):
            x, w, go = left(n, k), right(m, k), left(n, m)
            with torch.no_grad():
                check(ops.linear_fwd(x, [w], 0, 0, k, m, [1], [1.0], 1.0), x, w, k, (left.__name__, "map", k, m))
                check(ops.linear_bwd(go, [w], 0, 0, k, m, [1], [1.0], 1.0), go, w.t(), m, (left.__name__, "gradient", k, m))
        a, b = left(n, 64), right(n, 160)
        with torch.no_grad():
            check(ops.dense_wgrad(a, None, 0, b, 1.0, True, False)[0], a.t(), b.t(), n, (left.__name__, "weights"))
        x, w = left(130, 64), right(320, 64)
        with torch.no_grad():
            check(ops.dense_fwd(x, w, None, 1.0, 0)[0], x, w, 64, (left.__name__, "wide"))


@pytest.mark.parametrize("n", [1, 15, 33, 64, 65, 1025])
def test_tp_rows_shared_weight_gradient(n):
    """The gradient of weights shared by all rows: the column sum over the rows in one pass and in parts,
    two column tiles (352 columns), against float64. Each term is a sum of at most 25 products; the sum
    over n rows has at most n / 8 + 16 roundings a chain."""
    from flashcart_amd import o3
    C = 32
    g = torch.Generator(device=DEV).manual_seed(n)
    tp = o3.TensorProduct(2, 2, 2, C, C, shared_weights=True)
    a, b = (torch.randn(n, 9 * C, device=DEV, generator=g) for _ in range(2))
    w = torch.ones(tp.n_total_paths * C, device=DEV, requires_grad=True)
    out = tp(a, b, w)
    go = torch.randn(out.shape, device=DEV, generator=g)
    (gw,) = torch.autograd.grad(out, w, go)
    w64 = torch.ones(tp.n_total_paths * C, dtype=torch.float64, requires_grad=True)
    ref = O.tensor_product(a.double().cpu(), b.double().cpu(), w64, None, None, 2, 2, 2, C, C, False, True, False)
    (want,) = torch.autograd.grad(ref, w64, go.double().cpu())
    assert_close(gw, want, 0.0, (n / 8 + 41) * 2.0 ** -24 * 25 * n ** 0.5, "shared weight gradient")


@pytest.mark.parametrize("n,k,m,act", [(20001, 64, 64, 1), (9001, 256, 64, 1), (70, 20, 18, 1), (1, 64, 64, 1),
                                       # the wide output: columns in parts and whole, partial rows and chunks
                                       (1, 64, 256, 0), (129, 64, 2180, 0), (65665, 64, 260, 0)])
def test_dense_tiles(n, k, m, act):
    """Dense layers in each kernel's range, pre-activation, output and input gradient (with the SiLU derivative
    on the way in) against float64; a row that holds an infinity gives what IEEE sums give. The SiLU and its
    derivative change a value by at most twice its error; exp adds 2^-20 of the value."""
    ops = _ops()
    g = torch.Generator(device=DEV).manual_seed(n + m)
    x, w, go = (torch.randn(*s, device=DEV, generator=g) for s in ((n, k), (m, k), (n, m)))
    if n > 1:
        x[n - 1, 3] = float("inf")
    with torch.no_grad():
        out, pre = ops.dense_fwd(x, w, None, 0.125, act)
        gx = ops.dense_bwd(go, pre, w, 0.125, act)
    want_pre = 0.125 * (x.double() @ w.double().t())
    bound = 0.125 * _map_bound(x.double(), w.double(), k)
    rows = slice(0, max(1, n - 1))
    if act:
        z = want_pre.clone().requires_grad_(True)
        with torch.enable_grad():
            want = O.silu(z)
            (dz,) = torch.autograd.grad(want.sum(), z)
        assert bool(((pre.double() - want_pre).abs() <= bound)[rows].all())
        assert bool(((out.double() - want).abs() <= 2 * bound + 2.0 ** -20 * want.abs())[rows].all())
        a = go.double() * dz
        slack = 2 * go.double().abs() * bound + 2.0 ** -20 * go.double().abs()
    else:
        assert bool(((out.double() - want_pre).abs() <= bound)[rows].all())
        a, slack = go.double(), 0.0 * go.double()
    if n > 1:
        last = (pre if act else out)[n - 1]
        assert torch.equal(last.isnan(), want_pre[n - 1].isnan())
        assert torch.equal(last.isinf(), want_pre[n - 1].isinf())
    want_gx = 0.125 * (a @ w.double())
    gx_bound = 0.125 * _map_bound(a, w.double().t(), m) + 0.125 * (slack @ w.double().abs())
    assert bool(((gx.double() - want_gx).abs() <= gx_bound)[rows].all())


@pytest.mark.parametrize("n,m", [(1, 256), (129, 320), (128, 330)])
def test_wide_output_scaled_range(n, m):
    """The wide output layers where x W leaves float32's range and scale * x W does not (the weights are scaled
    before they are multiplied), against float64: dense layer and radial MLP. 1e38 is far enough from the limit that
    no partial sum of the scaled products overflows. The hidden layers' error, exp's included, is below 2^-18."""
    ops = _ops()
    g = torch.Generator(device=DEV).manual_seed(n)
    x, w = torch.randn(n, 64, device=DEV, generator=g) * 1e19, torch.randn(m, 64, device=DEV, generator=g) * 3e19
    scale = 2.0 ** -9 * 1.25
    with torch.no_grad():
        out, _ = ops.dense_fwd(x, w, None, scale, 0)
    want = scale * (x.double() @ w.double().t())
    assert float((want / scale).abs().max()) > 3.5e38 and float(want.abs().max()) < 1e38
    assert bool(((out.double() - want).abs() <= scale * _map_bound(x.double(), w.double(), 64)).all())

    x8, w0, w1 = (torch.randn(*s, device=DEV, generator=g) for s in ((n, 8), (64, 8), (64, 64)))
    w2 = torch.randn(m, 64, device=DEV, generator=g).clamp(-2.5, 2.5) * 1e38
    with torch.no_grad():
        out = ops.radial_mlp_fwd(x8, w0, 0.35, w1, 0.125, w2, scale)
    h2 = O.silu(0.125 * O.silu(0.35 * x8.double() @ w0.double().t()) @ w1.double().t())
    want = scale * (h2 @ w2.double().t())
    assert float((want / scale).abs().max()) > 3.5e38 and float(want.abs().max()) < 1e38
    bound = scale * (_map_bound(h2, w2.double(), 64) + 2.0 ** -18 * (h2.abs().amax() * w2.double().abs().sum(1)))
    assert bool(((out.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("n,m", [(1, 2176), (2041, 2176), (12033, 1088), (21761, 704), (30001, 160), (30001, 1088),
                                 (65536, 2176), (65537, 330)])
def test_radial_mlp_column_parts(n, m):
    """The radial MLP's output with its columns in one part and in several, as the numbers of row blocks and of
    columns have it, against float64. The hidden layers' error, exp's included, is below 2^-18."""
    ops = _ops()
    g = torch.Generator(device=DEV).manual_seed(n + m)
    x, w0, w1, w2 = (torch.randn(*s, device=DEV, generator=g) for s in ((n, 8), (64, 8), (64, 64), (m, 64)))
    with torch.no_grad():
        out = ops.radial_mlp_fwd(x, w0, 0.35, w1, 0.125, w2, 0.125)
    h2 = O.silu(0.125 * O.silu(0.35 * x.double() @ w0.double().t()) @ w1.double().t())
    w = w2.double()
    bound = 0.125 * (_map_bound(h2, w, 64) + 2.0 ** -18 * (h2.abs().amax() * w.abs().sum(1)))
    assert bool(((out.double() - 0.125 * (h2 @ w.t())).abs() <= bound).all())


@pytest.mark.parametrize("m", [(1 << 22) - 1, 1 << 22, (1 << 23) + 5])
def test_wide_output_of_millions_of_columns(m):
    """Rows of a wide output longer than 32-bit byte offsets within a row block reach (128 m 4 from 2^31 on): radial
    MLP and dense layer, two row blocks of which the second is partial, against float64. The hidden layers' error,
    exp's included, is below 2^-18."""
    ops = _ops()
    n = 130
    g = torch.Generator(device=DEV).manual_seed(m)
    x8, w0, w1 = (torch.randn(*s, device=DEV, generator=g) for s in ((n, 8), (64, 8), (64, 64)))
    w2 = torch.randn(m, 64, device=DEV, generator=g)
    h2 = O.silu(0.125 * O.silu(0.35 * x8.double() @ w0.double().t()) @ w1.double().t())
    with torch.no_grad():
        out = ops.radial_mlp_fwd(x8, w0, 0.35, w1, 0.125, w2, 0.125)
        dense, _ = ops.dense_fwd(h2.float(), w2, None, 0.125, 0)
    for c in range(0, m, 1 << 20):
        w = w2[c:c + (1 << 20)].double()
        want = 0.125 * (h2 @ w.t())
        bound = 0.125 * (_map_bound(h2, w, 64) + 2.0 ** -18 * (h2.abs().amax() * w.abs().sum(1)))
        for got in (out, dense):
            assert bool(((got[:, c:c + (1 << 20)].double() - want).abs() <= bound).all()), c


@pytest.mark.parametrize("pairs", [1, 37, 6001])
def test_dense_bwd_pairs_sizes(pairs):
    """The pair-summed input gradient with few pairs and with enough for its tiled kernel."""
    ops = _ops()
    k = 704
    g = torch.Generator(device=DEV).manual_seed(pairs)
    go = torch.randn(2 * pairs, k, device=DEV, generator=g)
    w = torch.randn(k, 64, device=DEV, generator=g)
    perm = torch.randperm(2 * pairs, device=DEV, generator=g).to(torch.int32)
    lo, hi = perm[:pairs].contiguous(), perm[pairs:].contiguous()
    with torch.no_grad():
        got = ops.dense_bwd_pairs(go, w, 0.5, lo, hi)
    a = go[lo.long()].double() + go[hi.long()].double()
    bound = 0.5 * _map_bound(go[lo.long()].abs().double() + go[hi.long()].abs().double(), w.double().t(), k)
    assert bool(((got.double() - 0.5 * (a @ w.double())).abs() <= bound).all())


@pytest.mark.parametrize("l1,l2,lo", [(2, 3, 3), (0, 3, 3)])
@pytest.mark.parametrize("degrees", [(9, 0, 41, 8), (300, 65, 1), (8,) * 40, (7,) * 40, (17, 16, 15) * 255])
def test_tp_conv_edge_groups_128(l1, l2, lo, degrees):
    """128-channel convolutions whose receivers are shared by four edge groups (two waves each): groups of
    unequal length, empty receivers, more edges than a wave stages indices of (64 a group), mean degrees around the 8
    where the groups begin and up to the 768 receivers where they end; all gradients, against float64."""
    C = 128
    n = len(degrees)
    ei = random_csr_graph(n, degrees, seed=n, allow_self=True)
    g = torch.Generator().manual_seed(n + l1)
    e = ei.shape[1]
    from oracle.cartesian import enumerate_paths
    P = len(enumerate_paths(l1, l2, lo, False))
    leaves64 = [torch.randn(*s, generator=g, dtype=torch.float64).requires_grad_(True)
                for s in ((n, (l1 + 1) ** 2 * C), (e, (l2 + 1) ** 2), (e, P * C))]
    ref = O.tensor_product(*leaves64, ei[0], ei[1], l1, l2, lo, C, 1)
    go = torch.randn(ref.shape, generator=g, dtype=torch.float64)
    want = torch.autograd.grad(ref, leaves64, go)
    from flashcart_amd import o3
    tp = o3.TensorProduct(l1, l2, lo, C, 1)
    leaves = [t.detach().float().to(DEV).requires_grad_(True) for t in leaves64]
    out = tp(*leaves, ei[0].to(DEV), ei[1].to(DEV))
    got = torch.autograd.grad(out, leaves, go.float().to(DEV))
    assert_close(out, ref, 2e-5, 2e-5 * (float(ref.abs().max()) + 1), "forward")
    for k, (a, b) in enumerate(zip(got, want)):
        assert_close(a, b, 2e-5, 2e-5 * (float(b.abs().max()) + 1), f"gradient {k}")


@pytest.mark.parametrize("l1,l2,lo", [(2, 3, 3), (2, 2, 2), (1, 1, 1)])
@pytest.mark.parametrize("n,degree", [(256, 8), (257, 8), (257, 16), (512, 31), (512, 32), (513, 32), (767, 8), (769, 8)])
def test_tp_conv_edge_group_limits_128(l1, l2, lo, n, degree):
    """Receivers and edges around the limits between one and four edge groups (products of which one, two or more
    workgroups fit a CU), against the same receivers among so many others that none is shared by groups; float32
    sums over `degree` edges in another order."""
    from flashcart_amd import o3
    C, more = 128, 800
    few = random_csr_graph(n, [degree], seed=n)
    both = torch.cat([few, torch.arange(n, n + more).expand(2, -1)], 1)
    tp = o3.TensorProduct(l1, l2, lo, C, 1)
    gen = torch.Generator(device=DEV).manual_seed(n + l1)

    def t(*shape):
        return torch.randn(*shape, device=DEV, generator=gen)

    e = both.shape[1]
    big = [t(n + more, (l1 + 1) ** 2 * C), t(e, (l2 + 1) ** 2), t(e, tp.n_total_paths * C)]
    rows = (n, few.shape[1], few.shape[1])
    go = None
    results = []
    for edges, leaves in ((both, big), (few, [a[:k] for a, k in zip(big, rows)])):
        leaves = [a.clone().requires_grad_(True) for a in leaves]
        out = tp(*leaves, edges[0].to(DEV), edges[1].to(DEV))
        go = t(*out.shape) if go is None else go
        grads = torch.autograd.grad(out, leaves, go[:out.shape[0]])
        results.append([out] + list(grads))
    for k, (want, got) in enumerate(zip(*results)):
        _close(got, want[:got.shape[0]], f"result {k}")


@pytest.mark.parametrize("n", [1, 7, 33, 257, 5003])
@pytest.mark.parametrize("k,m,act", [(3, 4, 0), (130, 65, 1), (64, 128, 0), (200, 64, 1)])
def test_wgrad_tiles(n, k, m, act):
    """Dense weight and bias gradients at row counts around the kernel's groups of 8, steps of 32 and parts of
    256, and column counts around its tiles, with an element-wise bound; then with an infinity and a NaN in
    the rows, which reach the sums they reach in IEEE arithmetic."""
    ops = _ops()
    g = torch.Generator(device=DEV).manual_seed(n + m)
    go, pre, x = (torch.randn(n, c, device=DEV, generator=g) for c in (m, m, k))
    a = go.double()
    if act:
        z = pre.double().requires_grad_(True)
        (dz,) = torch.autograd.grad(O.silu(z).sum(), z)
        a = a * dz
    slack = 2.0 ** -20 * a.abs() if act else 0.0 * a  # the derivative's exp
    with torch.no_grad():
        gw, gb = ops.dense_wgrad(go, pre if act else None, act, x, 0.5, True, True)
    bound = 0.5 * _map_bound(a.t(), x.double().t(), n) + 0.5 * (slack.t() @ x.double().abs())
    assert bool(((gw.double() - 0.5 * (a.t() @ x.double())).abs() <= bound).all())
    assert bool(((gb.double() - a.sum(0)).abs() <= (n / 8 + 8) * 2.0 ** -23 * a.abs().sum(0) + slack.sum(0)).all())
    go[n // 2, 0] = float("inf")
    x[n - 1, k - 1] = float("nan")
    with torch.no_grad():
        gw, _ = ops.dense_wgrad(go, pre if act else None, act, x, 0.5, True, False)
    a = go.double() * dz if act else go.double()
    want = 0.5 * (a.t() @ x.double())
    assert torch.equal(gw.isnan(), want.isnan()) and torch.equal(gw.isinf(), want.isinf())
    ok = want.isfinite()
    assert bool(((gw.double() - want).abs() <= bound)[ok].all())


@pytest.mark.parametrize("n,lin,lout,fin,fout,paths", [(1, 3, 3, 4, 4, [1] * 4), (37, 3, 2, 33, 65, [1, 2, 1, 1]),
                                                       (1001, 3, 3, 64, 128, [2, 1, 1, 1])])
def test_linear_wgrad_tiles(n, lin, lout, fin, fout, paths):
    """Rows in place in the packed features (components 1, 3, 5, 7 to a node) across the kernel's steps."""
    ops = _ops()
    g = torch.Generator(device=DEV).manual_seed(n)
    x = torch.randn(n, sum((2 * l + 1) * fin * paths[l] for l in range(lin + 1)), device=DEV, generator=g)
    go = torch.randn(n, (lout + 1) ** 2 * fout, device=DEV, generator=g)
    common = min(lin, lout)
    ws = [torch.empty(fout, fin * paths[l], device=DEV) for l in range(common + 1)]
    with torch.no_grad():
        got = ops.linear_wgrad(go, x, ws, lin, lout, fin, fout, paths, [1.0] * (common + 1), 1.0, [True] * (common + 1))
    io = oo = 0
    for l in range(common + 1):
        m, k = 2 * l + 1, fin * paths[l]
        a = go[:, oo:oo + m * fout].reshape(n * m, fout).double()
        b = x[:, io:io + m * k].reshape(n * m, k).double()
        assert bool(((got[l].double() - a.t() @ b).abs() <= _map_bound(a.t(), b.t(), n * m)).all()), f"rank {l}"
        io += m * k
        oo += m * fout


def _route_call(kind):
    """(operator, arguments) of one call with gradients through every differentiable input."""
    ops = _ops()
    gen = torch.Generator().manual_seed(11)

    def t(*shape):
        return torch.randn(*shape, generator=gen).to(DEV).requires_grad_(True)

    if kind == "conv":
        i, j = random_csr_graph(9, [4, 0, 3], seed=3)
        i, j = i.to(DEV).int(), j.to(DEV).int()
        n_paths = ops._n_paths(1, 1, 1, False)
        meta = ops.tp_meta(1, 1, 1, 8, 1, False, False)
        return ops.tp_fwd, (t(9, 32), t(i.numel(), 4), t(i.numel(), 8 * n_paths), i, j, 1, 1, 1, 8, 1, False, False, *meta)
    if kind == "dense":
        return ops.dense_fwd, (t(13, 8), t(16, 8), None, 0.3, 1)
    if kind == "norm":
        return ops.rms_norm, (t(7, 9 * 8), t(3, 8), 2, 1e-5)
    return ops.irreps_fwd, (unit_vectors(17, seed=2).float().to(DEV).requires_grad_(True), 2)


def _route_results(fn, args):
    """Outputs, gradients and second derivatives of a call, and the tensors it saves."""
    saved = []
    with torch.autograd.graph.saved_tensors_hooks(lambda s: saved.append(tuple(s.shape)) or s, lambda s: s):
        out = fn(*args)
    outs = [o for o in (out if isinstance(out, tuple) else (out,)) if o.requires_grad and o.numel()]
    leaves = [a for a in args if isinstance(a, torch.Tensor) and a.requires_grad]
    first = torch.autograd.grad(sum((o * o).sum() for o in outs), leaves, create_graph=True, allow_unused=True)
    second = torch.autograd.grad(sum((g * g).sum() for g in first if g is not None), leaves, allow_unused=True)
    return outs + [g for g in (*first, *second)], sorted(saved)


@pytest.mark.parametrize("kind", ["conv", "dense", "norm", "irreps"])
def test_operator_routes(kind):
    """A plain call and the registered operator: the same values, derivatives and saved tensors (bit for bit:
    the same kernels on the same inputs); vmap maps it, forward mode does the same and a tracer sees the operator."""
    from torch.fx.experimental.proxy_tensor import make_fx
    fn, args = _route_call(kind)
    assert fn._direct(args)
    got, saved = _route_results(fn, args)
    want, want_saved = _route_results(fn.op, args)
    assert saved == want_saved
    for k, (a, b) in enumerate(zip(got, want)):
        assert (a is None) == (b is None) and (a is None or torch.equal(a, b)), (kind, k)
    with torch.no_grad():
        a, b = fn(*args), fn.op(*args)
    a, b = (a, b) if isinstance(a, tuple) else ((a,), (b,))
    assert all(torch.equal(x, y) and not x.requires_grad for x, y in zip(a, b))

    mapped = torch.func.vmap(lambda x: fn(x, *args[1:]))(args[0].detach()[None])
    mapped = mapped if isinstance(mapped, tuple) else (mapped,)
    assert all(torch.equal(x, y[0]) for x, y in zip(a, mapped))

    def forward_mode(f):
        fwd = torch.autograd.forward_ad
        with fwd.dual_level():
            try:
                out = f(fwd.make_dual(args[0].detach(), torch.ones_like(args[0])), *args[1:])
                return fwd.unpack_dual(out[0] if isinstance(out, tuple) else out).tangent is None
            except RuntimeError as e:
                return str(e)

    assert forward_mode(fn) == forward_mode(fn.op)
    graph = make_fx(lambda x: fn(x, *args[1:]))(args[0].detach())
    assert any("flashcart" in str(n.target) for n in graph.graph.nodes)


def _operator_call(name):
    """Arguments of a small call of an operator, the differentiable ones leaves that require gradients (none for the
    operators without a formula of their own)."""
    ops = _ops()
    from flashcart_amd import _lib
    gen = torch.Generator().manual_seed(29)
    grads = getattr(ops, name).function is not None

    def t(*shape, low=None):
        v = torch.randn(*shape, generator=gen) if low is None else torch.rand(*shape, generator=gen) + low
        return v.to(DEV).requires_grad_(grads)

    i, j = (v.to(DEV).int() for v in random_csr_graph(9, [4, 0, 3], seed=3))
    e, radial = i.numel(), (_lib.BASIS_BESSEL, 8, 0.0, 5.0, 6)
    unit = unit_vectors(17, seed=2).float().to(DEV).requires_grad_(grads)
    meta = ops.tp_meta(1, 1, 1, 8, 1, False, False)
    conv = (t(9, 32), t(e, 4), t(e, 8 * meta[-1]), i, j, 1, 1, 1, 8, 1, False, False, *meta)
    maps = (t(12, 8), t(12, 8), None, None, None, 1, 1, 8, 12, [1, 1], [0.3, 0.2], 0.7)
    edges = (t(9, 3), t(e, 3), i, j, None, None, None, None, 2, *radial)
    mlp = (t(13, 8), t(64, 8), 0.3, t(64, 64), 0.2)
    return {
        "irreps_fwd": lambda: (unit, 2),
        "irreps_bwd": lambda: (t(17, 9), unit, 2),
        "irreps_dbwd": lambda: (t(17, 9), unit, t(17, 3), 2),
        "radial_fwd": lambda: (t(17, low=0.5), *radial),
        "radial_bwd": lambda: (t(17, low=0.5), t(17, 8), t(17), *radial),
        "edge_geometry": lambda: edges,
        "edge_geometry_bwd": lambda: (t(e, 9), t(e, 8), t(e), *edges, True),
        "tp_fwd": lambda: conv,
        "tp_bwd": lambda: (t(9, sum(meta[2])), *conv, False, True, True, True),
        "linear_fwd_op": lambda: (t(13, 32), *maps, t(13, 48)),
        "linear_bwd_op": lambda: (t(13, 48), *maps, t(13, 32)),
        "dense_fwd": lambda: (t(13, 8), t(16, 8), t(16), 0.3, 1),
        "dense_bwd": lambda: (t(13, 16), t(13, 16), t(16, 8), 0.3, 1),
        "radial_mlp_fwd": lambda: (*mlp, t(40, 64), 0.1),
        "radial_mlp_bwd": lambda: (t(13, 64), *mlp),
        "segment_sum": lambda: (t(13, 4), torch.tensor([0, 5, 5, 13], dtype=torch.int32, device=DEV),
                                torch.tensor([0] * 5 + [2] * 8, dtype=torch.int32, device=DEV)),
        "rms_norm": lambda: (t(7, 72), t(3, 8), 2, 1e-5),
        "rms_norm_bwd": lambda: (t(7, 72), t(7, 72), t(3, 8), t(7, low=0.5), 2),
        "gate": lambda: (t(7, 72), t(7, 24), 2, 1),
        "gate_bwd": lambda: (t(7, 72), t(7, 72), t(7, 24), 2, 1, True, True),
    }[name]()


def _operator_names():
    ops = _ops()
    return sorted(k for k, v in vars(ops).items() if isinstance(v, ops.Operator))


def _values_and_gradients(fn, args, leaves):
    """Outputs of a call and their gradients by ``leaves`` (a fixed cotangent)."""
    out = fn(*args)
    outs = [o for o in (out if isinstance(out, tuple) else (out,)) if o.numel()]
    diff = [o for o in outs if o.requires_grad]
    if not leaves:
        assert not diff
        return outs, []
    return outs, torch.autograd.grad(sum((o * (1.0 + o.detach())).sum() for o in diff), leaves, allow_unused=True)


@pytest.mark.parametrize("name", _operator_names())
def test_every_operator_route(name):
    """Every operator called plainly, through the registry, and with negated views for its floating-point arguments:
    the same values and gradients, bit for bit. The profiler sees the operator."""
    fn = getattr(_ops(), name)
    args = _operator_call(name)
    assert fn._direct(args)
    leaves = [a for a in args if isinstance(a, torch.Tensor) and a.requires_grad]
    got, grads = _values_and_gradients(fn, args, leaves)
    want, want_grads = _values_and_gradients(fn.op, args, leaves)
    assert len(got) == len(want) and all(torch.equal(a, b) for a, b in zip(got, want))
    assert all((a is None) == (b is None) and (a is None or torch.equal(a, b)) for a, b in zip(grads, want_grads))

    # the same values behind a negation: every floating-point argument, also a single element
    bases = [(-a.detach()).requires_grad_(a.requires_grad) if isinstance(a, torch.Tensor) and a.is_floating_point()
             else a for a in args]
    views = [torch._neg_view(b) if isinstance(b, torch.Tensor) and b.is_floating_point() else b for b in bases]
    neg, neg_grads = _values_and_gradients(
        fn, views, [b for b in bases if isinstance(b, torch.Tensor) and b.requires_grad])
    assert all(torch.equal(a, b) for a, b in zip(neg, want))
    assert all((a is None) == (b is None) and (a is None or torch.equal(a, -b)) for a, b in zip(neg_grads, want_grads))

    with torch.no_grad(), torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        fn(*args)
    assert any(ev.key.startswith("flashcart::") for ev in prof.key_averages())


@pytest.mark.parametrize("C", [32, 64, 128])
@pytest.mark.parametrize("l1,l2,lo", [(2, 3, 3), (0, 2, 2), (3, 3, 3)])
@pytest.mark.parametrize("degrees", [(1, 0, 2, 33, 66), (17, 16, 15) * 255])
def test_tp_conv_some_gradients(C, l1, l2, lo, degrees):
    """A convolution's backward asked for each subset of its gradients (other kernels for some subsets):
    the gradients of the full request up to its sums' rounding, and empty tensors for the rest."""
    ops = _ops()
    from flashcart_amd.o3._graph import build_graph
    ei = random_csr_graph(len(degrees), degrees, seed=C, allow_self=True)
    graph = build_graph(ei.to(DEV), len(degrees))
    g = torch.Generator(device=DEV).manual_seed(C + l1)
    meta = ops.tp_meta(l1, l2, lo, C, 1, False, False)
    n, e = len(degrees), ei.shape[1]
    in1, in2, w, go = (torch.randn(*s, device=DEV, generator=g) for s in (
        (n, (l1 + 1) ** 2 * C), (e, (l2 + 1) ** 2), (e, meta[-1] * C), (n, sum(meta[2]))))

    def run(*need):
        return ops.tp_bwd(go, in1, in2, w, graph.idx_i, graph.idx_j, l1, l2, lo, C, 1, False, False, *meta, False,
                          *need, graph.rowptr, graph.sender_perm, graph.sender_ptr, 0.7)

    # each gradient's terms in absolute value: the full request of the absolute operands bounds nothing (signed
    # coupling constants), so the bound is relative to the largest entry, as for the other products here
    want = run(True, True, True)
    for mask in range(1, 8):
        need = [bool(mask & b) for b in (1, 2, 4)]
        for k, (a, b, on) in enumerate(zip(run(*need), want, need)):
            if on:
                _close(a, b, f"gradient {k} of {need}")
            else:
                assert a.numel() == 0


@pytest.mark.parametrize("C", [32, 64, 128])
@pytest.mark.parametrize("degrees", [(4, 0, 2, 34, 66), (17, 16, 15) * 256])
def test_tp_conv_some_gradients_paired(C, degrees):
    """Each subset of the gradients with one weight row for two edges: as with the rows written out per edge (the same
    kernels, which read the same values), for pairs of arbitrary edges."""
    ops = _ops()
    from flashcart_amd.o3._graph import build_graph
    l1, l2, lo = 2, 3, 3
    ei = random_csr_graph(len(degrees), degrees, seed=C, allow_self=True)
    graph = build_graph(ei.to(DEV), len(degrees))
    g = torch.Generator(device=DEV).manual_seed(C)
    meta = ops.tp_meta(l1, l2, lo, C, 1, False, False)
    n, e = len(degrees), ei.shape[1]
    assert e % 2 == 0
    slot = torch.randperm(e, device=DEV, generator=g).to(torch.int32)
    in1, in2, w, go = (torch.randn(*s, device=DEV, generator=g) for s in (
        (n, (l1 + 1) ** 2 * C), (e, (l2 + 1) ** 2), (e // 2, meta[-1] * C), (n, sum(meta[2]))))

    def run(weights, pairs, *need):
        return ops.tp_bwd(go, in1, in2, weights, graph.idx_i, graph.idx_j, l1, l2, lo, C, 1, False, False, *meta, False,
                          *need, graph.rowptr, graph.sender_perm, graph.sender_ptr, 0.7, pairs)

    for mask in range(1, 8):
        need = [bool(mask & b) for b in (1, 2, 4)]
        for k, (a, b, on) in enumerate(zip(run(w, slot, *need), run(w[(slot >> 1).long()], None, *need), need)):
            if on:
                _close(a, b, f"gradient {k} of {need}")
            else:
                assert a.numel() == 0 and b.numel() == 0
