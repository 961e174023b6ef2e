"""The bf16 channel-mix variant of the sparse conv (precision 1: one bf16 MFMA per product in the node
expansion, the edge message and the node-expansion gradient, fp32 accumulation), against the fp64 oracle
(op level) and against the fp32-accurate path (whole model).  bf16 keeps 8 significant bits, so the
bound here is a bf16 one: 2e-2 relative (max-norm) at the op level, where every output sums 64 to 4160
rounded products; the measured errors are printed.  The variant must also be deterministic and really
differ from the fp32 path."""

import numpy as np
import pytest
import torch

from sparse_helpers import oracle_conv2, rel_inf

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOL_BF16 = 2e-2


@pytest.mark.parametrize("C", [64, 32, 128])
def test_bf16_conv2_op_against_oracle(C):
    from fsctep_amd import ops
    from fsctep_amd.graph import prepare_graph
    from test_sparse_gpu import _graph_with_edge_cases
    torch.manual_seed(3)
    N = 40
    src, dst = _graph_with_edge_cases(N, 400, 7)
    E = src.shape[0]
    x = torch.randn(N, 13, C, dtype=torch.float64)
    h = torch.randn(E, 64, dtype=torch.float64)
    v = torch.randn(E, 3, dtype=torch.float64)
    n = v / v.norm(dim=1, keepdim=True)
    L = torch.randn(6 * C * C, 64, dtype=torch.float64) / 8
    b = torch.randn(6 * C * C, dtype=torch.float64) * 0.1
    gr = prepare_graph(src.to(DEV), dst.to(DEV), torch.zeros(E, 3, device=DEV), N)
    order = torch.argsort(dst, stable=True)
    xo, ho, no = (t.clone().requires_grad_(True) for t in (x, h[order], n[order]))
    ref = oracle_conv2(xo, ho, no, L, b, src[order], dst[order], N, 1.0 / (E / N))
    G = torch.randn_like(ref)
    gx, gh, gn = torch.autograd.grad((ref * G).sum(), (xo, ho, no))
    bk1, bk6 = torch.ops.fsctep.sparse_prepare_weights(L.float().to(DEV), b.float().to(DEV), C)
    res = {}
    for prec in (0, 1):
        xd = x.float().to(DEV).requires_grad_(True)
        hd = h[order].float().to(DEV).requires_grad_(True)
        nd = n[order].float().to(DEV).requires_grad_(True)
        out = ops.sparse_conv_apply(xd, hd, nd, bk1, bk6, gr, precision=prec)
        grads = torch.autograd.grad(out, (xd, hd, nd), G.float().to(DEV))
        res[prec] = (out.detach(), *grads)
    errs = [rel_inf(a, r) for a, r in zip(res[1], (ref, gx, gh, gn))]
    print(f"C {C}: bf16 variant vs fp64 oracle: out {errs[0]:.2e}, dx {errs[1]:.2e}, dh {errs[2]:.2e}, dn {errs[3]:.2e}")
    assert max(errs) < TOL_BF16, errs
    assert rel_inf(res[1][0], res[0][0]) > 1e-5          # the bf16 products really ran
    assert rel_inf(res[0][0], ref) < 1e-5                 # and the default path is the fp32-accurate one


# the message gradient's channel chunks in four parts (up to 256 atoms), two (up to 2,047) and one
@pytest.mark.parametrize("N,E,C", [(40, 400, 64), (256, 1500, 32), (257, 1500, 64), (2047, 4000, 32), (2048, 4000, 32)])
def test_bf16_variant_rounds_the_channel_mix_alone(N, E, C):
    """With operands that bf16 holds (features +-1 in one channel a node, weights and radial values rounded to bf16) the
    channel mix is exact, so the outputs and the gradients of the radial values and directions, whose products run at
    fp32 accuracy, agree to 1e-5; the input gradient, which goes through the mix, to the bf16 bound."""
    from fsctep_amd import ops
    from fsctep_amd.graph import prepare_graph
    from test_sparse_gpu import _graph_with_edge_cases
    g = torch.Generator().manual_seed(N + C)
    bf = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64).bfloat16().double()
    src, dst = _graph_with_edge_cases(N, E, 11)
    E = src.shape[0]
    x = torch.zeros(N, 13, C, dtype=torch.float64)
    x[torch.arange(N)[:, None], torch.arange(13), torch.randint(0, C, (N, 1), generator=g)] = \
        torch.randint(0, 2, (N, 13), generator=g).double() * 2 - 1
    h, L, b = bf(E, 64), (bf(6 * C * C, 64) / 8), bf(6 * C * C) / 8
    v = torch.randn(E, 3, generator=g, dtype=torch.float64)
    n = (v / v.norm(dim=1, keepdim=True)).float().double()
    order = torch.argsort(dst, stable=True)
    xo, ho, no = (t.clone().requires_grad_(True) for t in (x, h[order], n[order]))
    ref = oracle_conv2(xo, ho, no, L, b, src[order], dst[order], N, 1.0 / (E / N))
    G = torch.randn(ref.shape, generator=g, dtype=torch.float64).float().double()
    gx, gh, gn = torch.autograd.grad((ref * G).sum(), (xo, ho, no))
    gr = prepare_graph(src.to(DEV), dst.to(DEV), torch.zeros(E, 3, device=DEV), N)
    bk1, bk6 = torch.ops.fsctep.sparse_prepare_weights(L.float().to(DEV), b.float().to(DEV), C)
    xd, hd, nd = (t.float().to(DEV).requires_grad_(True) for t in (x, h[order], n[order]))
    out = ops.sparse_conv_apply(xd, hd, nd, bk1, bk6, gr, precision=1)
    dx, dh, dn = torch.autograd.grad(out, (xd, hd, nd), G.float().to(DEV))
    assert max(rel_inf(a, r) for a, r in ((out.detach(), ref), (dh, gh), (dn, gn))) < 1e-5
    assert 1e-5 < rel_inf(dx, gx) < TOL_BF16


@pytest.mark.parametrize("prec", [0, 1])
def test_directions_of_any_length(prec):
    """The op takes any direction vectors: lengths from 0 to 50 (dP grows with the length's square), the default path
    to 1e-5 and the bf16 variant to the bf16 bound of every output, edges of each decade of length by themselves too
    (the gradient of a short direction is linear in the receiver gradient, that of a long one grows with it)."""
    from fsctep_amd import ops
    from fsctep_amd.graph import prepare_graph
    from test_sparse_gpu import _graph_with_edge_cases
    torch.manual_seed(5)
    C, N = 32, 40
    src, dst = _graph_with_edge_cases(N, 400, 9)
    E = src.shape[0]
    length = torch.logspace(-2, 1.7, E, dtype=torch.float64)[torch.randperm(E)]
    length[:5] = 0.0
    v = torch.randn(E, 3, dtype=torch.float64)
    n = v / v.norm(dim=1, keepdim=True) * length.unsqueeze(1)
    x, h = torch.randn(N, 13, C, dtype=torch.float64), torch.randn(E, 64, dtype=torch.float64)
    L, b = torch.randn(6 * C * C, 64, dtype=torch.float64) / 8, torch.randn(6 * C * C, dtype=torch.float64) * 0.1
    order = torch.argsort(dst, stable=True)
    xo, ho, no = (t.clone().requires_grad_(True) for t in (x, h[order], n[order]))
    ref = oracle_conv2(xo, ho, no, L, b, src[order], dst[order], N, 1.0 / (E / N))
    G = torch.randn_like(ref)
    gx, gh, gn = torch.autograd.grad((ref * G).sum(), (xo, ho, no))
    gr = prepare_graph(src.to(DEV), dst.to(DEV), torch.zeros(E, 3, device=DEV), N)
    bk1, bk6 = torch.ops.fsctep.sparse_prepare_weights(L.float().to(DEV), b.float().to(DEV), C)
    xd, hd, nd = (t.float().to(DEV).requires_grad_(True) for t in (x, h[order], n[order]))
    out = ops.sparse_conv_apply(xd, hd, nd, bk1, bk6, gr, precision=prec)
    dx, dh, dn = torch.autograd.grad(out, (xd, hd, nd), G.float().to(DEV))
    tol = TOL_BF16 if prec else 1e-5
    assert max(rel_inf(a, r) for a, r in zip((out.detach(), dx, dh, dn), (ref, gx, gh, gn))) < tol
    ls = length[order]
    for lo, hi in ((-1.0, 0.1), (0.1, 1.0), (1.0, 4.0), (4.0, 60.0)):
        m = (ls >= lo) & (ls < hi)
        assert m.any()
        assert rel_inf(dh.cpu()[m], gh[m]) < tol and rel_inf(dn.cpu()[m], gn[m]) < tol


def test_bf16_model_against_fp32_path_and_deterministic():
    import bench
    from fsctep_amd.sparse import energy_and_forces
    s = bench._system("sparse", 3000, 22)
    m = bench.build_model("sparse", torch.device(DEV))
    pos = torch.tensor(s.pos, dtype=torch.float32, device=DEV)
    A = torch.tensor(s.species, device=DEV)
    batch = torch.zeros(3000, dtype=torch.long, device=DEV)
    cell = torch.tensor(s.cell, dtype=torch.float32, device=DEV)
    g = m.prepare(torch.tensor(s.edge_src, device=DEV), torch.tensor(s.edge_dst, device=DEV),
                  torch.tensor(s.edge_shifts, dtype=torch.float32, device=DEV), 3000, A, pos=pos)
    e32, f32 = energy_and_forces(m, pos, batch, cell, g)
    m.channel_mix_precision = "bf16"
    e16, f16 = energy_and_forces(m, pos, batch, cell, g)
    e16b, f16b = energy_and_forces(m, pos, batch, cell, g)
    assert torch.equal(e16, e16b) and torch.equal(f16, f16b)
    er, fr = rel_inf(e16, e32), rel_inf(f16, f32)
    print(f"3000 atoms: bf16 variant vs fp32 path: energies {er:.2e}, forces {fr:.2e}")
    assert er > 1e-7 and er < 5e-2 and fr < 5e-2
    m.channel_mix_precision = "fp16"
    with pytest.raises(ValueError):
        energy_and_forces(m, pos, batch, cell, g)
