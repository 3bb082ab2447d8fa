"""The projection's backward on the fp16 matrix cores (csrc/fht_bwd.hip) against 64 bits."""
import math

import pytest
import torch

from lookupffn_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _hadamard(n):
    h = torch.ones(1, 1, dtype=torch.float64, device=DEV)
    while h.shape[0] < n:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h


def _inputs(B, H, D, R, T, seed=0):
    gen = torch.Generator(device=DEV).manual_seed(B + D + R + seed)
    rand = lambda *s: torch.randn(*s, generator=gen, device=DEV)
    return (1.5 * rand(B, H) + 0.3, rand(R, 4, D) / math.sqrt(D), rand(B, T * 8), rand(B, T), 1 + 0.1 * rand(H), 0.1 * rand(H))


def _reference(x, diag, z, g_score, ln_w=None, ln_b=None, eps=1e-5, decay=0.7):
    x, diag, z, g_score = (t.double() for t in (x, diag, z, g_score))
    (B, H), (R, J, D), T = x.shape, diag.shape, g_score.shape[1]
    if ln_w is not None:
        x = torch.nn.functional.layer_norm(x, (H,), ln_w.double(), ln_b.double(), eps)
    h = torch.nn.functional.pad(x, (0, D - H))
    z8 = z.view(B, T, 8)
    a = z8.abs()
    e = torch.exp(-2 * a)
    g = z8.sign() * (1 + a.sum(-1, keepdim=True) * 2 * e / (1 + e)) * (g_score / (1 + e).prod(-1)).unsqueeze(-1)
    g_z = torch.nn.functional.pad(g.reshape(B, T * 8), (0, R * D - T * 8))
    hd, g_x, g_diag = _hadamard(D), [], torch.zeros_like(diag)
    for r in range(R):
        u = [h]
        for s in range(J - 1):
            u.append((u[-1] * diag[r, s]) @ hd)
        gr = g_z[:, r * D:(r + 1) * D]
        t = decay * gr
        for s in range(J - 1, -1, -1):
            t = t @ hd
            g_diag[r, s] = (t * u[s]).sum(0)
            t = t * diag[r, s]
        g_x.append((t + (1 - decay) * gr)[:, :H])
    return sum(g_x), g_diag, g_z.sum(0)[:T * 8]


# Per transform a number's lo is rounded twice, by 2^-23 at most, and a sum in two times four instructions; seven transforms in a
# row, all of one sign: 7 * (2 * 2^-23 + 8 * 2^-24).  The score's gradient: a few roundings beside that.
REL = 7 * (2 * 2.0 ** -23 + 8 * 2.0 ** -24) + 1e-6


def _close(got, want):
    for g, w in zip(got, want):
        assert torch.isfinite(g).all() and ((g.double() - w.view(g.shape)).norm() / w.norm()).item() <= REL


# one, two and four rows to a tile, the last of them short; columns short of the transform's points and of the codes' groups; repeats
@pytest.mark.parametrize("B,H,D,R,T", [(300, 768, 1024, 1, 128), (5, 1024, 1024, 2, 200), (1, 516, 1024, 1, 3), (2100, 1000, 1024, 1, 126),
                                       (33, 500, 512, 1, 40), (1030, 512, 512, 2, 128), (70, 256, 256, 2, 64), (2051, 132, 256, 1, 31),
                                       (3, 256, 256, 4, 128)])
@pytest.mark.parametrize("with_ln", [False, True])
def test_against_64_bits(B, H, D, R, T, with_ln):
    x, diag, z, g_score, ln_w, ln_b = _inputs(B, H, D, R, T)
    z[0, :8] = 0
    ln = (ln_w, ln_b, 1e-5) if with_ln else ()
    got = ops.project_hash_bwd(x, diag, z, g_score, 0.7, 0.3, *ln)
    # (with LayerNorm one gradient of its output per repeat)
    _close((got[0].double().sum(0) if with_ln else got[0], *got[1:]), _reference(x, diag, z, g_score, *ln))
    again = ops.project_hash_bwd(x, diag, z, g_score, 0.7, 0.3, *ln)
    assert all(torch.equal(a, b) for a, b in zip(got, again))


@pytest.mark.parametrize("D", [256, 512, 1024])
def test_sizes_and_rows_of_their_own(D):
    """Inputs and gradients of any size, rows of very different sizes in one tile, and a row that is not finite stays alone."""
    x, diag, z, g_score, _, _ = _inputs(41, D, D, 1, D // 8)
    for sx, sd, sg in ((1e8, 1.0, 1e-20), (1e-12, 1e3, 1e10), (1.0, 1e-4, 1.0)):
        _close(ops.project_hash_bwd(x * sx, diag * sd, z, g_score * sg, 0.7, 0.3),
               _reference(x * sx, diag * sd, z, g_score * sg))
    base, _, _ = ops.project_hash_bwd(x, diag, z, g_score, 0.7, 0.3)
    g = g_score.clone()
    g[4] *= 1e-15
    g[9] *= 1e12
    g[14] = 0
    g[17, 1], g[22, 0] = float("nan"), float("inf")
    got, _, _ = ops.project_hash_bwd(x, diag, z, g, 0.7, 0.3)
    rows = [i for i in range(41) if i not in (4, 9, 14, 17, 22)]
    assert torch.equal(got.view(41, D)[rows], base.view(41, D)[rows]) and (got.view(41, D)[14] == 0).all()
    assert not torch.isfinite(got.view(41, D)[[17, 22]]).any()
    want = _reference(x, diag, z, g)[0]
    for i in (4, 9):
        assert ((got.view(41, D)[i].double() - want[i]).norm() / want[i].norm()).item() <= REL


@pytest.mark.parametrize("D", [256, 512, 1024])
def test_the_scores_gradient_far_from_zero(D):
    """One small value beside seven large ones: its gradient is exp(-2 |z|) times their sum, as exact far from zero as near it."""
    B, T = 400, D // 8
    x, diag, _, g_score, _, _ = _inputs(B, D, D, 1, T)
    gen = torch.Generator(device=DEV).manual_seed(D)
    z = torch.full((B, T, 8), 1e14, device=DEV)
    z[:, :, 3] = (0.5 + 14.5 * torch.rand(B, T, generator=gen, device=DEV)) * torch.randn(B, T, generator=gen, device=DEV).sign()
    z[z == 0] = 1.0
    g_x, _, _ = ops.project_hash_bwd(x, diag, z.view(B, T * 8), g_score, 0.0, 1.0)          # the gradient of z itself
    got, z3 = g_x.view(B, T, 8)[:, :, 3].double(), z[:, :, 3].double()
    e = torch.exp(-2 * z3.abs())
    want = z3.sign() * (1 + 2 * (7 * z[0, 0, 0].double() + z3.abs()) * e / (1 + e)) * (g_score.double() / (1 + e))
    # an ulp (2^-23) each for 2^t and the reciprocal, half of one for its correction, 1 + e twice, e / (1 + e), the sum's two last
    # additions, its product, 1 + it, the division and the last product: at most 2 * 2^-23 + 10 * 2^-24
    assert ((got - want) / want).abs().max() <= 14 * 2.0 ** -24
    # infinities, NaN and a sum beyond fp32 stay in their own row (a transform takes them through it)
    z[5, 7, 2], z[6, 1, 4], z[8, 0] = float("inf"), float("nan"), 3e38
    finite = torch.isfinite(ops.project_hash_bwd(x, diag, z.view(B, T * 8), g_score, 0.0, 1.0)[0].view(B, D)).all(-1)
    assert (~finite).nonzero().flatten().tolist() == [5, 6, 8]
