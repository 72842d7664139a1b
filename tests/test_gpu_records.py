"""The matrix-core product on digit planes (jm_mx.h, jm_mfma.hip) against
float64: its sums, its encoding and its range through the plugin product, and
the expert block whose products all take it.

Plugin shapes: 2048 columns split over 8 blocks of one super-stage (256 columns) and
unsplit, 768 columns unsplit (three super-stages) and split, 512 unsplit; Q4
groups of 64 and 32; a ragged last token tile."""

import numpy as np
import pytest
import torch

from conftest import banner
from joule_amd import q4_store as Q
from joule_amd.backend import HipBackend
from joule_amd.moe import HbmExpertStore, MoEShape
from joule_amd.synth import activations, router_weights, torch_store

pytestmark = pytest.mark.gpu

SHAPES = [(768, 2048, 40), (8192, 2048, 257), (8192, 768, 257), (2048, 768, 33), (4096, 512, 513)]


class Product:
    """One random Q4 matrix on the GPU, its nibbles and scales in float64."""

    def __init__(self, m, d, group, seed=0):
        g = torch.Generator(device="cuda")
        g.manual_seed(1000 * group + m + d + seed)
        self.m, self.d, self.group = m, d, group
        self.packed = torch.randint(0, 256, (m * d // 2,), generator=g, device="cuda", dtype=torch.uint8)
        self.scales = (torch.rand(m * d // group, generator=g, device="cuda") * 0.01 + 0.002).to(torch.float16)
        n = self.packed.cpu().numpy()
        sc = self.scales.cpu().numpy().view(np.uint16)
        self.W = torch.from_numpy(Q.dequantize(sc, n, m * d, group).reshape(m, d)).cuda().double()

    def __call__(self, X):
        out = torch.empty((X.shape[0], self.m), device="cuda")
        HipBackend().q4_gemm(out, X.contiguous(), self.packed, self.scales.view(torch.int16), self.m, self.d, self.group)
        torch.cuda.synchronize()
        return out

    def terms(self, X):
        """[groups, T, m] the groups' exact contributions."""
        T, ng = X.shape[0], self.d // self.group
        x = X.double().view(T, ng, self.group).transpose(0, 1)
        w = self.W.view(self.m, ng, self.group).permute(1, 2, 0)
        return torch.stack([x[g] @ w[g].contiguous() for g in range(ng)])


def _float32_bound(t):
    """Rounding of the sums alone, per element: a group's sum is rounded at
    most twice (the last plane, the scale's multiply-add), a running sum over
    consecutive groups once per group and per column split (at most 8): 2^-24
    (2 sum |term| + (groups + 8) R), R the largest sum over consecutive
    groups."""
    pre = torch.cat([torch.zeros_like(t[:1]), t.cumsum(0)])
    R = pre.amax(0) - pre.amin(0)
    return 2.0 ** -24 * (2 * t.abs().sum(0) + (t.shape[0] + 8) * R)


@pytest.mark.parametrize("group", [64, 32])
@pytest.mark.parametrize("m,d,T", SHAPES)
@pytest.mark.parametrize("sign", ["one", "mixed"])
def test_sums_round_like_float32(gpu, m, d, T, group, sign):
    """Integer tokens of 15 bits, which the encoding holds exactly, so that
    only the sums round.  Tokens of one sign need the -8 of the nibbles inside
    the groups: taken once for all groups, the running sum is up to 100 R."""
    banner(f"records sums {m}x{d} T={T} G={group} {sign}")
    p = Product(m, d, group)
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    X = torch.randint(28000, 32768, (T, d), generator=g, device="cuda").float()
    if sign == "mixed":
        X = X * (torch.randint(0, 2, (T, d), generator=g, device="cuda") * 2 - 1)
    X = X / 32768
    got = p(X)
    t = p.terms(X)
    over = ((got.double() - t.sum(0)).abs() / _float32_bound(t)).max().item()
    print(f"  largest error / bound {over:.3f}", flush=True)
    assert over <= 1.0


@pytest.mark.parametrize("group", [64, 32])
@pytest.mark.parametrize("m,d,T", [(768, 2048, 40), (8192, 768, 257)])
@pytest.mark.parametrize("kind", ["spikes", "constant"])
def test_values_are_held_to_half_a_step(gpu, m, d, T, group, kind):
    """A value is held to half a step, at most its group's largest / 507374.
    With one value per group that is the error of its term; in a row of one
    value every group holds it alike, and the result is off by that factor.
    On top, the sums' rounding."""
    banner(f"records step {m}x{d} T={T} G={group} {kind}")
    p = Product(m, d, group)
    g = torch.Generator(device="cuda")
    g.manual_seed(7)
    if kind == "constant":
        X = (1.0 + torch.rand((T, 1), generator=g, device="cuda")).expand(T, d).contiguous()
    else:
        X = torch.zeros((T, d // group, group), device="cuda")
        at = torch.randint(0, group, (T, d // group, 1), generator=g, device="cuda")
        X.scatter_(2, at, 1.0 + torch.rand((T, d // group, 1), generator=g, device="cuda"))
        X = X.view(T, d)
    got = p(X)
    t = p.terms(X)
    held = t.sum(0).abs() if kind == "constant" else t.abs().sum(0)
    over = ((got.double() - t.sum(0)).abs() / (held / 507374 + _float32_bound(t))).max().item()
    print(f"  largest error / bound {over:.3f}", flush=True)
    assert over <= 1.0


@pytest.mark.parametrize("group", [64, 32])
@pytest.mark.parametrize("mean", [0.0, 3.0])
def test_product_error(gpu, group, mean):
    """N(mean, 1) tokens.  Each value's rounding is uniform within half a step,
    at most max / 507374 of its group, and independent: the error of an
    element has the variance sum of (max / 507374)^2 / 3 w^2, and the largest
    of 10^5 lies within 6 of its standard deviations; on top, the sums'
    rounding.  A lost digit plane, plane scale or correction is 30 times
    this at the least (a step of the plane above)."""
    banner(f"records error G={group} mean={mean}")
    m, d, T = 2048, 2048, 70
    p = Product(m, d, group)
    g = torch.Generator(device="cuda")
    g.manual_seed(11)
    X = torch.randn((T, d), generator=g, device="cuda") + mean
    got = p(X)
    t = p.terms(X)
    mx = X.double().abs().view(T, d // group, group).amax(2)
    sd = ((mx / 507374) ** 2 / 3 @ p.W.view(m, d // group, group).square().sum(2).T.contiguous()).sqrt()
    over = ((got.double() - t.sum(0)).abs() / (6 * sd + _float32_bound(t))).max().item()
    rel = ((got.double() - t.sum(0)).norm() / t.sum(0).norm()).item()
    print(f"  largest error / bound {over:.3f}, rel err {rel:.2e}", flush=True)
    assert over <= 1.0


@pytest.mark.parametrize("scale", [4e-34, 1e-30, 1e30, 1e36])
@pytest.mark.parametrize("kind", ["constant", "normal"])
def test_product_over_the_float_range(gpu, scale, kind):
    """test_product_error's bound and test_values_are_held_to_half_a_step's at
    the ends of the float32 range: a step is at least 2^-126, and the sums over
    unsigned nibbles and their correction stay finite where the result is."""
    banner(f"records range {scale} {kind}")
    m, d, T, group = 768, 2048, 40, 64
    p = Product(m, d, group)
    g = torch.Generator(device="cuda")
    g.manual_seed(13)
    if kind == "constant":
        X = (1.0 + torch.rand((T, 1), generator=g, device="cuda")).expand(T, d)
    else:
        X = torch.randn((T, d), generator=g, device="cuda")
    X = (X.double() * scale).float().contiguous()
    got = p(X)
    t = p.terms(X)
    half = (X.double().abs().view(T, d // group, group).amax(2) / 507374).clamp_min(2.0 ** -127)
    if kind == "constant":
        held = t.sum(0).abs() * (half / X.double().abs().view(T, d // group, group).amax(2)).amax(1, keepdim=True)
    else:
        held = 6 * ((half ** 2 / 3) @ p.W.view(m, d // group, group).square().sum(2).T.contiguous()).sqrt()
    assert torch.isfinite(got).all()
    over = ((got.double() - t.sum(0)).abs() / (held + _float32_bound(t))).max().item()
    rel = ((got.double() - t.sum(0)).norm() / t.sum(0).norm()).item()
    print(f"  largest error / bound {over:.3f}, rel err {rel:.2e}", flush=True)
    assert over <= 1.0
    # the block integers of the int8 form, 16 bits, at the lower end too
    assert rel <= 2.0 ** -15


@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("group", [64, 32])
def test_non_finite_values_stay_in_their_row(gpu, group, value):
    """A non-finite value makes its token's whole row non-finite (every weight
    row reads it) and leaves the other rows as they are."""
    banner(f"records non-finite {value} G={group}")
    p = Product(768, 2048, group)
    g = torch.Generator(device="cuda")
    g.manual_seed(17)
    X = torch.randn((70, 2048), generator=g, device="cuda")
    clean = p(X)
    bad = [0, 33, 69]
    for i, b in enumerate(bad):
        X[b, (0, 1000, 2047)[i]] = value
    got = p(X)
    assert not torch.isfinite(got[bad]).any()
    keep = [i for i in range(70) if i not in bad]
    assert torch.equal(got[keep], clean[keep])


class Block:
    """A one-layer block whose experts all take the matrix-core branch."""

    def __init__(self, d, m, group):
        self.shape = MoEShape(d, m, 16, 8, True, f"d{d}-m{m}")
        blob, offsets = torch_store(self.shape, 1, group)
        self.group = group
        self.store = HbmExpertStore(self.shape, 1, blob, offsets, group)
        self.store.set_router(torch.from_numpy(router_weights(self.shape, 0)[None]).cuda())
        self.store.set_dense_min(1)

    def __call__(self, x):
        sh = self.shape
        self.top = torch.empty((x.shape[0], sh.topk), dtype=torch.int32, device="cuda")
        self.tw = torch.empty((x.shape[0], sh.topk), device="cuda")
        out = self.store.layer_ffn_batch(0, x, topk_idx=self.top, topk_w=self.tw)
        torch.cuda.synchronize()
        return out

    def exact(self, x):
        """float64, with the routing of the call before."""
        sh, out = self.shape, torch.zeros(x.shape, dtype=torch.float64, device="cuda")
        for e in range(sh.E):
            W = [torch.from_numpy(Q.dequantize(sc.cpu().numpy().view(np.uint16), pk.cpu().numpy(), n, self.group)
                                  .reshape(r)).cuda().double()
                 for (sc, pk, n), r in zip(self.store.ensure(0, e), ((sh.m, sh.d), (sh.m, sh.d), (sh.d, sh.m)))]
            tok, slot = torch.where(self.top == e)
            xe = x[tok].double()
            act = torch.nn.functional.silu(xe @ W[0].T) * (xe @ W[1].T)
            out.index_add_(0, tok, self.tw[tok, slot].double().unsqueeze(1) * (act @ W[2].T))
        return out


@pytest.mark.parametrize("d,m,group,B", [(512, 256, 32, 40), (1024, 256, 64, 70), (2048, 768, 32, 65), (2048, 768, 64, 130),
                                         (1024, 512, 64, 97), (2048, 2048, 64, 33)])
@pytest.mark.parametrize("mean", [0.0, 2.0])
def test_block_error(gpu, d, m, group, B, mean):
    """Largest error of a token over its largest output at most 2e-5, the bar
    of the five-digit kernels (whose step, max / 489335, lies between the
    records' max / 507375 and max / 253688).  A lost plane, scale or
    correction in either product costs at least 32 steps."""
    banner(f"records block d={d} m={m} G={group} B={B} mean={mean}")
    blk = Block(d, m, group)
    try:
        x = torch.from_numpy(activations(B, d, seed=d + m)).cuda() + mean
        got = blk(x).double()
        assert blk.store.dense_tiles() == int(((torch.bincount(blk.top.flatten().long()) + 31) // 32).sum())
        want = blk.exact(x)
        err = ((got - want).abs().amax(1) / want.abs().amax(1)).max().item()
        print(f"  max rel err {err:.2e}", flush=True)
        assert err <= 2e-5
    finally:
        blk.store.close()


@pytest.mark.parametrize("group", [64, 32])
def test_block_non_finite_tokens(gpu, group):
    """On the matrix-core branch: a token whose act leaves the float32 range
    comes out non-finite as a whole (every hidden row reads it), a NaN token is
    routed nowhere and comes out 0, and the other tokens keep their bits."""
    banner(f"records block non-finite G={group}")
    blk = Block(1024, 768, group)
    try:
        x = torch.from_numpy(activations(70, 1024, seed=3)).cuda()
        clean = blk(x)
        x[5] *= 1e25
        x[40, 100] = float("nan")
        got = blk(x)
        assert not torch.isfinite(got[5]).any()
        assert (blk.top[40] == -1).all() and (got[40] == 0).all()
        keep = [b for b in range(70) if b not in (5, 40)]
        assert torch.equal(got[keep], clean[keep])
    finally:
        blk.store.close()
