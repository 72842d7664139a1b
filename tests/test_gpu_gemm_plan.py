"""Every form of the bf16 projections' GEMM (128- and 256-row tile in 1, 2 and
4 column ranges, with and without the RMSNorm, three matrices in one call) at
token counts that end inside a 64-token tile, the form asserted through
jm_gemm_plan."""

import ctypes

import numpy as np
import pytest
import torch

from joule_amd import _lib
from joule_amd.decoder import DecoderShape, DecoderWeights, HipDecoder, KVCacheSet
from joule_amd.dense import DenseFfnStore, dense_ffn_shape
from joule_amd.synth import activations, decoder_weights, fill_kv
from oracle import decoder as D

pytestmark = pytest.mark.gpu

NARROW, WIDE = 0, 1


def plan(rows, K, B):
    kz = ctypes.c_int()
    return _lib.lib().jm_gemm_plan(*rows, K, B, ctypes.byref(kz)), kz.value


@pytest.mark.parametrize("d,m,B,gu,dn", [(4096, 12288, 33, (WIDE, 4), (NARROW, 4)), (4096, 12288, 65, (WIDE, 2), (NARROW, 4)),
                                         (4096, 12288, 257, (WIDE, 1), (WIDE, 4)), (2048, 4096, 161, (NARROW, 1), (NARROW, 4)),
                                         (2048, 6144, 63, (NARROW, 2), (NARROW, 4)), (2048, 8192, 270, (WIDE, 1), (NARROW, 2))])
def test_block_forms(d, m, B, gu, dn):
    """The dense FFN against float64, largest error of a token over its largest
    output.  A token value is off by at most 2^-18 of itself (bf16 hi + lo), so
    a sum of K such terms by a standard deviation of 2^-18 / sqrt(3) of its
    own; the row's largest of 2048 or more sums is 3.5 of those, and the
    largest error of 10^6 within 6: 2^-18 per product, three products."""
    print(f"[gemm plan] block d={d} m={m} B={B}", flush=True)
    assert plan((m, m, 0), d, B) == gu and plan((d, 0, 0), m, B) == dn
    store = DenseFfnStore(d, m, 1)
    g = torch.Generator(device="cuda")
    g.manual_seed(B)
    w1, w2 = ((torch.randn((1, m, d), generator=g, device="cuda") * 0.03).to(torch.bfloat16) for _ in range(2))
    w3 = (torch.randn((1, d, m), generator=g, device="cuda") * 0.03).to(torch.bfloat16)
    store.set_weights(w1, w2, w3)
    x = torch.from_numpy(activations(B, d)).cuda()
    got = store.layer_ffn_batch(0, x).double()
    xd = x.double()
    gate, up = xd @ w1[0].double().T, xd @ w2[0].double().T
    want = (torch.nn.functional.silu(gate) * up) @ w3[0].double().T
    err = ((got - want).abs().amax(1) / want.abs().amax(1)).max().item()
    print(f"  max rel err {err:.2e}", flush=True)
    assert err <= 3 * 2.0 ** -18
    store.close()


@pytest.mark.parametrize("d,H,KH,B,want", [(1024, 32, 32, 129, (WIDE, 2)), (1024, 32, 32, 321, (WIDE, 1)),
                                           (4096, 32, 8, 130, (WIDE, 4)), (1024, 8, 2, 97, (NARROW, 4))])
def test_qkv_forms(d, H, KH, B, want):
    """q, k and v of one call (the norm weight, the sums of squares per range,
    the third matrix's rows) against the oracle: the tokens' outputs and the
    cache rows that the call appends."""
    print(f"[gemm plan] qkv d={d} H={H} KH={KH} B={B}", flush=True)
    assert plan((H * 128, KH * 128, KH * 128), d, B) == want
    shape = DecoderShape(n_layers=1, moe=dense_ffn_shape(d, 512), n_heads=H, n_kv=KH, maxT=512, qk_norm_type=1)
    weights = DecoderWeights(shape, **decoder_weights(shape, norm_jitter=0.1))
    kv = KVCacheSet(shape, 1)
    fill_kv(kv.data)
    torch.cuda.synchronize()
    w = {k: v.float().cpu().numpy() for k, v in weights.t.items()}
    oracle = D.OracleDecoder(1, d, H, KH, 128, shape.eps, 1, False, w, None)
    dec = HipDecoder(DenseFfnStore(d, 512, 1), weights, graph=False)
    kv_h = [(kv.data[0, 0, 0].float().cpu().numpy(), kv.data[0, 0, 1].float().cpu().numpy())]
    x = activations(B, d, seed=B)
    got = dec.decode_layers_batch(torch.from_numpy(x).cuda(), list(range(B)), kv, seqs=[0] * B).cpu().numpy()
    ref = np.concatenate([oracle.decode_layers_batch(x[i:i + 1], [i], [kv_h]) for i in range(B)])
    rel = (np.abs(got - ref).max(axis=1) / np.abs(ref).max(axis=1)).max()
    print(f"  max rel err {rel:.2e}", flush=True)
    assert rel <= 1e-3                              # the decoder's bar
    for j in (0, 1):
        r = kv_h[0][j][:B]
        lim = np.abs(r) * 2.0 ** -7 + 1e-4 * np.abs(r).max(axis=-1, keepdims=True)      # one bf16 unit
        assert np.all(np.abs(kv.data[0, 0, j, :B].float().cpu().numpy() - r) <= lim)
    dec.store.close()
