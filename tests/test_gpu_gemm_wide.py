"""The wide-tile projection GEMM (k_gemm_bf16_wide: 256 weight rows x 64
tokens per block) at the edges of its token tile, through the dense FFN: at d
= 2048, m = 6144 and 257 to 320 tokens the gate/up product takes it.

Bar of the block, per token: a product term is off by at most 2^-18 of itself
(the tokens' bf16 hi + lo split), so a sum of K terms by 2^-18 sum|term|,
which for N(0, 1) data is about 2^-18 x 0.8 sqrt(K) x the sum's own scale,
under 2^-18 x 9 of a row's largest of 2048 sums; three products follow one
another: 27 x 2^-18 = 1.03e-4."""

import numpy as np
import pytest
import torch

from joule_amd.dense import DenseFfnStore
from joule_amd.synth import activations
from oracle import decoder as D
from test_gpu_dense import TOL, _dense_model

pytestmark = pytest.mark.gpu

BLOCK_TOL = 27 * 2.0 ** -18


@pytest.mark.parametrize("B", [257, 288, 289, 320])
def test_wide_tile_edges(B):
    d, m = 2048, 6144
    print(f"[gemm wide] block B={B}", flush=True)
    store = DenseFfnStore(d, m, 1)
    g = torch.Generator(device="cuda")
    g.manual_seed(B)
    w1, w2 = ((torch.randn((1, m, d), generator=g, device="cuda") * 0.03).to(torch.bfloat16) for _ in range(2))
    w3 = (torch.randn((1, d, m), generator=g, device="cuda") * 0.03).to(torch.bfloat16)
    store.set_weights(w1, w2, w3)
    x = torch.from_numpy(activations(B, d))
    got = store.layer_ffn_batch(0, x.cuda()).cpu().double()
    f = [w[0].cpu().double() for w in (w1, w2, w3)]
    xd = x.double()
    gate, up = xd @ f[0].T, xd @ f[1].T
    want = (gate / (1 + torch.exp(-gate)) * up) @ f[2].T
    err = ((got - want).abs().amax(1) / want.abs().amax(1)).max().item()
    print(f"  max rel err {err:.2e}", flush=True)
    assert err <= BLOCK_TOL
    store.close()


def test_wide_tile_prefill():
    """With the norm weight and the sums of squares: a 257-token prompt
    through 2 dense layers against one decode step per position; layer 1's
    cache rows show layer 0's output of every token."""
    L, d, m, V, T = 2, 2048, 6144, 1000, 257
    dec, oracle, kv = _dense_model(L=L, d=d, m=m, H=8, KH=2, maxT=T, B=1, V=V)
    g = torch.Generator(device="cuda")
    g.manual_seed(78)
    emb = (torch.randn((V, d), generator=g, device="cuda") * 0.5).to(torch.bfloat16)
    lm = (torch.randn((V, d), generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    dec.weights.t["embed"] = emb
    dec._w = dec.weights.kernel_w()
    dec.set_lm_head(lm)
    prompt = np.random.default_rng(6).integers(0, V, size=T).tolist()
    kv_seq = [(kv.data[0, l, 0].float().cpu().numpy(), kv.data[0, l, 1].float().cpu().numpy()) for l in range(L)]
    print(f"[gemm wide] prefill T={T}", flush=True)
    logits = torch.empty(V, dtype=torch.float32, device="cuda")
    dec.prefill_layers(torch.tensor(prompt, dtype=torch.int32, device="cuda"), kv, 0, logits)
    torch.cuda.synchronize()
    E = emb.float().cpu().numpy()
    hid = None
    for t, tok in enumerate(prompt):
        hid = oracle.decode_layers_batch(D.embed_lookup(E, [tok]), [t], [kv_seq])
    want = D.lm_head(lm.float().cpu().numpy(), hid)[0]
    rel = np.abs(logits.cpu().numpy() - want).max() / np.abs(want).max()
    print(f"  last-position logits max rel err {rel:.2e}", flush=True)
    assert rel < TOL
    for l in range(L):
        for j in (0, 1):
            r = kv_seq[l][j][:T]
            lim = np.abs(r) * 2.0 ** -7 + 1e-4 * np.abs(r).max(axis=-1, keepdims=True)    # one bf16 unit
            assert np.all(np.abs(kv.data[0, l, j, :T].float().cpu().numpy() - r) <= lim)
    dec.store.close()
