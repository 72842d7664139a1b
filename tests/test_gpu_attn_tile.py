"""The query-tiled attention of a prompt's positions (k_attn_tile) against the
oracle's per-position attention: every ratio of query to KV heads, token
counts around the 64-row tiles and around the count that selects the kernel
(tokens x KV heads of 320), prefixes that start inside a 32-position tile; and that a non-finite token
reaches no earlier position."""

import numpy as np
import pytest
import torch

from joule_amd.decoder import DecoderShape, DecoderWeights, HipDecoder, KVCacheSet
from joule_amd.dense import DenseFfnStore, dense_ffn_shape
from joule_amd.synth import activations, decoder_weights, fill_kv
from oracle import decoder as D

pytestmark = pytest.mark.gpu

TOL = 1e-3          # the decoder's bar: max relative error against the oracle, per token
DIM, M = 1024, 512


def _model(H, KH, maxT, qk=1):
    shape = DecoderShape(n_layers=1, moe=dense_ffn_shape(DIM, M), n_heads=H, n_kv=KH, maxT=maxT, qk_norm_type=qk)
    t = decoder_weights(shape, norm_jitter=0.1)
    weights = DecoderWeights(shape, **t)
    kv = KVCacheSet(shape, 1)
    fill_kv(kv.data)
    torch.cuda.synchronize()
    w = {k: v.float().cpu().numpy() for k, v in weights.t.items()}
    return HipDecoder(DenseFfnStore(DIM, M, 1), weights, graph=False), D.OracleDecoder(1, DIM, H, KH, 128, shape.eps, qk, False, w, None), kv


def _run(dec, x, p0, kv):
    B = x.shape[0]
    out = dec.decode_layers_batch(torch.from_numpy(x).cuda(), list(range(p0, p0 + B)), kv, seqs=[0] * B)
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("H,KH,qk,B,p0", [(8, 8, 1, 39, 0), (8, 8, 1, 40, 0), (8, 8, 2, 65, 31), (8, 8, 0, 64, 97),
                                          (8, 4, 0, 80, 0), (8, 4, 1, 97, 130), (8, 2, 2, 161, 0), (8, 2, 1, 176, 95),
                                          (8, 1, 1, 319, 3), (8, 1, 1, 320, 0), (8, 1, 0, 333, 128)])
def test_tiles_match_oracle(H, KH, qk, B, p0):
    print(f"[attn tile] H={H} KH={KH} qk={qk} B={B} p0={p0}", flush=True)
    dec, oracle, kv = _model(H, KH, 512, qk)
    kv_h = [(kv.data[0, 0, 0].float().cpu().numpy(), kv.data[0, 0, 1].float().cpu().numpy())]
    x = activations(B, DIM, seed=B + p0)
    got = _run(dec, x, p0, kv)
    want = np.concatenate([oracle.decode_layers_batch(x[i:i + 1], [p0 + i], [kv_h]) for i in range(B)])
    rel = (np.abs(got - want).max(axis=1) / np.abs(want).max(axis=1)).max()
    print(f"  max rel err {rel:.2e}", flush=True)
    assert rel <= TOL
    dec.store.close()


@pytest.mark.parametrize("bad,value", [(0, np.nan), (19, np.inf), (40, np.nan), (63, -np.inf)])
def test_non_finite_token_stays_causal(bad, value):
    print(f"[attn tile] non-finite token {bad}", flush=True)
    dec, _, kv = _model(8, 8, 256)
    x = activations(64, DIM, seed=9)
    clean = _run(dec, x, 3, kv)
    x[bad, 5] = value
    got = _run(dec, x, 3, kv)
    assert np.isfinite(clean).all()
    assert np.array_equal(got[:bad], clean[:bad])
    assert not np.isfinite(got[bad:]).all(axis=1).any()
    dec.store.close()


@pytest.mark.parametrize("H,KH,B,p0", [(32, 32, 15, 300), (32, 32, 16, 300), (8, 8, 43, 130), (8, 8, 44, 130)])
def test_one_head_each_on_both_sides_of_the_rule(H, KH, B, p0):
    """One query head per KV head takes the tiled kernel from 16 tokens and 352
    tokens x KV heads."""
    test_tiles_match_oracle(H, KH, 1, B, p0)
