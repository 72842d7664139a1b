"""The dense branch's units at the edges of its kernels against the oracle:
contractions of one, two, three and eight super-stages of 256 columns, Q4
groups of 64 and 32, more units than resident blocks (so that blocks take
several) and ragged last tiles; and its activation encoding over the range of
float magnitudes.

Bar: normwise per token, 1e-3 (the block's), as test_gpu_parity.py's."""

import numpy as np
import pytest
import torch

from conftest import banner
from joule_amd.moe import MoEShape
from joule_amd.synth import activations
from test_gpu_parity import TOL, Layer, _rel, _run_block

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,m,group,B", [(512, 256, 32, 40), (1024, 256, 64, 70), (512, 512, 32, 97), (2048, 768, 32, 65),
                                         (512, 768, 32, 1000), (1024, 256, 64, 1100), (2048, 2048, 64, 33)])
def test_units_match_oracle(gpu, oracle_lib, d, m, group, B):
    banner(f"dense units d={d} m={m} G={group} B={B}")
    layer = Layer(MoEShape(d, m, 16, 8, True, f"d{d}-m{m}"), group, 1, oracle_lib)
    try:
        layer.store.set_dense_min(1)
        x = activations(B, d, seed=d + m + B)
        out, top, tw = _run_block(layer, 0, x)
        counts = np.bincount(top.ravel(), minlength=16)
        assert layer.store.dense_tiles() == int(((counts + 31) // 32).sum())
        rout, rtop, _ = layer.oracle(0).forward(x, n_threads=8)
        assert np.array_equal(top, rtop)
        err = _rel(out, rout)
        print(f"  max rel err {err:.3e}", flush=True)
        assert err <= TOL
    finally:
        layer.store.close()


@pytest.mark.parametrize("scale", [1e-30, 1e-6, 1.0, 65536.0, 1e9])
def test_units_follow_the_activations_magnitude(gpu, oracle_lib, scale):
    """Groups whose largest value is just under and at a power of two (where
    the encoding's exponent steps), zero groups, and tokens at the given
    scale; the router sees the same logits up to the scale, so only the
    dense product and its encoding differ from scale 1.  At 1e9 SwiGLU is
    linear or zero; at 1e-30 act underflows to 0 in float32 on both sides."""
    banner(f"dense units, activations of scale {scale}")
    layer = Layer(MoEShape(1024, 256, 16, 8, True, "d1024-m256"), 64, 1, oracle_lib)
    try:
        layer.store.set_dense_min(1)
        x = activations(48, 1024, seed=5)
        x[:, 64:128] = 0.0
        x[::2, 0] = np.nextafter(np.float32(4.0), np.float32(0.0))
        x[1::2, 0] = 4.0
        x = (x * np.float32(scale)).astype(np.float32)
        out, top, _ = _run_block(layer, 0, x)
        assert layer.store.dense_tiles() > 0
        rout, rtop, _ = layer.oracle(0).forward(x, n_threads=8)
        assert np.array_equal(top, rtop)
        assert np.isfinite(out).all()
        if np.abs(rout).max() == 0.0:
            assert np.abs(out).max() == 0.0
        else:
            err = _rel(out, rout)
            print(f"  max rel err {err:.3e}", flush=True)
            assert err <= TOL
    finally:
        layer.store.close()
