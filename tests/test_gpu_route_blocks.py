"""The batch router's blocks of 8 tokens (2048 tokens and more outside the wide router's range: more than
32 experts or top-k above 4), with a partial last block: routing bit for bit against the oracle, the layer
on it with both kinds of records, the block forward's norm inside it. Hidden sizes in rising order, since
those above 1024 other than 2880 share one kernel whose LDS grows with them."""
import numpy as np
import pytest

from silentotithrandousha_amd import GpuMoeDispatcher
from silentotithrandousha_amd import synthetic as syn
from tests.helpers import assert_bit_exact, assert_rel_l2

pytestmark = pytest.mark.gpu


def _check(orc, H, E, k, T, quant, seed):
    L = syn.make_layer(H, 96, E, seed=seed, scale_lo=117, scale_hi=121, router_sigma=0.1)
    gamma = np.linspace(0.5, 1.5, H).astype(np.float32)
    d = GpuMoeDispatcher(H, 96, 7.0)
    try:
        d.preload_layer(0, L)
        d.preload_norm(0, gamma, 1e-5)
        x = syn.hidden(T, H, seed=seed + 1)
        want_l = orc.router_logits(L["router_w"], L["router_b"], x, E, H)
        idx, w, logits = d.router_topk(0, x, k, want_logits=True, n_experts=E)
        assert_bit_exact(logits, want_l, "router logits (canonical order)")
        widx, ww, _, _ = orc.topk(want_l, k)
        assert np.array_equal(idx, widx)
        assert_rel_l2(w, ww, "top-k weights", 1e-6)
        assert_rel_l2(d.layer_forward(0, x, k), orc.moe_layer(x, L, k)[0], "layer")
        if quant:
            d.set_act_quant(1)
            assert_rel_l2(d.layer_forward(0, x, k), orc.moe_layer_mxfp6(x, L, k)[0], "layer, MXFP6 activations", 2e-4)
        n = orc.rms_norm(x, gamma, 1e-5)
        assert np.array_equal(d.block_forward(0, x, k), (x + d.layer_forward(0, n, k)).astype(np.float32))
    finally:
        d.close()


@pytest.mark.parametrize("H,E,k", [(96, 40, 8), (544, 200, 2), (1024, 40, 8), (1536, 32, 5), (2048, 40, 4), (2560, 128, 4), (2880, 40, 8)])
@pytest.mark.parametrize("quant", [False, True])
def test_eight_token_blocks(orc, H, E, k, quant):
    _check(orc, H, E, k, 2053, quant, 900 + H + E)


# MXFP6 records with the norm inside the router: a token a block, and the wide router
@pytest.mark.parametrize("H,E,k,T", [(544, 8, 2, 100), (2880, 16, 4, 1025), (1024, 32, 4, 771)])
def test_quantised_block_forward(orc, H, E, k, T):
    _check(orc, H, E, k, T, True, 950 + H)
