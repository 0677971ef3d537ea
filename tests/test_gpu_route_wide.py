"""The router of larger batches (logits on the f32 MFMA, grouping in a kernel of its own) against the
oracle's canonical order, bit for bit, and the layer on top of it."""
import numpy as np
import pytest

from silentotithrandousha_amd import GpuMoeDispatcher
from silentotithrandousha_amd import synthetic as syn
from tests.helpers import assert_bit_exact, assert_rel_l2

pytestmark = pytest.mark.gpu


# H: one step and many, K tails inside a load; E: one group, not a multiple of 16, two; T: a partial
# last workgroup, one token in it, several workgroups of the grouping
@pytest.mark.parametrize("H,E,k,T", [(32, 3, 2, 1040), (96, 8, 1, 1025), (544, 17, 4, 1129), (2048, 16, 2, 1333), (2880, 32, 4, 1043),
                                     (3072, 31, 3, 1111)])
def test_wide_router_bit_exact(orc, H, E, k, T):
    L = syn.make_layer(H, 96, E, seed=800 + H + E, scale_lo=117, scale_hi=121, router_sigma=0.1)
    d = GpuMoeDispatcher(H, 96, 7.0)
    try:
        d.preload_layer(0, L)
        x = syn.hidden(T, H, seed=801 + T)
        x[3, :], x[5, H - 1], x[6, 0], x[7, :] = 0.0, np.nan, np.inf, 1e-38  # zeros, NaN, inf, products below f32's normals
        want = orc.router_logits(L["router_w"], L["router_b"], x, E, H)
        idx, w, logits = d.router_topk(0, x, k, want_logits=True, n_experts=E)
        assert_bit_exact(logits, want, "router logits (canonical order)")
        widx, ww, _, _ = orc.topk(want, k)
        assert np.array_equal(idx, widx)
        assert_rel_l2(w, ww, "top-k weights", 1e-6)
        # the layer on it: the kernel's records and grouping
        x = syn.hidden(T, H, seed=802 + T)
        want, _, _, _ = orc.moe_layer(x, L, k)
        assert_rel_l2(d.layer_forward(0, x, k), want, "layer")
        # a prefix below the kernel's range takes the other router: the same tokens, the same bits
        for a, b in zip(d.router_topk(0, x, k, want_logits=True, n_experts=E), d.router_topk(0, x[:40], k, want_logits=True, n_experts=E)):
            assert np.array_equal(a[:40], b)
        gamma = np.linspace(0.5, 1.5, H).astype(np.float32)
        d.preload_norm(0, gamma, 1e-5)
        n = orc.rms_norm(x, gamma, 1e-5)
        assert np.array_equal(d.block_forward(0, x, k), (x + d.layer_forward(0, n, k)).astype(np.float32))
        d.set_adaptive_topk(True, 1, 0.3, 0.05, 0.6)  # dropped slots
        n_dropped = int((d.router_topk(0, x, k)[0] < 0).sum())
        big = d.layer_forward(0, x, k)
        parts = np.concatenate([d.layer_forward(0, x[i:i + 64], k) for i in range(0, T, 64)])
        assert k == 1 or n_dropped > 0
        assert_rel_l2(big, parts, "adaptive", 3e-4)  # the batches may take GEMMs of 3 or 6 terms: 2^-13 of a block
    finally:
        d.close()


@pytest.mark.parametrize("T,E,k", [(895, 32, 2), (896, 32, 2), (1024, 2, 1), (1025, 2, 1), (2047, 7, 1), (2048, 7, 1), (2049, 7, 1)])
def test_switch_to_the_wide_router(orc, T, E, k):
    """The two routers on either side of a switch give the same bits; for 32 experts, which one ran shows in
    the launches: their grouping does not fit k_route's LDS at this hidden size, so it needs k_bucket
    (kernel 1), which the wide router's own grouping does without."""
    H = 256
    L = syn.make_layer(H, 96, E, seed=830, scale_lo=117, scale_hi=121, router_sigma=0.1)
    d = GpuMoeDispatcher(H, 96, 7.0)
    try:
        d.preload_layer(0, L)
        x = syn.hidden(T, H, seed=831)
        d.set_timing(True)
        d.reset_timing()
        y = d.layer_forward(0, x, k)
        d.synchronize()
        assert d.get_timing(1)[1] == (1 if E == 32 and T < 896 else 0)
        d.set_timing(False)
        want = orc.router_logits(L["router_w"], L["router_b"], x, E, H)
        idx, w, logits = d.router_topk(0, x, k, want_logits=True, n_experts=E)
        assert_bit_exact(logits, want, "router logits (canonical order)")
        widx, ww, _, _ = orc.topk(want, k)
        assert np.array_equal(idx, widx)
        assert_rel_l2(w, ww, "top-k weights", 1e-6)
        assert_rel_l2(y, orc.moe_layer(x, L, k)[0], "layer")
    finally:
        d.close()
