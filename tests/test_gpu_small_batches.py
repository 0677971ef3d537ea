"""The six-term streamed GEMM that batches of fewer than 4 entries per expert take by default:
against the fp32 oracle and against the per-tile GEMV path (bf16 hi + lo operands) it stands in
for, at the edges of its 8-entry chunks and over ragged shapes."""
import ctypes

import numpy as np
import pytest

from silentotithrandousha_amd import DeviceBuffer, GpuMoeDispatcher
from silentotithrandousha_amd import synthetic as syn
from silentotithrandousha_amd._ffi import check, lib
from tests.helpers import assert_rel_l2, rel_l2

pytestmark = pytest.mark.gpu

# The GEMV's operands are within 2^-17 of each value, the six terms within 2^-28 of each block's
# maximum: their products differ by about 1e-5 relative on these layers, whose pre-activations the
# SwiGLU passes on without the large gains of wider scales.
GEMV_TOL = 4e-5


def _pair(d, x, k):
    got = d.layer_forward(0, x, k)
    d.set_batch_gemm(0)
    ref = d.layer_forward(0, x, k)
    d.set_batch_gemm(1)
    return got, ref


# H, I, E, k, T, router sigma: the forms the rule (fine_ahead) takes: 23 and 24 steps, K not a multiple of
# 128 on either side, the smallest experts, 128 and 256 experts, experts of 1 to 8, 9, 17 and 31 entries (a
# large router spread sends every token to the same experts), the largest average below 4
FINE = [(2880, 2880, 8, 4, 6, 0.1), (3072, 3072, 8, 4, 3, 0.1), (3072, 1056, 8, 1, 31, 0.1), (544, 3072, 8, 1, 31, 0.1),
        (3040, 512, 8, 1, 31, 0.1), (2080, 2432, 16, 2, 12, 0.1), (1024, 1024, 128, 4, 48, 0.1), (352, 3072, 256, 1, 200, 0.1),
        (2304, 2304, 16, 2, 8, 40.0), (2304, 2304, 16, 2, 9, 40.0), (2304, 2304, 16, 2, 17, 40.0), (2304, 2304, 16, 2, 31, 40.0)]
# and forms it leaves to the GEMV: small experts at any count of tokens, few weights in all, K past 3072
GEMV = [(96, 96, 8, 2, 5, 0.1), (64, 64, 8, 4, 3, 0.1), (160, 224, 8, 1, 31, 0.1), (512, 512, 64, 4, 50, 0.1),
        (256, 256, 32, 4, 31, 0.1), (256, 128, 256, 4, 255, 0.1), (2880, 2880, 8, 1, 2, 0.1), (3104, 1056, 8, 1, 31, 0.1)]


@pytest.mark.parametrize("H,I,E,k,T,sigma,fine", [c + (True,) for c in FINE] + [c + (False,) for c in GEMV])
def test_small_batch_matches_oracle_and_gemv(orc, H, I, E, k, T, sigma, fine):
    assert T * k < 4 * E
    L = syn.make_layer(H, I, E, seed=600 + T + H, scale_lo=117, scale_hi=121, router_sigma=sigma)
    d = GpuMoeDispatcher(H, I, 7.0)
    try:
        d.preload_layer(0, L)
        x = syn.hidden(T, H, seed=601 + T)
        if sigma > 1:
            x = x[:1] + 1e-3 * x  # tokens alike: the same experts for all of them
        got, ref = _pair(d, x, k)
        assert np.array_equal(got, ref) != fine  # which of the two ran: their last bits differ
        want, _, idx, _ = orc.moe_layer(x, L, k)
        gidx, _ = d.router_topk(0, x, k)
        assert np.array_equal(gidx, idx)
        if sigma > 1:
            assert np.bincount(idx[idx >= 0].ravel()).max() == T
        e_new, e_gemv = assert_rel_l2(got, want, "default", 2e-5), assert_rel_l2(ref, want, "GEMV", 2e-5)
        print(f"oracle: default {e_new:.2e}, GEMV {e_gemv:.2e}; apart {rel_l2(got, ref):.2e}")
        assert rel_l2(got, ref) < GEMV_TOL
        d.set_local_group(0)  # grouped by the router instead of the GEMM's workgroups
        assert np.array_equal(d.layer_forward(0, x, k), got)
    finally:
        d.close()


def test_small_batch_outliers_and_extremes(orc):
    """Activations that a block scale serves worst: one value of a block a thousand times the rest,
    magnitudes from 2^-100 to 2^60, zero rows, and a non-finite value (NaN in its token alone)."""
    H, I, E, k, T = 3072, 512, 8, 1, 31
    L = syn.make_layer(H, I, E, seed=640, scale_lo=117, scale_hi=121, router_sigma=0.1)
    x = syn.hidden(T, H, seed=641)
    x[0, ::32] *= 1000.0
    x[1] *= np.float32(2.0**-100)
    x[2, :64] *= np.float32(2.0**60)
    x[3] = 0.0
    d = GpuMoeDispatcher(H, I, 7.0)
    try:
        d.preload_layer(0, L)
        got, ref = _pair(d, x, k)
        assert not np.array_equal(got, ref)
        want = orc.moe_layer(x, L, k)[0]
        for t in range(T):
            assert_rel_l2(got[t], want[t], f"token {t}", 2e-5)
            assert rel_l2(got[t], ref[t]) < GEMV_TOL
        x[4, 7] = np.nan
        bad = d.layer_forward(0, x, k)
        assert not np.isfinite(bad[4]).any()
        keep = [t for t in range(T) if t != 4]
        assert np.array_equal(bad[keep], got[keep])
    finally:
        d.close()


@pytest.mark.parametrize("gain", [100.0, 1000.0])
def test_small_batch_values_beside_an_outlier(orc, gain):
    """Every block of x holds one value `gain` times the rest, which no weight reads: the outputs are the
    small values' alone. Within the bound of the bf16 hi + lo operands (2^-17 of each value); terms cut
    at 2^-18 of the block's maximum were 4e-5 and 3e-4 off."""
    H, I, E, k = 3072, 512, 8, 1
    L = syn.make_layer(H, I, E, seed=645, scale_lo=117, scale_hi=121, router_sigma=0.1)
    L["gu_blocks"][..., 0] &= 0xF0  # value 0 of each block of 32
    x = syn.hidden(31, H, seed=646)
    x[:, ::32] *= gain
    d = GpuMoeDispatcher(H, I, 7.0)
    try:
        d.preload_layer(0, L)
        got, ref = _pair(d, x, k)
        want = orc.moe_layer(x, L, k)[0]
        assert not np.array_equal(got, ref)
        assert_rel_l2(ref, want, "GEMV", 8e-6)
        assert_rel_l2(got, want, "six terms", 8e-6)
    finally:
        d.close()


def test_small_batch_adaptive_unaligned_and_replayed(orc):
    """Adaptive top-k's dropped slots; an x that is not 16-byte aligned (the GEMV path); a graph
    captured after one eager call, replayed between eager calls of other sizes."""
    H, I, E = 1024, 1536, 32
    L = syn.make_layer(H, I, E, seed=650, scale_lo=117, scale_hi=121, router_sigma=0.2)
    d = GpuMoeDispatcher(H, I, 7.0)
    try:
        d.preload_layer(0, L)
        x = syn.hidden(20, H, seed=651)
        d.set_adaptive_topk(True, 1, 0.7, 0.4, 0.85)
        want, _, idx, _ = orc.moe_layer(x, L, 4, adaptive=orc.Adaptive(1, 1, 0.7, 0.4, 0.85))
        assert (idx < 0).any()
        got, ref = _pair(d, x, 4)
        assert not np.array_equal(got, ref)
        assert_rel_l2(got, want, "adaptive", 2e-5)
        assert rel_l2(got, ref) < GEMV_TOL
        d.set_adaptive_topk(False)
        d.layer_forward(0, syn.hidden(123, H, seed=652), 4)  # the largest call first: the graph's workspace stays
        eager = d.layer_forward(0, x, 4)
        flat = DeviceBuffer.from_array(np.concatenate([np.zeros(1, np.float32), x.ravel()]))
        y = DeviceBuffer(x.nbytes)
        check(lib().moe_layer_forward_device(d.ctx, 0, ctypes.c_void_p(flat.ptr + 4), 20, 4, ctypes.c_void_p(y.ptr), None))
        d.synchronize()
        d.set_batch_gemm(0)
        assert np.array_equal(y.download(np.float32, x.shape), d.layer_forward(0, x, 4))
        d.set_batch_gemm(1)
        xd, g = DeviceBuffer.from_array(x), ctypes.c_void_p()
        check(lib().moe_graph_begin(d.ctx))
        try:
            d.layer_forward_device(0, xd, 20, 4, y)
        finally:
            check(lib().moe_graph_end(d.ctx, ctypes.byref(g)))
        try:
            for rep in range(3):
                check(lib().moe_memset_device(ctypes.c_void_p(y.ptr), 0xFF, x.nbytes))
                check(lib().moe_graph_launch(d.ctx, g))
                d.synchronize()
                assert np.array_equal(y.download(np.float32, x.shape), eager), f"replay {rep}"
                d.layer_forward(0, syn.hidden(3 + 60 * rep, H, seed=660 + rep), 4)
        finally:
            check(lib().moe_graph_destroy(g))
    finally:
        d.close()


# H: a router of one and of two loads per lane, the runtime chain (2048), padding (H < 64 NQ); T: the
# streamed forms, the wide router (2053 tokens; x at a 4-byte alignment: 8-token blocks with a partial
# one); k: each unrolled combine and the loop
@pytest.mark.parametrize("H,E,k,T", [(96, 8, 1, 5), (544, 8, 2, 40), (2048, 16, 3, 9), (2880, 8, 4, 2053), (1024, 8, 8, 33)])
def test_block_norm_in_router_and_residual_in_combine(orc, H, E, k, T):
    """The batch's block forward gives the same bits as x + layer_forward(oracle RMSNorm(x)), also
    for rows of zeros and of huge values and for x at a 4-byte alignment."""
    L = syn.make_layer(H, 96, E, seed=660 + H, scale_lo=117, scale_hi=121, router_sigma=0.1)
    rng = np.random.default_rng(661)
    gamma = (1 + 0.2 * rng.standard_normal(H)).astype(np.float32)
    d = GpuMoeDispatcher(H, 96, 7.0)
    try:
        d.preload_layer(0, L)
        d.preload_norm(0, gamma, 1e-5)
        x = (3 * syn.hidden(T, H, seed=662)).astype(np.float32)
        x[1], x[2] = 0.0, 1e15 * x[2]
        ref = (x + d.layer_forward(0, orc.rms_norm(x, gamma, 1e-5), k)).astype(np.float32)
        assert np.array_equal(d.block_forward(0, x, k), ref)
        flat, out = DeviceBuffer.from_array(np.concatenate([np.zeros(1, np.float32), x.ravel()])), DeviceBuffer(x.nbytes)
        check(lib().moe_block_forward_device(d.ctx, 0, ctypes.c_void_p(flat.ptr + 4), T, k, ctypes.c_void_p(out.ptr), None))
        d.synchronize()
        assert np.array_equal(out.download(np.float32, x.shape), ref)
    finally:
        d.close()
