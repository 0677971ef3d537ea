"""The per-expert host calls, which run one record without an expert list: over the K splits of the
tile-per-workgroup kernel and on the chunked kernel past it, against the oracle."""
import numpy as np
import pytest

from silentotithrandousha_amd import GpuMoeDispatcher
from silentotithrandousha_amd import synthetic as syn
from tests.helpers import assert_rel_l2

pytestmark = pytest.mark.gpu


# H, I: one block of one step, blocks that end inside a step and inside a scale word, whole words, the
# largest K of the split (3072), K past it
@pytest.mark.parametrize("H,I", [(32, 32), (96, 160), (2880, 2880), (3072, 224), (224, 3072), (3104, 96), (96, 3104), (512, 544)])
def test_one_expert_matches_oracle(orc, H, I):
    L = syn.make_layer(H, I, 3, seed=700 + H + I, scale_lo=117, scale_hi=121, router=False)
    d = GpuMoeDispatcher(H, I, 7.0)
    try:
        d.preload_layer(0, L)
        xs = syn.hidden(3, H, seed=701)
        for e in (2, 0, 1):  # another expert and another x each call
            want = orc.expert_ffn(xs[e], *syn.expert_slice(L, e), H, I)[0]
            got = d.dispatch_expert_preloaded(xs[e], 0, e)
            assert_rel_l2(got, want, f"expert {e}", 2e-5)  # bf16 hi + lo operands: 2^-17 of each value
            assert np.array_equal(d.dispatch_expert(xs[e], *syn.expert_slice(L, e)), got)
    finally:
        d.close()
