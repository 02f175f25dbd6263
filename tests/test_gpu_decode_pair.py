"""One token through layers whose shared expert is stored in another format than
the routed ones: both sides' gate/up rows in one launch, by the strided and by
the unit-aligned kernel, at one and two units per lane, from the narrowest
experts to a shared expert wider than all the routed ones together, and with
several times more rows than waves in flight, so that the weight rings wrap.

Tolerance: three-level activations carry 24 bits of a block's largest value
and the block dots are exact integers, so TOL (5e-6) is the bar of every
product; the two kernels form the same sums and agree bit for bit."""
import numpy as np
import pytest

from gpu_util import TOL, assert_routing_equal, rel_err, run_gpu

pytestmark = pytest.mark.gpu

Q4_0, Q5_0, Q8_0 = 2, 6, 8


@pytest.mark.parametrize("hidden,inter,shared_inter", [(512, 64, 64), (4160, 128, 128), (2048, 64, 1024), (4160, 2048, 2048),
                                                       (2048, 4096, 4096)])
@pytest.mark.parametrize("dt,shared_dt", [(Q4_0, Q5_0), (Q4_0, Q8_0), (Q5_0, Q4_0), (Q5_0, Q8_0), (Q8_0, Q4_0),
                                          (Q8_0, Q5_0)])
def test_shared_expert_in_another_format(oracle, dt, shared_dt, hidden, inter, shared_inter):
    from moe_amd import _lib as L
    from moe_amd import synth
    from moe_amd.layer import Context

    shape = synth.scaled(synth.SHAPES["qwen2_moe"], hidden=hidden, inter=inter, shared_inter=shared_inter,
                         n_experts=8, expert_dt=dt, shared_dt=shared_dt)
    host = synth.build_host_layer(shape, 5)
    layer = synth.make_layer(Context(0), host)
    x = synth.activations(6, 1, hidden)
    out, sel, w, _, _ = oracle.from_host_layer(host).forward(x)
    got = []
    prev = L.lib().moe_debug_decode_kernel(1)
    try:
        for choice in (1, 2):
            assert L.lib().moe_debug_decode_kernel(choice) >= 0
            layer.set_mode(4)
            assert L.lib().moe_debug_layer_path(layer.handle, 1) == 4
            g = run_gpu(layer, x)
            assert_routing_equal(g, sel, w, f"kernel {choice}")
            assert rel_err(g["out"], out) <= TOL
            got.append(g["out"])
    finally:
        L.lib().moe_debug_decode_kernel(prev)
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
