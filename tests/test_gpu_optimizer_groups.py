"""The optimizer's tied groups at the edges of a wavefront: 1, 63, 64, 65 and 200 entries."""
import numpy as np
import pytest

import oracle
from heliox_amd import Sim, build_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [1, 63, 64, 65, 200])
def test_adam_group_sizes(gpu_lib, size):
    print(f"case adam group of {size}", flush=True)
    spec = build_config(5, 2, 5.0)
    g = Sim()
    g.load_model_from_spec(spec, add_monitors=False)
    g.tape_begin(100)
    g.finitialize(-65.0)
    g.run(100.25 * spec.dt)
    g.adjoint(np.arange(2), np.full((100, 2), -60.0))
    grad, w0 = g.gradient("pas", "g_pas"), g.get_array("pas", "g_pas").copy()
    opt = g.adam_create(0.9, 0.999, 1e-8)
    groups = [np.arange(3, 3 + size), np.arange(300, 300 + size)]
    for inst in groups:
        g.adam_add_group(opt, "pas", "g_pas", inst)
    g.adam_step(opt, 1e-6, 1.0)
    w1 = g.get_array("pas", "g_pas")
    ww, m, v = np.array([w0[i[0]] for i in groups]), np.zeros(2), np.zeros(2)
    oracle.adam_step(ww, np.concatenate([grad[i] for i in groups]), np.full(2, size, np.int32), m, v, 1, 1e-6, 1.0)
    for k, inst in enumerate(groups):
        assert np.allclose(w1[inst], ww[k], rtol=1e-14, atol=0)
    assert np.array_equal(np.delete(w1, np.concatenate(groups)), np.delete(w0, np.concatenate(groups)))
    _, mg, vg = g.adam_state(opt, 2)
    assert np.allclose(mg, m, rtol=1e-14, atol=0) and np.allclose(vg, v, rtol=1e-14, atol=0)
    left = g.gradient("pas", "g_pas")
    assert np.all(left[np.concatenate(groups)] == 0.0)
