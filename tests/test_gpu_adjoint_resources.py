"""The kernels that a scene is held to the scratch limits of: those that it launches."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("nder", [1, 2, 3, 4, 8, 16])
def test_the_adjoint_is_checked_at_the_width_it_runs_at(gpu, nder, bits):
    """A forward render runs the scene's own width, the density adjoint that of one lane."""
    f = gpu.lib.dtrt_test_kernel_resources
    f.argtypes = [C.c_int, C.c_int, C.c_char_p, C.c_int, C.c_void_p, C.c_int]
    names, vals = C.create_string_buffer(40 * 32), np.zeros((32, 5), np.uint64)
    n = f(nder, bits, names, 40, vals.ctypes.data, 32)
    assert 0 < n <= 32
    got = {names.raw[i * 40:i * 40 + 40].split(b"\0")[0].decode(): vals[i] for i in range(n)}
    assert len(got) == n
    assert {"k_ad_bounce<%d>" % nder, "k_ad_edges<%d>" % nder, "k_ad_bounce<1>/adjoint", "k_adj_bounce<1>", "k_adj_list<1>"} <= set(got)
    assert [k for k in got if k.startswith("k_adj_")] == [k for k in got if k.startswith("k_adj_") and k.endswith("<1>")]
