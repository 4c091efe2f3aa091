"""Which links the drop-in calls bring to the GPU: compat's oe reads even
sites' links only, so a call that keeps nothing brings only those.  Whatever
was brought before, every call uses the caller's links of that call, and the
link cache holds all of them.  Tolerance: FP64, as the hopping tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture
def hp():
    from plqcd_amd import hopping
    yield hopping
    hopping.lib().plqcd_hip_cache_gauge(0)
    hopping.set_mode(hopping.HOP_COMPAT)
    hopping.finalize_plqcd()


@pytest.mark.parametrize("cache", [0, 1])
@pytest.mark.parametrize("mode", [0, 1])
def test_each_call_uses_its_own_links(hp, mode, cache):
    import oracle
    L = (4, 6, 4, 8)
    V = int(np.prod(L))
    hp.init_dims(L)
    hp.set_mode(mode)
    hp.lib().plqcd_hip_cache_gauge(cache)
    q = hp.random_spinor(V, 7)
    half = V // 2
    for turn, calls in enumerate(("oe", "oe eo", "eo oe all", "oe all", "all oe eo")):
        u = hp.random_gauge_su3(V, 20 + turn)  # another field, and with the cache another turn of it
        hp.lib().plqcd_hip_gauge_changed()
        want = oracle.hopping_full(q, u, L, mode)
        for call in calls.split():
            out = hp.spinor_field(V)
            {"eo": hp.hopping_matrix_eo, "oe": hp.hopping_matrix_oe, "all": hp.hopping_matrix}[call](q, out, u)
            part = {"eo": slice(0, half), "oe": slice(half, V), "all": slice(0, V)}[call]
            assert np.abs(out[part] - want[part]).max() < 1e-13 * np.abs(want).max(), (turn, call)


def test_cache_switched_on_after_half_the_links(hp):
    """oe without the cache brings half the links; with the cache switched on
    then, the next calls must not take that half for all of them."""
    import oracle
    L = (4, 4, 6, 4)
    V = int(np.prod(L))
    hp.init_dims(L)
    hp.set_mode(hp.HOP_COMPAT)
    q, u = hp.random_spinor(V, 8), hp.random_gauge_su3(V, 9)
    want = oracle.hopping_full(q, u, L, hp.HOP_COMPAT)
    out = hp.spinor_field(V)
    hp.hopping_matrix_oe(q, out, u)
    hp.lib().plqcd_hip_cache_gauge(1)
    hp.hopping_matrix_oe(q, out, u)
    hp.hopping_matrix_eo(q, out, u)
    assert np.abs(out - want).max() < 1e-13 * np.abs(want).max()
