"""GPU: what one context's tuning may not decide for another: the form of the
derivative and of the Peierls phase on the grids that have a choice."""
import numpy as np
import pytest

import edus

pytestmark = pytest.mark.gpu

A = np.array([[4.1, 4.1, 0.0], [2.4, -2.4, 0.0], [0.0, 0.0, 20.0]])


def _engine(nb, n, **more):
    rng = np.random.default_rng(nb)
    h = rng.standard_normal((n * n, nb, nb)) + 1j * rng.standard_normal((n * n, nb, nb))
    return edus.Engine(nb, n, n, 0.1 * (h + h.conj().transpose(0, 2, 1)), A=A, filledbands=nb // 2, **more)


@pytest.mark.parametrize("n", [90, 96])
@pytest.mark.parametrize("nb,layout,form", [(9, edus.LAYOUT_FULL, 0), (12, edus.LAYOUT_HERMITIAN, 0),
                                            (10, edus.LAYOUT_FULL, 1), (14, edus.LAYOUT_HERMITIAN, 1)])
def test_phase_form_is_the_peierls_context_s_own(n, nb, layout, form):
    """By its planes (96 and more: one launch), whatever a length-gauge context of
    as many planes was timed to."""
    print("case", n, nb, layout, flush=True)
    length = _engine(nb, n, layout=layout)
    forms = [_engine(nb, n, layout=layout, peierls=True).get_tuning().grad_fused for _ in range(2)]
    assert forms == [form, form]
    t = length.get_tuning()  # and the length-gauge context's choice does not move with it
    assert _engine(nb, n, layout=layout).get_tuning().grad_fused == t.grad_fused


@pytest.mark.parametrize("n,nb", [(120, 3), (96, 5), (48, 7)])
def test_a_group_keeps_its_members_form(n, nb):
    a = _engine(nb, n)
    for form in (0, 1):
        t = a.get_tuning()
        t.grad_fused = form
        a.set_tuning(t)
        assert a.clone().get_tuning().grad_fused == form


@pytest.mark.parametrize("n", [96, 120])
def test_tuning_leaves_no_state(n):
    """A context starts from rho = 0, also where H0 holds a NaN."""
    h = np.zeros((n * n, 2, 2), dtype=complex)
    h[5, 0, 0] = np.nan
    eng = edus.Engine(2, n, n, h, A=A, filledbands=1)
    assert not eng.get_state().any()
