"""ParamSpec.apply: the scheme with the parameters' new values."""
import numpy as np
import pytest

from rt_amd import diff, schemes
from rt_amd import scheme as S


def test_apply_sets_every_value_and_nothing_else():
    sch = schemes.echelle(2, 4)
    spec = diff.echelle_design_params(sch)
    v = spec.values(sch) * 1.01 + 1e-3
    got = spec.apply(sch, v)
    assert np.array_equal(spec.values(got), v)
    assert np.array_equal(spec.apply(got, spec.values(sch)).table, sch.table)


def test_apply_counts_surfaces_from_the_end_and_refuses_others():
    sch = schemes.echelle(2, 4)
    n = sch.n_surf
    for s in (0, n - 1, -1, -n):
        assert diff.ParamSpec([diff.Param(s, S.S_DIST)]).apply(sch, [7.5]).surfaces[s].distance[0] == 7.5
    for s in (n, -n - 1, -2 * n):
        with pytest.raises(IndexError):
            diff.ParamSpec([diff.Param(s, S.S_DIST)]).apply(sch, [7.5])
