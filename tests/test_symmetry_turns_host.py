"""Symmetries of scans whose views coincide (several turns, repeated views), as
tests/test_symmetry_host.py checks them for one turn: the permutations of the
views compose as the symmetries do, so that the representatives' classes hold
every view exactly once."""
import numpy as np
import pytest

from test_symmetry_host import apply, scan, tables, turn  # noqa: F401 (tables: fixture)


def turns(n, per_turn):
    return 2 * np.pi * np.arange(n) / per_turn


CASES = {
    # nx, ny, angles, allowed, symmetries
    "2 turns, rectangle": (40, 30, turns(720, 360), 0x55, 4),
    "2 turns, square": (40, 40, turns(720, 360), 0xff, 8),
    "2 turns, linspace": (40, 30, np.linspace(0, 4 * np.pi, 720, endpoint=False), 0x55, 4),
    "3 turns, rectangle": (40, 30, turns(1080, 360), 0x55, 4),
    "3 turns, square": (32, 32, turns(3000, 1000), 0xff, 8),
    "2 turns of an odd count": (32, 31, turns(62, 31), 0x55, 2),
    "3 turns, turned start": (32, 32, 0.37 + turns(180, 60), 0xff, 4),
    "2 turns of 30 + 1/2, square": (32, 32, turns(61, 30.5), 0xff, 2),
    "tiled": (32, 32, np.tile(turn(60), 3), 0xff, 8),
    "repeated": (32, 32, np.repeat(turn(60), 2), 0xff, 8),
    "one turn and a quarter": (32, 32, turns(75, 60), 0xff, None),
    "a turn and its first view twice more": (32, 32, np.r_[turn(60), 2 * np.pi, 4 * np.pi], 0xff, None),
}


@pytest.mark.parametrize("name", list(CASES))
def test_symmetry_tables_of_coincident_views(tables, name):  # noqa: F811
    nx, ny, ang, allowed, want = CASES[name]
    nu = 64
    views = np.array(scan(ang, nu))
    op, rep, rep_view, view, tile, owner = tables(nx, ny, nu, views, allowed)
    nh, n_p = len(op), len(views)
    if want is not None:
        assert nh == want, op
    if nh == 1:
        return
    view, rep_view = view.reshape(n_p, nh), rep_view.reshape(len(rep), nh)
    assert sorted(rep_view[rep_view >= 0]) == list(range(n_p))  # one writer per view
    probe = np.array([1.0, 2.0])
    for i, a in enumerate(op):
        assert sorted(view[:, i]) == list(range(n_p))
        for v in range(n_p):
            assert np.allclose(apply(a, *views[v][:2]), views[view[v, i]][:2], atol=1e-8, rtol=0)
        for j, b in enumerate(op):
            ab = [k for k, c in enumerate(op) if np.allclose(apply(c, *probe), apply(a, *apply(b, *probe)))]
            assert len(ab) == 1
            assert np.array_equal(view[view[:, j], i], view[:, ab[0]]), (a, b)


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_views_that_are_no_numbers_have_no_symmetries(tables, bad):  # noqa: F811
    ang = turn(60)
    views = np.array(scan(ang, 64))
    views[17] = bad
    views[40, 0] = bad
    op, *_ = tables(32, 32, 64, views, 0xff)
    assert list(op) == [0]
