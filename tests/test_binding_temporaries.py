"""Host arrays that the binding has to copy for a call (not contiguous) live until the call returns."""
import weakref

import numpy as np
import pytest

import cdns


class Library:
    """Stands for the C library: at each call, are the copies that were made for it still there?"""

    def __init__(self, copies):
        self.copies, self.calls = copies, []

    def __getattr__(self, name):
        def call(*args):
            self.calls.append((name, len(self.copies), [c() is not None for c in self.copies]))
            return 0

        return call


CALLS = {
    "cdns_curl": (lambda ch, v, s, b: ch.curl(v), 1),
    "cdns_cross_product": (lambda ch, v, s, b: ch.cross_product(v, v), 2),
    "cdns_nonlinear_term": (lambda ch, v, s, b: ch.nonlinear_term(v), 1),
    "cdns_solve_modes": (lambda ch, v, s, b: ch.solve_modes(s, b, v, np.zeros((5, 2, 3, 6), np.complex128)[..., ::2]), 4),
}


@pytest.mark.parametrize("name", list(CALLS))
def test_copies_of_strided_arrays_outlive_the_call(monkeypatch, name):
    copies = []
    contiguous = np.ascontiguousarray

    def tracked(a, *more):
        c = contiguous(a, *more)
        if c is not a:
            copies.append(weakref.ref(c))
        return c

    lib = Library(copies)
    monkeypatch.setattr(cdns, "lib", lambda path=None: lib)
    monkeypatch.setattr(cdns.np, "ascontiguousarray", tracked)
    ch = object.__new__(cdns.Channel)
    ch._h, ch.cfg, ch.nzk, ch.nj, ch.nkx = None, {}, 5, 4, 3
    vector = np.zeros((5, 4, 3, 6), np.complex128)[..., ::2]
    scalar = np.zeros((5, 4, 6), np.complex128)[..., ::2]
    boundary = np.zeros((5, 2, 6), np.complex128)[..., ::2]
    call, count = CALLS[name]
    call(ch, vector, scalar, boundary)
    assert [c for c in lib.calls if c[0] == name] == [(name, count, [True] * count)]


def test_arrays_of_a_call_are_freed_with_their_last_reference(monkeypatch):
    """Not by the cycle collector some time later: a restart's arrays are hundreds of megabytes."""
    import gc

    monkeypatch.setattr(cdns, "lib", lambda path=None: Library([]))
    ch = object.__new__(cdns.Channel)
    ch._h, ch.cfg, ch.nzk, ch.nj, ch.nkx = None, {}, 5, 4, 3
    gc.disable()
    try:
        v = np.zeros((5, 4, 3, 3), np.complex128)
        ch.set_state("velocity", v)
        out = ch.get_state("velocity")
        refs = [weakref.ref(v), weakref.ref(out)]
        del v, out
        assert [r() is None for r in refs] == [True, True]
    finally:
        gc.enable()
