"""Atom counts past 32-bit indices are an argument error of the pair terms (before any device work)."""

import ctypes

import pytest

from torchff import _lib


@pytest.mark.parametrize("mode", range(6))
def test_too_many_atoms_is_an_argument_error(mode):
    lib = _lib.load(require_gpu=False)
    word = ctypes.c_longlong(0)
    p = ctypes.addressof(word)  # (not read: the count is refused first)
    rc = lib.tff_pair_energy(1, mode, p, 2 ** 31, None, None, 0, None, 0, p, p, p, p, 1, 1.0, 1.0, 1.0, 0, 1.0, p, None,
                             None, None, None, None, p, 8, None)
    assert rc != 0 and b"natoms" in lib.tff_last_error()
