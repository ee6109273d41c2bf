"""The compiled Python binding against the ctypes one: the same functions,
arguments and statuses, and errors instead of truncated arguments."""

from __future__ import annotations

import pytest

from tensorforge_amd import _native

FAKE = 0x1000  # never dereferenced: every call below fails validation or is empty


def test_binding_functions_are_library_functions_of_the_same_arity():
    binding = _native.launch()
    names = [name for name in dir(binding) if name.startswith("tf_")]
    assert len(names) >= 25 and set(names) <= set(_native.SIGNATURES)
    for name in names:
        with pytest.raises(TypeError, match=f"expected {len(_native.SIGNATURES[name])} arguments"):
            getattr(binding, name)(*[0] * (len(_native.SIGNATURES[name]) + 1))


@pytest.mark.parametrize(("name", "args"), [
    ("tf_linear_kstream", (FAKE, 64, FAKE, 64, FAKE, 64, 65, 64, 64, 2, None)),
    ("tf_linear_kstream", (FAKE, 64, FAKE, 64, FAKE, 64, 0, 64, 64, 2, None)),
    ("tf_rms_norm", (FAKE, FAKE, FAKE, 4, 64, -1.0, 2, None)),
    ("tf_rms_norm", (None, FAKE, FAKE, 4, 64, 1e-5, 2, None)),
    ("tf_argmax_rows", (FAKE, 1 << 40, 0, 64, 2, FAKE, None)),
])
def test_binding_and_ctypes_agree(name, args):
    library = _native.library()
    want = getattr(library, name)(*args)
    message = library.tf_last_error()
    assert getattr(_native.launch(), name)(*args) == want
    assert library.tf_last_error() == message


def test_binding_rejects_values_it_cannot_pass():
    call = _native.launch().tf_argmax_rows
    with pytest.raises(OverflowError):
        call(FAKE, 64, 1 << 33, 64, 2, FAKE, None)
    with pytest.raises(OverflowError):
        call(FAKE, 1 << 70, 1, 64, 2, FAKE, None)
    with pytest.raises(TypeError):
        call("pointer", 64, 1, 64, 2, FAKE, None)
