"""The callables of csrc/fastcall.c in the place of ctypes functions: every kind of argument arrives as ctypes hands it over, and what they
do not take goes to ctypes (CPU only: the functions that are called are ctypes callbacks)."""
import ctypes as ct
import sysconfig

import numpy as np
import pytest

KIND = {'P': ct.c_void_p, 'i': ct.c_int, 'f': ct.c_float}


# (imported by the tests: a process that loads these libraries before torch, which other files import, has two HIP runtimes)
@pytest.fixture
def cm():
    from deepnet_amd import cudamat
    return cudamat


@pytest.fixture
def fastcall():
    return pytest.importorskip('deepnet_amd._fastcall')


def pair(cm, fastcall, kinds):
    """A fast callable and the ctypes function beside it, both of a callback that notes its arguments."""
    seen = []
    kind = kinds.lstrip('v')
    proto = ct.CFUNCTYPE(None if kinds.startswith('v') else ct.c_int, *[KIND[k] for k in kind])

    def note(*args):
        seen.append(args)
        return None if kinds.startswith('v') else len(seen)
    slow = proto(note)
    return fastcall.Function(ct.cast(slow, ct.c_void_p).value, kinds, (ct.POINTER(cm.cudamat),), slow), slow, seen


def test_arguments_arrive_in_their_places(cm, fastcall):
    from deepnet_amd import cudamat_conv as cc
    letters = {cm._M: 'P', cm._f: 'f', cm._i: 'i', cm._u: 'i'}
    tables = ((cm._cudamat, cm._SIGNATURES), (cc._ConvNet, {n: (None, a) for n, a in cc._SIGNATURES.items()}))
    signatures = {('' if res is not None else 'v') + ''.join(letters[a] for a in args) for lib, table in tables
                  for name, (res, args) in table.items() if isinstance(getattr(lib, name), fastcall.Function)}
    assert len(signatures) > 10
    for kinds in sorted(signatures):
        fast, slow, seen = pair(cm, fastcall, kinds)
        mats = [cm.cudamat() for _ in kinds]
        value = dict(P=lambda j: ct.pointer(mats[j]), i=lambda j: -7 * j - 3, f=lambda j: 0.1 * j + 1e-3)
        args = [value[k](j) for j, k in enumerate(kinds.lstrip('v'))]
        first, second = fast(*args), slow(*args)
        assert (first, second) == ((None, None) if kinds.startswith('v') else (1, 2)), kinds
        assert seen[0] == seen[1] and len(seen[0]) == len(args), kinds


def test_other_arguments_go_to_ctypes(cm, fastcall):
    fast, slow, seen = pair(cm, fastcall, 'PPif')
    mat = cm.cudamat()
    p = ct.pointer(mat)
    for args in ((None, p, 3, 1.5), (ct.byref(mat), p, 3, 1.5), (p, ct.addressof(mat), 3, 2), (p, p, np.int64(4), np.float64(0.5)),
                 (p, p, True, 1.0), (p, p, 2 ** 32 + 5, 1.0), (ct.pointer(cm.rnd_struct()), p, ct.c_int(3), ct.c_float(1.5))):
        del seen[:]
        outcome = []
        for f in (fast, slow):
            try:
                f(*args)
                outcome.append(None)
            except (TypeError, ct.ArgumentError) as e:
                outcome.append(type(e))
        assert outcome[0] == outcome[1] and len(seen) in (0, 2) and seen[:1] == seen[1:], args
    for bad in ((p, p, 3), (p, p, 'x', 1.0), (p, 2.5, 3, 1.0)):
        with pytest.raises((TypeError, ct.ArgumentError)):
            fast(*bad)
    assert fast.argtypes == slow.argtypes and cm._cudamat.dot.argtypes == cm._SIGNATURES['dot'][1]
    with pytest.raises(KeyError):
        fastcall.Function(1, 'ffff', (), slow)


def test_the_module_is_named_for_its_interpreter(fastcall):
    """(another version of Python does not find it, and takes ctypes)"""
    assert fastcall.__file__.endswith('/_fastcall' + sysconfig.get_config_var('EXT_SUFFIX'))


def test_what_ctypes_functions_take_besides_calls(cm, fastcall):
    fast, slow, seen = pair(cm, fastcall, 'Pf')
    assert ct.cast(fast, ct.c_void_p).value == ct.cast(slow, ct.c_void_p).value
    assert fast(None, 1.5) == 1 and fast(None, 1.5) == 2
    fast.errcheck = lambda result, func, args: result + 100          # (what is set, counts from the next call on)
    assert fast(None, 2.5) == 103 and slow(None, 2.5) == 104 and fast.errcheck is slow.errcheck
    assert [s[1] for s in seen] == [1.5, 1.5, 2.5, 2.5]
    del fast.errcheck
    assert fast(None, 2.5) == 5
    with pytest.raises(TypeError):
        fast.argtypes = 3
