"""Format descriptors as objects: copies, pickles and their C struct."""
import copy
import pickle

import pytest

import lofloat_amd as lof


class Named(lof.FloatFormatDescriptor):
    """A subclass with attributes and a slot of its own."""
    __slots__ = ("family", "__dict__")


def _named():
    f = Named(8, 3, 7, lof.InfBehavior(1), lof.NaNBehavior(0), lof.Signedness(0),
              lof.formats.P3109_InfChecker(8), lof.formats.P3109_NaNChecker(8))
    f.family, f.note = "e4m3", "weights"
    return f


@pytest.mark.parametrize("used", [False, True])
@pytest.mark.parametrize("clone", [copy.copy, copy.deepcopy,
                                   lambda f: pickle.loads(pickle.dumps(f))],
                         ids=["copy", "deepcopy", "pickle"])
def test_copies_keep_a_subclasss_attributes(clone, used):
    f = _named()
    if used:
        f.c_format()
    g = clone(f)
    assert type(g) is Named and g.as_tuple() == f.as_tuple()
    assert (g.family, g.note) == ("e4m3", "weights")
    assert bytes(g.c_format()) == bytes(f.c_format())


def test_a_changed_c_struct_changes_no_format():
    f = _named()
    for c in (f.c_format(), lof.AccumSpec(fmt=f).c_accum().fmt):
        c.bias = 3
    assert f.bias == f.c_format().bias == lof.AccumSpec(fmt=f).c_accum().fmt.bias == 7
