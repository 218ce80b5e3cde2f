"""The fingerprint of an integrand's owner while another thread gives the owner
an attribute (its first call does): here the attribute name does it, at the
moment it is looked at."""
from tensormesh_amd.forms import _owner_key


class Name(str):
    """An attribute name whose inspection adds an attribute to its owner."""

    def startswith(self, *args):
        self.owner.__dict__["_added"] = 1
        return super().startswith(*args)


class Owner:
    pass


def test_an_attribute_added_meanwhile():
    o = Owner()
    o.E = 2.0
    want = _owner_key(o, 0, set())
    o = Owner()
    name = Name("E")
    name.owner = o
    o.__dict__[name] = 2.0
    assert _owner_key(o, 0, set()) == want
    assert o._added == 1 and _owner_key(o, 0, set()) == want
