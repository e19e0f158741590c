"""The ABI version goes up with the entry points of include/yee.h: a binding of another version is refused when it loads, so
a declaration added or taken away under the same number would be found by a missing symbol at best."""
from opensol_amd import _lib
from tests.test_abi import declared_functions

# entry points declared at each version whose declarations changed
DECLARED = {19: 20, 20: 22, 21: 24, 22: 25}


def test_version_goes_up_with_the_declared_entry_points():
    assert len(declared_functions()) == DECLARED[_lib.ABI_VERSION]
