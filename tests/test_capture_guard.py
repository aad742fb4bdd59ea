"""No cyclic collection runs inside a graph capture."""
import gc

import pytest

from nv_genai_amd.utils.runtime import capture_guard


@pytest.mark.parametrize("on", [True, False])
def test_no_collection_inside_a_capture(on):
    was = gc.isenabled()
    (gc.enable if on else gc.disable)()
    try:
        with pytest.raises(KeyError), capture_guard():
            assert not gc.isenabled()
            with capture_guard():
                assert not gc.isenabled()
            assert not gc.isenabled()
            raise KeyError
        assert gc.isenabled() == on
    finally:
        (gc.enable if was else gc.disable)()
