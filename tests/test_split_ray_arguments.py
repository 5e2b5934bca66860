"""lts_trace_rays_split checks its arguments before any HIP call, as lts_trace_rays does."""
import ctypes

import pytest

from test_capi_null_arguments import LTS_E_ARG, lib  # noqa: F401  (fixture)

P = ctypes.c_void_p(16)  # never dereferenced


@pytest.mark.parametrize("args", [(None, None, None, 4, None, None), (None, P, None, 4, P, P), (None, None, P, 4, P, P),
                                  (None, P, P, -1, P, P), (None, P, P, (1 << 26) + 1, P, P), (None, P, P, 4, None, P)])
def test_bad_arguments_are_refused(lib, args):  # noqa: F811
    assert lib.lts_trace_rays_split(*args) == LTS_E_ARG
    assert lib.lts_last_error(None) == b"bad trace_rays arguments"
