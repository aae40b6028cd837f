"""The tuning a context starts with: a wave of the shadow-ray kernel fetches new
rays at 16 idle lanes, and the Python defaults are the library's."""
import pytest

pytestmark = pytest.mark.gpu


def test_defaults():
    import risltc_amd
    ctx = risltc_amd.Context(0)
    try:
        start = ctx.get_tuning().as_dict()
        assert start["trace_refill"] == 16
        ctx.set_tuning(wave_width=64, cull_chunk=5, lds_lights=0, trace_refill=64)
        assert ctx.get_tuning().trace_refill == 64
        ctx.set_tuning()
        assert ctx.get_tuning().as_dict() == start
    finally:
        ctx.close()
