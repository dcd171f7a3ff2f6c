"""Whether a built library is taken for one of the sources as they are."""
import __graft_entry__ as ge
import pytest


def test_library_built_with_other_flags_is_refused(monkeypatch):
    """Packed FP32 instructions allowed, or accumulators elsewhere: another library from the same sources."""
    built = ge.source_hash()
    for left_out in ("-packed-fp32-ops", "-amdgpu-mfma-vgpr-form=1"):
        with monkeypatch.context() as m:
            m.setattr(ge, "HIPCC_FLAGS", [f for f in ge.HIPCC_FLAGS if f != left_out])
            assert ge.source_hash() != built
            with pytest.raises(RuntimeError, match="not built from the current sources"):
                ge.check_built()
