"""The build entry point on hosts without the reference's sources: an absent or
an empty reference directory builds the library and skips the host oracle."""
import __graft_entry__ as entry


def test_reference_sources(tmp_path):
    assert not entry.reference_sources(tmp_path / "absent")
    assert not entry.reference_sources(tmp_path)
    (tmp_path / "src").mkdir()
    assert not entry.reference_sources(tmp_path)
    (tmp_path / "src" / "host_reference.hpp").write_text("")
    assert entry.reference_sources(tmp_path)
