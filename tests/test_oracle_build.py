"""The oracle builds where the reference's sources are absent, also when their
directory is there and empty; the reference harness is then left out."""
import oracle as O


def test_oracle_builds_without_reference_sources(tmp_path, monkeypatch):
    monkeypatch.setattr(O, "REFERENCE", str(tmp_path), raising=False)
    O.build()
