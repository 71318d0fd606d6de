"""Tests against the reference's own transport are skipped, with the reason,
where it is not built and cannot be; a tree that has its sources says what to
run."""
import pytest

import refbind as rb


def test_missing_reference(tmp_path, monkeypatch):
    monkeypatch.setattr(rb, "REF_DIR", str(tmp_path))
    monkeypatch.setattr(rb, "_libs", {})
    monkeypatch.setattr(rb, "REF_SOURCES", str(tmp_path / "none"), raising=False)
    for debug in (True, False):
        with pytest.raises(pytest.skip.Exception, match="no reference sources"):
            rb.reference(debug)
    (tmp_path / "src" / "moqui").mkdir(parents=True)
    monkeypatch.setattr(rb, "REF_SOURCES", str(tmp_path / "src"), raising=False)
    for debug in (True, False):
        with pytest.raises(FileNotFoundError, match="make -C oracle"):
            rb.reference(debug)
    with pytest.raises(FileNotFoundError):   # the oracle's sources are in the tree
        rb.oracle()
