"""``default_split_pages``: splits of fewer than 16 pages are few, and rows with
more pages than those splits cover keep the 16-page rule."""
import pytest

from care_kv.attention import default_split_pages


@pytest.mark.parametrize("short_splits", [8, 16])
@pytest.mark.parametrize("rows", [1, 2, 4, 8, 12, 32, 64, 128, 512])
def test_short_splits_are_few(monkeypatch, rows, short_splits):
    monkeypatch.delenv("CAREKV_DECODE_MIN_WGS", raising=False)
    for pages in range(1, 2100):
        sp = default_split_pages(pages, rows, step=4, short_splits=short_splits)
        assert sp % 4 == 0 and 4 <= sp <= 256
        if sp < 16:
            assert -(-pages // sp) <= short_splits, (pages, rows, sp)
        if pages > 12 * short_splits:  # past what the short splits cover, splits are no shorter than 16 pages
            assert 16 <= sp <= default_split_pages(pages, rows), (pages, rows, sp)


def test_step_16_is_unchanged(monkeypatch):
    monkeypatch.delenv("CAREKV_DECODE_MIN_WGS", raising=False)
    for pages in (1, 32, 250, 512, 2048):
        for rows in (1, 4, 32, 256, 1024):
            sp = default_split_pages(pages, rows)
            want = max(16, min(256, -(-pages // 2), pages * rows // 1024))
            assert sp == (want + 15) // 16 * 16 == default_split_pages(pages, rows, short_splits=8)
