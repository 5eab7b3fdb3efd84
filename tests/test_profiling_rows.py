"""The byte counts that profiling.py's summary expects of one UPDATE_OLD (12
fields in one dispatch), by the fields' layout (no GPU)."""
import argparse
import os
import sqlite3
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "pllcart3d_amd"))
import profiling  # noqa: E402

COPY = "void pllc::k_copy_pairs<double>(pllc::Dims, pllc::CopyPairs<double>, long)"


def _summary(tmp_path, capsys, fetch, write, **kw):
    con = sqlite3.connect(str(tmp_path / "t.db"))
    con.execute("create table kernels (name text, dispatch_id int, stream_id int, start int, end int)")
    con.execute("insert into kernels values (?, 1, 1, 0, 1000)", (COPY,))
    con.commit()
    con.close()
    for f, c, v in (("f.db", "FETCH_SIZE", fetch), ("w.db", "WRITE_SIZE", write)):
        con = sqlite3.connect(str(tmp_path / f))
        con.execute("create table counters_collection (kernel_name text, dispatch_id int, counter_name text, value real)")
        con.execute("insert into counters_collection values ('k_copy_pairs<double>', 1, ?, ?)", (c, v))
        con.commit()
        con.close()
    profiling.summary(argparse.Namespace(**dict(dict(trace=str(tmp_path / "t.db"), fetch=str(tmp_path / "f.db"),
                                                     write=str(tmp_path / "w.db"), bytes=8, row=None), **kw)))
    return capsys.readouterr().out


def _pitched(nx, ny, row, b):
    """KiB fetched and written for 12 fields whose rows of `row` values start
    with k = 1 on a 128-byte line: whole lines read; written in 32-byte
    pieces, one for k = 0 and those that hold k = 1 .. nz + 1."""
    lines, pieces = -(-row * b // 128), 1 + -(-(row - 1) * b // 32)
    return 12 * nx * ny * lines * 128 / 1024, 12 * nx * ny * pieces * 32 / 1024


@pytest.mark.parametrize("nx, ny, row, b", [(262, 130, 130, 8), (526, 84, 83, 8), (306, 102, 129, 8), (526, 84, 83, 4)])
def test_pitched_rows(tmp_path, capsys, nx, ny, row, b):
    f, w = _pitched(nx, ny, row, b)
    out = _summary(tmp_path, capsys, f, w, points=nx * ny * row, row=row, bytes=b)
    assert "factors are 1.000 (fetch) and 1.000 (write)" in out


def test_packed_fields(tmp_path, capsys):
    """Fewer than 1.5 million points: the fields' own bytes, whatever the row."""
    kib = 12 * 134 * 66 * 66 * 8 / 1024
    out = _summary(tmp_path, capsys, kib, kib, points=134 * 66 * 66, row=66)
    assert "factors are 1.000 (fetch) and 1.000 (write)" in out


def test_row_goes_with_points(tmp_path, capsys):
    f, w = _pitched(262, 130, 130, 8)
    assert "factors are 1.000" in _summary(tmp_path, capsys, f, w, points=262 * 130 * 130)   # the default grid's row
    for kw in (dict(points=526 * 84 * 83), dict(points=526 * 84 * 83, row=130)):
        for g in ("t.db", "f.db", "w.db"):
            os.remove(str(tmp_path / g))
        with pytest.raises(SystemExit):
            _summary(tmp_path, capsys, 1.0, 1.0, **kw)
