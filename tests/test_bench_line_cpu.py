"""The benchmark's result line: one JSON line on stdout that a reader of a few
kilobytes can hold, the long tables on stderr."""
import json

import bench


def test_long_tables_go_to_stderr(capsys):
    table = {"S7": {f: {"ms": 0.123456, "within": True} for f in "abcdefghijklmnopqrstuvwxyz"}}
    line = {"metric": "m", "value": 1.5, "config": {"index": "int32"}, "formats": {"CSR": {}},
            "precision_sweep": table, "large_configs": table}
    bench.emit(dict(line))
    out, err = capsys.readouterr()
    assert out.count("\n") == 1 and err.count("\n") == 1
    assert json.loads(out) == {k: line[k] for k in ("metric", "value", "config", "formats")}
    assert json.loads(err) == {"precision_sweep": table, "large_configs": table}


def test_left_out_tables(capsys):
    bench.emit({"metric": "m", "value": 1.5, "precision_sweep": None})
    out, err = capsys.readouterr()
    assert json.loads(out) == {"metric": "m", "value": 1.5, "precision_sweep": None}
    assert err == ""
