"""The table of tuned options: each operation's best is the fastest of the
rows measured beside it."""
from sable_amd import autotune


def test_best_is_the_fastest_row():
    table = autotune.load_table()
    assert {"spmv", "spmm_n128"} <= set(table)
    for key, entry in table.items():
        row = min(entry["rows"], key=lambda r: r["ms"])
        assert entry["best"] == {k: row[k] for k in entry["best"]}, key
