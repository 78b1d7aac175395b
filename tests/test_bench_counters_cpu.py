"""bench.py uses a committed counter table only beside times of the code it was
taken from, and never reports a share of a peak above 1 (no GPU)."""
import bench

ROWS = """kernel | per_step | avg_us | hbm_MB | valu_issue
k_flux<0, 0> | 3.00 | 1000.0 | 2000.0 | 0.500
k_flux<2, 0> | 1.00 | 2000.0 | 8000.0 | 0.800
k_shock | 1.00 | 500.0 | 1000.0 | 0.100
"""


def table(folder, key):
    (folder / "w_plain_fp64_counters.txt").write_text(ROWS + bench.KEY_LINE + key + "\n")
    return bench.read_counter_summary("w", "plain_fp64", folder)


def test_counters_of_other_code_are_not_used(tmp_path):
    assert bench.read_counter_summary("w", "plain_fp64", tmp_path)[0] is None
    cs, why = table(tmp_path, bench.kernel_key())
    assert why is None and set(cs["rows"]) == {"k_flux<0, 0>", "k_flux<2, 0>", "k_shock"}
    cs, why = table(tmp_path, "0" * 16)
    assert cs is None and "other code" in why
    (tmp_path / "w_plain_fp64_counters.txt").write_text(ROWS)
    cs, why = bench.read_counter_summary("w", "plain_fp64", tmp_path)
    assert cs is None and "other code" in why


def test_key_follows_code_and_not_comments(tmp_path, monkeypatch):
    src = tmp_path / "flash-x_amd" / "csrc"
    src.mkdir(parents=True)
    (tmp_path / "flash-x_amd" / "Makefile").write_text("FLAGS := -O3  # fast\n")
    (src / "a.hip").write_text("int f() { return 1; }  // one\n/* two\n lines */\n")
    monkeypatch.setattr(bench, "ROOT", tmp_path)
    key = bench.kernel_key()
    (src / "a.hip").write_text("int f() {\n  return 1;\n}\n")
    (tmp_path / "flash-x_amd" / "Makefile").write_text("# flags\nFLAGS := -O3\n")
    assert bench.kernel_key() == key
    (src / "a.hip").write_text("int f() { return 2; }\n")
    assert bench.kernel_key() != key
    (src / "a.hip").write_text("int f() { return 1; }\n")
    (tmp_path / "flash-x_amd" / "Makefile").write_text("FLAGS := -O2\n")
    assert bench.kernel_key() != key


def test_shares_above_one_are_not_reported(tmp_path):
    cs, _ = table(tmp_path, bench.kernel_key())
    # 14 GB in 4 launches; 15 GB in all
    got, why = bench.counter_fractions(cs, 1.25e-3, 6e-3)
    assert why is None
    assert abs(got["traffic"] - 3.5e9) < 1.0
    assert abs(got["hbm"] - 3.5e9 / 1.25e-3 / 8e12) < 1e-12
    assert abs(got["path"] - 15e9 / 6e-3 / 8e12) < 1e-12
    assert abs(got["valu"] - (0.5 * 3000 + 0.8 * 2000) / 5000) < 1e-12 and got["column"] == "valu_issue"
    for avg_s, step_s in ((0.4e-3, 6e-3), (1.25e-3, 1.8e-3)):
        got, why = bench.counter_fractions(cs, avg_s, step_s)
        assert set(got.values()) == {None} and "above 1" in why
    assert bench.counter_fractions(None, 1.0, 1.0) == (dict(traffic=None, hbm=None, valu=None, column=None, path=None), None)
