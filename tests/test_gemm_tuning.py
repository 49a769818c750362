"""Saved tile tables across builds (no GPU needed)."""
import quantit_amd as qa


def test_numbers_that_changed_their_kernel_are_timed_anew(tmp_path):
    old = tmp_path / "old.json"
    old.write_text('{"gemm_variants": {\n  "f64 old a": 0,\n  "f64 old b": 5,\n  "f64 old c": 1,\n  "f64 old d": 3\n}}\n')
    qa.gemm_tuning_load(old)
    out = tmp_path / "out.json"
    qa.gemm_tuning_save(out)
    text = out.read_text()
    assert '"f64 old c": 1' in text and '"f64 old d": 3' in text
    assert "f64 old a" not in text and "f64 old b" not in text


def test_a_table_of_this_build_comes_back(tmp_path):
    mine, out = tmp_path / "mine.json", tmp_path / "out.json"
    mine.write_text('{"tiles": [64, 32], "gemm_variants": {\n  "f64 new a": 5,\n  "f64 new b": 0\n}}\n')
    qa.gemm_tuning_load(mine)
    for _ in range(2):
        qa.gemm_tuning_save(out)
        assert out.read_text().startswith('{"tiles": [64, 32], "gemm_variants": {')
        assert '"f64 new a": 5' in out.read_text() and '"f64 new b": 0' in out.read_text()
        qa.gemm_tuning_load(out)
