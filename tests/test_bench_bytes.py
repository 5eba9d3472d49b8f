"""The bytes that bench.py counts for a stage: what its kernels move once."""
import importlib.util
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _bench():
    spec = importlib.util.spec_from_file_location("bench_module", os.path.join(ROOT, "bench.py"))
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


def test_pair_search_reads_records_and_table():
    """Key and record of every particle, the cell table, and no candidate array."""
    b = _bench()
    assert b.stage_bytes("candidates", 1000, 64, 4096, 3) == 20 * 1000 + 4 * 4097
    assert b.stage_bytes("candidates", 1000, 64, 0, 3, True, "bins") == 20 * 1000 + 4
