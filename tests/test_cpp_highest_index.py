"""The largest delta index of a serving request (tests/cpp/highest_index_test.cpp), on the CPU."""
from test_cpp_host import run


def test_highest_index():
    out = run("highest_index_test")
    assert "highest index: 0 failures" in out
