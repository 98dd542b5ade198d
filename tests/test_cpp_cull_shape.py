"""The rule for the flat cull's workgroups (tests/cpp/cull_shape_test.cpp), on the CPU."""
from test_cpp_host import run


def test_workgroup_size_by_rows():
    out = run("cull_shape_test")
    assert "cull shape: 0 failures" in out
