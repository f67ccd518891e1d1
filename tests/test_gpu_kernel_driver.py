"""The profiling driver runs what the dispatcher launches, and names it."""

import pytest

from flashlite_amd import kernel_driver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("args,name", [
    (["--shape", "2", "8", "512"], "br32_rows"),
    (["--shape", "2", "8", "512", "--config", "6"], "br32_kv512_w4_quarters"),
    (["--shape", "2", "8", "333", "--dtype", "bf16", "--head-dim", "128"], "br32_rows"),
    (["--shape", "2", "8", "4096"], "br256_bc64_w8_slot"),
])
def test_names_what_it_launches(cuda, capsys, args, name):
    kernel_driver.main(args + ["--iters", "2"])
    assert f" {name}" in capsys.readouterr().out
