"""Which kernels a step launches: the marks of the mixed stage tiles are made
where something reads them, and tile shapes are tuned per stage kernel."""
import json
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def launches():
    r = subprocess.run([sys.executable, os.path.join(os.path.dirname(os.path.abspath(__file__)), "kernel_launches.py")],
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    return json.loads(r.stdout.split("\n")[-2])


@pytest.mark.parametrize("case,marks", [
    ("bubble", 1), ("bubble, one stream", 1),  # the mixed tiles go to the general kernel
    # constant reconstruction: no other kernel, marks for the overlap alone
    ("bubble, constant", 1), ("bubble, constant, one stream", 0),
    ("gas", 0), ("gas, inactive cells", 1), ("gas, inactive cells, constant", 0),
])
def test_marks_of_the_stage_tiles(launches, case, marks):
    n = launches[case]
    assert n.get("k_dt") == 1  # one step was seen
    assert n.get("k_tile_mixed", 0) == marks, n


@pytest.mark.parametrize("case,trials", [("tuned by its like", 0), ("tuned by constant", 16),
                                         ("tuned by characteristic", 16)])
def test_tile_shapes_are_tuned_for_the_kernel_that_runs(launches, case, trials):
    """Four trials of each of the four shapes, then the two stages of a step."""
    assert launches[case]["k_stage_u"] == trials + 2, launches[case]


@pytest.mark.parametrize("way", ["upload", "initialize"])
def test_inactive_cells_that_are_gone_cost_nothing(launches, way):
    """Marks and the general stage kernel while there are inactive cells, and
    neither once the solver's material IDs are set anew without any."""
    n = launches["gas again, " + way]
    assert n["with"]["k_tile_mixed"] == 1 and n["with"]["k_stage"] == n["with"]["k_stage_u"] == 2, n
    assert "k_tile_mixed" not in n["without"] and "k_stage" not in n["without"] and n["without"]["k_stage_u"] == 2, n


@pytest.mark.parametrize("case,copies", [("new materials", 2), ("new materials, roe as well", 1)])
def test_material_tables_are_written_where_they_are_read(launches, case, copies):
    """A new table goes to the translation units whose kernels its solver runs
    (each loads its code at the first write), without a wait in between."""
    n = launches[case]
    assert n.get("hipMemcpyToSymbolAsync", 0) == copies and "hipMemcpyToSymbol" not in n, n
