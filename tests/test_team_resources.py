"""The register budget of the kernels in which a workgroup of wavefronts takes a query or a node, on the compiler's own output (no GPU
needed): held to so many registers that four teams of four are on a CU (two on long rows and with the largest sets), and spilling
where the row and the set do not fit them -- no more than measured, and in the hop loops only in the widest."""
import shutil

import pytest

from cuhnsw_amd import kernel_report

pytestmark = pytest.mark.skipif(shutil.which(kernel_report.HIPCC) is None, reason="hipcc is not installed")

# kernel -> (wavefronts per SIMD at least, scratch bytes per lane at most, scratch accesses in the hop loops at most)
LIMITS = {
    "search_fast_kernel<dot,1,2,team>": (4, 0, 0),
    "search_fast_kernel<dot,1,5,team>": (4, 0, 0),
    "search_fast_kernel<dot,1,8,team>": (4, 28, 0),
    "search_fast_kernel<l2,2,2,team>": (4, 0, 0),
    "search_fast_kernel<l2,2,5,team>": (4, 0, 0),
    "search_fast_kernel<dot,2,8,team>": (4, 88, 18),
    "search_fast_kernel<l2,4,4,team>": (4, 40, 7),
    "search_fast_kernel<l2,4,8,team>": (4, 120, 51),
    "search_fast_kernel<l2,0,5,team>": (2, 0, 0),
    "search_fast_kernel<l2,0,16,team>": (2, 36, 7),
    "build_search_kernel<dot,1,2,team>": (4, 0, 0),
    "build_search_kernel<dot,2,3,team>": (4, 0, 0),
    "build_search_kernel<l2,2,4,team>": (4, 0, 0),
    "build_search_kernel<l2,4,4,team>": (4, 28, 1),
    "build_search_kernel<l2,0,4,team>": (2, 0, 0),
}


@pytest.fixture(scope="module")
def report():
  return kernel_report.compile_kernels(kernel_report.TEAMS)


@pytest.mark.parametrize("name", sorted(LIMITS))
def test_team_kernel_keeps_its_register_budget(report, name):
  waves, scratch, in_loops = LIMITS[name]
  r = report[name]
  assert r["waves_per_simd"] >= waves, r
  assert r["scratch_bytes_per_lane"] <= scratch, r
  assert r["scratch_instructions_in_hop_loops"] <= in_loops, r


@pytest.mark.parametrize("name", sorted(LIMITS))
def test_rows_of_a_list_are_in_flight_together(report, name):
  assert report[name]["loads_in_turn"] <= 3, report[name]
