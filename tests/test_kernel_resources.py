"""The register budget of the first-pass search kernels, checked on the compiler's own output (no GPU needed).

The sorted-set search is held to a fixed number of wavefronts per SIMD and runs 7 to 12 % slower when the register
allocator reloads a spilled register inside its hop loop; small source changes anywhere in the kernel decide that.
So every change is checked here: wavefronts per SIMD, scratch bytes per lane, and scratch-memory instructions inside
the hop loops (the innermost loops that hold both the sorted-set insert and a fetch from global memory)."""
import shutil

import pytest

from cuhnsw_amd import kernel_report

pytestmark = pytest.mark.skipif(shutil.which(kernel_report.HIPCC) is None, reason="hipcc is not installed")

# kernel -> (wavefronts per SIMD at least, scratch bytes per lane at most, scratch accesses in the hop loops at most: none)
LIMITS = {
    "search_fast_kernel<dot,1,5>": (7, 68),
    "search_fast_kernel<dot,1,5,trails>": (7, 56),
    "search_fast_kernel<l2,1,5>": (7, 60),
    "search_fast_kernel<dot,2,5>": (7, 60),
    "search_fast_kernel<l2,2,5>": (7, 88),
    "search_fast_kernel<l2,2,5,trails>": (7, 76),
    "search_fast_kernel<dot,1,2>": (7, 0),
    "search_fast_kernel<dot,2,8>": (5, 36),
    "search_fast_kernel<dot,2,2>": (7, 20),
    "search_fast_kernel<l2,2,2>": (7, 20),
    # (a wavefront with a SIMD to itself: nothing spills, however wide the instance)
    "search_fast_kernel<dot,1,5,few>": (1, 0),
    "search_fast_kernel<l2,2,2,few>": (1, 0),
    "search_fast_kernel<l2,0,5,few>": (1, 0),
    "search_fast_kernel<l2,4,5>": (5, 20),
    "search_fast_kernel<l2,0,7,few>": (1, 0),
    "search_fast_kernel<dot,0,8,few>": (1, 0),
    # the other sizes of the set
    "search_fast_kernel<dot,1,3>": (7, 0),
    "search_fast_kernel<dot,1,4>": (7, 36),
    "search_fast_kernel<dot,2,4>": (7, 20),
    "search_fast_kernel<l2,2,3>": (7, 20),
    "search_fast_kernel<l2,2,4>": (7, 36),
    "search_fast_kernel<l2,2,4,trails>": (7, 24),
    "search_fast_kernel<dot,1,6>": (6, 36),
    "search_fast_kernel<l2,1,6>": (7, 48),
    "search_fast_kernel<dot,2,6>": (7, 60, 7),  # (a few reloads in the loop, and still faster than six wavefronts)
    "search_fast_kernel<l2,2,6>": (7, 44),
    "search_fast_kernel<l2,2,6,trails>": (6, 20),
    "search_fast_kernel<dot,1,7>": (5, 0),
    "search_fast_kernel<l2,2,7>": (5, 0),
    "search_fast_kernel<dot,2,4,few>": (1, 0),
    "search_fast_kernel<l2,0,6,few>": (1, 0),
}


@pytest.fixture(scope="module")
def report():
  return kernel_report.compile_kernels(kernel_report.FIRST_PASS)


@pytest.mark.parametrize("name", sorted(LIMITS))
def test_first_pass_kernel_keeps_its_register_budget(report, name):
  waves, scratch, in_loops = (LIMITS[name] + (0,))[:3]
  r = report[name]
  assert r["waves_per_simd"] >= waves, r
  assert r["scratch_bytes_per_lane"] <= scratch, r
  assert r["scratch_instructions_in_hop_loops"] <= in_loops, r


@pytest.mark.parametrize("name", sorted(n for n in LIMITS if "few" in n))
def test_rows_are_in_flight_together(report, name):
  """A wavefront with a SIMD to itself has nobody to wait for its loads beside: the rows of a distance pass, fp16 included,
  are asked for before the first of them is waited for (each in turn, and a search takes twice its time)."""
  assert report[name]["loads_in_turn"] <= 2, report[name]


def test_loop_analysis_sees_a_spill_inside_a_loop():
  """The control-flow analysis itself, on a hand-written listing: a query loop around a hop loop that holds a
  fetch and the insert; the scratch access in the hop loop counts, the ones outside it do not."""
  isa = """
kern:
  s_mov_b32 s0, 0
.LBB0_1:
  scratch_load_dword v1, off, off
  s_cbranch_scc1 .LBB0_5
.LBB0_2:
  global_load_dword v5, v[6:7], off
  v_med3_f32 v0, v1, v2, v3
  s_cbranch_vccz .LBB0_4
.LBB0_3:
  scratch_load_dword v2, off, off offset:4
.LBB0_4:
  s_cbranch_scc0 .LBB0_2
.LBB0_5:
  scratch_store_dword off, v1, off
  s_cbranch_scc0 .LBB0_1
.LBB0_6:
  s_endpgm
.Lfunc_end0:
"""
  assert kernel_report.loop_scratch_accesses(isa, "kern") == (1, 3)
  # a loop over rows inside the hop loop, which bounds their keys: not an insert, the hop loop is still the one around it
  rows = """  s_cbranch_vccz .LBB0_4
.LBB0_31:
  global_load_dwordx4 v[8:11], v[6:7], off
  v_med3_f32 v0, v1, -s2, s2
  s_cbranch_scc1 .LBB0_31
"""
  assert kernel_report.loop_scratch_accesses(isa.replace("  s_cbranch_vccz .LBB0_4\n", rows), "kern") == (1, 3)
