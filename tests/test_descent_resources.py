"""The register budget of the kernel that makes a batch's descents four to a wavefront, on the compiler's own output (no GPU
needed): five of its wavefronts on a SIMD, 20 480 queries a round."""
import shutil

import pytest

from cuhnsw_amd import kernel_report

pytestmark = pytest.mark.skipif(shutil.which(kernel_report.HIPCC) is None, reason="hipcc is not installed")


def test_descents_of_large_batches_keep_five_wavefronts_per_simd():
  report = kernel_report.compile_kernels(kernel_report.DESCENTS)
  assert len(report) == 4
  for name, r in report.items():
    assert r["waves_per_simd"] >= 5 and r["scratch_bytes_per_lane"] == 0, (name, r)
