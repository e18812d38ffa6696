"""A traffic figure is reported for the kernels that it was measured on and for no others: every source that the device code is made
of counts towards the digest."""
import os
import re

import bench

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cuhnsw_amd", "csrc")
HOST_ONLY = {"index_file.h", "options.h", "host_staging.h"}  # files, options and the pinned blocks


def test_every_source_of_the_device_code_is_in_the_digest():
  seen, todo = set(), ["instances.hip"]
  while todo:
    name = todo.pop()
    if name in seen or name in HOST_ONLY:
      continue
    seen.add(name)
    with open(os.path.join(CSRC, name)) as f:
      todo += re.findall(r'^#include "([^"]+)"', f.read(), re.M)
  assert "kernels.h" in seen and seen == set(bench.KERNEL_SOURCES)
