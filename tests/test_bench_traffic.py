"""bench.py's traffic figure: counted on kernels that the library has, with the
template arguments they have, and reported only for the launch it was counted on."""
import glob
import os
import re

import bench
from opesci import compilation


def test_traffic_is_of_kernels_that_exist():
    source = ''.join(open(p).read() for p in sorted(glob.glob(os.path.join(compilation.CSRC, '*.hip'))))
    kernels = {}
    for m in re.finditer(r'template <([^>]*)>\s*__global__ __launch_bounds__\([^;{]*?\) void (\w+)\(', source):
        kernels[m.group(2)] = m.group(1).count(',') + 1
    records = bench.traffic_records()
    assert records
    for rec in records:
        name, args = re.match(r'(\w+)<(.*)>$', rec['kernel']).groups()
        assert kernels.get(name) == args.count(',') + 1, rec


def test_traffic_only_of_the_launch_that_ran():
    default = bench.committed_traffic(bench.workload(256, 4, 'native', False, True))
    assert default > 15 * 4 * 256 ** 3
    assert bench.committed_traffic(bench.workload(256, 4, 'native', True, True)) > 20 * 4 * 256 ** 3
    for other in (bench.workload(256, 4, 'native', False, True, fused=True), bench.workload(256, 4, 'native', False, False, gather=True),
                  bench.workload(255, 4, 'native', False, True), bench.workload(256, 4, 'fp16', False, True)):
        assert bench.committed_traffic(other) is None
