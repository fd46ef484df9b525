"""When the AWQ decoders launch a cached plan (by the shapes the measurements of awq._op_takes_plan name)."""
import pytest

from mpserve_amd.awq import _op_takes_plan


@pytest.mark.parametrize("k,n,m,buckets,rows,group,takes", [
    # whole blocks: always
    (1024, 64, 120, 40, 64, 0, True), (256, 64, 4096, 30, 64, 0, True), (512, 256, 1024, 9, 2048, 128, True),
    # narrow rows: between half as many buckets as CUs and as many
    (512, 1024, 128, 110, 1024, 0, False), (256, 600, 60, 124, 600, 0, False), (256, 1000, 60, 131, 1000, 0, True),
    (256, 4096, 8, 279, 4096, 0, False),
    # blocks of a wide weight are narrow too: 5000 columns in blocks of 40
    (256, 1000, 5000, 100, 1000 * 125, 0, False),
    # flat rows: from 6 elements a substream
    (256, 8, 1500, 8, 8, 0, False), (256, 600, 300, 97, 600, 0, True), (512, 8, 3000, 8, 8, 0, False),
    (512, 40, 3000, 32, 40, 0, True),
    # groups of other sizes
    (1024, 100, 1024, 86, 400, 256, False), (256, 4096, 4096, 407, 262144, 64, True), (256, 100, 1024, 138, 1600, 64, True),
    (256, 8, 1500, 8, 8, 1500, False), (1024, 600, 1500, 71, 600, 1500, True),
    # no slab path
    (1024, 4096, 4096, 400, 524288, 32, False), (300, 4096, 4096, 100, 4096, 0, False), (256, 64, 64, 0, 64, 0, False),
])
def test_rule(k, n, m, buckets, rows, group, takes):
    assert _op_takes_plan(k, n, m, buckets, rows, group, 256) is takes
