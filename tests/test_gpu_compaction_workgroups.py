"""Lane compaction in workgroups of 256 and 512 lanes (grids that leave CUs
empty in workgroups of 1,024): bit-identical to the uncompacted loop, ragged
last workgroups included."""

import numpy as np
import pytest

from palladium_amd.emit import launch_geometry
from palladium_amd.emit.compact import workgroup_for
from test_gpu_compaction import _collatz

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4096, 4097, 65_536, 65_600, 131_072, 131_073])
def test_every_workgroup_size_equals_the_plain_loop(monkeypatch, n):
    print(f"[compact] n={n}", flush=True)
    rng = np.random.default_rng(n)
    x = rng.integers(1, 200_000, n).astype(np.int32)
    x[::97] = 1
    f = rng.standard_normal(n).astype(np.float32)
    call = _collatz(n)
    bound = call.bound(x, f)
    assert bound.geometry.block == workgroup_for(n) and "__syncthreads" in bound.hip_source
    assert launch_geometry(bound.spec).blocks == -(-n // workgroup_for(n))
    got = call(x, f)
    monkeypatch.setenv("PALLADIUM_WHILE_COMPACTION", "0")
    for g, w in zip(got, _collatz(n)(x, f)):
        np.testing.assert_array_equal(g, w)
