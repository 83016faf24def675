"""Host copies through pinned buffers that an earlier copy of another size made:
every byte arrives, whichever copy came first."""
import numpy as np
import pytest

import oracle as O
import perks_amd as P

pytestmark = pytest.mark.gpu

MIB = 1 << 20


@pytest.mark.parametrize("order", [(8, 36, 9, 100), (35, 8, 30, 37), (100, 30, 8, 36), (30, 31, 16, 8)])
def test_sizes_in_turn(gpu, order):
    P.release()  # the first copy makes the set
    for mib in order:
        cells = mib * MIB // 4 + 3
        print(f"[host-copy] order={order} {mib} MiB", flush=True)
        field = O.uniform(cells, mib, -1.0, 1.0, np.float32).reshape(1, 1, cells)
        got, _ = P.j3d_run(field, 0, method="plain", boundary="zero")
        assert got.tobytes() == field.tobytes()
