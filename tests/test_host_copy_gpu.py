"""Host arrays of the host entry points go to the device and back in pieces of
4 MiB through 4 pinned buffers, from 8 MiB on: every byte arrives at the sizes
around those counts, from pageable and pinned memory, with several callers at
once, and the steps between see the whole field."""
import threading

import numpy as np
import pytest

import oracle as O
import perks_amd as P

pytestmark = pytest.mark.gpu

MIB = 1 << 20


@pytest.mark.parametrize("cells", [8 * MIB // 4 - 1, 8 * MIB // 4, 8 * MIB // 4 + 1, 16 * MIB // 4, 16 * MIB // 4 + 3,
                                   35 * MIB // 4 - 5])
@pytest.mark.parametrize("pinned", [False, True])
def test_bytes_arrive(gpu, cells, pinned):
    torch = gpu
    print(f"[host-copy] cells={cells} pinned={pinned}", flush=True)
    field = O.uniform(cells, 7, -1.0, 1.0, np.float32).reshape(1, 1, cells)
    if pinned:
        field = torch.from_numpy(field).pin_memory().numpy()
    got, _ = P.j3d_run(field, 0, method="plain", boundary="zero")
    assert got.tobytes() == field.tobytes()


def test_callers_at_once(gpu):
    fields = [O.uniform(130 * 200 * 201, 20 + i, -1.0, 1.0, np.float64).reshape(130, 200, 201) for i in range(4)]
    st = O.stencil_from_shape(P.shape_info("3d7pt"), "clamp")
    got = [None] * len(fields)

    def call(i):
        got[i] = P.j3d_run(fields[i], 3, method="plain", boundary="clamp")[0]

    threads = [threading.Thread(target=call, args=(i,)) for i in range(len(fields))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for f, g in zip(fields, got):
        assert g.tobytes() == O.iterate(f, st, 3).tobytes()


def test_release_between_calls(gpu):
    field = O.uniform(9 * MIB // 4, 3, -1.0, 1.0, np.float32).reshape(1, 1, -1)
    for _ in range(2):
        got, _ = P.j3d_run(field, 0, method="plain", boundary="zero")
        assert got.tobytes() == field.tobytes()
        P.release()
