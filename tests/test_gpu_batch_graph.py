"""A batch whose captured launches are replayed while the jobs that nucleate
come and go (held, released, finished, removed, admitted): the graph has the
nucleation kernel or not, launches with a due job before and after each change.
Every job gives the bits of the plain path alone."""
import numpy as np
import pytest
import torch

from pfpa import model as M
from pfpa.batch import PF_STORAGE_F32, PF_STORAGE_F64, Batch, make_desc

from test_gpu_batch import NUC_DX, nuc_fields, plain, rand_fields

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", [PF_STORAGE_F64, PF_STORAGE_F32])
@pytest.mark.parametrize("launch_steps", [1, 3])
def test_graph_with_and_without_nucleation(gpu, launch_steps, storage):
    dtype = torch.float64 if storage == PF_STORAGE_F64 else torch.float32
    desc = dict(nucleation=True, seed=77, nuc_every=4, nuc_dx=NUC_DX)
    s, sn = M.make_setup(130, 71, bc=0), M.make_setup(64, 48, bc=1)
    f, fn, fm = rand_fields(130, 71, 0, 1), nuc_fields(64, 48, 1, 7), nuc_fields(64, 48, 1, 8)
    b = Batch(storage, pool_bytes=64 << 20)
    b.set_launch_steps(launch_steps)
    j = b.add(make_desc(s, 1 << 30, instance=1), f)
    jn = b.add(make_desc(sn, 1 << 30, instance=2, **desc), fn)

    def check():
        for k, setup, fields, kw in ((j, s, f, {}),
                                     (jn, sn, fn, dict(nucleation=True, seed=77, nuc_every=4,
                                                       nuc_dx=NUC_DX, instance=2)),
                                     (jm, sn, fm, dict(nucleation=True, seed=77, nuc_every=4,
                                                       nuc_dx=NUC_DX, instance=3))):
            if k is None:
                continue
            got, want = b.read(k), plain(setup, fields, b.poll(k)[0], dtype, **kw)
            for q in range(4):
                assert np.array_equal(got[q].astype(np.float64), want[q]), (k, b.poll(k), q)

    jm = None
    b.run(9, 4)                                  # with: two replays and one launch alone
    check()
    before = b.poll(jn)[0]
    b.hold(jn)
    b.run(8, 4)                                  # without
    assert b.poll(jn)[0] == before
    check()
    b.hold(jn, False)
    b.run(4, 4)                                  # with again
    assert b.poll(jn)[0] > before
    check()
    b.hold(jn)
    jm = b.add(make_desc(sn, 11, instance=3, **desc), fm)   # finishes within the replays
    b.run(12, 4)
    assert b.poll(jm) == (11, False)
    check()
    b.remove(jm)
    jm = None
    b.run(8, 4)                                  # without
    b.hold(jn, False)
    b.run(5, 4)
    check()
    b.close()
