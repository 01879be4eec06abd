"""Jobs of both precisions side by side in a pool too small for all of them: memory one precision's jobs
give back is taken by the other's while both run, and every root is bit for bit the one it has alone."""
import numpy as np
import pytest
import torch

from muscle.serve import LeafBank, Server, tree_nodes
from tests.gpu_util import host
from tests.test_gpu_serve import job_bytes, small_trees

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("room", [1, 4])
def test_shared_pool(room):
    bank = LeafBank(seed=11)
    specs = []
    for s in range(400, 410):
        specs += small_trees([s], dtype="c64" if s % 2 else "c32", n_nodes=(60, 120), size_log2=(6, 15))
    leaves = [bank.leaves(spec, np.random.default_rng(21 + i)) for i, spec in enumerate(specs)]

    def run(srv, jobs):
        ids = [(i, srv.submit_prepared(srv.prepare(leaves[i], tree_nodes(specs[i])))) for i in jobs]
        out = []
        for i, jid in ids:
            assert srv.wait(jid, timeout=120.0)["status"] == 0
            out.append(host(srv.result(jid)))
            srv.release(jid)
        return out

    alone = Server(pool_gib=4)
    want = [run(alone, [i])[0] for i in range(len(specs))]
    alone.close()
    # the tables of a job take less than 4 MB beside its results
    pool = room * max(job_bytes(s) for s in specs) + (4 << 20) * room
    srv = Server(pool_gib=pool / 2**30)
    for _ in range(3):
        for i, got in enumerate(run(srv, range(len(specs)))):
            assert (got == want[i]).all(), i
    torch.cuda.synchronize()
    srv.close()
