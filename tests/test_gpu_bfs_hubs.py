"""BFS drivers on graphs whose vertices' degrees lie around the sizes where
the kernels split a vertex's neighbours (first neighbours of a row, work
items of a hub), against the CPU BFS."""
import numpy as np
import pytest

import oracle
import spmspv_amd as sa

pytestmark = pytest.mark.gpu


def hub_graph(n, hub_degrees, seed):
    """Symmetric CSR of n vertices: vertex i < len(hub_degrees) is joined to
    hub_degrees[i] random others, and a path joins half of the vertices."""
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    r, c = [], []
    for i, d in enumerate(hub_degrees):
        others = rng.choice(np.arange(len(hub_degrees), n), size=d, replace=False)
        r += [i] * d
        c += others.tolist()
    path = rng.permutation(n)[: n // 2]
    r += path[:-1].tolist()
    c += path[1:].tolist()
    A = sp.csr_matrix((np.ones(len(r), np.float32), (r, c)), shape=(n, n))
    A = ((A + A.T) > 0).astype(np.float32).tocsr()
    A.sort_indices()
    return A


@pytest.mark.parametrize("nsrc", [3, 64])
@pytest.mark.parametrize("hubs", [(7, 8, 9, 263, 264, 265), (255, 256, 257, 520, 4000), (1,)])
def test_bfs_multi_hub_degrees(gpu, hubs, nsrc):
    n = 5003
    A = hub_graph(n, hubs, len(hubs))
    M = sa.Matrix(n, n, A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data)
    cp, ri, _ = oracle.csr_to_csc(n, n, A.indptr, A.indices, A.data)
    srcs = np.random.default_rng(nsrc).integers(0, n, nsrc).astype(np.int32)
    srcs[0] = 0
    lev = sa.DeviceArray(n * nsrc, np.int32)
    for _ in range(2):  # the second call finds the first one's state
        M.A.bfs_multi(srcs, lev)
        got = lev.to_host().reshape(n, nsrc)
        for i, s in enumerate(srcs):
            ref, _ = oracle.bfs(n, cp, ri, int(s))
            np.testing.assert_array_equal(got[:, i], ref, err_msg=f"source {s}")


@pytest.mark.parametrize("graphs", [0, 1])
@pytest.mark.parametrize("policy", [0, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("n,hubs", [(5003, (7, 8, 9, 263, 264, 265)), (40961, (255, 256, 257, 520, 30000))])
def test_bfs_hub_degrees(gpu, n, hubs, policy, graphs):
    A = hub_graph(n, hubs, len(hubs))
    M = sa.Matrix(n, n, A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data)
    cp, ri, _ = oracle.csr_to_csc(n, n, A.indptr, A.indices, A.data)
    lev = sa.DeviceArray(n, np.int32)
    for src in (0, len(hubs) - 1, n - 1):
        st = M.A.bfs(src, lev, policy=policy, use_graphs=graphs)
        ref, _ = oracle.bfs(n, cp, ri, src)
        np.testing.assert_array_equal(lev.to_host(), ref)
        assert int(st[3]) == int((ref >= 0).sum())
