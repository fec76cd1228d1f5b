"""IVF probe selection on the GPU against the CPU oracle: the centroid store (digits'
exponents and norms) and each query's nprobe nearest cells, bit-exact, ties to the
lower cell id; then search_ivf by nprobe end to end."""
import numpy as np
import pytest
import torch

import oracle
import scratchtape_amd as st
from scratchtape_amd import knn

pytestmark = pytest.mark.gpu
D = 256


def run_probe(dev, cent, queries, nprobe):
    c = knn.Centroids(torch.from_numpy(cent).to(dev))
    got = c.probe(torch.from_numpy(queries).to(dev), nprobe).cpu().numpy()
    return c, got


def test_centroid_store_matches_the_oracle(dev):
    rng = np.random.default_rng(31)
    cent = rng.standard_normal((61, D)).astype(np.float32)  # 61: a partial last block of 8
    cent[0] = 0.0
    cent[1] *= np.float32(2.0 ** -60)
    cent[2] *= np.float32(2.0 ** 60)
    cent[3] = np.where(np.arange(D) < 2, 1.0, 0.0)  # max at the top of the int16 range
    cent[4] = -cent[3]
    c = knn.Centroids(torch.from_numpy(cent).to(dev))
    _, wexp, wnorm = oracle.knn_centroid_prep(cent)
    np.testing.assert_array_equal(c.cexp.cpu().numpy(), wexp)
    np.testing.assert_array_equal(c.cnorm.cpu().numpy(), wnorm)
    assert c.digits.numel() == 8 * 4096


@pytest.mark.parametrize("nlist,nq,nprobe", [(5, 3, 5), (8, 1, 1), (300, 7, 8), (1000, 130, 16), (1537, 64, 3)])
def test_probe_matches_the_oracle(dev, nlist, nq, nprobe):
    rng = np.random.default_rng(nlist * 7 + nq)
    cent = rng.standard_normal((nlist, D)).astype(np.float32)
    queries = rng.standard_normal((nq, D)).astype(np.float32)
    _, got = run_probe(dev, cent, queries, nprobe)
    np.testing.assert_array_equal(got, oracle.knn_probe(cent, queries, nprobe))


# Slices of 2, 4, 6 and 12 tiles of 16 centroids, slot counts around the merge's powers of two (1 to 64, and 65),
# last slices of one tile, one to many query groups.
@pytest.mark.parametrize("nlist,nq", [(16, 70), (33, 5), (130, 3), (1000, 65), (1041, 257), (2048, 3), (2049, 130),
                                      (4090, 40), (4100, 330), (6145, 64), (12480, 64), (12481, 10)])
def test_probe_slices_and_merge_layouts(dev, nlist, nq):
    rng = np.random.default_rng(nlist + nq)
    cent = rng.standard_normal((nlist, D)).astype(np.float32)
    cent[nlist // 2:nlist // 2 + 12] = cent[0]  # ties within and across slices
    queries = rng.standard_normal((nq, D)).astype(np.float32)
    queries[0] = cent[0]
    for nprobe in (1, 7, 16):
        _, got = run_probe(dev, cent, queries, nprobe)
        np.testing.assert_array_equal(got, oracle.knn_probe(cent, queries, nprobe))


# More (slice, query group) pairs than CUs: workgroups that walk several query groups, with last groups and tiles of
# one query, groups that do not divide among them, and 65 slices (the merge's general path).
@pytest.mark.parametrize("nlist,nq", [(1000, 2753), (4100, 777), (12288, 321), (12480, 330)])
def test_probe_workgroups_walk_query_groups(dev, nlist, nq):
    rng = np.random.default_rng(nlist + nq)
    cent = rng.standard_normal((nlist, D)).astype(np.float32)
    cent[nlist // 2:nlist // 2 + 80] = cent[0]  # crowded slots: more than 64 equal candidates
    queries = rng.standard_normal((nq, D)).astype(np.float32)
    queries[0] = queries[nq - 1] = cent[0]
    queries[nq // 2] = 0.0
    for nprobe in (8, 16):
        _, got = run_probe(dev, cent, queries, nprobe)
        np.testing.assert_array_equal(got, oracle.knn_probe(cent, queries, nprobe))


def test_captured_probe_without_room_for_the_query_digits(dev):
    # 2,624 queries of 6 slices leave an arena of 1.25 x 2,624 x 4,632 bytes: room for the candidates of 3,008 queries
    # (more than 256 pairs) but not for their digits, which a capture may not grow the arena for.
    st.lib().st_scratch_release()
    g = torch.Generator(device=dev).manual_seed(9)
    c = knn.Centroids(torch.randn((1000, D), generator=g, device=dev))
    queries = torch.randn((3008, D), generator=g, device=dev)
    c.probe(queries[:2624].contiguous(), 8)
    out = torch.empty((3008, 8), dtype=torch.int32, device=dev)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        c.probe(queries, 8, out=out)
    want = c.probe(queries, 8)  # grows the arena
    for _ in range(3):
        out.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(c.probe(queries, 8), want)
    del graph
    torch.cuda.synchronize()
    st.lib().st_scratch_release()


def test_captured_probe_of_fewer_queries_than_before(dev):
    # 320 queries over 2,048 cells take 32 slices (320 x 32 x 772 bytes of candidates, and a quarter more of arena), 256
    # queries 64 smaller ones (256 x 64 x 772), which a capture has no room for: they take larger slices instead.
    st.lib().st_scratch_release()
    g = torch.Generator(device=dev).manual_seed(10)
    c = knn.Centroids(torch.randn((2048, D), generator=g, device=dev))
    queries = torch.randn((320, D), generator=g, device=dev)
    want = c.probe(queries, 16)
    few = queries[:256].contiguous()
    out = torch.empty((256, 16), dtype=torch.int32, device=dev)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        c.probe(few, 16, out=out)
    for _ in range(3):
        out.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want[:256])
        assert torch.equal(c.probe(few, 16), want[:256])  # eager: grows the arena the first time
    del graph
    torch.cuda.synchronize()
    st.lib().st_scratch_release()


def test_probe_edge_cases(dev):
    rng = np.random.default_rng(32)
    nlist = 200
    cent = rng.standard_normal((nlist, D)).astype(np.float32)
    cent *= np.exp2(rng.integers(-30, 31, nlist)).astype(np.float32)[:, None]  # magnitudes 2^-30 .. 2^30
    cent[10] = 0.0
    cent[77] = cent[12]   # duplicates: equal dd, ties to the lower id
    cent[150] = cent[12]
    queries = rng.standard_normal((40, D)).astype(np.float32)
    queries *= np.exp2(rng.integers(-30, 31, 40)).astype(np.float32)[:, None]
    queries[0] = 0.0                 # ranks by centroid norm
    queries[1] = cent[12]            # the duplicated centroid itself
    queries[2] = cent[33]
    queries[3] = np.float32(1e6) * np.sign(rng.standard_normal(D)).astype(np.float32)
    for nprobe in (1, 4, 16):
        _, got = run_probe(dev, cent, queries, nprobe)
        np.testing.assert_array_equal(got, oracle.knn_probe(cent, queries, nprobe))
    assert list(got[1, :3]) == [12, 77, 150] and got[2, 0] == 33


def test_probe_at_the_benchmark_shape(dev):
    # 12288 cells, 256 queries, 8 probes: the scan benchmark's batch.
    g = torch.Generator(device=dev).manual_seed(5)
    cent = torch.randn((12288, D), generator=g, device=dev)
    queries = torch.randn((256, D), generator=g, device=dev)
    got = knn.Centroids(cent).probe(queries, 8).cpu().numpy()
    np.testing.assert_array_equal(got, oracle.knn_probe(cent.cpu().numpy(), queries.cpu().numpy(), 8))


def test_probe_in_several_query_chunks(dev):
    # 600,000 cells: a dd chunk holds 64 queries, so 130 queries take three chunks.
    g = torch.Generator(device=dev).manual_seed(6)
    nlist = 600_000
    cent = torch.randn((nlist, D), generator=g, device=dev)
    queries = torch.randn((130, D), generator=g, device=dev)
    c = knn.Centroids(cent)
    got = c.probe(queries, 16).cpu().numpy()
    parts = np.concatenate([c.probe(queries[a:b].contiguous(), 16).cpu().numpy() for a, b in ((0, 63), (63, 130))])
    np.testing.assert_array_equal(got, parts)
    sample = [0, 63, 64, 127, 128, 129]  # each side of each chunk boundary, against the oracle
    prep = oracle.knn_centroid_prep(cent.cpu().numpy())
    want = oracle.knn_probe(None, queries.cpu().numpy()[sample], 16, prep=prep)
    np.testing.assert_array_equal(got[sample], want)


def test_search_ivf_by_nprobe_end_to_end(dev):
    rng = np.random.default_rng(33)
    ncells = 48
    sizes = rng.integers(0, 2500, ncells)
    cell_start = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    cent = rng.standard_normal((ncells, D)).astype(np.float32)
    # Keys scattered around their cell's centroid, stored cell-contiguous.
    keys = (np.repeat(cent, sizes, axis=0) + 0.8 * rng.standard_normal((int(cell_start[-1]), D))).astype(np.float32)
    store = knn.KnnStore2bit.from_keys(torch.from_numpy(keys).to(dev), cell_start)
    store.set_centroids(torch.from_numpy(cent).to(dev))
    queries = (cent[rng.integers(0, ncells, 20)] + 0.8 * rng.standard_normal((20, D))).astype(np.float32)
    idx, dist = store.search_ivf(torch.from_numpy(queries).to(dev), 6)
    probes = oracle.knn_probe(cent, queries, 6)
    widx, wdist = oracle.knn_search(store.codes.cpu().numpy(), store.scales.cpu().numpy(), cell_start, queries, probes)
    np.testing.assert_array_equal(idx.cpu().numpy(), widx)
    np.testing.assert_array_equal(dist.cpu().numpy(), wdist)


@pytest.mark.parametrize("case", ["all_equal", "many_equal_nearest", "near_equal_nearest", "one_cell_last_round"])
def test_probe_selection_under_ties_and_round_edges(dev, case):
    # Equal or near-equal distances fill the selection's candidate buffer past one
    # wave (many_equal, near_equal) or past its capacity (all_equal: 3000 candidates);
    # 12289 cells leave one cell for the second round of 12288.
    rng = np.random.default_rng(34)
    nlist = 12289 if case == "one_cell_last_round" else 3000
    cent = rng.standard_normal((nlist, D)).astype(np.float32)
    queries = rng.standard_normal((5, D)).astype(np.float32)
    if case == "all_equal":
        cent[:] = cent[0]
    elif case in ("many_equal_nearest", "near_equal_nearest"):
        idx = rng.choice(nlist, 300, replace=False)
        cent[idx] = queries[0]
        if case == "near_equal_nearest":
            cent[idx] += np.float32(1e-4) * rng.standard_normal((300, D)).astype(np.float32)
    else:
        cent[12288] = queries[1]
    for nprobe in (1, 8, 16):
        _, got = run_probe(dev, cent, queries, nprobe)
        np.testing.assert_array_equal(got, oracle.knn_probe(cent, queries, nprobe))
    if case == "all_equal":
        assert list(got[0]) == list(range(16))
    if case == "one_cell_last_round":
        assert got[1, 0] == 12288


def test_probe_random_indexes(dev):
    # Seeded random indexes: 1..5000 cells, magnitudes 2^-25 .. 2^25 on both sides, duplicated
    # centroids (ties to the lower id), zero queries, nprobe 1..16.
    rng = np.random.default_rng(35)
    for _ in range(8):
        nlist = int(rng.choice([int(rng.integers(1, 100)), int(rng.integers(100, 5000))]))
        nq = int(rng.integers(1, 300))
        nprobe = int(rng.integers(1, min(16, nlist) + 1))
        cent = (rng.standard_normal((nlist, D)) * np.exp2(rng.integers(-25, 26, (nlist, 1)))).astype(np.float32)
        if rng.random() < 0.5:
            cent[rng.integers(0, nlist, max(1, nlist // 10))] = cent[int(rng.integers(0, nlist))]
        queries = (rng.standard_normal((nq, D)) * np.exp2(rng.integers(-25, 26, (nq, 1)))).astype(np.float32)
        queries[0] = 0.0
        _, got = run_probe(dev, cent, queries, nprobe)
        np.testing.assert_array_equal(got, oracle.knn_probe(cent, queries, nprobe))
