"""Batched binary (Hamming) searches, the matrix-core scan, against the CPU oracle: ids and
scores bit-exact under the lowest-index tie-break.

Batches of 4 or more queries over 512- or 1024-dim sign-packed rows take the MFMA scans: up to 64
queries the stream kernel, once per set of 32, and more the tile kernel. The cases cover both row
sizes on both kernels, partial query groups and sets (17, 33, 100), a batch over two launches (130),
k from 1 to 1000 (Hamming scores tie massively at the k-th place), a partial last tile, queries
whose bits are all clear or all set, and duplicated rows."""

import numpy as np
import pytest

import oracle
from helpers import assert_topk_equivalent, normalized

pytestmark = pytest.mark.gpu


def search(capi, words, dim, queries, k):
    n = words.shape[0]
    store = capi.store_desc(capi.DeviceArray.from_host(words), n, dim, capi.BINARY)
    desc = capi.search_desc(store, capi.DeviceArray.from_host(queries), queries.shape[0], k)
    idx, val, flags = capi.search(desc)
    assert not flags.any(), "candidate overflow on a random corpus"
    return idx, val


@pytest.mark.parametrize("n,dim,batch,k", [
    (70_001, 512, 4, 10),
    (70_001, 512, 33, 100),
    (70_001, 512, 100, 10),      # the tile kernel at 512 bits
    (70_001, 1024, 17, 1),
    (120_007, 1024, 32, 10),
    (120_007, 1024, 100, 100),
    (60_013, 1024, 130, 10),
    (60_013, 1024, 32, 1000),
])
def test_batched_hamming_bit_exact(gpu, n, dim, batch, k):
    capi = gpu
    corpus = normalized(n, dim, 300 + batch)
    queries = normalized(batch, dim, 400 + batch)
    words = oracle.pack_binary(corpus)
    idx, val = search(capi, words, dim, queries, k)
    ref = oracle.scores_hamming(words, oracle.pack_binary(queries), dim)
    assert_topk_equivalent(idx, val, ref, k)


def test_batched_hamming_extreme_queries_and_duplicates(gpu):
    capi = gpu
    n, dim, k = 50_000, 1024, 64
    base = normalized(700, dim, 11)
    corpus = base[np.arange(n) % 700]  # 700 classes of identical rows
    queries = normalized(8, dim, 12)
    queries[0] = 1.0   # every bit set
    queries[1] = -1.0  # every bit clear
    queries[2] = -queries[3]  # complementary pair
    words = oracle.pack_binary(corpus)
    idx, val = search(capi, words, dim, queries, k)
    ref = oracle.scores_hamming(words, oracle.pack_binary(queries), dim)
    assert_topk_equivalent(idx, val, ref, k)


# rows of 32, 48 and 96 bytes: words read past chunk boundaries, a last copy of half a kilobyte (384
# bits); the dense, threshold and (2,000,003 rows) sketch phases, streamed and on the tile kernel
@pytest.mark.parametrize("n,dim,batch,k", [
    (3_001, 256, 4, 10),
    (70_001, 256, 17, 100),
    (70_001, 256, 100, 10),
    (70_001, 384, 4, 10),
    (120_007, 384, 33, 100),
    (60_013, 768, 32, 1000),
    (120_007, 768, 130, 10),
    (2_000_003, 768, 20, 100),
    (8_000_003, 384, 5, 10),
])
def test_short_rows_bit_exact(gpu, n, dim, batch, k):
    capi = gpu
    rng = np.random.default_rng(dim + batch)
    words = rng.integers(0, 2**32, (n, dim // 32), dtype=np.uint32)
    words[n // 3] = words[7]  # a tie across the corpus
    queries = normalized(batch, dim, 900 + dim)
    qbits = oracle.pack_binary(queries)
    words[n - 1] = qbits[0]  # the best row is the last one
    d_words, d_queries = capi.DeviceArray.from_host(words), capi.DeviceArray.from_host(queries)
    desc = capi.search_desc(capi.store_desc(d_words, n, dim, capi.BINARY), d_queries, batch, k, capi.COSINE)
    idx, val, flags = capi.search(desc)
    assert not flags.any()
    for first in range(0, batch, 16):  # (the oracle's scores of 8M rows a few queries at a time)
        part = slice(first, first + 16)
        ref_idx, ref_val = oracle.topk(oracle.scores_hamming(words, qbits[part], dim), k)
        assert np.array_equal(idx[part], ref_idx) and np.array_equal(val[part], ref_val)
