"""The split prefill's partials: no two query tiles of a launch share a region of the workspace, whatever number of
parts each of them has (a tile has a part per key tile where it sees fewer tiles than there are parts)."""
import random


def test_block_sparse_unequal_parts(walk):
    """Query tiles that see fewer key tiles than there are parts beside ones that see more."""
    counts = [[9, 10, 12, 16], [9, 9, 12, 9], [1, 2, 9, 10, 12, 40], [40, 3, 1], [2, 7, 5, 30]]
    got = walk([(16, 2, 32768, 64, 64, c) for c in counts] + [(16, 2, 16384, 150, 2048, c) for c in counts] +
               [(8, 2, 12000, 300, 512, c) for c in counts] + [(4, 1, 60000, 100, 100, c) for c in counts])
    assert got["worst"] == 16 and got["mixed"] >= 15


def test_dense_unequal_parts(walk):
    """Dense prompts from position 0: the first tiles have fewer key tiles than there are parts."""
    got = walk([(2, 2, 0, 3072, 3072, []), (2, 2, 0, 4096, 4096, []), (2, 2, 0, 3500, 8192, []), (1, 1, 0, 8192, 8192, [])])
    assert got["mixed"] == 4


def test_any_launch(walk):
    """Head counts, positions, chunk sizes and visible counts at random, on whole and partitioned CU counts."""
    r = random.Random(7)
    mixed = 0
    for n_cu in (256, 64, 32):
        cases = []
        for _ in range(3000):
            nkv = r.choice([1, 1, 2, 2, 3, 4, 8])
            nh = nkv * r.choice([1, 2, 4, 8, 16])
            n = int(2 ** r.uniform(0, 13.2))
            pos = r.choice([0, int(2 ** r.uniform(0, 18))])
            see = [int(2 ** r.uniform(0, 7)) for _ in range(r.choice([0, 1, 3, 8, 17]))]
            cases.append((nh, nkv, pos, n, r.choice([n, n, max(n, 2048)]), see))
        mixed += walk(cases, n_cu)["mixed"]
    assert mixed > 500
