"""The upper refit passes on lists that do not fit their LDS copy (2560 nodes),
bit-exact against the CPU oracle.  Spheres are placed by their Morton codes so
that deep chains of nodes cross the border of every 512-leaf chunk (the list of
a 65,536-leaf span) or of every span (the list of the top pass); the test
counts the nodes of those lists in the oracle's tree."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests.test_gpu_lbvh import check_equal, gpu_build, oracle_build
from visrtx_amd import _native as N

CHUNK, SPAN, LIST, LEAF = 512, 1 << 16, 2560, 0x80000000


def _centres(codes):
    """Points whose 10-bit grid cells have these Morton codes, where the
    scene's centroids span [0, 1]^3."""
    q = np.zeros((3, len(codes)), np.uint32)
    for b in range(10):
        for a in range(3):
            q[a] |= ((codes >> np.uint32(3 * b + 2 - a)) & np.uint32(1)) << np.uint32(b)
    return ((q.T.astype(np.float32) + np.float32(0.5)) / np.float32(1024)).astype(np.float32)


def _chained(step, chains):
    """Spheres with a chain of chains[j - 1] nodes across the border before
    sorted leaf j * step: the codes P, P ^ 1, P ^ 2, P ^ 4, ... of the j-th of
    128 cells, P last before the border; copies of the cell's largest code fill
    up to the next border."""
    pattern = 0b01010101010101010101010

    def cell(j):
        bits = 1 << np.arange(chains[j - 1], dtype=np.int64)
        p = (j << 23) | pattern
        return np.sort(np.concatenate([[p], p ^ bits])), p

    parts, at = [], 0
    for j in range(1, len(chains) + 1):
        codes, p = cell(j)
        below = int((codes <= p).sum())
        fill = j * step - below - at
        assert fill >= 0
        parts += [np.full(fill, parts[-1][-1] if parts else 0), codes]
        at += fill + len(codes)
    n = (len(chains) + 1) * step
    parts.append(np.full(n - 1 - at, parts[-1][-1]))
    codes = np.concatenate(parts).astype(np.uint32)
    c = np.concatenate([_centres(codes), np.ones((1, 3), np.float32)])
    c[0] = 0.0      # with the last one: the corners of the code space
    rng = np.random.default_rng(len(chains))
    r = (rng.integers(1, 64, n) / np.float32(1 << 14)).astype(np.float32)
    order = rng.permutation(n)
    return c[order], r[order]


def _crossing(child, first, step, borders):
    """Nodes of the tree whose leaves lie on both sides of a border (leaf
    first + k * step, k = 1 .. borders)."""
    seen = set()
    for k in range(1, borders + 1):
        b, node = first + k * step, 0
        while True:
            seen.add(node)
            left, right = (int(x) for x in child[node])
            gamma = left & ~LEAF    # the last leaf of the left child
            if b - 1 == gamma:
                break
            node = left if b <= gamma else right
    return seen


def _build(step, chains, limit_pass):
    c, r = _chained(step, chains)
    o = oracle_build(orc.ORC_SPHERE, c, radius=r)
    n = len(c)
    top = _crossing(o["child"], 0, SPAN, (n - 1) // SPAN)
    if limit_pass == "top":
        return c, r, o, len(top)
    inner = _crossing(o["child"], 0, CHUNK, SPAN // CHUNK - 1)
    return c, r, o, len(inner - top)


CASES = {
    # one span: 127 borders with a chain each, the 127 nodes over the cells, and
    # with chains of under 23 the one that parts the last cell from the corner
    "span_2560": (CHUNK, [20] * 19 + [19] * 108, "span", 2560),
    "span_2561": (CHUNK, [20] * 20 + [19] * 107, "span", 2561),
    "span_long": (CHUNK, [23] * 127, "span", 127 * 24),
    # 112 spans: 111 borders, the 111 nodes over the cells, and the corner's
    "top_2560": (SPAN, [23] * 6 + [22] * 105, "top", 2560),
    "top_2561": (SPAN, [23] * 7 + [22] * 104, "top", 2561),
}


@pytest.mark.parametrize("case", ["span_2560", "span_2561", "span_long"])
def test_lists_have_the_intended_lengths(case):
    step, chains, which, want = CASES[case]
    assert _build(step, chains, which)[3] == want


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(CASES))
def test_lists_at_and_past_the_lds_limit(require_gpu, case):
    step, chains, which, want = CASES[case]
    c, r, o, count = _build(step, chains, which)
    print(f"[refit lists] {case}: {len(c)} spheres, list of {count}", flush=True)
    assert count == want and (count > LIST) == (case not in ("span_2560", "top_2560"))
    check_equal(gpu_build(N.VRX_SPHERE, c, radius=r), o, len(c))
