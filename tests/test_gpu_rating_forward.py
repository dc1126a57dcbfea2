"""The learned rating's weights on their way to the GPU: several weight sets one after the other,
through the kernel that packs them and the memory that is kept between calls. The scores of a graph
equal the quantised logits of its features with the same weights, each set's logits are the 64-bit
MLP's on the BF16 operands within the forward's rounding, and partitions alternate between weight
sets without a trace of the other one."""
import numpy as np
import pytest

import kahip_amd as K
import oracle.rating as R

pytestmark = pytest.mark.gpu


def weights(seed):
    r = np.random.default_rng(seed)
    w = (r.standard_normal(K.MLP_PARAMS) * 0.2).astype(np.float32)
    w[:512] += np.float32(seed) * np.float32(0.125)
    return w


@pytest.fixture(scope="module")
def mesh():
    g = K.Graph.rgg(60001, 5)
    host = g.to_host()
    yield g, host
    g.free()


@pytest.mark.parametrize("first", [0, 1, 2])
def test_scores_are_the_quantised_logits(mesh, first):
    _, (x, a, vw, ew) = mesh
    f = K.edge_features(x, a, vw, ew, 300, 9)
    seen = []
    for i in range(3):
        w = weights((first + i) % 3)
        score = K.edge_scores(x, a, vw, ew, K.RATING_LEARNED, w, 300, 9)
        assert np.array_equal(score, R.quantize_logit(K.mlp_forward(f, w)))
        seen.append(score)
    assert not np.array_equal(seen[0], seen[1]) and not np.array_equal(seen[1], seen[2])


def test_alternating_partitions(mesh):
    g, _ = mesh
    want = {}
    for i in range(24):
        s = i % 3
        part, _ = g.partition(3, seed=2, rating=K.RATING_LEARNED, mlp_weights=weights(s),
                              cluster_rounds=4)
        assert np.array_equal(want.setdefault(s, part), part), (i, s)


@pytest.mark.parametrize("row", [0, 511, 512, 575, 576, 4671, 4672, 4735, 4736, 4799, 4800])
def test_every_part_of_the_pack(row):
    """One parameter of each block's ends, with the others fixed: the logits change as the 64-bit
    MLP's do (weights and features that are exact in BF16, so only sums round)."""
    r = np.random.default_rng(3)
    f = (r.integers(0, 16, (100, 8)) / 4.0).astype(np.float32)
    w = (r.integers(-4, 5, K.MLP_PARAMS) / 8.0).astype(np.float32)
    w[row] = 2.0
    p = w.astype(np.float64)
    h1 = np.maximum((f[:, :, None] * p[:512].reshape(64, 8).T[None]).sum(1) + p[512:576], 0.0)
    h1 = R.bf16_round(h1)
    h2 = np.maximum((h1[:, :, None] * p[576:4672].reshape(64, 64).T[None]).sum(1) + p[4672:4736],
                    0.0)
    z = (h2 * p[4736:4800]).sum(1) + p[4800]
    got = K.mlp_forward(f, w)
    # fp32 sums of at most 64 products, two layers: 128 roundings of 2^-24 relative to the terms
    scale = (np.abs(h2) * np.abs(p[4736:4800])).sum(1) + np.abs(h1).sum(1) + 1.0
    assert np.all(np.abs(got - z) <= 128 * 2.0 ** -24 * 64 * scale)
