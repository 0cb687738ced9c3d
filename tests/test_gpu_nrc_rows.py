"""The learned cache's encoding, which gives each eighth of the chip two
levels, and the table gradient, whose lanes share a row: at 1, 8, 9 and 16
levels (none, one or two levels an eighth), tables small enough that only the
hash is used and large enough that dense levels are among them, and row counts
around the 16-, 128- and 256-row pieces; and inference in slices (of 2^18
rows) against the same rows alone."""
import numpy as np
import pytest
import torch

import rtxamd
from nrc_reference import HIDDEN, OUT_PAD, WIDTH, Reference, random_inputs

pytestmark = pytest.mark.gpu

LO, HI = (-1.0, -2.0, 0.0), (3.0, 2.0, 1.5)


@pytest.fixture(scope="module")
def renderer():
    r = rtxamd.Renderer(0)
    yield r
    r.close()


def copying_mlp(info, cols):
    """Identity layers and an output layer that picks the input columns."""
    mlp = np.zeros(info.mlpParams, np.float32)
    for l in range(HIDDEN):
        mlp[l * WIDTH * WIDTH:(l + 1) * WIDTH * WIDTH] = np.eye(WIDTH, dtype=np.float32).reshape(-1)
    out = mlp[HIDDEN * WIDTH * WIDTH:].reshape(OUT_PAD, WIDTH)
    for o, c in enumerate(cols):
        out[o, c] = 1.0
    return mlp


@pytest.mark.parametrize("levels,log2,rows", [(1, 8, 1), (8, 13, 15), (9, 8, 17), (16, 19, 129), (9, 19, 256),
                                              (16, 8, 257), (8, 16, 1023)])
def test_encoding_and_table_gradient(renderer, levels, log2, rows):
    renderer.nrc_create(LO, HI, seed=3, levels=levels, log2TableSize=log2, trainBatch=1024)
    info = renderer.nrc_info()
    rng = np.random.default_rng(levels + rows)
    grid = rng.uniform(0.0, 1.0, (info.levels, info.tableSize, 2)).astype(np.float32)
    x = random_inputs(rows, LO, HI, rng)
    ref = Reference(info)
    enc = ref.encode(torch.from_numpy(x), torch.from_numpy(grid)).detach().numpy()
    last = 2 * levels - 1
    for cols in ([0, 1, last], [last - 1, last, 42]):
        mlp = copying_mlp(info, cols)
        renderer.nrc_set_params(grid, mlp)
        assert np.array_equal(renderer.nrc_infer(x), np.maximum(enc[:, cols], 0.0))
    # the output is the feature itself (positive, so every ReLU passes): d loss
    # / d feature is d loss / d output, rounded to BF16 once (2^-8) and copied
    # through the identity layers; the weights and their FP32 sums add less
    target = rng.uniform(0.0, 2.0, (rows, 3)).astype(np.float32)
    renderer.nrc_set_params(grid, copying_mlp(info, [0, 1, last]))
    _, ggrid, _ = renderer.nrc_gradients(x, target)
    tg = torch.from_numpy(grid).requires_grad_(True)
    loss = Reference.loss(ref.forward(torch.from_numpy(x), tg, torch.from_numpy(copying_mlp(info, [0, 1, last]))),
                          torch.from_numpy(target))
    loss.backward()
    want = tg.grad.numpy()
    assert np.all(ggrid[want == 0] == 0)
    assert np.linalg.norm(ggrid - want) <= 2.0 ** -7 * np.linalg.norm(want)


@pytest.mark.parametrize("n", [1 << 18, (1 << 18) + 1, (1 << 22) + 77])
def test_inference_in_slices(renderer, n):
    renderer.nrc_create(LO, HI, seed=3, levels=8, log2TableSize=12)
    rng = np.random.default_rng(1)
    x = np.tile(random_inputs(4099, LO, HI, rng), ((n + 4098) // 4099, 1))[:n]
    got = renderer.nrc_infer(x)
    once = renderer.nrc_infer(x[:4099])
    assert np.array_equal(got, np.tile(once, ((n + 4098) // 4099, 1))[:n])
