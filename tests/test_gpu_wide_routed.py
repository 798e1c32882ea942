"""Models wide enough (2048 columns) for the forms of up to 16 rows in which the router's product and the choice of experts are part of the launch that makes their input, and the list
of rows by expert part of gate and up: whole steps against the restatements in oracle/, with identity experts, experts in groups, experts weighted at their input, one and four streams."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import fomunex_common as fomunex  # noqa: E402
import gulidra_common as gulidra  # noqa: E402
import natatar_common as natatar  # noqa: E402
from pimosun_common import layered, m40, write_folder  # noqa: E402
from test_gpu_gulidra import assert_logits  # noqa: E402


def gulidra_model(width):
    g = gulidra
    return g, g.od, g.model(101, width, [(g.attention(4, 2, 32, 32), g.experts(16, 2, 4, 48)), (g.lightning(2, 32, 32, [0.9, 0.99]), g.dense(64)), (g.attention(3, 1, 24, 40), g.experts(5, 3, 3, 33))])


def natatar_model(width, streams):
    g = natatar
    return g, g.sd, g.model(101, width, streams, [(g.attention(4, 2, 32, 32, v_mix=False), g.experts(12, 3, 48, (4, 2), 1.7)), (g.delta(2, 1, 32, 32, 3), None),
                                                  (g.attention(3, 1, 24, 40, v_mix=False), g.experts(7, 2, 33))])


def fomunex_model(width):
    """All experts first, a choice last: a close call decided otherwise in bf16 is then seen by no later token."""
    g = fomunex
    return g, g.pd, g.model(101, width, [(g.attention(3, 1, 24, 40, 70, 30.0), g.experts(4, 4, 33, 0.8)), (g.mixing(2, 32), g.dense(64)), (g.attention(4, 2, 32, 32, 20, 9.0), g.experts(16, 4, 48, 1.5))],
                            eps=1e-3)


def random_tensors(common, cfg):
    """Experts that matter (a wrong choice, or one's weight for another's, moves the logits by more than their limit), and scores that differ where they are sigmoids."""
    T = common.random_tensors(cfg, 5)
    for n in T:
        if ".mlp.e" in n and n.endswith("down"):
            T[n] *= {"Gulidra": 1, "Natatar": 3, "Fomunex": 8}[cfg["architecture"]]
        if n.endswith("mlp.router") and cfg["architecture"] == "Fomunex":
            T[n] *= 0.5
    return T


@pytest.fixture(scope="module")
def ctx():
    yield m40.Context(0)


# rows of a step by sequence: one and four rows, sixteen of one sequence and of three, more rows (whose feed-forward is launched apart) in between
STEPS = [{0: 1}, {0: 4}, {1: 16}, {2: 9, 1: 6, 0: 1}, {0: 1, 1: 1, 2: 1}, {2: 17}, {0: 5, 1: 1}, {0: 1, 2: 1}] + 6 * [{0: 1, 1: 1, 2: 1}] + [{0: 2, 1: 14}, {0: 16}, {2: 4, 1: 4}]


@pytest.mark.parametrize("of,sizes", [(gulidra_model, (2048,)), (gulidra_model, (2072,)), (natatar_model, (2048, 4)), (natatar_model, (2056, 1)), (fomunex_model, (2048,)), (fomunex_model, (4096,))])
def test_steps_of_few_rows(ctx, tmp_path, of, sizes):
    common, restatement, cfg = of(*sizes)
    folder = write_folder(tmp_path, cfg, random_tensors(common, cfg))
    reference = restatement.Model.load(folder)
    rng = np.random.default_rng(sum(sizes))
    tokens, want, margins = [], [], []
    for s in range(3):
        tokens.append(rng.integers(0, cfg["vocab"], sum(step.get(s, 0) for step in STEPS)))
        q = reference.sequence()
        want.append(q.feed(tokens[-1].tolist()))
        margins.append(np.array(q.margins))
    m = layered.LayeredModel.open(ctx, folder, "bfloat16", 512, 4)
    at, got, rows = [0, 0, 0], [], []
    for step in STEPS:
        got.append(m.step([(s, tokens[s][at[s]:at[s] + n], range(n)) for s, n in step.items()]))
        for s, n in step.items():
            rows += [(s, at[s] + k) for k in range(n)]
            at[s] += n
    assert_logits(np.concatenate(got), np.stack([want[s][p] for s, p in rows]), "bfloat16", np.array([margins[s][p] for s, p in rows]), (of.__name__, sizes))
    m.close()
