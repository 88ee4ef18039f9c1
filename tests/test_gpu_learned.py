"""The frontier predictor's HIP kernels against the float64 oracle, and the
learned schedule end to end (reports unchanged, predictions measured)."""
import numpy as np
import pytest

import oracle
from oracle import mlp_ref
from ngap_amd import NgapError, learned, synth
from ngap_amd.mlp import MLP

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, flush=True)


@pytest.fixture(scope="module")
def mlp():
    m = MLP(0, seed=3)
    yield m
    m.close()


def test_forward_and_gradient_match_oracle(mlp):
    rng = np.random.default_rng(0)
    p = mlp.params.astype(np.float64)
    for n in (1, 17, 300):
        x = rng.normal(size=(n, 264)).astype(np.float32)
        t = rng.normal(size=n).astype(np.float32)
        say("mlp forward/gradient", n)
        y = mlp.predict(x)
        y_ref, _ = mlp_ref.forward(p, x.astype(np.float64))
        assert np.allclose(y, y_ref, rtol=1e-4, atol=1e-4)   # FP32 vs float64
        g, loss = mlp.gradient(x, t)
        g_ref, loss_ref = mlp_ref.gradient(p, x.astype(np.float64), t.astype(np.float64))
        assert np.isclose(loss, loss_ref, rtol=1e-4)
        scale = np.abs(g_ref).max()
        assert np.max(np.abs(g - g_ref)) <= 1e-4 * scale + 1e-6


def test_pair_inference_equals_dense(mlp):
    rng = np.random.default_rng(1)
    hist = rng.random((40, 256)).astype(np.float32)
    hist /= hist.sum(1, keepdims=True)
    stats = rng.random((7, 8)).astype(np.float32)
    pairs = np.stack([rng.integers(0, 7, 500), rng.integers(0, 40, 500)], 1)
    say("mlp pairs")
    y1 = mlp.predict_pairs(hist, stats, pairs)
    y2 = mlp.predict(learned.features(hist, stats, pairs))
    assert np.array_equal(y1, y2)


def test_training_fits_a_known_function():
    rng = np.random.default_rng(2)
    x = rng.random((20000, 264)).astype(np.float32)
    t = (3 * x[:, 0] - 2 * x[:, 260] + x[:, 100] * x[:, 101]).astype(np.float32)
    m = MLP(0, seed=5)
    say("mlp training")
    l0 = float(np.mean((m.predict(x) - t) ** 2))
    loss = m.train(x, t, epochs=20, batch=512, lr=2e-3)
    l1 = float(np.mean((m.predict(x) - t) ** 2))
    assert l1 < 0.05 * l0 and loss < 0.05 * l0
    m.close()


def test_learned_schedule_end_to_end(engine):
    rng = np.random.default_rng(9)
    groups = synth.batch_groups(rng, 48, lo=50, hi=8000)
    chunk = 1 << 14
    train = synth.drifting_input(np.random.default_rng(10), 1 << 20, chunk, 1e-3, groups, 16)
    test = synth.drifting_input(np.random.default_rng(11), 1 << 19, chunk, 1e-3, groups, 16)
    stats = learned.group_stats(groups)
    engine.load_groups(groups, 2)
    say("traces")
    engine.set_input(train, chunk)
    pairs, y = learned.collect_traces(engine, train, chunk, len(groups))
    x = learned.features(learned.window_hist(train, chunk), stats, pairs)
    m = MLP(0, seed=1)
    say("train", x.shape)
    m.train(x, y, epochs=8, batch=2048, lr=2e-3)
    engine.set_input(test, chunk)
    tp, ty = learned.collect_traces(engine, test, chunk, len(groups))
    pred = m.predict_pairs(learned.window_hist(test, chunk), stats, tp)
    mae = float(np.mean(np.abs(pred - ty)))
    base = float(np.mean(np.abs(y.mean() - ty)))   # a predictor without features
    say("mae", mae, "constant predictor", base)
    assert mae < base
    S = len(test) // chunk
    cost = np.zeros((len(groups), S * learned.windows_per_chunk(chunk)))
    cost[tp[:, 0], tp[:, 1]] = learned.predicted_cost(pred)
    waves = engine.batched_waves()
    assert waves > 0
    tasks, tcost = learned.schedule_from_costs(cost, len(groups), S, chunk, waves=waves)
    # the predicted peak sizes the worklist spill area below the static
    # default of 65,536 items per wave (the memory the network saves)
    assert learned.spill_capacity(pred, tcost) < 65536
    want, _ = oracle.run(groups, test, chunk)
    say("learned schedule run")
    st = engine.run(algorithm="nonblockingallgroups", schedule="batched", precompute_depth=2,
                    unique=True, tasks=tasks, spill_capacity=learned.spill_capacity(pred, tcost),
                    fallback=True)
    assert np.array_equal(engine.reports(), want)
    assert st["num_tasks"] == len(tasks)
    ctasks, ccost = learned.cross_schedule_from_costs(cost, S, chunk, waves=waves)
    say("learned all-group schedule run")
    st = engine.run(algorithm="nonblockingallgroups", schedule="batched", precompute_depth=2,
                    unique=True, tasks=ctasks, spill_capacity=learned.spill_capacity(pred, ccost),
                    fallback=True)
    assert np.array_equal(engine.reports(), want)
    assert st["num_tasks"] == len(ctasks)
    m.close()


@pytest.mark.parametrize("n", [15, 16, 31, 32, 33, 512, 16384 + 1, 40000])
def test_gradient_tiles_match_oracle(n):
    """Sizes around a tile (32 samples), and several tiles per workgroup."""
    rng = np.random.default_rng(n)
    m = MLP(0, seed=4)
    p = m.params.astype(np.float64)
    x = rng.normal(size=(n, 264)).astype(np.float32)
    t = rng.normal(size=n).astype(np.float32)
    say("mlp tiles", n)
    y_ref, _ = mlp_ref.forward(p, x.astype(np.float64))
    assert np.allclose(m.predict(x), y_ref, rtol=1e-4, atol=1e-4)
    g, loss = m.gradient(x, t)
    g_ref, loss_ref = mlp_ref.gradient(p, x.astype(np.float64), t.astype(np.float64))
    assert np.isclose(loss, loss_ref, rtol=1e-4)
    assert np.max(np.abs(g - g_ref)) <= 1e-4 * np.abs(g_ref).max() + 1e-6
    m.close()


@pytest.mark.parametrize("n", [1, 15, 16, 17, 64, 49153, 100000])
def test_pairs_rounds_match_dense(mlp, n):
    """Pairs around a wave's round (16) and a full grid of rounds (49,152)."""
    rng = np.random.default_rng(n)
    hist = rng.random((33, 256)).astype(np.float32) / 128
    stats = rng.random((17, 8)).astype(np.float32)
    pairs = np.stack([rng.integers(0, 17, n), rng.integers(0, 33, n)], 1)
    say("mlp pairs", n)
    y = mlp.predict_pairs(hist, stats, pairs)
    assert np.array_equal(y, mlp.predict(learned.features(hist, stats, pairs)))
    for bad in ((17, 0), (0, 33)):
        wrong = pairs.copy()
        wrong[n // 2] = bad
        with pytest.raises(NgapError, match="pair out of range"):
            mlp.predict_pairs(hist, stats, wrong)


def test_training_steps_match_oracle():
    """Mini-batches with a remainder, shuffled rows, Adam: parameters after
    two epochs against the same steps in float64."""
    rng = np.random.default_rng(6)
    n, batch = 1000, 300
    x = rng.random((n, 264)).astype(np.float32)
    t = x[:, 0].astype(np.float32)
    m = MLP(0, seed=8)
    p = m.params.astype(np.float64)
    say("mlp training steps")
    loss = m.train(x, t, epochs=2, batch=batch, lr=1e-3, seed=11)
    z, idx, step = 11, list(range(n)), 0
    mom, var = np.zeros_like(p), np.zeros_like(p)
    for _ in range(2):
        for i in range(n - 1, 0, -1):
            z = (z * 6364136223846793005 + 1442695040888963407) & (2**64 - 1)
            j = (z >> 33) % (i + 1)
            idx[i], idx[j] = idx[j], idx[i]
        total = 0.0
        for a in range(0, n, batch):
            rows = idx[a:a + batch]
            g, l = mlp_ref.gradient(p, x[rows].astype(np.float64), t[rows].astype(np.float64))
            total += l * len(rows)
            step += 1
            mom = 0.9 * mom + 0.1 * g
            var = 0.999 * var + 0.001 * g * g
            p = p - 1e-3 * (mom / (1 - 0.9**step)) / (np.sqrt(var / (1 - 0.999**step)) + 1e-8)
    # eight steps of at most 1e-3 per parameter, each to FP32 accuracy but for
    # parameters whose gradient is itself rounding noise
    assert np.linalg.norm(m.params - p) <= 1e-5 * np.linalg.norm(p)
    assert np.isclose(loss, total / n, rtol=1e-4)
    m.close()
