"""Powers by the shorter way against the definition they stand for, bit for bit: enough inputs that some (three in 100,000)
lie so near the middle of two floats that only the definition settles them, exponents on both sides of the line (16)
from which the definition is always taken, results down to the smallest and up to the largest floats."""
import numpy as np
import pytest
import torch

from gpu_util import bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("alpha", [1e-3, 0.25, 0.6, 0.999, 1.0001, 2.0, 7.5, 16.0])
@pytest.mark.parametrize("push", [False, True])
def test_powers_bit_exact(alpha, push):
    from mindrl_amd.core import PriorityReplayBuffer
    from oracle import orc
    n = 1 << 19
    rng = np.random.default_rng(int(alpha * 1000))
    pr = np.exp(rng.uniform(-88 / max(alpha, 1.0), 88 / max(alpha, 1.0), n)).astype(np.float32)
    pr[::3] = (1.0 + 1e-3 * rng.normal(size=pr[::3].size)).astype(np.float32)
    pr[:10] = [0.0, 1.0, 1e-38, 1e-45, 2.9e38, 2.0, 0.5, np.float32(1.0) - np.float32(2.0 ** -24),
               np.float32(1.0) + np.float32(2.0 ** -23), np.float32(np.sqrt(0.5))]
    g = PriorityReplayBuffer(alpha, n, 4, [(1,)], [torch.int32], seed0=1)
    rows = torch.zeros(n, 1, dtype=torch.int32).cuda()
    if push:  # four powers per lane
        g.insert(rows, priorities=torch.from_numpy(pr).cuda())
    else:  # one power per thread
        g.insert(rows)
        g.update_priorities(torch.arange(n).cuda(), torch.from_numpy(pr).cuda())
    s, _ = g.export_tree()
    want = orc.powf_array(pr, alpha)
    bad = np.nonzero(bits(s[n:]) != bits(want))[0]
    assert bad.size == 0, (pr[bad[:5]], s[n:][bad[:5]], want[bad[:5]])
    g.destroy()


@pytest.mark.parametrize("beta", [0.0, 0.4, 1.0, 16.0, 16.5, 40.0])
def test_weights_bit_exact(beta):
    from mindrl_amd.core import PriorityReplayBuffer
    from oracle import orc
    n, batch = 4096, 2048
    rng = np.random.default_rng(7)
    pr = np.exp(rng.uniform(-1, 1, n)).astype(np.float32)
    g = PriorityReplayBuffer(1.0, n, batch, [(1,)], [torch.int32], seed0=1)
    c = orc.OraclePER(1.0, n, [(1,)], [np.int32], seed=1)
    rows = np.zeros((n, 1), np.int32)
    g.insert(torch.from_numpy(rows).cuda(), priorities=torch.from_numpy(pr).cuda())
    c.push([rows], n, pr)
    u = rng.random(batch).astype(np.float32)
    for path in (1, 2):
        g.set_option("sample_path", path)
        w = g.sample(beta, uniforms=torch.from_numpy(u).cuda())[1].cpu().numpy()
        assert np.array_equal(bits(w), bits(c.sample(batch, beta, u)[1])), beta
    g.destroy()
