"""Which calls replay a captured graph: several layers, and a single layer
whose tokens go one by one through many kernels (an e8m0 byte outside the
matrix-core path's range).  A single layer of few kernels is launched directly.
Read off the runtime calls that torch's profiler traces."""
import numpy as np
import pytest

from cpubrrr_amd import MoeBlock, MoeConfig, synth

pytestmark = pytest.mark.gpu


def graph_launches(blk, n_layers, x, n_tok):
    from torch.profiler import ProfilerActivity, profile
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        blk.forward_device(0, n_layers, x.data_ptr(), n_tok)
        blk.sync()
    calls = {e.key: e.count for e in p.key_averages()}
    if "hipLaunchKernel" not in calls and "hipGraphLaunch" not in calls:
        pytest.skip("the profiler traces no runtime calls here")
    return calls.get("hipGraphLaunch", 0)


@pytest.mark.parametrize("special,n_layers,n_tok,graphs", [
    (False, 1, 1, 0),
    (False, 1, 40, 0),
    (False, 2, 3, 1),
    (True, 1, 10, 0),          # 30 kernels
    (True, 1, 11, 1),          # 33
])
def test_graph_or_direct(gpu, special, n_layers, n_tok, graphs):
    print(f"case launch rule special={special} layers={n_layers} n_tok={n_tok}", flush=True)
    import torch
    d, dff, ne, k = 480, 480, 8, 4
    L = synth.gptoss_layer(d, dff, ne, k, seed=31)
    if special:
        L["gate"].reshape(-1, 17)[::97, 0] = 0
    X = np.stack([synth.token(d, 31, i) for i in range(n_tok)])
    with MoeBlock(MoeConfig.gptoss(d=d, n_expert=ne, top_k=k, d_ff=dff, n_layer=2, max_tokens=40)) as blk:
        blk.load_layer(0, L)
        blk.load_layer(1, L)
        x = torch.from_numpy(X).cuda()
        torch.cuda.synchronize()
        assert graph_launches(blk, n_layers, x, n_tok) == graphs
        if special:                                        # a second x, token by token: the same kernels, the same bits
            y = torch.from_numpy(X).cuda()
            torch.cuda.synchronize()
            for i in range(n_tok):
                blk.forward_device(0, 1, y[i].data_ptr(), 1)
            blk.sync()
            assert torch.equal(x, y)
