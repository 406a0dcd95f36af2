"""GPU parity of the batched (n_tok > 1) path at the sizes where its kernels for
small batches begin and end: few tokens, expert counts that are no whole
groups, rows that are no whole chunks, and both sides of each size rule.  The
expected outputs are grouped_ref's: the reference's combine, with the
reference's serial fp32 logits, of per-token decode's expert rows."""
import numpy as np
import pytest

from cpubrrr_amd import MoeBlock, MoeConfig, synth
from tests.grouped_ref import BatchCheck, grouped_expect

pytestmark = pytest.mark.gpu


def check(L, cfg, X, family):
    with MoeBlock(cfg) as blk:
        blk.load_layer(0, L)
        Y, _ = blk.forward(0, X)
        bc = BatchCheck()
        for i in range(X.shape[0]):
            _, tr = blk.forward(0, X[i], trace=True)
            ye, _, _ = grouped_expect(L, X[i], tr, family)
            bc.add(Y[i], ye, X[i], (i,))
        bc.done()


@pytest.mark.parametrize("d,dff,ne,k,n_tok", [
    (96, 96, 2, 2, 2),          # one block of the router's chain, fewer experts than a group
    (416, 64, 20, 4, 3),        # 13 blocks, 20 experts
    (3840, 64, 33, 3, 5),       # the longest row, 33 experts
    (1088, 96, 16, 1, 17),
    (448, 64, 128, 4, 128),     # the last size of the small batch's router kernel in long chunks
    (448, 64, 128, 4, 129),     # the first in short chunks
    (416, 64, 120, 2, 137),     # 13 blocks, half a chunk at the end, experts and tokens that are no whole groups
    (1568, 64, 128, 2, 133),    # more than the steps requested ahead
    (768, 64, 128, 4, 129),     # a row that is whole rounds of the register sets, in short chunks
    (1536, 64, 16, 2, 3),       # and in long ones
    (448, 64, 128, 4, 256),     # the last in short chunks
    (448, 64, 128, 4, 257),     # the first of the other kernel
])
def test_mxfp4_small_batches(gpu, d, dff, ne, k, n_tok):
    print(f"case small batch d={d} dff={dff} ne={ne} k={k} n_tok={n_tok}", flush=True)
    L = synth.gptoss_layer(d, dff, ne, k, seed=21, zipf=1.1)
    X = np.stack([synth.token(d, 21, i) for i in range(n_tok)])
    check(L, MoeConfig.gptoss(d=d, n_expert=ne, top_k=k, d_ff=dff, max_tokens=n_tok), X, "gptoss")


@pytest.mark.parametrize("d,dff,ne,k,n_tok,down,same", [
    (256, 256, 8, 2, 3, 14, False),         # one superblock in each matrix
    (512, 512, 16, 8, 5, 12, False),
    (768, 768, 20, 1, 7, 14, False),        # an odd superblock count, top-1
    # one token nine times: an expert's second tile.  (Copies of a token share its expf ulps, so
    # BatchCheck's share of bit-exact tokens, taken from ten tokens on, would say nothing.)
    (512, 1536, 16, 4, 9, 12, True),
    (1280, 768, 16, 4, 16, 14, False),      # four pairs per expert: the last size of the few-token kernels
    (1280, 768, 16, 4, 17, 14, False),      # the first of the matrix-core tiles
    (512, 2048, 16, 2, 4, 14, False),       # d_ff beyond the few-token down kernel
    (4096, 1536, 8, 2, 7, 14, False),       # the few-token kernels at their widest: 512 threads, more than 64 KB of LDS
    (4096, 1536, 8, 4, 8, 12, True),        # and with full tiles
])
def test_kq_small_batches(gpu, d, dff, ne, k, n_tok, down, same):
    print(f"case kq small batch d={d} dff={dff} ne={ne} k={k} n_tok={n_tok} down={down}", flush=True)
    L = synth.qwen_layer(d, dff, ne, k, seed=22, down_type=down)
    X = np.stack([synth.token(d, 22, 0 if same else i) for i in range(n_tok)])
    check(L, MoeConfig.qwen3(d=d, n_expert=ne, top_k=k, d_ff=dff, max_tokens=n_tok, down_type=down), X, "qwen")


@pytest.mark.parametrize("ne,k,n_tok", [(32, 4, 5), (128, 8, 64), (128, 8, 65)])    # one launch up to 64 tokens, two beyond
def test_batched_selection_ties(gpu, ne, k, n_tok):
    """Equal logits (equal router rows): the lowest index wins, as in the reference."""
    print(f"case batched selection ties ne={ne} k={k} n_tok={n_tok}", flush=True)
    L = synth.gptoss_layer(384, 64, ne, k, seed=23)
    W = L["router_w"].reshape(ne, 384)
    W[: ne // 2] = W[ne // 2:]                       # every logit twice
    W[1] = W[2] = W[0]                               # and one four times
    X = np.stack([synth.token(384, 23, i) for i in range(n_tok)])
    check(L, MoeConfig.gptoss(d=384, n_expert=ne, top_k=k, d_ff=64, max_tokens=n_tok), X, "gptoss")


# the matrix-core tiles: k-parts of 15 blocks cut short in either sub-part, row tiles that are no
# whole workgroup in gate/up (4) and down (8), several tiles per expert
@pytest.mark.parametrize("d,dff,ne,k,n_tok", [
    (32 * 15, 32 * 16, 4, 2, 70),
    (32 * 16, 32 * 23, 4, 4, 33),
    (32 * 31, 32 * 5, 8, 4, 65),
    (32 * 24, 32 * 30, 3, 3, 40),
])
def test_mxfp4_tiles(gpu, d, dff, ne, k, n_tok):
    print(f"case tiles d={d} dff={dff} ne={ne} k={k} n_tok={n_tok}", flush=True)
    L = synth.gptoss_layer(d, dff, ne, k, seed=24, zipf=1.1)
    X = np.stack([synth.token(d, 24, i) for i in range(n_tok)])
    check(L, MoeConfig.gptoss(d=d, n_expert=ne, top_k=k, d_ff=dff, max_tokens=n_tok), X, "gptoss")


@pytest.mark.parametrize("d,kept", [(4096, True), (8192, False)])
def test_router_copy_only_for_the_batched_path(gpu, d, kept):
    """The transposed router copy (4 n_expert d bytes a layer) belongs to handles that can take the batched path."""
    print(f"case router copy d={d}", flush=True)
    import torch
    ne, layers = 256, 32
    used = []
    for tokens in (1, 1, 2):                         # the first handle also brings in the library's code
        before = torch.cuda.mem_get_info()[0]
        with MoeBlock(MoeConfig.qwen3(d=d, n_expert=ne, top_k=8, d_ff=256, n_layer=layers, max_tokens=tokens)):
            used.append(before - torch.cuda.mem_get_info()[0])
    copy = 4 * ne * d * layers
    assert (used[2] - used[1] >= copy // 2) == kept, (used, copy)
