"""Batched pi0.5 denoise loop (batch >= 2) on the MI355X vs the CPU fp32 oracle: the group kernels (2 to 16
samples) and the stage engine (more, long prefixes, workspaces without room for the groups).

Tolerance (the acceptance tolerance for bf16 operands with fp32 accumulation vs the fp32 oracle, on the
final actions of every sample): max-abs <= 2e-2 and mean-abs <= 2e-3.
"""
import numpy as np
import pytest
import torch

from tests import pi05_case as P
from tests import stage_engine as SE
from flashact_amd import pi05

MAX_ABS, MEAN_ABS = 2e-2, 2e-3

pytestmark = pytest.mark.gpu


def _check(c, gpu, **kw):
    ref = P.run_oracle(c)
    out, kc, vc = P.run_gpu_batched(c, gpu, **kw)
    ws = pi05.workspace(gpu, c["batch"], c["Tv"], pi05.lmax_for(c["Lp"], c["Tv"]))
    assert pi05.read_status(ws) == 0
    assert np.isfinite(out).all()
    for b in range(c["batch"]):
        st = P.parity(out[b, :c["Tv"]], ref[b])
        print(f"B={c['batch']} sample {b} NL={c['NL']} Lp={c['Lp']} Tv={c['Tv']} S={c['S']}: {st}", flush=True)
        assert st["max_abs"] <= MAX_ABS and st["mean_abs"] <= MEAN_ABS, (b, st)
    return out, ref, kc, vc


def test_batched_two_samples(gpu):
    _check(P.make_case(NL=2, Lp=968, Tv=50, S=2, batch=2), gpu)


# Lp + Tv: 54, 50, 364, 1109 end inside a 128-key chunk of the stage engine (the last chunk masked, its V^T
# tail group zeroed), 256 fills every chunk exactly (no masking at all); below on the groups, whose chunks are
# of the prefix alone, and in test_stage_engine_small_batches on the stage engine
@pytest.mark.parametrize("B,Lp,Tv,S", [(3, 37, 17, 2), (2, 0, 50, 1), (5, 300, 64, 1), (2, 1100, 9, 2),
                                      (2, 206, 50, 1)])
def test_batched_edge_shapes(gpu, B, Lp, Tv, S):
    _check(P.make_case(NL=2, Lp=Lp, Tv=Tv, S=S, batch=B, seed=B + Lp + Tv), gpu)


# Every group shape (batch 2, 3-4, 5-8, 9-16: one or two samples on one, two or four XCDs; odd batches leave
# a group with one sample or none) and the stage engine past them (17), at one and four token tiles,
# prefixes that end on, before and after a 64-key unit of the attention, and prefixes long enough
# (Lp > 1024) for a second segment of units per key chunk.
@pytest.mark.parametrize("B,Lp,Tv,S,NL", [(2, 64, 1, 2, 1), (2, 1030, 64, 1, 1), (3, 65, 16, 2, 2), (4, 1200, 33, 1, 1),
                                         (5, 63, 64, 1, 1), (8, 1025, 17, 1, 2), (9, 0, 49, 1, 1), (16, 129, 10, 2, 1),
                                         (17, 70, 9, 1, 1)])
def test_batched_group_shapes(gpu, B, Lp, Tv, S, NL):
    _check(P.make_case(NL=NL, Lp=Lp, Tv=Tv, S=S, batch=B, seed=B + Lp + Tv), gpu)


# Long prefixes of 9 to 16 samples run on whichever kernel is faster there, short horizons on the stage
# engine: each side of the rule, and the shortest prefix past it at 9 samples (2689) and its neighbour.
@pytest.mark.parametrize("B,Lp,Tv,owner", [(9, 2688, 10, SE.PI05_GROUP), (9, 2689, 10, SE.PI05_STAGE),
                                          (16, 8100, 1, SE.PI05_STAGE), (12, 4200, 33, SE.PI05_GROUP),
                                          (12, 8128, 64, SE.PI05_GROUP), (8, 8100, 1, SE.PI05_GROUP)])
def test_batched_long_prefixes(gpu, B, Lp, Tv, owner):
    c = P.make_case(NL=1, Lp=Lp, Tv=Tv, S=1, batch=B, seed=B + Tv)
    _check(c, gpu)
    ws = pi05.workspace(gpu, B, Tv, pi05.lmax_for(Lp, Tv))
    assert SE.owner(ws) == owner


def _check_stage(c, gpu, ws=None):
    ref = P.run_oracle(c)
    ws = ws if ws is not None else pi05.workspace(gpu, c["batch"], c["Tv"], pi05.lmax_for(c["Lp"], c["Tv"]))
    out = P.run_gpu_batched(c, gpu, ws=ws)[0]
    assert pi05.read_status(ws) == 0 and SE.owner(ws) == SE.PI05_STAGE
    for b in range(c["batch"]):
        st = P.parity(out[b, :c["Tv"]], ref[b])
        print(f"stage B={c['batch']} sample {b} NL={c['NL']} Lp={c['Lp']} Tv={c['Tv']} S={c['S']}: {st}", flush=True)
        assert st["max_abs"] <= MAX_ABS and st["mean_abs"] <= MEAN_ABS, (b, st)
    return out


# The stage engine where it serves: past 16 samples, several token tiles (the last one partial or full, up to
# the 4096 tokens of a launch), layers after layers, prefixes of none to more than eight key chunks.
@pytest.mark.parametrize("B,Lp,Tv,S,NL", [(17, 1100, 50, 2, 3), (18, 0, 64, 2, 2), (40, 206, 50, 2, 2), (64, 70, 64, 2, 2),
                                         (64, 300, 2, 2, 2)])
def test_stage_engine_large_batches(gpu, B, Lp, Tv, S, NL):
    _check_stage(P.make_case(NL=NL, Lp=Lp, Tv=Tv, S=S, batch=B, seed=B + Lp + Tv), gpu)


def test_stage_engine_full_depth(gpu):
    _check_stage(P.make_case(NL=18, Lp=968, Tv=50, S=10, batch=17, seed=5), gpu)


# The shapes of test_batched_edge_shapes and the first of this file, and more than 8 samples, on a workspace
# without room for the groups.
@pytest.mark.parametrize("B,Lp,Tv,S", [(2, 968, 50, 2), (3, 37, 17, 2), (2, 0, 50, 1), (5, 300, 64, 1), (2, 1100, 9, 2),
                                      (2, 206, 50, 1), (12, 1100, 17, 2)])
def test_stage_engine_small_batches(gpu, B, Lp, Tv, S):
    c = P.make_case(NL=2, Lp=Lp, Tv=Tv, S=S, batch=B, seed=B + Lp + Tv)
    ws = SE.zeroed(SE.need(lambda w: P.run_gpu_batched(c, gpu, ws=w), gpu), gpu)
    first = _check_stage(c, gpu, ws)
    assert np.array_equal(P.run_gpu_batched(c, gpu, ws=ws)[0], first)


def test_batched_repeats_on_one_workspace(gpu):
    """Launches of different group shapes, of the batch-1 kernel and of the stage engine (a workspace too
    small for the groups) on one workspace, each against its first result."""
    cs = [P.make_case(NL=1, Lp=90, Tv=20, S=2, batch=B, seed=B) for B in (2, 4, 8, 16)]
    n = max(pi05.workspace(gpu, c["batch"], 20, 112).numel() for c in cs)
    raw = torch.zeros(n + 256, dtype=torch.uint8, device=gpu)
    ws = raw[(-raw.data_ptr()) % 256:][:n]
    first = {}
    for r in range(2):
        for c in cs:
            out = P.run_gpu_batched(c, gpu, ws=ws)[0]
            assert pi05.read_status(ws) == 0
            assert np.array_equal(out, first.setdefault(c["batch"], out))
        one = P.run_gpu(P.make_case(NL=1, Lp=90, Tv=20, S=2, seed=2), gpu, ws=ws)[0]
        assert np.abs(one - first.setdefault(1, one)).max() <= MAX_ABS  # the exchange parity moves its last bit
    small = ws[:(8 << 20)]  # room for the stage engine at batch 2 only
    out = P.run_gpu_batched(cs[0], gpu, ws=small)[0]
    assert np.abs(out - first[2]).max() <= MAX_ABS


def test_batched_baseline_config2(gpu):
    """The batch-16 benchmark workload vs the fp32 oracle: batch 16, 18 layers, Lp=968, Tv=50, 10 steps."""
    _check(P.make_case(NL=18, Lp=968, Tv=50, S=10, batch=16), gpu)


def test_batched_matches_bs1_kernel(gpu):
    """Sample i of a batched launch agrees with the batch-1 kernel run on sample i alone."""
    c = P.make_case(NL=2, Lp=200, Tv=50, S=2, batch=3, seed=7)
    g = P.gpu_tensors(c, gpu)
    outb = P.run_gpu_batched(c, gpu, g)[0]
    for b in range(3):
        g1 = P.gpu_tensors(c, gpu)
        out1 = P.run_gpu(c, gpu, g1, sample=b)[0]
        assert np.abs(out1 - outb[b]).max() <= MAX_ABS


def test_batched_padded_rows_untouched(gpu):
    c = P.make_case(NL=1, Lp=100, Tv=10, S=1, batch=2)
    out = P.run_gpu_batched(c, gpu, xt_rows=16)[0]
    assert np.all(out[:, 10:] == 0.0)


def test_batched_suffix_cache_rows(gpu):
    """Each sample's suffix K/V rows land in its own slice of the stacked caches; the prefix is untouched."""
    c = P.make_case(NL=1, Lp=64, Tv=8, S=1, batch=2)
    out, ref, kc, vc = _check(c, gpu)
    kc = kc.float().cpu()
    vc = vc.float().cpu()
    w = c["w"]
    for b in range(2):
        x = c["inp"]["noise"][b] @ w["w_ain"].T + w["b_ain"]
        m = c["mods"][0, 0, 0]
        h = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * (1 + m[:1024]) + m[1024:2048]
        k = h @ w["wk"][0].float().T
        v = h @ w["wv"][0].float().T
        cos, sin = c["cos"], c["sin"]
        k = torch.cat([k[:, :128] * cos - k[:, 128:] * sin, k[:, 128:] * cos + k[:, :128] * sin], -1)
        assert torch.allclose(kc[b, 0, 64:72], k, atol=3e-2, rtol=3e-2)
        assert torch.allclose(vc[b, 0, :, 64:72].T, v, atol=3e-2, rtol=3e-2)
        assert torch.equal(kc[b, 0, :64], c["inp"]["kpre"][b, 0].float())


# Every group shape with full, partial and absent samples, and the stage engine: the rows of this step's keys
# and values that a launch leaves in the caches, of every sample and layer, against the batch-1 kernel's.
# More layers than XCDs of a group, since they take turns writing them; the rows before and behind stay.
# bf16 rows of layers whose inputs differ by their own bf16 operands: the bound of the test above.
@pytest.mark.parametrize("B,Lp,Tv", [(2, 70, 33), (3, 64, 64), (4, 37, 17), (5, 129, 50), (8, 70, 9), (9, 65, 16),
                                    (16, 40, 37), (17, 70, 9)])
def test_batched_cache_rows_of_every_layer(gpu, B, Lp, Tv):
    NL = 6
    c = P.make_case(NL=NL, Lp=Lp, Tv=Tv, S=2, batch=B, seed=B + Lp)
    g, g1 = P.gpu_tensors(c, gpu), P.gpu_tensors(c, gpu)
    for k, v in g["caches"]:  # rows that no launch may touch or use
        k[:, Lp + Tv:], v[..., Lp + Tv:] = 7.0, 7.0
    _, kc, vc = P.run_gpu_batched(c, gpu, g)
    ws = pi05.workspace(gpu, B, Tv, g["Lmax"])
    assert pi05.read_status(ws) == 0
    assert SE.owner(ws) == (SE.PI05_GROUP if B <= 16 else SE.PI05_STAGE)
    for b in range(B):
        _, k1, v1 = P.run_gpu(c, gpu, g1, sample=b)
        k, v = kc[b].float(), vc[b].float()
        for l in range(NL):
            assert torch.allclose(k[l, Lp:Lp + Tv], k1[l, Lp:Lp + Tv].float(), atol=3e-2, rtol=3e-2), (b, l)
            assert torch.allclose(v[l, :, Lp:Lp + Tv], v1[l, :, Lp:Lp + Tv].float(), atol=3e-2, rtol=3e-2), (b, l)
        assert torch.equal(k[:, :Lp], c["inp"]["kpre"][b].float().to(gpu))
        assert torch.equal(v[..., :Lp], c["inp"]["vpre"][b].float().transpose(1, 2).to(gpu))
        assert (k[:, Lp + Tv:] == 7).all() and (v[..., Lp + Tv:] == 7).all()
