"""MolmoAct2 flow loop on the MI355X vs the CPU fp32 oracle (parity gate).

Tolerance (the acceptance tolerance for bf16 operands with fp32 accumulation vs the fp32 oracle, on the
final actions, integrated dims [0, adim)): max-abs <= 2e-2 and mean-abs <= 2e-3.
"""
import numpy as np
import pytest

from tests import ma2_case as C
from tests import stage_engine as SE
from flashact_amd import ma2

MAX_ABS, MEAN_ABS = 2e-2, 2e-3

pytestmark = pytest.mark.gpu


def _check(c, gpu, **kw):
    ref = C.run_oracle(c)
    out = C.run_gpu(c, gpu, **kw)
    ws = ma2.workspace(gpu, c["batch"], c["Tv"], ma2.lkmax_for(c["Lk"]))
    assert ma2.read_status(ws) == 0
    assert np.isfinite(out).all()
    for b in range(c["batch"]):
        st = C.parity(out[b, :c["Tv"]], ref[b], c["adim"])
        print(f"B={c['batch']} sample {b} NL={c['NL']} Lk={c['Lk']} Tv={c['Tv']} S={c['S']}: {st}", flush=True)
        assert st["max_abs"] <= MAX_ABS and st["mean_abs"] <= MEAN_ABS, (b, st)
        # dims past adim are left as they were (the noise is zero there)
        assert np.all(out[b, :c["Tv"], c["adim"]:] == c["inp"]["noise"][b, :, c["adim"]:].numpy())
    return out, ref


def test_ma2_small(gpu):
    _check(C.make_case(NL=2, Lk=493, Tv=30, S=2), gpu)


def test_ma2_config4_bs1(gpu):
    """The MolmoAct2 benchmark workload at batch 1: 36 layers, Lk=493, Tv=30, adim=6, 10 steps."""
    _check(C.make_case(NL=36, Lk=493, Tv=30, S=10), gpu)


# Batch 1 runs the XCD-local kernel up to Tv = 32 and Lk = 1024: (1, 512, 32) fills every token lane
# and context rank; (1, 65, 17) leaves one token in the second token tile and a ragged key chunk. The
# others run the group kernels (one sample with 40 tokens too).
@pytest.mark.parametrize("B,Lk,Tv,S,adim", [(1, 1, 1, 2, 6), (2, 700, 64, 1, 32), (3, 37, 17, 2, 5),
                                            (1, 128, 16, 1, 6), (2, 129, 33, 1, 1), (1, 512, 32, 2, 6),
                                            (1, 65, 17, 2, 7), (1, 300, 40, 2, 6)])
def test_ma2_edge_shapes(gpu, B, Lk, Tv, S, adim):
    _check(C.make_case(NL=2, Lk=Lk, Tv=Tv, S=S, adim=adim, batch=B, seed=Lk + Tv), gpu)


# Contexts past 512 rows at batch 1: one key in the 17th chunk (513), a ragged chunk (777), every rank
# attending (1024) and the first context of the group kernel. Two steps: one Euler step of dt = 1 with
# unit gates sits at 2e-3 mean-abs from its bf16 operands alone (the stage-engine kernel 2.3e-3 at
# Lk = 1025, Tv = 5), two at 1.5e-3.
@pytest.mark.parametrize("Lk,Tv", [(513, 30), (777, 17), (1024, 32), (1025, 5)])
def test_ma2_long_context(gpu, Lk, Tv):
    _check(C.make_case(NL=2, Lk=Lk, Tv=Tv, S=2, seed=Lk), gpu)


def test_ma2_long_context_keeps_whole_partial_sums(gpu):
    """Past 512 keys the batch-1 kernel's exchanged partial sums are whole fp32 values: launches whose
    exchanges carry other parities (one layer and one step make three, so the parity of the second
    exchange buffer flips from launch to launch) give the same bits, also after the kernel of the shorter
    contexts has used the workspace."""
    import torch
    c = C.make_case(NL=1, Lk=600, Tv=32, S=1, adim=32, seed=3)
    short = C.make_case(NL=1, Lk=90, Tv=32, S=1, adim=32, seed=4)
    n = ma2.workspace(gpu, 1, 32, ma2.lkmax_for(600)).numel()
    raw = torch.zeros(n + 256, dtype=torch.uint8, device=gpu)
    ws = raw[(-raw.data_ptr()) % 256:][:n]
    first = C.run_gpu(c, gpu, ws=ws)
    for again in range(3):
        assert np.array_equal(C.run_gpu(c, gpu, ws=ws), first), again
    C.run_gpu(short, gpu, ws=ws)
    assert np.array_equal(C.run_gpu(c, gpu, ws=ws), first)
    assert np.array_equal(C.run_gpu(c, gpu, ws=ws), first)
    assert ma2.read_status(ws) == 0


# Batch 1, layer counts whose next layer is the same (1) and an odd one, a single token, a full second token
# tile and the last row of the first, contexts that leave ranks without keys: the layer's weights lie in LDS
# regions that other stages and the next layer reuse. Four steps, as for the groups below.
@pytest.mark.parametrize("NL,Lk,Tv", [(1, 33, 1), (1, 1024, 32), (3, 512, 17), (3, 40, 16)])
def test_ma2_batch1_layers(gpu, NL, Lk, Tv):
    _check(C.make_case(NL=NL, Lk=Lk, Tv=Tv, S=4, seed=NL + Lk), gpu)


# Every group shape (batch 1-4, 5-8, 9-16, two or four token tiles per sample) with groups of one sample, of
# none and full, token counts on either side of the tiles, context chunks that are empty, ragged and
# longer than one softmax segment, and the stage engine past them (17). Four steps: at two, bf16 operands
# alone leave 1.4e-3 mean-abs, and 1.1e-3 to 2.1e-3 over a sample of 30 values (the stage engine's 17 x 5
# tokens); the error falls with the step length.
@pytest.mark.parametrize("B,Lk,Tv,adim", [(1, 33, 33, 6), (2, 1, 32, 6), (3, 700, 16, 6), (4, 1100, 64, 6),
                                          (5, 129, 17, 32), (8, 513, 49, 6), (9, 64, 30, 6), (16, 300, 31, 6),
                                          (12, 65, 50, 1), (17, 50, 5, 6)])
def test_ma2_group_shapes(gpu, B, Lk, Tv, adim):
    _check(C.make_case(NL=2, Lk=Lk, Tv=Tv, S=4, adim=adim, batch=B, seed=B + Lk + Tv), gpu)


def _check_stage(c, gpu, ws=None):
    ref = C.run_oracle(c)
    ws = ws if ws is not None else ma2.workspace(gpu, c["batch"], c["Tv"], ma2.lkmax_for(c["Lk"]))
    out = C.run_gpu(c, gpu, ws=ws)
    assert ma2.read_status(ws) == 0 and SE.owner(ws) == SE.MA2_STAGE
    for b in range(c["batch"]):
        st = C.parity(out[b, :c["Tv"]], ref[b], c["adim"])
        print(f"stage B={c['batch']} sample {b} NL={c['NL']} Lk={c['Lk']} Tv={c['Tv']} S={c['S']}: {st}", flush=True)
        assert st["max_abs"] <= MAX_ABS and st["mean_abs"] <= MEAN_ABS, (b, st)
        assert np.all(out[b, :c["Tv"], c["adim"]:] == c["inp"]["noise"][b, :, c["adim"]:].numpy())
    return out


# The stage engine where it serves, past 16 samples: its small tiles (up to 64 tokens, split-K sums in place)
# and its large ones, partial and full, up to 2048 tokens. Four steps, as for the groups.
@pytest.mark.parametrize("B,Lk,Tv,adim,NL", [(17, 300, 3, 32, 3), (64, 33, 1, 32, 2), (17, 493, 30, 6, 2), (20, 1100, 33, 6, 2),
                                            (32, 129, 64, 32, 2)])
def test_ma2_stage_engine_large_batches(gpu, B, Lk, Tv, adim, NL):
    _check_stage(C.make_case(NL=NL, Lk=Lk, Tv=Tv, S=4, adim=adim, batch=B, seed=B + Lk + Tv), gpu)


def test_ma2_stage_engine_full_depth(gpu):
    _check_stage(C.make_case(NL=36, Lk=493, Tv=30, S=10, batch=17, seed=6), gpu)


# Batches that fit the groups, on a workspace without room for them (the stage engine needs less up to 64
# tokens): its small tiles with one to four waves per cross-attention item. Run twice: the split-K counters
# are back at zero.
@pytest.mark.parametrize("B,Lk,Tv,adim", [(1, 300, 40, 6), (1, 1025, 5, 32), (2, 129, 30, 6), (3, 37, 17, 5), (1, 128, 64, 32)])
def test_ma2_stage_engine_small_batches(gpu, B, Lk, Tv, adim):
    c = C.make_case(NL=2, Lk=Lk, Tv=Tv, S=4, adim=adim, batch=B, seed=B + Lk + Tv)
    ws = SE.zeroed(SE.need(lambda w: C.run_gpu(c, gpu, ws=w), gpu), gpu)
    first = _check_stage(c, gpu, ws)
    assert np.array_equal(C.run_gpu(c, gpu, ws=ws), first)


def test_ma2_groups_repeat_on_one_workspace(gpu):
    """Launches of different group shapes and of the stage engine (a workspace with no room for the groups)
    on one workspace, each against its first result."""
    import torch
    cs = [C.make_case(NL=1, Lk=90, Tv=Tv, S=2, batch=B, seed=B) for B, Tv in ((2, 20), (3, 40), (6, 20), (6, 40), (12, 20))]
    n = max(ma2.workspace(gpu, c["batch"], c["Tv"], 96).numel() for c in cs)
    raw = torch.zeros(n + 256, dtype=torch.uint8, device=gpu)
    ws = raw[(-raw.data_ptr()) % 256:][:n]
    first = {}
    for r in range(2):
        for i, c in enumerate(cs):
            out = C.run_gpu(c, gpu, ws=ws)
            assert ma2.read_status(ws) == 0
            assert np.array_equal(out, first.setdefault(i, out))
    out = C.run_gpu(cs[0], gpu, ws=ws[:(8 << 20)])
    assert np.abs(out - first[0]).max() <= MAX_ABS


def test_ma2_batch16(gpu):
    """The MolmoAct2 benchmark workload at batch 16 (on the groups) at full depth, 36 layers x 10 steps, every
    sample against the oracle (benchmarks/molmoact2/eval_numerics.py:147-159 is the reference's
    fidelity check of the same loop)."""
    _check(C.make_case(NL=36, Lk=493, Tv=30, S=10, batch=16), gpu)


def test_ma2_batch16_shallow(gpu):
    """Batch 16 at 2 layers and 2 steps: a quick first signal before the full-depth case."""
    _check(C.make_case(NL=2, Lk=493, Tv=30, S=2, batch=16), gpu)


def test_ma2_batched_matches_single(gpu):
    c = C.make_case(NL=2, Lk=200, Tv=30, S=2, batch=3, seed=5)
    g = C.gpu_tensors(c, gpu)
    outb = C.run_gpu(c, gpu, g)
    for b in range(3):
        out1 = C.run_gpu(c, gpu, g, samples=[b])[0]
        assert np.abs(out1 - outb[b]).max() <= MAX_ABS


def test_ma2_deterministic(gpu):
    c = C.make_case(NL=2, Lk=300, Tv=30, S=2)
    g = C.gpu_tensors(c, gpu)
    assert np.array_equal(C.run_gpu(c, gpu, g), C.run_gpu(c, gpu, g))


def test_ma2_padded_rows_untouched(gpu):
    c = C.make_case(NL=1, Lk=50, Tv=10, S=1)
    out = C.run_gpu(c, gpu, xt_rows=16)
    assert np.all(out[:, 10:] == 0.0)
