"""GPU parity: the HIP path, called through the C ABI, against the CPU oracle on
the same seeded inputs. Routing (top-k indices, expert counts/offsets,
permutation) must be bit-exact; outputs within the tolerance in moe_case.TOL."""
import numpy as np
import pytest
import torch

from flash_distributed_moe_amd import _lib, synth
from flash_distributed_moe_amd.flashMoeLauncher import MoeKernelLauncher
from oracle import oracle
from tests.moe_case import GpuCase

pytestmark = pytest.mark.gpu


def run_case(cfg, seed=7907, sched=_lib.SCHED_STREAM, sample=None, inplace=False):
    print("case", cfg.name, "T", cfg.T, "H", cfg.H, "E", cfg.E, "k", cfg.k, "I", cfg.I,
          cfg.dtype, "seed", seed, "sched", sched, flush=True)
    case = GpuCase(cfg, seed, sched)
    try:
        x = case.inp["tokens"]
        out = case.run(inplace=inplace)
        routing = case.launcher.routing(cfg.T)
        case.check_routing(x, routing)
        ids = None
        if sample is not None and sample < cfg.T:
            ids = np.unique(np.linspace(0, cfg.T - 1, sample).astype(np.int64))
        err = case.check_outputs(x, out, ids)
        print("  max rel err %.3e" % err, flush=True)
        return case, out
    finally:
        case.close()


def test_tiny_f32():
    run_case(synth.CONFIGS["tiny_f32"])


def test_tiny_f32_matches_golden(golden_dir):
    import os

    g = np.load(os.path.join(golden_dir, "ref_tiny_f32.npz"))
    cfg = synth.CONFIGS["tiny_f32"]
    case = GpuCase(cfg, int(g["seed"]))
    try:
        out = case.run().cpu().numpy()
        r = case.launcher.routing(cfg.T)
        assert np.array_equal(r["topk_idx"], g["topk_idx"])
        np.testing.assert_allclose(r["topk_w"], g["topk_w"], rtol=2e-6)
        assert np.max(np.abs(out - g["out"])) <= 2e-5 * np.max(np.abs(g["out"]))
    finally:
        case.close()


# AUTO takes the streaming variant at this size; the tiled one is asked for by name
@pytest.mark.parametrize("seed,sched", [(7907, _lib.SCHED_STREAM), (1, _lib.SCHED_STREAM),
                                        (2, _lib.SCHED_STREAM), (7907, _lib.SCHED_AUTO), (7907, _lib.SCHED_TILED)])
def test_qwen3_30b_decode(seed, sched):
    run_case(synth.CONFIGS["qwen3_30b_decode"], seed=seed, sched=sched)


@pytest.mark.parametrize("sched", [_lib.SCHED_STREAM, _lib.SCHED_TILED])
def test_qwen3_30b_decode_inplace(sched):
    run_case(synth.CONFIGS["qwen3_30b_decode"], inplace=True, sched=sched)


@pytest.mark.parametrize("sched", [_lib.SCHED_STREAM, _lib.SCHED_TILED])
@pytest.mark.parametrize("T", [1, 3, 17, 65, 130])
def test_ragged_token_counts_bf16(T, sched):
    cfg = synth.CONFIGS["qwen3_30b_decode"].replace(T=T, name="ragged")
    run_case(cfg, seed=T, sched=sched)


@pytest.mark.parametrize("shape", [
    # T, H, E, k, I, dtype
    (5, 64, 16, 4, 32, "f32"),
    (7, 128, 8, 8, 64, "f32"),      # k == E
    (33, 256, 32, 1, 96, "bf16"),   # top-1
    (40, 192, 200, 6, 160, "bf16"),  # E not a multiple of 64
    (100, 64, 4, 2, 32, "bf16"),    # > 64 rows per expert: several row tiles
    (64, 64, 4, 2, 32, "bf16"),     # small batch whose experts get ~32 rows: early tasks re-run with more row blocks
    (48, 128, 2, 1, 64, "bf16"),    # ~24 rows per expert, top-1
    (60, 128, 3, 3, 64, "f32"),     # k == E: 60 rows in every expert
])
def test_odd_shapes(shape):
    T, H, E, k, I, dt = shape
    run_case(synth.MoeConfig("odd", T, H, E, k, I, dt), seed=T + H)


@pytest.mark.parametrize("shape", [
    # T, H, E, k, I, hot: bf16 layers with H % 256 == 0 run the logit chains on the
    # matrix core, 16 tokens x 16 experts per workgroup, in stages of 256 k whose
    # loads go out eight stages at a time
    (17, 768, 24, 3, 64, 0),      # three stages; last token group and last expert group partly empty
    (65, 2304, 60, 5, 96, 0),     # nine stages: a second, short batch of loads
    (130, 512, 200, 6, 160, 0),   # 9 x 13 groups
    (1, 4096, 16, 2, 64, 0),      # one token, sixteen stages
    (200, 1024, 48, 4, 64, 3),    # router bias
    (40, 768, 24, 3, 64, 0),      # early gate/up tasks (T <= 64, T*k >= E) behind the same router
    (64, 512, 72, 8, 32, 2),      # the same with 4.5 expert groups and a bias
    (60, 256, 16, 2, 64, 2),      # early tasks; the two hot experts hold far more than 16 rows and start over
    (150, 512, 128, 8, 64, 0),    # early tasks behind three 64-token mask words
    (150, 256, 64, 4, 64, 1),     # early tasks; the hot expert holds all 150 tokens: its one tile is walked in 64-row steps
    (100, 512, 128, 8, 32, 2),    # the same with two hot experts of 100 rows
    (250, 512, 128, 8, 64, 0),    # 12 to 24 rows per expert: early tasks of two row blocks
    (230, 256, 64, 4, 64, 1),     # the same with a hot expert of 230 rows
])
def test_matrix_core_router_shapes(shape):
    T, H, E, k, I, hot = shape
    run_case(synth.MoeConfig("mcr", T, H, E, k, I, "bf16", hot=hot), seed=T + E)


def test_router_bias_hot_experts_small():
    cfg = synth.MoeConfig("hot", 256, 256, 16, 4, 64, "bf16", hot=2)
    run_case(cfg, seed=3)


def test_relaunch_and_smaller_batch():
    """Counters return to zero by themselves: launch twice, then a smaller batch."""
    cfg = synth.CONFIGS["qwen3_30b_decode"]
    case = GpuCase(cfg, sched=_lib.SCHED_STREAM)
    try:
        x = case.inp["tokens"]
        a = case.run()
        b = case.run()
        assert torch.equal(a, b)
        small = x[:20].contiguous()
        c = case.run(tokens=small)
        r = case.launcher.routing(20)
        case.check_routing(small, r)
        assert torch.equal(c, a[:20])       # tokens are independent
        assert case.launcher.status() == (0, 3)
    finally:
        case.close()


@pytest.mark.parametrize("sched", [_lib.SCHED_STREAM, _lib.SCHED_AUTO])
def test_relaunch_across_batch_sizes(sched):
    """One launcher, batches that take different paths one after the other (early
    gate/up tasks, the ordinary ticket order, one token, and with AUTO the tiled
    variant): every launch leaves the counters as the next one needs them."""
    cfg = synth.MoeConfig("seq", 600, 512, 64, 4, 128, "bf16")
    case = GpuCase(cfg, seed=11, sched=sched)
    try:
        x = case.inp["tokens"]
        full = case.run()
        case.check_routing(x, case.launcher.routing(cfg.T))
        case.check_outputs(x, full, np.arange(0, cfg.T, 7))
        for T in (150, 600, 40, 1, 190, 300, 64):
            part = x[:T].contiguous()
            out = case.run(tokens=part)
            case.check_routing(part, case.launcher.routing(T))
            case.check_outputs(part, out, np.arange(0, T, 3))
        assert case.launcher.status()[0] == 0
    finally:
        case.close()


@pytest.mark.parametrize("shape", [
    # T, H, E, k, I: the tiled variant (MFMA 16x16x32, both of its pipelines) forced on small problems
    (300, 256, 8, 2, 128),      # ragged last row tile (75 rows per expert on average)
    (700, 512, 4, 2, 256),      # several 256-row tiles per expert, ragged tail
    (64, 256, 200, 6, 128),     # E > 128: two expert slabs in the router; tiny tiles
    (1, 256, 8, 2, 128),        # a single token
    (1100, 256, 8, 2, 128),     # ~275 rows per expert: tall tiles (a tail of <= 64 rows joins the full tile)
    (1180, 512, 4, 1, 256),     # ~295 rows per expert, top-1; some experts beyond 320 rows (tile + tail tile)
    (4100, 256, 200, 6, 128),   # more than one round of 16-token router tasks: 32-token tasks, two expert slabs, ragged last task
    (900, 768, 8, 2, 384),      # twelve and six 64-k stages: the packed weights' deeper pipeline past its first and last stages
    (2500, 512, 8, 1, 640),     # ~312 rows per expert: tiles of nine and ten 32-row blocks on three token buffers
])
def test_tiled_variant_forced(shape):
    T, H, E, k, I = shape
    cfg = synth.MoeConfig("tiled", T, H, E, k, I, "bf16")
    print("tiled forced", shape, flush=True)
    case = GpuCase(cfg, seed=T + E, sched=_lib.SCHED_TILED)
    try:
        assert case.launcher.sched_for(T) == _lib.SCHED_TILED
        x = case.inp["tokens"]
        out = case.run()
        case.check_routing(x, case.launcher.routing(T))
        err = case.check_outputs(x, out)
        print("  max rel err %.3e" % err, flush=True)
        # the streaming variant on the same inputs agrees on routing bit for bit
        other = GpuCase(cfg, seed=T + E, sched=_lib.SCHED_STREAM, inputs=case.inp)
        try:
            out2 = other.run()
            r1, r2 = case.launcher.routing(T), other.launcher.routing(T)
            assert np.array_equal(r1["topk_idx"], r2["topk_idx"])
            assert np.array_equal(r1["perm"], r2["perm"])
            # Outputs: the streaming variant sums float rows and rounds once; the tiled one
            # rounds each slot's down-projection row to bf16 first (relative 2^-9 each, the
            # weights sum to 1), then both round the sum to bf16. Per token the two may
            # therefore differ by a bf16 ulp or two (2^-7 relative) of the row's largest
            # element, and by no more.
            a, b = out.float(), out2.float()
            ulp = a.abs().max(dim=1, keepdim=True).values * 2.0 ** -7
            worst = float(((a - b).abs() / ulp).max())
            print("  tiled vs streaming: %.2f bf16 ulps of the row maximum" % worst, flush=True)
            assert worst <= 2.0          # measured: at most 1.00
        finally:
            other.close()
        # the tiled variant reading the packed weight copy computes the same bits
        packed = GpuCase(cfg, seed=T + E, sched=_lib.SCHED_TILED, inputs=case.inp, pack_weights=True)
        try:
            assert packed.launcher.sched_for(T) == _lib.SCHED_TILED
            assert torch.equal(packed.run(), out)
        finally:
            packed.close()
    finally:
        case.close()


@pytest.mark.parametrize("rows", [1, 33, 64, 65, 96, 97, 128, 129, 160, 161, 192, 193, 224, 225, 256, 257, 288,
                                  289, 320, 321, 640, 641, 961])
@pytest.mark.parametrize("I", [128, 192 * 2, 640])
def test_tiled_tile_heights(rows, I):
    """Every number of 32-row blocks a tile can have, at both edges, alone and as one of several tiles
    of an expert (k == E: both experts hold every row), with 2,
    6 and 10 stages of 64 k in the down projection and 4 in the gate/up one: on row-major weights
    against the oracle, and the packed weights must give the same bits (through the register-staged
    pipeline with two sets of registers, but for the 2 stages and tiles of more than 256 rows)."""
    check_tile_heights(rows, 256, I)


@pytest.mark.parametrize("rows", [1, 33, 64])
@pytest.mark.parametrize("H,I", [(512, 512), (2304, 2048), (2048, 2304)])
def test_tiled_short_tiles_of_many_stages(rows, H, I):
    """Tiles of up to 64 rows with 32 and 36 stages of 64 k, where the register-staged pipeline takes
    four sets of registers, and with 8, where it still takes two."""
    check_tile_heights(rows, H, I)


@pytest.mark.parametrize("rows", [1, 70, 161, 300, 330])
@pytest.mark.parametrize("H,I", [(128, 128), (192, 160), (320, 224), (448, 352), (576, 672), (64 * 9, 32 * 9)])
def test_tiled_ragged_columns(rows, H, I):
    """Hidden sizes that are no multiple of a task's 256 columns and intermediate sizes that are none of
    its 128 (a wave's columns exist or not as a whole), with k an even or an odd number of 32-k steps
    (the last stage of the odd ones starts 32 k early and multiplies its second half only; h rows are
    padded to whole lines), on every depth of the staged pipeline."""
    check_tile_heights(rows, H, I)


@pytest.mark.parametrize("T,H,E,k,I,hot,edges", [
    (70, 192, 2, 2, 160, 0, False),       # one tile of three 32-row blocks; odd 32-k steps
    (161, 320, 2, 2, 224, 0, True),       # k of 3.5 stages; norm and residual
    (330, 448, 2, 2, 352, 0, False),      # two tiles an expert
    (330, 576, 5, 3, 672, 2, False),
    (400, 512, 4, 2, 160, 0, False),      # only I is ragged
    (900, 320, 16, 2, 256, 3, True),      # only H is, in no whole stage of the logit chains
    (70000, 128, 4, 1, 160, 0, False),    # beyond the short prologue
])
@pytest.mark.parametrize("packed", [False, True])
def test_tiled_ragged_equals_the_streaming_variant(T, H, E, k, I, hot, edges, packed):
    """Layers whose columns do not divide into the tiled variant's tasks are held in as many bits there as in
    the streaming variant, which serves their small batches: the same sums in the same order, float rows that
    carry their gate weight, one rounding. So the same bits."""
    cfg = synth.MoeConfig("ragged", T, H, E, k, I, "bf16", hot=hot)
    print("ragged", T, H, E, k, I, packed, flush=True)
    dev = torch.device("cuda:0")
    norm = synth.normal_torch(5, 9, (H,), 0.25, torch.float32, dev).add_(1.0).to(torch.bfloat16) if edges else None
    make = lambda sched, inputs: GpuCase(cfg, seed=T + I, sched=sched, inputs=inputs, pack_weights=packed,
                                         norm_weight=norm, residual=edges)
    a = make(_lib.SCHED_STREAM, None)
    try:
        assert a.launcher.split_blocks_for(T) == 0
        want = a.run()
        b = make(_lib.SCHED_TILED, a.inp)
        try:
            assert b.launcher.sched_for(T) == _lib.SCHED_TILED
            assert torch.equal(b.run(), want)
            assert torch.equal(b.run(), want)
        finally:
            b.close()
    finally:
        a.close()


def tiled_start(case):
    """How the tiled kernel gets from tokens to row tiles, and its records of kind 0 (logits) and 6 (selections), from a
    traced launch, which starts as one without a trace does."""
    case.launcher.trace_enable(1 << 17)
    case.run()
    kinds = np.bincount(case.launcher.trace_read()["kind"], minlength=7)
    case.launcher.trace_enable(0)
    return "tickets" if kinds[1] else "chains" if kinds[6] else "tokens", int(kinds[0]), int(kinds[6])


# chains: logit chains of 16 tokens x 32 experts, on 256 workgroups; tokens: router tasks of all experts, in slabs of 128;
# tickets: router, scan and scatter one after the other
@pytest.mark.parametrize("T,H,E,k,start", [
    (40, 128, 17, 3, "tokens"),
    (1000, 192, 33, 2, "tokens"),
    (1536, 320, 70, 8, "tokens"),
    (1537, 320, 70, 8, "tokens"),
    (1000, 512, 256, 6, "tokens"),
    (1536, 768, 33, 2, "tokens"),
    (1537, 768, 33, 2, "tokens"),
    (2048, 128, 256, 2, "tokens"),    # the last size whose mask words fit LDS
    (2049, 128, 256, 2, "tickets"),   # the first whose do not
    (40, 768, 17, 3, "chains"),       # a group of experts with one expert
    (1000, 832, 33, 2, "chains"),     # a last 256-k stage that is partly empty
    (1024, 768, 100, 4, "tokens"),
    (1025, 768, 100, 4, "tokens"),
    (1024, 1024, 100, 4, "chains"),   # 256 workgroups with a chain task each
    (1025, 1024, 100, 4, "tokens"),   # one slab does not pay for a second round
    (513, 512, 64, 4, "chains"),
    (512, 256, 64, 4, "chains"),      # the last size that needs no more than 256 k
    (513, 256, 64, 4, "tokens"),
    (512, 192, 64, 4, "tokens"),      # less than 256 k
    (509, 128, 200, 17, "chains"),    # two slabs of 128 k; a last selection of one token
    (557, 384, 200, 6, "chains"),     # two slabs against one round
    (600, 384, 200, 6, "chains"),     # ... against two rounds, of which the second is short
    (900, 1024, 160, 4, "chains"),
    (1040, 1728, 256, 4, "chains"),   # ... against three
    (1040, 1664, 256, 4, "tokens"),   # chains too short for that
    (4096, 2176, 8, 1, "chains"),     # a selection for every wave of the launch
    (4097, 2176, 8, 1, "tokens"),     # router tasks of 32 tokens, the last of one
])
def test_tiled_starts(T, H, E, k, start):
    """The ways the tiled kernel gets from tokens to row tiles, at the edges of their ranges: routing
    tables bit for bit, outputs against the oracle, and the same from a second launch."""
    cfg = synth.MoeConfig("starts", T, H, E, k, 128, "bf16", hot=3)
    print("tiled starts", T, H, E, k, start, flush=True)
    case = GpuCase(cfg, seed=T + E, sched=_lib.SCHED_TILED)
    try:
        assert case.launcher.sched_for(T) == _lib.SCHED_TILED
        out = case.run()
        case.check_routing(case.inp["tokens"], case.launcher.routing(T))
        case.check_outputs(case.inp["tokens"], out, nthreads=4)
        assert torch.equal(case.run(), out)
        up = lambda a, b: -(-a // b)
        got = tiled_start(case)
        assert got[0] == start
        if start == "chains":
            assert got[1:] == (up(T, 16) * up(E, 32), up(T, 4))
    finally:
        case.close()


@pytest.mark.parametrize("T,H,E,k,start", [
    (4099, 192, 128, 32, "tickets"),  # 32-token router tasks, the last of 3 tokens; the most slots
    (4100, 128, 200, 17, "tickets"),  # two slabs of experts, the second partly empty; more slots than a row has lanes
    (2100, 64, 40, 5, "streaming"),   # too few k for the tiled variant: one token to a wave
    (2100, 128, 40, 5, "tokens"),     # 16-token tasks, the last of 4 tokens
    (601, 128, 200, 17, "tokens"),    # ... of two slabs; the last of 9 tokens
    (509, 128, 200, 17, "chains"),    # selections spread over the workgroups, the last of one token
    (511, 256, 120, 17, "chains"),    # ... of three tokens
    (407, 128, 200, 17, "chains"),    # ... of two tokens a wave, the last of one
    (409, 128, 200, 17, "chains"),    # the first size of so many winners with four; the last of one token
    (32, 256, 120, 32, "split-k"),    # every workgroup picks the winners, four tokens to each of its waves
    (32, 256, 200, 1, "split-k"),     # ... of which each lane holds 16 experts
    (16, 256, 256, 9, "split-k"),     # ... two tokens
    (15, 512, 129, 32, "split-k"),    # ... the last wave one
    (17, 256, 256, 9, "split-k"),     # the first size of more than 128 experts whose winners are picked once
    (32, 256, 200, 32, "split-k"),
    (33, 256, 120, 17, "split-k"),    # the first size whose winners are picked once
    (1, 256, 97, 32, "split-k"),
])
@pytest.mark.parametrize("admitted", ["all", "three"])
def test_router_winners(T, H, E, k, start, admitted):
    """Equal logits (every expert's row of the router weights twice, so the lower index wins) and experts that
    are never admitted (a bias of -inf leaves three, fewer than k): winners and weights against the oracle."""
    cfg = synth.MoeConfig("winners", T, H, E, k, 128, "bf16")
    print("winners", T, H, E, k, start, admitted, flush=True)
    inp = synth.make_inputs_torch(cfg, T + k, torch.device("cuda:0"))
    inp["gate"][E // 2:2 * (E // 2)] = inp["gate"][:E // 2].clone()
    if admitted == "three":
        inp["bias"] = torch.full((E,), -float("inf"), device="cuda:0")
        inp["bias"][[1, E // 2 + 1, E - 1]] = 0.0
    case = GpuCase(cfg, sched=_lib.SCHED_AUTO if start == "split-k" else _lib.SCHED_TILED, inputs=inp)
    tiled = start in ("chains", "tokens", "tickets")
    try:
        assert (case.launcher.sched_for(T) == _lib.SCHED_TILED) == tiled
        assert (case.launcher.split_blocks_for(T) != 0) == (start == "split-k")
        case.run()
        routing = case.launcher.routing(T)
        if tiled:
            got = tiled_start(case)
            assert got[0] == start
            if start == "chains":
                assert got[2] == -(-T // (2 if E > 128 and T <= 24 * k else 4))
        hw = case.host_weights()
        idx, w = oracle.gate(inp["tokens"].float().cpu().numpy(), hw["gate"], k, bias=hw["bias"])
        assert (idx < 0).any() == (admitted == "three" and k > 3)
        assert np.array_equal(routing["topk_idx"], idx)
        np.testing.assert_allclose(routing["topk_w"], w, rtol=2e-6, atol=1e-7)  # as in GpuCase.check_routing
    finally:
        case.close()


def check_tile_heights(rows, H, I):
    cfg = synth.MoeConfig("heights", rows, H, 2, 2, I, "bf16")
    print("tile heights", rows, H, I, flush=True)
    case = GpuCase(cfg, seed=rows + I, sched=_lib.SCHED_TILED)
    try:
        out = case.run()
        case.check_routing(case.inp["tokens"], case.launcher.routing(rows))
        case.check_outputs(case.inp["tokens"], out, nthreads=4)
        packed = GpuCase(cfg, seed=rows + I, sched=_lib.SCHED_TILED, inputs=case.inp, pack_weights=True)
        try:
            assert torch.equal(packed.run(), out)
        finally:
            packed.close()
    finally:
        case.close()


@pytest.mark.parametrize("rows,H,I", [
    (1, 128, 128), (15, 128, 128), (16, 192, 160), (17, 320, 224), (33, 128, 288), (49, 448, 128), (64, 256, 352),
    (65, 576, 672), (81, 64 * 9, 32 * 9), (96, 256, 256), (97, 320, 160), (193, 192, 224), (400, 512, 416),
])
def test_tiled_float32(rows, H, I):
    """The float32 tiled kernel at the edges of its tiles (16 to 96 rows), column blocks (128 of I, 256 of
    H) and k (even and odd numbers of 32-k steps): row-major weights against the oracle, and the packed
    copy must give the same bits."""
    cfg = synth.MoeConfig("tiled_f32", rows, H, 2, 2, I, "f32")
    print("tiled float32", rows, H, I, flush=True)
    case = GpuCase(cfg, seed=rows + I, sched=_lib.SCHED_TILED)
    try:
        assert case.launcher.sched_for(rows) == _lib.SCHED_TILED
        out = case.run()
        case.check_routing(case.inp["tokens"], case.launcher.routing(rows))
        case.check_outputs(case.inp["tokens"], out, nthreads=4)
        assert torch.equal(case.run(), out)
        packed = GpuCase(cfg, seed=rows + I, sched=_lib.SCHED_TILED, inputs=case.inp, pack_weights=True)
        try:
            assert torch.equal(packed.run(), out)
        finally:
            packed.close()
    finally:
        case.close()


@pytest.mark.parametrize("H,I,one_a_cu", [(512, 256, True), (512, 288, False), (576, 256, False)])
def test_tiled_float32_one_workgroup_a_cu(H, I, one_a_cu):
    """128 row tiles: with two tasks each in both projections there are as many as CUs, and the first workgroup of
    each takes them; with three in either everybody draws."""
    cfg = synth.MoeConfig("one_a_cu", 640, H, 128, 2, I, "f32")
    print("tiled float32, tasks", H, I, flush=True)
    case = GpuCase(cfg, seed=H + I, sched=_lib.SCHED_TILED)
    try:
        out = case.run()
        case.check_routing(case.inp["tokens"], case.launcher.routing(640))
        case.check_outputs(case.inp["tokens"], out, nthreads=4)
        case.launcher.trace_enable(1 << 14)
        assert torch.equal(case.run(), out)
        rec = case.launcher.trace_read()
        case.launcher.trace_enable(0)
        for kind, tasks in ((3, 128 * -(-I // 128)), (4, 128 * -(-H // 256))):
            at = rec[rec["kind"] == kind]
            assert len(at) == tasks
            if one_a_cu:
                assert at["worker"].max() < torch.cuda.get_device_properties(0).multi_processor_count
    finally:
        case.close()


def same_values(want, got, scale=None):
    """The same infinities and NaN, and finite values within the tolerance of float32 layers, each against
    the root mean square of its own token row (or of `scale`, a part of its columns)."""
    assert torch.equal(torch.isnan(want), torch.isnan(got))
    assert torch.equal(torch.isposinf(want), torch.isposinf(got)) and torch.equal(torch.isneginf(want), torch.isneginf(got))
    fin = torch.isfinite(want)
    w, g = torch.where(fin, want, 0.0).double(), torch.where(fin, got, 0.0).double()
    part = slice(None) if scale is None else scale
    rms = (w[:, part].pow(2).sum(1, keepdim=True) / fin[:, part].sum(1, keepdim=True).clamp(min=1)).sqrt()
    worst = ((w - g).abs() - 2e-5 * w.abs() - 2e-5 * rms)[:, part]
    assert float(worst.max()) <= 0.0


def test_tiled_float32_values_without_bf16_parts():
    """Infinities, NaN, values that round to infinity in bf16 and tiny ones among the expert weights: the
    float32 tiled kernel gives what the streaming kernel's float32 instructions give, element by element:
    the same infinities and NaN, and finite values within the tolerance of float32 layers."""
    cfg = synth.MoeConfig("tiled_f32", 300, 256, 8, 2, 160, "f32")
    dev = torch.device("cuda:0")
    inp = synth.make_inputs_torch(cfg, 5, dev)
    f1, f2 = inp["ffn1"], inp["ffn2"]
    f1[0, 3, 7] = float("inf")
    f1[0, cfg.I + 70, 250] = -float("inf")
    f1[1, 5, 9] = float("nan")
    f1[2, 11, 0] = 3.4e38
    f1[2, cfg.I + 11, 1] = 1e-38
    f2[2, 17, 3] = float("inf")
    ref = GpuCase(cfg, seed=5, sched=_lib.SCHED_STREAM, inputs=inp)
    case = GpuCase(cfg, seed=5, sched=_lib.SCHED_TILED, inputs=inp)
    try:
        want, got = ref.run(), case.run()
        assert torch.isnan(want).any() and torch.isinf(want).any() and torch.isfinite(want).any()
        same_values(want, got)
        # rows that no such weight reaches: a wrong ordinary value shows
        assert int((torch.isfinite(want).all(1) & (want.abs().amax(1) < 1e3)).sum()) >= 5
        broken = got + 1e-3 * (got.abs() < 1e3)
        with pytest.raises(AssertionError):
            same_values(want, broken)
    finally:
        case.close()
        ref.close()


def test_tiled_float32_tiny_weights():
    """Down rows of 1e-28 to 1e-36 of the usual size, one expert a token, so that nothing larger is added: the
    streaming kernel's values, also where the low parts of such weights are beyond bf16. The same for up rows,
    and zeros among them stay zeros."""
    cfg = synth.MoeConfig("tiled_f32", 90, 256, 3, 1, 160, "f32")
    inp = synth.make_inputs_torch(cfg, 6, torch.device("cuda:0"))
    inp["ffn2"][:, 20:40] *= 1e-28
    inp["ffn2"][:, 40:120] *= 1e-30
    inp["ffn2"][:, 128:160] *= 1e-33
    inp["ffn2"][:, 160:200] *= 1e-35
    inp["ffn2"][:, 200:210] = 0.0
    inp["ffn2"][:, 210:220] *= 1e-36
    inp["ffn1"][:, cfg.I + 40:cfg.I + 60] *= 1e-35
    ref = GpuCase(cfg, seed=6, sched=_lib.SCHED_STREAM, inputs=inp)
    case = GpuCase(cfg, seed=6, sched=_lib.SCHED_TILED, inputs=inp)
    try:
        want, got = ref.run(), case.run()
        assert 0.0 < float(want[:, 40:120].abs().max()) < 1e-29 and 0.0 < float(want[:, 210:220].abs().max()) < 1e-35
        assert not got[:, 200:210].any()
        for part in ((0, 20), (20, 40), (40, 120), (120, 128), (128, 160), (160, 200), (210, 220), (220, 256)):
            print("  columns", part, flush=True)
            same_values(want, got, slice(*part))
        rows = int(ref.launcher.routing(cfg.T)["counts"].sum())
        h = [torch.from_numpy(np.array(c.launcher.intermediate(cfg.T)))[:rows] for c in (ref, case)]
        same_values(*h, slice(0, 40))
        same_values(*h, slice(40, 60))
    finally:
        case.close()
        ref.close()


@pytest.mark.parametrize("T,k,H,I,every", [(40, 1, 128, 128, 0), (97, 2, 192, 160, 0), (200, 2, 320, 224, 0),
                                           (290, 1, 448, 288, 0), (97, 3, 192, 160, 5), (290, 3, 320, 224, 3), (96, 3, 128, 128, 1)])
def test_tiled_float32_infinite_tokens(T, k, H, I, every):
    """Tokens that hold infinities or values beyond bf16, in the first, a middle and the last row of tiles of
    one to six row blocks, a few of a tile or (`every`) more than the 16 rows that are multiplied again
    together: the gate/up rows and the outputs of the streaming kernel, those of the tokens beside them included."""
    cfg = synth.MoeConfig("tiled_f32", T, H, 3, k, I, "f32")
    print("tiled float32, infinite tokens", T, k, H, I, every, flush=True)
    inp = synth.make_inputs_torch(cfg, T, torch.device("cuda:0"))
    x = inp["tokens"]
    x[0, 5], x[T // 2, H - 1], x[T - 1, 64] = float("inf"), -float("inf"), 3.4e38
    if every:
        x[::every, 9] = float("inf")
    ref = GpuCase(cfg, seed=T, sched=_lib.SCHED_STREAM, inputs=inp)
    case = GpuCase(cfg, seed=T, sched=_lib.SCHED_TILED, inputs=inp)
    try:
        want, got = ref.run(), case.run()
        same_values(want, got)
        rows = int(ref.launcher.routing(T)["counts"].sum())  # (no expert is chosen for a logit of minus infinity)
        h = [torch.from_numpy(np.array(c.launcher.intermediate(T)))[:rows] for c in (ref, case)]
        assert not torch.isfinite(h[0]).all()
        same_values(*h)
    finally:
        case.close()
        ref.close()


def test_tiled_float32_infinite_tokens_hold_up_no_one_else():
    """One infinite token sends a row block of each of its experts through the float32 instructions again, a
    wave on its own. The launch may take 1.5 times as long for that."""
    cfg = synth.MoeConfig("tiled_f32", 320, 2048, 16, 2, 768, "f32")
    case = GpuCase(cfg, seed=3, sched=_lib.SCHED_TILED)
    try:
        x, out = case.inp["tokens"], torch.empty_like(case.inp["tokens"])

        def us():
            times = []
            for _ in range(25):
                a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                a.record()
                case.launcher.launch(x, out)
                b.record()
                b.synchronize()
                times.append(a.elapsed_time(b) * 1e3)
            return sorted(times)[12]

        us()
        plain = us()
        x[100, 5] = float("inf")
        poisoned = us()
        print("  %.0f us, with an infinite token %.0f" % (plain, poisoned), flush=True)
        assert not torch.isfinite(out[100]).any() and torch.isfinite(out[:100]).all()
        assert poisoned <= 1.5 * plain
    finally:
        case.close()


@pytest.mark.parametrize("dtype,E,k,H,I", [("bf16", 16, 2, 512, 4096), ("f32", 16, 2, 512, 2048), ("bf16", 12, 3, 256, 8192)])
@pytest.mark.parametrize("packed", [False, True])
def test_split_k_down_rows_of_8_kib(dtype, E, k, H, I, packed):
    """Down rows of whole 8 KiB are walked in equal stretches by batches that reach most experts, as by smaller
    ones. (With one run of gate/up steps a wave, those are the same in both:) a token's sums are the same bits."""
    cfg = synth.MoeConfig("stretches", 2 * E, H, E, k, I, dtype)
    case = GpuCase(cfg, seed=I, pack_weights=packed)
    try:
        small = (E - 1) // k
        assert case.launcher.split_blocks_for(small) == case.launcher.split_blocks_for(cfg.T) == 1
        out = case.run()
        case.check_outputs(case.inp["tokens"], out)
        assert torch.equal(case.run(tokens=case.inp["tokens"][:small].contiguous()), out[:small])
    finally:
        case.close()


@pytest.mark.parametrize("E,k,H,I,split,stream", [
    (128, 8, 4096, 640, (1, 8, 15), (16, 24, 32, 128)),   # 2560 gate/up tasks for 256 CUs
    (128, 8, 4096, 608, (1, 16, 31), (32, 64)),           # 2432
    (16, 2, 4096, 4096, (1, 8, 15), (16, 64)),
    (128, 8, 4032, 640, (1, 16, 32, 128), ()),            # rows of another pitch
])
def test_row_major_float32_rows_of_16_kib(E, k, H, I, split, stream):
    """Row-major float32 layers whose gate/up rows are whole 16 KiB leave the split-k kernel to smaller batches:
    from two rows an expert on, and from one where a workgroup has ten tasks. Packed ones do not."""
    dev = torch.device("cuda:0")
    w = [torch.empty(s, dtype=torch.float32, device=dev) for s in ((E, H), (E, 2 * I, H), (E, H, I))]  # never read
    for packed in (False, True):
        l = MoeKernelLauncher()
        l.create(*w, 256, l.getDistributedUniqueId(True), 0, 1, top_k=k, pack_weights=False, prepacked=packed)
        try:
            assert [l.split_blocks_for(t) for t in split] == [1] * len(split)
            assert [l.split_blocks_for(t) for t in stream] == [int(packed)] * len(stream)
        finally:
            l.destroy()


@pytest.mark.parametrize("dtype,packed,E,k,H,I,rows", [
    ("f32", True, 128, 8, 512, 256, 10), ("f32", True, 64, 4, 512, 256, 10), ("f32", True, 16, 2, 512, 2048, 10),
    ("f32", True, 60, 4, 512, 512, 14), ("f32", True, 39, 4, 512, 512, 16), ("f32", True, 8, 2, 1024, 1024, 16),
    ("f32", False, 96, 4, 512, 2048, 10), ("f32", False, 64, 4, 512, 1024, 10), ("f32", False, 64, 4, 512, 1408, 16),
    ("f32", False, 40, 5, 1344, 736, 16), ("f32", False, 32, 4, 512, 768, 22), ("f32", False, 16, 2, 512, 2048, 22),
    ("f32", False, 8, 2, 512, 2048, 26), ("f32", False, 8, 2, 512, 1792, 22),
    ("bf16", False, 40, 5, 1344, 736, 14), ("bf16", False, 24, 3, 640, 2016, 20), ("bf16", False, 16, 2, 320, 160, 26),
    ("bf16", True, 16, 2, 320, 160, 26),
])
def test_auto_takes_the_tiled_variant_from_its_line_on(dtype, packed, E, k, H, I, rows):
    """Layers with few tasks stay on the streaming variant for more rows an expert."""
    dt, dev = torch.bfloat16 if dtype == "bf16" else torch.float32, torch.device("cuda:0")
    w = [torch.empty(s, dtype=dt, device=dev) for s in ((E, H), (E, 2 * I, H), (E, H, I))]  # never read
    l = MoeKernelLauncher()
    line = -(-rows * E // k)
    l.create(*w, line + 1, l.getDistributedUniqueId(True), 0, 1, top_k=k, pack_weights=False, prepacked=packed)
    try:
        assert [l.sched_for(t) for t in (line - 1, line, line + 1)] == [_lib.SCHED_STREAM] + [_lib.SCHED_TILED] * 2
    finally:
        l.destroy()


@pytest.mark.parametrize("E,k,last", [(128, 4, 256), (96, 4, 336), (64, 2, 512)])
def test_auto_row_major_leaves_the_streaming_variant_with_the_split_k_kernel(E, k, last):
    """AUTO sends row-major bf16 batches of 14 to 24 rows an expert to the streaming variant for its
    split-k kernel only. That kernel starts with at most half of the 256 CUs on the logit chains
    (16 tokens x 16 experts each): `last` tokens. From 14 rows an expert on, a batch it does not
    start for is the tiled variant's, and so is every one of them while a trace is written."""
    cfg = synth.MoeConfig("auto", 24 * E // k, 256, E, k, 128, "bf16")
    line = -(-14 * E // k)   # tokens from which an expert has 14 rows on average
    case = GpuCase(cfg, seed=E)
    try:
        sched = case.launcher.sched_for
        above = max(last + 1, line)
        print("row-major AUTO", E, k, "split-k up to", last, "tiled from", above, flush=True)
        assert sched(last) == _lib.SCHED_STREAM
        assert [sched(t) for t in (above, above + 16, cfg.T)] == [_lib.SCHED_TILED] * 3
        x = case.inp["tokens"]
        out = case.run()
        case.check_routing(x, case.launcher.routing(cfg.T))
        case.check_outputs(x, out, nthreads=4)
        case.launcher.trace_enable(1 << 16)
        assert sched(line) == _lib.SCHED_TILED
        case.launcher.trace_enable(0)
        assert sched(line) == (_lib.SCHED_STREAM if line <= last else _lib.SCHED_TILED)
    finally:
        case.close()


@pytest.mark.parametrize("name,T", [("qwen3_30b_decode", 64), ("qwen3_30b_decode", 100),
                                    ("tiny_f32", 16)])
def test_packed_weights_equal_unpacked(name, T):
    """The packed second copy of the expert weights changes where bytes are read
    from, not what is computed."""
    cfg = synth.CONFIGS[name].replace(T=T)
    a = GpuCase(cfg, seed=11, sched=_lib.SCHED_STREAM)
    try:
        b = GpuCase(cfg, seed=11, sched=_lib.SCHED_STREAM, inputs=a.inp, pack_weights=True)
        try:
            out_a, out_b = a.run(), b.run()
            assert torch.equal(out_a, out_b)
            b.check_routing(b.inp["tokens"], b.launcher.routing(T))
            b.check_outputs(b.inp["tokens"], out_b, None if T <= 64 else np.arange(0, T, 7))
            # refresh after an in-place weight change
            b.inp["ffn2"].mul_(2.0)
            b.launcher.refresh_weights()
            a_out2, b_out2 = a.run(), b.run()
            assert torch.equal(a_out2, b_out2)
            b.inp["ffn2"].mul_(0.5)
        finally:
            b.close()
    finally:
        a.close()


@pytest.mark.parametrize("name,T,sched", [("qwen3_30b_decode", 64, _lib.SCHED_STREAM),
                                          ("qwen3_30b_decode", 700, _lib.SCHED_TILED),
                                          ("tiny_f32", 16, _lib.SCHED_STREAM),
                                          # several row tiles an expert: their tasks share the weights
                                          ("qwen3_30b_decode", 1500, _lib.SCHED_STREAM),
                                          ("tiny_f32", 600, _lib.SCHED_STREAM)])
def test_prepacked_weights_equal_unpacked(name, T, sched):
    """Weights packed in place by the caller (no second copy anywhere, the
    launcher's workspace holds no weight-sized region) give the same bits as the
    row-major tensors and as the launcher's own packed copy."""
    import ctypes

    cfg = synth.CONFIGS[name].replace(T=T)
    a = GpuCase(cfg, seed=11, sched=sched)
    try:
        out_a = a.run()
        packed_inp = dict(a.inp)
        packed_inp["ffn1"] = a.inp["ffn1"].clone()
        packed_inp["ffn2"] = a.inp["ffn2"].clone()
        a.launcher.pack_weights_in_place(packed_inp["ffn1"], packed_inp["ffn2"])
        torch.cuda.synchronize()
        assert not torch.equal(packed_inp["ffn1"], a.inp["ffn1"])     # it really is another layout
        b = GpuCase(cfg, seed=11, sched=sched, inputs=packed_inp, prepacked=True)
        try:
            assert torch.equal(b.run(), out_a)
            b.check_routing(b.inp["tokens"], b.launcher.routing(T))
            # workspace: nothing weight-sized
            d = _lib.LayerDesc()
            d.experts, d.hidden, d.intermediate, d.top_k = cfg.E, cfg.H, cfg.I, cfg.k
            d.dtype = _lib.BF16 if cfg.dtype == "bf16" else _lib.F32
            d.max_tokens, d.sched, d.flags = T, sched, _lib.FLAG_WEIGHTS_PREPACKED
            n_pre, n_copy = ctypes.c_size_t(0), ctypes.c_size_t(0)
            assert _lib.load().flashMoeWorkspaceBytes(ctypes.byref(d), ctypes.byref(n_pre)) == 0
            d.flags = _lib.FLAG_PACK_WEIGHTS
            assert _lib.load().flashMoeWorkspaceBytes(ctypes.byref(d), ctypes.byref(n_copy)) == 0
            esz = 2 if cfg.dtype == "bf16" else 4
            assert n_copy.value - n_pre.value >= 3 * cfg.E * cfg.H * cfg.I * esz
        finally:
            b.close()
        c = GpuCase(cfg, seed=11, sched=sched, inputs=a.inp, pack_weights=True)
        try:
            assert torch.equal(c.run(), out_a)
        finally:
            c.close()
    finally:
        a.close()


@pytest.mark.parametrize("blocks,shape", [
    (1, (1, 256, 8, 2, 128)),            # one k-step a wave; most workgroups without a task
    (1, (1, 256, 8, 8, 256)),            # one down task to a workgroup (eight parts)
    (1, (10, 512, 8, 1, 352)),           # eleven down k-steps over four waves; early gate/up tasks of unused experts
    (1, (33, 768, 32, 4, 160)),          # three k-steps a wave, five in the down projection; two mask words of experts
    (1, (64, 2048, 64, 8, 416, 4)),      # four experts with 64 rows: tiles of one expert among the rest; a full window
    (1, (67, 2304, 16, 2, 128, 2)),      # ragged tiles; nine k-steps a wave, more than the window
    (1, (72, 256, 256, 9, 128)),         # every expert slot in use; two mask words
    (1, (128, 256, 256, 9, 128, 3)),     # 1152 routing entries, all workgroups busy with routing or early tasks
    (2, (80, 256, 8, 1, 128)),           # ten rows an expert: tiles of two row blocks, most with one block in use
    (2, (128, 256, 8, 1, 128)),          # 16 rows an expert: the second block empty, full or anywhere between
    (2, (190, 768, 16, 2, 352, 2)),      # 23.75 rows an expert; ragged tiles of up to 32 rows, two experts with several
    (2, (256, 512, 96, 8, 160, 4)),      # 2048 routing entries: the tables are full
    (0, (40, 256, 4, 1, 128)),           # too few router weights for the loads nobody needs
    (0, (98, 256, 8, 2, 256)),           # 24.5 rows an expert
])
def test_split_k_small_batches(blocks, shape):
    _check_split_k(blocks, shape, "bf16")


@pytest.mark.parametrize("blocks,shape", [
    (1, (1, 128, 16, 2, 128)),           # one k-step a wave in either projection; 64-column tasks in pairs, one pair
    (1, (3, 192, 16, 2, 160)),           # an odd number of 64-column tasks: eight parts of a down task; odd k-steps
    (1, (16, 256, 8, 2, 128)),           # tiny: most workgroups without a task
    (1, (1, 2048, 16, 8, 768)),          # one token, full windows
    (1, (33, 1344, 40, 5, 736)),         # 21 column blocks of 64; 84 and 46 k-steps over the eight waves
    (1, (77, 320, 16, 2, 160)),          # 9.6 rows an expert, ragged last chunk of the chains
    (1, (64, 2048, 64, 8, 416, 4)),      # four experts with 64 rows: several tiles each
    (1, (127, 256, 256, 9, 128, 3)),     # 512 chain tasks: four waves of each routing workgroup; two mask words
    (0, (129, 256, 256, 9, 128)),        # 544 of them: the streaming kernel
    (0, (36, 256, 4, 1, 128)),           # too few router weights for the loads nobody needs
])
def test_split_k_small_batches_float32(blocks, shape):
    _check_split_k(blocks, shape, "f32")


def _check_split_k(blocks, shape, dtype):
    """Small batches (bf16: at most 24 rows an expert, float32: fewer than 10): the split-k kernel at the edges of its k
    parts, tiles and tables, on row-major weights against the oracle; the packed copy gives the same
    bits, and so does a second launch (every counter is back at zero). `blocks`: the 16-row blocks
    of its tiles, 0 just outside its range (another kernel runs, the packed copy's may differ)."""
    T, H, E, k, I = shape[:5]
    cfg = synth.MoeConfig("split", T, H, E, k, I, dtype, hot=shape[5] if len(shape) > 5 else 0)
    print("split-k", dtype, shape, flush=True)
    case = GpuCase(cfg, seed=T + E)
    try:
        assert case.launcher.split_blocks_for(T) == blocks
        out = case.run()
        case.check_routing(case.inp["tokens"], case.launcher.routing(T))
        case.check_outputs(case.inp["tokens"], out, nthreads=4)
        assert torch.equal(case.run(), out)
        packed = GpuCase(cfg, seed=T + E, inputs=case.inp, pack_weights=True)
        try:
            assert packed.launcher.split_blocks_for(T) == blocks
            if blocks:
                assert torch.equal(packed.run(), out)
        finally:
            packed.close()
    finally:
        case.close()
