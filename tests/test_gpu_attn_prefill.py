"""GPU parity of the causal flash-attention prefill against the fp32 oracle.

Contract: |gpu - oracle| <= 2e-3 + 1e-2*|oracle| elementwise, oracle =
benchmarks/src/bin/attention_microbench.rs:665-702 generalised to GQA on the cache.
"""
import ctypes
import math
import threading

import numpy as np
import pytest

import oracle
from tests._util import D, assert_close_attn, normal_f16, rng

pytestmark = pytest.mark.gpu

SCALE = 1.0 / math.sqrt(D)


def _run(torch, q, kc, vc, qs, kv_len=None):
    import grout_amd

    dq = torch.from_numpy(q).cuda()
    dk = torch.from_numpy(kc).cuda()
    dv = torch.from_numpy(vc).cuda()
    out = torch.empty_like(dq)
    grout_amd.attend_prefill(dq, dk, dv, out, qs, kv_len=kv_len)
    torch.cuda.synchronize()
    return out.cpu().numpy()


def _case(seed, hq, hkv, S, qs, MS, scale_rows=None):
    g = rng(seed)
    q = normal_f16(g, (S, hq, D))
    kc = normal_f16(g, (hkv, MS, D))
    vc = normal_f16(g, (hkv, MS, D))
    if scale_rows is not None:
        idx = g.random((hkv, MS)) < scale_rows
        kc[idx] = (kc[idx].astype(np.float32) * 8).astype(np.float16)
    return q, kc, vc


@pytest.mark.parametrize("hq,hkv,S,qs,MS,seed", [
    (16, 8, 512, 0, 512, 1),      # config c1
    (4, 2, 17, 0, 17, 2),         # tiny, ragged
    (4, 2, 64, 5, 80, 3),         # query_start > 0 on a padded cache
    (8, 8, 100, 0, 128, 4),       # MHA (G = 1), ragged
    (64, 8, 130, 0, 160, 5),      # G = 8 (Qwen3-32B heads)
    (32, 8, 1, 0, 1, 6),          # single row
    (32, 8, 257, 1000, 1400, 7),  # chunked suffix far into the cache
    (12, 4, 200, 0, 200, 8),      # G = 3 (workgroups straddle position tiles)
])
def test_prefill_matches_oracle(gpu, hq, hkv, S, qs, MS, seed):
    import torch

    q, kc, vc = _case(seed, hq, hkv, S, qs, MS)
    out = _run(torch, q, kc, vc, qs)
    ref = oracle.attn_prefill_f32(q, kc, vc, SCALE, kv_len=qs + S, query_start=qs)
    assert_close_attn(out, ref, f"prefill hq={hq} hkv={hkv} S={S} qs={qs}")


def test_prefill_first_row_is_v0(gpu):
    """Row 0 at position 0 sees only key 0: p = 1, l = 1, out = V[kvh, 0] exactly."""
    import torch

    q, kc, vc = _case(40, 8, 2, 96, 0, 96)
    out = _run(torch, q, kc, vc, 0)
    for h in range(8):
        assert np.array_equal(out[0, h].view(np.uint16), vc[h // 4, 0].view(np.uint16))


def test_prefill_outlier_keys(gpu):
    """1% of K rows scaled x8 (config c5's online-softmax stress), S=1024."""
    import torch

    q, kc, vc = _case(41, 64, 8, 1024, 0, 1024, scale_rows=0.01)
    out = _run(torch, q, kc, vc, 0)
    ref = oracle.attn_prefill_f32(q, kc, vc, SCALE, kv_len=1024, query_start=0)
    assert_close_attn(out, ref, "prefill outliers")


def test_chunked_prefill_equals_full(gpu):
    """src/model.rs:6134-6205 invariant: a suffix prefill at query_start>0 over the
    cached prefix equals the same rows of a full prefill."""
    import torch

    q, kc, vc = _case(42, 32, 8, 384, 0, 384)
    full = _run(torch, q, kc, vc, 0)
    cut = 200
    part = _run(torch, np.ascontiguousarray(q[cut:]), kc, vc, cut)
    assert_close_attn(part, full[cut:].astype(np.float32), "chunked vs full", atol=1e-3, rtol=0)


def test_gqa_equals_mha_with_repeated_kv(gpu):
    import torch

    hq, hkv, S = 8, 2, 150
    q, kc, vc = _case(43, hq, hkv, S, 0, S)
    out = _run(torch, q, kc, vc, 0)
    kr = np.ascontiguousarray(np.repeat(kc, hq // hkv, axis=0))
    vr = np.ascontiguousarray(np.repeat(vc, hq // hkv, axis=0))
    out_mha = _run(torch, q, kr, vr, 0)
    assert np.array_equal(out.view(np.uint16), out_mha.view(np.uint16))


@pytest.mark.parametrize("S", [2048])
def test_prefill_long_sampled_rows(gpu, S):
    """Qwen3-4B heads at S=2048; oracle on a stride sample of rows."""
    import torch

    q, kc, vc = _case(44, 32, 8, S, 0, S)
    out = _run(torch, q, kc, vc, 0)
    ref = oracle.attn_prefill_f32(q, kc, vc, SCALE, kv_len=S, query_start=0, row_begin=3,
                                  row_step=61)
    rows = np.arange(3, S, 61)
    assert_close_attn(out[rows], ref[rows], "prefill S=2048 sampled")


@pytest.mark.parametrize("S,G,qs", [(1024, 4, 0), (700, 2, 300)])
def test_small_grid_workgroup_shape_is_bit_identical(gpu, S, G, qs):
    """Grids of at most one 4-tile workgroup per CU run those, grids of more than
    two per CU 8-tile workgroups; every wavefront computes the same thing in
    both, so a problem and the same problem with more KV heads appended (which
    pushes the grid past the threshold) agree bit for bit on the shared heads."""
    import torch

    cus = torch.cuda.get_device_properties(0).multi_processor_count
    per_head = -(-(-(-S // 32) * G) // 4)  # 4-tile workgroups
    hkv_small = cus // per_head
    hkv_big = 2 * cus // per_head + 1
    assert hkv_small >= 2 and per_head * hkv_small <= cus and per_head * hkv_big > 2 * cus
    print(f"[prefill 4/8 waves] S={S} G={G} Hkv {hkv_small} vs {hkv_big}", flush=True)
    q, kc, vc = _case(400 + S, hkv_big * G, hkv_big, S, qs, qs + S)
    small = _run(torch, np.ascontiguousarray(q[:, :hkv_small * G]), np.ascontiguousarray(kc[:hkv_small]),
                 np.ascontiguousarray(vc[:hkv_small]), qs)
    big = _run(torch, q, kc, vc, qs)
    assert np.array_equal(small.view(np.uint16), big[:, :hkv_small * G].view(np.uint16))
    ref = oracle.attn_prefill_f32(np.ascontiguousarray(q[:, :hkv_small * G]), kc[:hkv_small],
                                  vc[:hkv_small], SCALE, kv_len=qs + S, query_start=qs,
                                  row_step=37)
    assert_close_attn(small[::37], ref[::37], "4-wavefront workgroups, sampled rows")


@pytest.mark.parametrize("S,G,hkv,qs", [
    (1000, 4, 8, 0),    # one round of 4-tile workgroups, ragged last tile
    (1024, 8, 8, 0),    # two rounds: 512 workgroups on 256 CUs
    (33, 3, 2, 700),    # a handful of workgroups, tasks past the end, 12 tiles
    (65, 1, 5, 0),      # behind 520 keys: walks of 9 and 10 tiles
    (65, 1, 90, 0),     # shortest walks, 1 and 2 tiles: too many heads for the short form
])
def test_narrow_workgroups_are_bit_identical(gpu, S, G, hkv, qs):
    """4-tile workgroups (computing and copying wavefronts apart) against the
    8-tile grid, which the same problem takes once more KV heads fill the GPU
    several times over: the shared heads agree bit for bit."""
    import torch

    cus = torch.cuda.get_device_properties(0).multi_processor_count
    n_pos = -(-S // 32)
    hkv_big = hkv * (-(-4 * cus // (-(-n_pos * G // 8) * hkv)))
    print(f"[prefill narrow] S={S} G={G} Hkv {hkv} vs {hkv_big}", flush=True)
    # Past the short form's 8 key tiles, or past its one workgroup per CU.
    kv_pad = 520 if _short_form_applies(cus, hkv * G, S, qs, qs + S) else 0
    g = torch.Generator(device="cuda").manual_seed(500 + S)
    q, kc, vc = (torch.randn(s, generator=g, device="cuda", dtype=torch.float16)
                 for s in ((S, hkv_big * G, D), (hkv_big, qs + S + kv_pad, D), (hkv_big, qs + S + kv_pad, D)))
    import grout_amd

    def run(heads):
        out = torch.full((S, heads * G, D), float("nan"), dtype=torch.float16, device="cuda")
        a = [t.contiguous() for t in (q[:, :heads * G], kc[:heads], vc[:heads])] + [out]
        # The C entry point without a workspace: these shapes never split their keys.
        status = grout_amd.lib().grout_attn_prefill(
            *(t.data_ptr() for t in a), SCALE, heads * G, heads, D, S, qs + S + kv_pad, qs + kv_pad,
            kc.shape[1], torch.cuda.current_stream().cuda_stream)
        assert status == 0
        torch.cuda.synchronize()
        return out.view(torch.int16)

    assert torch.equal(run(hkv), run(hkv_big)[:, :hkv * G])


@pytest.mark.parametrize("hq,hkv,S,qs,kv_len,MS", [
    (32, 8, 7, 12001, None, 12008),  # one packed tile a head, last cache row in use
    (64, 8, 10, 5000, None, 5100),   # three tiles, the last with 16 rows
    (6, 2, 33, 2000, None, 2100),    # G = 3: positions straddle tiles; 4 tiles, one row in the last
    (16, 8, 1, 1000, None, 1001),    # one row, 16 key tiles
    (5, 5, 129, 700, None, 900),     # G = 1: 5 tiles, a second workgroup with one
    (8, 1, 300, 1000, None, 1300),   # 19 workgroups
    (32, 8, 20, 3000, 2900, 3100),   # kv_len before the first position: no causal mask at all
    (32, 8, 20, 3000, 3005, 3100),   # and inside the rows
])
def test_key_split_matches_oracle(gpu, hq, hkv, S, qs, kv_len, MS):
    """Few rows behind many keys: keys split over workgroups, f32 partials merged
    by a second launch; K outliers move the splits' maxima apart."""
    import torch

    import grout_amd

    kv = qs + S if kv_len is None else kv_len
    nbytes = grout_amd.lib().grout_attn_prefill_workspace_bytes(hq, hkv, D, S, kv, qs, MS)
    tile_bytes = 32 * (D + 2) * 4 * hkv * -(-S * (hq // hkv) // 32)
    assert nbytes >= 2 * tile_bytes and nbytes % tile_bytes == 0, "shape does not split"
    print(f"[prefill key split] hq={hq} hkv={hkv} S={S} qs={qs} kv_len={kv} splits {nbytes // tile_bytes}", flush=True)
    q, kc, vc = _case(600 + S, hq, hkv, S, qs, MS, scale_rows=0.01)
    out = _run(torch, q, kc, vc, qs, kv_len=kv)
    ref = oracle.attn_prefill_f32(q, kc, vc, SCALE, kv_len=kv, query_start=qs)
    assert_close_attn(out, ref, f"key split hq={hq} hkv={hkv} S={S} qs={qs} kv_len={kv}")


def test_key_split_workspace_and_capture(gpu):
    """A workspace of NaNs or of too few bytes does not show in the output; a
    captured call takes no scratch and replays to the unsplit result."""
    import torch

    import grout_amd

    hq, hkv, S, qs = 32, 8, 5, 4000
    q, kc, vc = (torch.from_numpy(a).cuda() for a in _case(650, hq, hkv, S, qs, qs + S))
    L = grout_amd.lib()
    nbytes = L.grout_attn_prefill_workspace_bytes(hq, hkv, D, S, qs + S, qs, qs + S)
    assert nbytes > 0

    def run(ws, n):
        out = torch.full_like(q, float("nan"))
        assert L.grout_attn_prefill_ws(
            q.data_ptr(), kc.data_ptr(), vc.data_ptr(), out.data_ptr(), SCALE, hq, hkv, D, S, qs + S, qs,
            qs + S, None, ws, n, torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        return out

    ws = torch.full((nbytes // 4,), float("nan"), device="cuda")
    split = run(ws.data_ptr(), nbytes)
    assert torch.equal(split, run(ws.data_ptr(), nbytes))
    unsplit = run(None, 0)
    assert torch.equal(unsplit, run(ws.data_ptr(), nbytes - 4))
    assert_close_attn(split.cpu().numpy(), unsplit.float().cpu().numpy(), "split vs unsplit", atol=1e-3, rtol=0)
    out = torch.empty_like(q)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        grout_amd.attend_prefill(q, kc, vc, out, qs)
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        grout_amd.attend_prefill(q, kc, vc, torch.empty_like(q), qs)
        torch.cuda.synchronize()
        assert torch.equal(out, unsplit)


@pytest.mark.parametrize("hq,hkv,S", [
    (1, 1, 4000),  # 32 workgroups, the lightest with one row tile
    (2, 1, 2000),  # two query heads packed
])
def test_key_split_with_empty_splits(gpu, hq, hkv, S):
    """A prompt from position 0 whose first row blocks have fewer key tiles than
    there are splits: workgroups without a tile leave partials of weight 0, and
    every partial that the merge reads has been written (the workspace is NaN)."""
    import torch

    import grout_amd

    L = grout_amd.lib()
    nbytes = L.grout_attn_prefill_workspace_bytes(hq, hkv, D, S, S, 0, S)
    n_tiles = -(-S * (hq // hkv) // 32)
    splits = nbytes // (32 * (D + 2) * 4 * hkv * n_tiles)
    # Workgroups take 4 row tiles, heaviest first: the lightest has the remainder.
    lightest_rows = 32 * ((n_tiles - 1) % 4 + 1)
    assert splits > -(-(lightest_rows // (hq // hkv)) // 64), "no split is empty"
    print(f"[prefill empty splits] hq={hq} hkv={hkv} S={S} splits {splits}", flush=True)
    h = _case(670 + hq, hq, hkv, S, 0, S, scale_rows=0.01)
    q, kc, vc = (torch.from_numpy(a).cuda() for a in h)
    out = torch.full_like(q, float("nan"))
    ws = torch.full((nbytes // 4,), float("nan"), device="cuda")
    assert L.grout_attn_prefill_ws(
        q.data_ptr(), kc.data_ptr(), vc.data_ptr(), out.data_ptr(), SCALE, hq, hkv, D, S, S, 0, S, None,
        ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    ref = oracle.attn_prefill_f32(*h, SCALE, kv_len=S, query_start=0)
    assert_close_attn(out.cpu().numpy(), ref, f"empty splits hq={hq} S={S}")


def test_key_split_on_two_streams(gpu):
    """Split launches of two problems on two streams at once: each takes scratch
    of its own stream, so both give what they give alone."""
    import torch

    import grout_amd

    hq, hkv = 32, 8
    problems = []
    for i, (S, qs) in enumerate(((7, 9000), (61, 5000))):
        q, kc, vc = (torch.from_numpy(a).cuda() for a in _case(680 + i, hq, hkv, S, qs, qs + S))
        assert grout_amd.lib().grout_attn_prefill_workspace_bytes(hq, hkv, D, S, qs + S, qs, qs + S) > 0
        ref = torch.empty_like(q)
        grout_amd.attend_prefill(q, kc, vc, ref, qs)
        outs = [torch.full_like(q, float("nan")) for _ in range(40)]
        problems.append((torch.cuda.Stream(), q, kc, vc, ref, outs, qs))
    torch.cuda.synchronize()
    print("[prefill key split] two streams", flush=True)
    for i in range(40):
        for stream, q, kc, vc, _, outs, qs in problems:
            with torch.cuda.stream(stream):
                grout_amd.attend_prefill(q, kc, vc, outs[i], qs)
    torch.cuda.synchronize()
    for _, _, _, _, ref, outs, _ in problems:
        assert all(torch.equal(o, ref) for o in outs)


_GLOBAL, _THREAD_LOCAL = 0, 1  # hipStreamCaptureMode


def _capture_around(torch, stream, mode, call, own_thread):
    """Runs `call` (in a thread of its own or here) while `stream`, a raw handle,
    is captured; True if the graph was built and its kernel runs on replay."""
    import grout_amd

    L = grout_amd.lib()
    flag = torch.zeros((1,), dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    stream, error = ctypes.c_void_p(stream), []

    def guarded():
        try:
            call()
        except Exception as e:  # the capture is ended before it is raised
            error.append(e)

    assert L.hipStreamBeginCapture(stream, mode) == 0
    if own_thread:
        t = threading.Thread(target=guarded)
        t.start()
        t.join()
    else:
        guarded()
    recorded = L.grout_set_position_async(flag.data_ptr(), 7, stream)
    graph = ctypes.c_void_p()
    ended = L.grout_graph_end(stream, ctypes.byref(graph))
    if error:
        raise error[0]
    assert recorded == 0 and ended == 0, f"the capture was broken: {recorded}, {ended}"
    assert L.grout_graph_launch(graph, stream) == 0
    torch.cuda.synchronize()
    L.grout_graph_destroy(graph)
    return int(flag.item()) == 7


@pytest.mark.parametrize("oom", [False, True])
@pytest.mark.parametrize("mode,own_thread", [(_GLOBAL, True), (_GLOBAL, False), (_THREAD_LOCAL, False)])
def test_key_split_scratch_leaves_other_captures_alone(gpu, mode, own_thread, oom):
    """An eager call whose scratch the allocator does not have at hand, while
    another stream is captured: it splits (or, with no memory left, runs unsplit)
    and the capture goes on."""
    import torch

    import grout_amd

    hq, hkv, S, qs = 32, 8, 300, 4000
    q, kc, vc = (torch.from_numpy(a).cuda() for a in _case(651, hq, hkv, S, qs, qs + S))
    L = grout_amd.lib()
    nbytes = L.grout_attn_prefill_workspace_bytes(hq, hkv, D, S, qs + S, qs, qs + S)
    assert nbytes > (4 << 20)
    ref, out = torch.empty_like(q), torch.full_like(q, float("nan"))
    if oom:
        assert L.grout_attn_prefill(
            q.data_ptr(), kc.data_ptr(), vc.data_ptr(), ref.data_ptr(), SCALE, hq, hkv, D, S, qs + S, qs, qs + S,
            torch.cuda.current_stream().cuda_stream) == 0
    else:
        grout_amd.attend_prefill(q, kc, vc, ref, qs)
    torch.cuda.synchronize()
    captured, side = torch.cuda.Stream(), torch.cuda.Stream()

    total = torch.cuda.get_device_properties(0).total_memory

    def call():
        if oom:
            torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (1 << 20)) / total)
        try:
            with torch.cuda.stream(side):
                grout_amd.attend_prefill(q, kc, vc, out, qs)
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)

    torch.cuda.empty_cache()
    reserved = torch.cuda.memory_reserved()
    print(f"[prefill scratch] capture mode {mode} own thread {own_thread} oom {oom}", flush=True)
    assert _capture_around(torch, captured.cuda_stream, mode, call, own_thread)
    assert oom or torch.cuda.memory_reserved() > reserved, "the allocator had the scratch at hand"
    assert torch.equal(out, ref)


@pytest.mark.parametrize("mode,own_thread", [(_GLOBAL, True), (_GLOBAL, False), (_THREAD_LOCAL, False)])
def test_key_split_on_the_legacy_stream_beside_a_blocking_capture(gpu, mode, own_thread):
    """An eager call on the default stream while a blocking stream is captured,
    where HIP does not say whether the default stream captures: it runs unsplit."""
    import torch

    import grout_amd

    hq, hkv, S, qs = 32, 8, 5, 4000
    q, kc, vc = (torch.from_numpy(a).cuda() for a in _case(652, hq, hkv, S, qs, qs + S))
    L = grout_amd.lib()
    assert L.grout_attn_prefill_workspace_bytes(hq, hkv, D, S, qs + S, qs, qs + S) > 0
    ref, out = torch.empty_like(q), torch.full_like(q, float("nan"))
    legacy = torch.cuda.default_stream()
    assert L.grout_attn_prefill(
        q.data_ptr(), kc.data_ptr(), vc.data_ptr(), ref.data_ptr(), SCALE, hq, hkv, D, S, qs + S, qs, qs + S,
        legacy.cuda_stream) == 0

    def call():
        with torch.cuda.stream(legacy):
            grout_amd.attend_prefill(q, kc, vc, out, qs)

    blocking = ctypes.c_void_p()
    assert L.hipStreamCreate(ctypes.byref(blocking)) == 0
    print(f"[prefill legacy stream] capture mode {mode} own thread {own_thread}", flush=True)
    try:
        assert _capture_around(torch, blocking.value, mode, call, own_thread)
    finally:
        assert L.hipStreamDestroy(blocking) == 0
    assert torch.equal(out, ref)


def _short_form_applies(cus, hq, S, qs, kv_len):
    """The host rule of the short form: every 32-row block needs at most 8 key
    tiles of 64, and one workgroup per (query head, row block) fits the CUs."""
    n_blocks = -(-S // 32)
    return min(kv_len, qs + 32 * n_blocks) <= 8 * 64 and n_blocks * hq <= cus


@pytest.mark.parametrize("hq,hkv,S,qs,MS,kv_len,seed", [
    (16, 8, 50, 40, 96, None, 11),    # rows 40..63's second tile holds none of their keys
    (8, 2, 512, 0, 512, None, 12),    # 8 key tiles in the last row block, G = 4
    (32, 8, 256, 0, 256, None, 13),   # 256 workgroups: one per CU on MI355X
    (4, 1, 300, 200, 512, 480, 14),   # kv_len short of query_start + q_len (rows past it see 480 keys)
    (21, 7, 321, 7, 400, None, 15),   # ragged: a partial last row block, G = 3
    (16, 8, 1, 511, 512, None, 17),   # one row over 512 keys: every wavefront holds a tile
    (8, 4, 32, 480, 512, None, 18),   # one full row block at the end of the range
])
def test_short_prefill_matches_oracle(gpu, hq, hkv, S, qs, MS, kv_len, seed):
    """Launches small enough for the short form (one workgroup per query head
    and 32-row block, one key tile per wavefront, partials merged in LDS)."""
    import torch

    kv = qs + S if kv_len is None else kv_len
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert _short_form_applies(cus, hq, S, qs, kv), "shape outside the short form"
    print(f"[short prefill] hq={hq} hkv={hkv} S={S} qs={qs} kv_len={kv}", flush=True)
    q, kc, vc = _case(seed, hq, hkv, S, qs, MS)
    out = _run(torch, q, kc, vc, qs, kv_len=kv)
    ref = oracle.attn_prefill_f32(q, kc, vc, SCALE, kv_len=kv, query_start=qs)
    assert_close_attn(out, ref, f"short prefill hq={hq} hkv={hkv} S={S} qs={qs} kv_len={kv}")


def test_short_prefill_boundary_agrees_with_grid(gpu):
    """The same problem on both sides of the short form's CU rule: the short
    launch and the grid launch (one more query head pushes the grid past one
    workgroup per CU) agree within the attention tolerance on the shared heads."""
    import torch

    cus = torch.cuda.get_device_properties(0).multi_processor_count
    S, G = 256, 2
    hq_short = (cus // (S // 32)) // G * G
    hq_grid = hq_short + G
    assert _short_form_applies(cus, hq_short, S, 0, S) and not _short_form_applies(cus, hq_grid, S, 0, S)
    print(f"[short prefill boundary] hq {hq_short} vs {hq_grid}", flush=True)
    q, kc, vc = _case(16, hq_grid, hq_grid // G, S, 0, S)
    short = _run(torch, np.ascontiguousarray(q[:, :hq_short]), np.ascontiguousarray(kc[:hq_short // G]),
                 np.ascontiguousarray(vc[:hq_short // G]), 0)
    grid = _run(torch, q, kc, vc, 0)
    assert_close_attn(short, grid[:, :hq_short].astype(np.float32), "short vs grid")
    ref = oracle.attn_prefill_f32(q, kc, vc, SCALE, kv_len=S, query_start=0, row_step=13)
    assert_close_attn(grid[::13], ref[::13], "grid, sampled rows")
