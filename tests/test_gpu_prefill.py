"""Prefill chunks on matrix cores (fr_hip_run_batch).

The reference has no multi-token path beyond run()'s burst of at most 8: its
client cuts a prompt into bursts (client/fronk_client.h:41-42) and each burst
is run() (backends/ref.c:57-98). So row t of a chunk must equal, within the F32
tolerance, what ref returns for token t: checked against the oracle's
restatement of ref on host copies of the same synthetic slices, and against
this library's own run() on the same tokens. At the full 512-token size,
size-independent properties hold bit for bit: a repeat run is identical,
permuting the tokens permutes the rows, and doubling every gate doubles every
output (a power of two commutes with every rounding on the path).
"""
import numpy as np
import pytest

import fronk_amd as fa
import oracle
from fixtures import oracle_request, slice_view, softmax_gates, sparse_unit, zipf_routes
from test_gpu_parity import check_close

pytestmark = pytest.mark.gpu

SEED = 0x5EED0005


@pytest.fixture(scope="module")
def eng():
    e = fa.Engine(0)
    yield e
    for b in range(20):
        e.release(b)


def load(eng, hidden, blocks, layers=1, fmt=fa.FMT_Q4KT):
    for b in range(20):
        eng.release(b)
    for b in blocks:
        assert eng.synthetic(b, hidden, fmt, layers, SEED) == fa.OK


def host_units(lay, blocks, layer, experts):
    """Sparse host copies of the owned synthetic blocks (None where a block is
    not owned) holding the slices of `experts` at `layer`."""
    used = sorted(set(int(e) for e in np.asarray(experts).ravel()))
    units = [None] * 20
    for b in blocks:
        u = sparse_unit(lay)
        for e in used:
            slice_view(u, lay, layer, e)[:] = oracle.synth_slice(lay, SEED, b, layer, e)
        units[b] = u
    return units


def oracle_rows(lay, blocks, layer, experts, gates, x):
    units = host_units(lay, blocks, layer, experts)
    rows = []
    for t0 in range(0, x.shape[0], 8):
        sl = slice(t0, min(t0 + 8, x.shape[0]))
        rc, ref = oracle.ref_run(units, fa.FMT_Q4KT, False, oracle_request(layer, experts[sl], gates[sl], x[sl]))
        assert rc == 0
        rows.append(ref[:sl.stop - sl.start])
    return np.concatenate(rows)


def chunk(rng, tokens, hidden, pool=None):
    """Top-10 routes per token. With a pool, Zipf(1.1) popularity over it, so
    that hot experts take several 16-token tiles and cold ones a single token."""
    if pool is None:
        experts = np.stack([rng.choice(512, 10, replace=False) for _ in range(tokens)]).astype(np.uint16)
    else:
        experts = np.asarray(pool, np.uint16)[zipf_routes(rng, tokens, experts=len(pool))]
    gates = np.zeros((tokens, 11), np.float32)
    gates[:, :10] = softmax_gates(rng, tokens)
    x = rng.standard_normal((tokens, hidden)).astype(np.float32)
    return experts, gates, x


def run_ok(eng, layer, experts, gates, x):
    print(f"prefill tokens={x.shape[0]} hidden={x.shape[1]} layer={layer}", flush=True)
    rc, y = eng.run_batch(layer, experts, gates, x)
    assert rc == fa.OK, rc
    return y


def run_bursts(eng, layer, experts, gates, x):
    out = []
    for t0 in range(0, x.shape[0], 8):
        rc, y = eng.run(layer, experts[t0:t0 + 8], gates[t0:t0 + 8], x[t0:t0 + 8], fa.MODE_F32)
        assert rc == fa.OK
        out.append(y)
    return np.concatenate(out)


@pytest.mark.parametrize("hidden,tokens,blocks", [
    (4096, 40, tuple(range(20))),
    (2560, 24, (0, 7, 19)),
    (2304, 24, (0, 5, 19)),
])
def test_prefill_rows_match_oracle(eng, hidden, tokens, blocks):
    """Hot experts span several tiles, cold ones hold one token; at hidden 2560
    and 2304 only 3 slices are owned, and at 2304 (9 super-blocks) the last
    down workgroup (512 outputs) has idle wavefronts."""
    lay = oracle.layout(hidden, fa.FMT_Q4KT)
    load(eng, hidden, blocks)
    rng = np.random.default_rng(hidden + tokens)
    pool = rng.choice(512, 40, replace=False)
    experts, gates, x = chunk(rng, tokens, hidden, pool)
    counts = np.bincount(experts.ravel(), minlength=512)
    assert counts.max() > 16 and counts[counts > 0].min() < 16   # several tiles, and partial ones
    y = run_ok(eng, 0, experts, gates, x)
    s = eng.sample()
    assert s.unique_experts == len(set(experts.ravel().tolist())) and s.blocks == len(blocks)
    ref = oracle_rows(lay, blocks, 0, experts, gates, x)
    check_close(ref, y, fa.MODE_F32, ("prefill", hidden))
    check_close(run_bursts(eng, 0, experts, gates, x), y, fa.MODE_F32, ("prefill vs run", hidden))


def test_prefill_512_tokens_properties(eng):
    """The chunk size of the prefill workload: 512 tokens, uniform top-10 over
    512 experts, 20 owned slices, hidden 4096, layer 1."""
    hidden, tokens, layer = 4096, 512, 1
    lay = oracle.layout(hidden, fa.FMT_Q4KT)
    load(eng, hidden, range(20), layers=2)
    rng = np.random.default_rng(512)
    experts, gates, x = chunk(rng, tokens, hidden)
    y = run_ok(eng, layer, experts, gates, x)
    assert np.isfinite(y).all()
    again = run_ok(eng, layer, experts, gates, x)
    assert np.array_equal(y.view(np.uint32), again.view(np.uint32))
    perm = rng.permutation(tokens)
    yp = run_ok(eng, layer, experts[perm], gates[perm], x[perm])
    assert np.array_equal(yp.view(np.uint32), y[perm].view(np.uint32))
    y2 = run_ok(eng, layer, experts, 2 * gates, x)
    assert np.array_equal(y2.view(np.uint32), (2 * y).view(np.uint32))
    sample = np.arange(0, tokens, 64)
    ref = oracle_rows(lay, range(20), layer, experts[sample], gates[sample], x[sample])
    check_close(ref, y[sample], fa.MODE_F32, "prefill 512 sample")
    check_close(run_bursts(eng, layer, experts[:16], gates[:16], x[:16]), y[:16], fa.MODE_F32, "prefill vs run")


def test_prefill_48_layers_resident(eng):
    """The resident node of the prefill workload: 48 layers of 20 owned
    blocks in HBM (108.7 GB), a 512-token chunk on the last layer, whose
    slices sit at the top of each block's 5.4 GB. Sampled rows against the
    oracle; every row finite; a repeat is bit-identical."""
    hidden, tokens, layer = 4096, 512, 47
    lay = oracle.layout(hidden, fa.FMT_Q4KT)
    print("prefill: 20 blocks x 48 layers resident", flush=True)
    load(eng, hidden, range(20), layers=48)
    try:
        rng = np.random.default_rng(4847)
        experts, gates, x = chunk(rng, tokens, hidden)
        y = run_ok(eng, layer, experts, gates, x)
        assert np.isfinite(y).all()
        assert np.array_equal(run_ok(eng, layer, experts, gates, x).view(np.uint32), y.view(np.uint32))
        sample = np.arange(5, tokens, 73)
        ref = oracle_rows(lay, range(20), layer, experts[sample], gates[sample], x[sample])
        check_close(ref, y[sample], fa.MODE_F32, "prefill layer 47 of 48")
    finally:
        for b in range(20):
            eng.release(b)


def test_prefill_error_paths(eng):
    hidden = 4096
    load(eng, hidden, (0, 1))
    rng = np.random.default_rng(5)
    experts, gates, x = chunk(rng, 20, hidden)
    y = run_ok(eng, 0, experts, gates, x)
    assert eng.run_batch(0, experts[:0], gates[:0], x[:0])[0] == fa.INVALID
    dup = experts.copy()
    dup[3, 1] = dup[3, 0]
    assert eng.run_batch(0, dup, gates, x)[0] == fa.INVALID
    big = experts.copy()
    big[2, 4] = 512
    assert eng.run_batch(0, big, gates, x)[0] == fa.INVALID
    assert eng.run_batch(0, experts, gates, x, fa.MODE_F64)[0] == fa.UNSUPPORTED
    assert eng.run_batch(1, experts, gates, x)[0] == fa.STATE
    assert eng.run_batch(0, experts, gates, x[:, :2560])[0] == fa.INVALID
    bad = x.copy()
    bad[7, 100] = np.inf
    rc, yb = eng.run_batch(0, experts, gates, bad)
    assert rc == fa.NUMERIC and not yb.any()
    # The status word is cleared per launch: the next good chunk succeeds.
    assert np.array_equal(run_ok(eng, 0, experts, gates, x).view(np.uint32), y.view(np.uint32))
    assert eng.synthetic(2, hidden, fa.FMT_Q8, 1, SEED) == fa.OK
    assert eng.run_batch(0, experts, gates, x)[0] == fa.UNSUPPORTED
    eng.release(2)


def cut_of(eng, experts, gates, x):
    """[gslices, gdown] of the plan's BatchHeader: the kernels the chunk takes."""
    return eng.batch_plan(0, experts, gates, x, fa.MODE_F32)[72:80].view(np.uint32).tolist()


def hot_and_cold(experts):
    """The expert of most tokens and one of the fewest."""
    count = np.bincount(experts.ravel(), minlength=512)
    return [int(np.argmax(count)), int(np.flatnonzero(count == count[count > 0].min())[0])]


# The chunks below run on prefill_gate_up_few and prefill_down_few, or on
# prefill_gate_up<4> and prefill_down with tiles of 16 to 64 tokens.
BOTH = pytest.mark.parametrize("hidden,nblk,tokens,pool,cut", [(4096, 2, 24, 30, [0, 0]), (2560, 20, 320, 300, [4, 1])])


@BOTH
@pytest.mark.parametrize("which", ["d", "dmin"])
def test_prefill_large_down_scales(eng, hidden, nblk, tokens, pool, cut, which):
    """Down super-blocks whose d (or dmin) is 4 or more in magnitude (4, -5, 6, 100,
    and 65504, the largest fp16) in slices of a hot expert and of a cold one, some
    super-blocks of a slice and slices side by side: with d the down kernels
    take those slices on their scaled path. The chunk's rows and run()'s against the
    oracle."""
    blocks = tuple(range(nblk))
    lay = oracle.layout(hidden, fa.FMT_Q4KT)
    load(eng, hidden, blocks)
    rng = np.random.default_rng(4444)
    experts, gates, x = chunk(rng, tokens, hidden, rng.choice(512, pool, replace=False))
    assert cut_of(eng, experts, gates, x) == cut
    chosen = hot_and_cold(experts)
    rows = np.unique(np.concatenate([np.flatnonzero((experts == e).any(axis=1))[:9] for e in chosen] + [np.arange(3)]))
    units = host_units(lay, blocks, 0, experts[rows])
    edits = ((5, 3, 0x4400), (17, 9, 0xC500), (0, 0, 0x4600), (31, hidden // 256 - 1, 0x5640), (12, 6, 0x7BFF))
    for b, e in [(1, chosen[0]), (1, chosen[1]), (nblk - 2, chosen[0])]:
        view = slice_view(units[b], lay, 0, e)
        for neuron, sb, v in edits:
            off = 2 * lay.proj + neuron * lay.down_row + 144 * sb + (2 if which == "dmin" else 0)
            view[off:off + 2] = np.array([v], np.uint16).view(np.uint8)
        assert eng.refresh(b, units[b], 0, e) == fa.OK
    y = run_ok(eng, 0, experts, gates, x)
    ref = []
    for i in range(0, len(rows), 8):
        part = rows[i:i + 8]
        rc, r = oracle.ref_run(units, fa.FMT_Q4KT, False, oracle_request(0, experts[part], gates[part], x[part]))
        assert rc == 0
        ref.append(r[:len(part)])
    # y is one neuron's h at d = 65504, whose own dot may nearly cancel: a chunk and
    # run() differ by up to the sum of their distances from the oracle.
    check_close(np.concatenate(ref), y[rows], fa.MODE_F32, ("prefill large down scales", which))
    check_close(np.concatenate(ref), run_bursts(eng, 0, experts[rows], gates[rows], x[rows]), fa.MODE_F32, ("run", which))


@pytest.mark.parametrize("seed,blocks,tokens,pool,cut", [
    (5, (0, 1), 40, 40, [0, 0]), (6, (0, 1), 40, 40, [0, 0]), (7, (3,), 40, 40, [0, 0]),
    (5, tuple(range(20)), 320, 300, [4, 1]), (6, tuple(range(20)), 320, 300, [4, 1]),
])
def test_prefill_down_operand_parts_agree(eng, seed, blocks, tokens, pool, cut):
    """The down's two f16 parts of d*h sum to it: every token within 2e-6 of the
    oracle (of a large chunk, 40 of them). fp32 sums of 20 terms whose magnitudes
    add up to a few times the result leave about 1e-6 at most; a hi part that one
    use rounds differently from the other (2^-11 of one product) shows as 3e-6
    and more in some token of each of the small chunks."""
    hidden = 4096
    lay = oracle.layout(hidden, fa.FMT_Q4KT)
    load(eng, hidden, blocks)
    rng = np.random.default_rng(seed)
    experts, gates, x = chunk(rng, tokens, hidden, rng.choice(512, pool, replace=False))
    assert cut_of(eng, experts, gates, x) == cut
    y = run_ok(eng, 0, experts, gates, x)
    rows = np.arange(40) * (tokens // 40)
    ref = oracle_rows(lay, blocks, 0, experts[rows], gates[rows], x[rows])
    for i, t in enumerate(rows):
        rc, err = oracle.compare(ref[i], y[t])
        assert rc == 0 and err[0] <= 2e-6, (seed, t, err)


@BOTH
def test_prefill_bad_scales_and_x(eng, hidden, nblk, tokens, pool, cut):
    """A non-finite x, and one non-finite d or dmin in a gate, an up or a down row
    of the last slice of a hot expert's or a cold one's, each end in FR_NUMERIC
    with y untouched; the restored chunk is bit-identical."""
    blocks = tuple(range(nblk))
    lay = oracle.layout(hidden, fa.FMT_Q4KT)
    load(eng, hidden, blocks)
    rng = np.random.default_rng(78)
    experts, gates, x = chunk(rng, tokens, hidden, rng.choice(512, pool, replace=False))
    assert cut_of(eng, experts, gates, x) == cut
    good = run_ok(eng, 0, experts, gates, x)
    for v in (np.inf, np.nan):
        bad = x.copy()
        bad[tokens - 1, hidden - 1] = v
        rc, y = eng.run_batch(0, experts, gates, bad)
        assert rc == fa.NUMERIC and not y.any()
    chosen = hot_and_cold(experts)
    units = host_units(lay, blocks[-1:], 0, chosen)
    b = blocks[-1]
    for e in chosen:
        view = slice_view(units[b], lay, 0, e)
        keep = view.copy()
        for off in (0, lay.proj + 31 * lay.gu_row + lay.gu_row - 144 + 2, 2 * lay.proj, 2 * lay.proj + 32 * lay.down_row - 144 + 2):
            view[off:off + 2] = np.array([0x7C00], np.uint16).view(np.uint8)
            assert eng.refresh(b, units[b], 0, e) == fa.OK
            print(f"non-finite scale at {off} of expert {e}", flush=True)
            rc, y = eng.run_batch(0, experts, gates, x)
            assert rc == fa.NUMERIC and not y.any(), (e, off)
            view[:] = keep
            assert eng.refresh(b, units[b], 0, e) == fa.OK
    assert np.array_equal(run_ok(eng, 0, experts, gates, x).view(np.uint32), good.view(np.uint32))


@pytest.mark.parametrize("hidden,nblk,tokens,pool,slices,down", [
    (2560, 20, 200, 300, 4, 1),    # tiles of one to four 16-token tiles, all with partial ends
    (2304, 7, 700, 512, 4, 0),     # nine super-blocks; the last workgroup's fourth wavefront has no slice
    (2304, 10, 900, 512, 2, 1),
    (2304, 7, 1600, 512, 4, 1),
    (2304, 6, 160, 512, 2, 0),
    (2560, 18, 130, 512, 4, 0),    # two wavefronts of the last workgroup without a slice
    (256, 20, 600, 100, 4, 1),     # one super-block
    (256, 1, 2600, 512, 0, 0),     # one super-block and slice
    (4096, 3, 24, 30, 0, 0),       # few workgroups
])
def test_prefill_gate_up_cuts(eng, hidden, nblk, tokens, pool, slices, down):
    """Each way the routed gate/up is cut into workgroups, with either down, at odd
    sizes: rows against the oracle, and a repeat bit for bit."""
    blocks = tuple(range(20 - nblk, 20))
    lay = oracle.layout(hidden, fa.FMT_Q4KT)
    load(eng, hidden, blocks)
    rng = np.random.default_rng(hidden + tokens)
    experts, gates, x = chunk(rng, tokens, hidden, rng.choice(512, pool, replace=False))
    assert cut_of(eng, experts, gates, x) == [slices, down]
    y = run_ok(eng, 0, experts, gates, x)
    assert np.array_equal(y, run_ok(eng, 0, experts, gates, x))
    rows = rng.choice(tokens, 7, replace=False)
    ref = oracle_rows(lay, blocks, 0, experts[rows], gates[rows], x[rows])
    check_close(ref, y[rows], fa.MODE_F32, ("cut", hidden, nblk))


@pytest.mark.parametrize("tokens,blocks", [(n, (0, 7)) for n in (1, 60, 63, 64, 130, 300)] + [(520, tuple(range(20)))])
def test_prefill_run_batch_equals_resident_plan(eng, tokens, blocks):
    """fr_hip_run_batch's way up and down (copy kernels up to 1 MB of plan, which
    64 tokens at hidden 4096 pass; 512 KB pieces above) leaves y what a resident
    plan gives, bit for bit; and after a call that fails, fr_hip_batch_output
    reports that call's status."""
    import ctypes as C

    import torch
    hidden = 4096
    load(eng, hidden, blocks)
    rng = np.random.default_rng(tokens)
    experts, gates, x = chunk(rng, tokens, hidden)
    assert cut_of(eng, experts, gates, x) == ([0, 0] if tokens < 100 else [2, 0] if tokens < 500 else [4, 1])
    y = run_ok(eng, 0, experts, gates, x)
    plan = eng.batch_plan(0, experts, gates, x, fa.MODE_F32)
    dev = torch.from_numpy(plan).to("cuda")
    torch.cuda.synchronize()
    ref, status = np.zeros_like(x), C.c_uint()
    assert fa.lib().fr_hip_batch_launch(plan.ctypes.data, dev.data_ptr(), None) == fa.OK
    assert fa.lib().fr_hip_batch_output(None, fa.fptr(ref), x.size, C.byref(status)) == fa.OK
    assert status.value == 0 and np.array_equal(y.view(np.uint32), ref.view(np.uint32))
    x[-1, -1] = np.inf
    assert eng.run_batch(0, experts, gates, x)[0] == fa.NUMERIC
    assert fa.lib().fr_hip_batch_output(None, None, 0, C.byref(status)) == fa.OK and status.value != 0


def test_prefill_captured_launch_records_kernels_only(eng):
    """A captured fr_hip_batch_launch holds kernel nodes alone: a memset node has
    given wrong results on replays after the first."""
    import ctypes as C

    import torch
    hidden = 4096
    load(eng, hidden, (0, 7))
    rng = np.random.default_rng(9)
    experts, gates, x = chunk(rng, 40, hidden)
    run_ok(eng, 0, experts, gates, x)   # the scratch is grown before the capture
    plan = eng.batch_plan(0, experts, gates, x, fa.MODE_F32)
    dev = torch.from_numpy(plan).to("cuda")
    torch.cuda.synchronize()
    s, g = torch.cuda.Stream(), torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(g, stream=s, capture_error_mode="thread_local"):
        assert fa.lib().fr_hip_batch_launch(plan.ctypes.data, dev.data_ptr(), C.c_void_p(s.cuda_stream)) == fa.OK
    with open("/proc/self/maps") as f:
        hip = C.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))
    graph, n = C.c_void_p(g.raw_cuda_graph()), C.c_size_t()
    assert hip.hipGraphGetNodes(graph, None, C.byref(n)) == 0 and n.value
    nodes = (C.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(graph, nodes, C.byref(n)) == 0
    for node in nodes:
        kind = C.c_int()
        assert hip.hipGraphNodeGetType(C.c_void_p(node), C.byref(kind)) == 0
        assert kind.value == 0, kind.value   # hipGraphNodeTypeKernel


@pytest.mark.parametrize("tokens", [40, 130])
def test_prefill_replayed_launch_keeps_its_status(eng, tokens):
    """A captured fr_hip_batch_launch reports its own status at every replay, with
    fr_hip_run_batch calls (by copy kernel at 40 tokens, in pieces at 130) and
    eager work between the replays: a failing chunk's replay after a good
    run_batch still fails, a good one after a failing run_batch still passes."""
    import ctypes as C

    import torch
    hidden, lib = 4096, fa.lib()
    load(eng, hidden, (0, 7))
    rng = np.random.default_rng(tokens)
    experts, gates, x = chunk(rng, tokens, hidden)
    bad = x.copy()
    bad[3, 5] = np.inf
    good = run_ok(eng, 0, experts, gates, x)
    plans = [eng.batch_plan(0, experts, gates, v, fa.MODE_F32) for v in (x, bad)]
    dev = torch.from_numpy(plans[0]).to("cuda")
    torch.cuda.synchronize()
    s, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s, capture_error_mode="thread_local"):
        assert lib.fr_hip_batch_launch(plans[0].ctypes.data, dev.data_ptr(), C.c_void_p(s.cuda_stream)) == fa.OK
    for rep in range(4):
        fails = rep % 2 == 0
        print(f"replay {rep}", flush=True)
        rc, _ = eng.run_batch(0, experts, gates, x if fails else bad)
        assert rc == (fa.OK if fails else fa.NUMERIC)
        dev.copy_(torch.from_numpy(plans[1 if fails else 0]))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        y, status = np.zeros_like(x), C.c_uint()
        assert lib.fr_hip_batch_output(None, fa.fptr(y), x.size, C.byref(status)) == fa.OK
        assert (status.value != 0) == fails and np.array_equal(y, np.zeros_like(x) if fails else good), rep


def test_prefill_buffers_count_as_hot_allocations(eng):
    """Every buffer that a chunk grows is in the sample's hot_allocations: the
    scratch (four buffers) by the launch, run_batch's plan and y by its first
    call at a size, none by the second."""
    import torch
    hidden, lib = 2560, fa.lib()
    load(eng, hidden, ())
    assert eng.close() == fa.OK   # the next engine has no scratch
    fa.Engine(0)
    load(eng, hidden, (0,))
    experts, gates, x = chunk(np.random.default_rng(1), 20, hidden)
    plan = eng.batch_plan(0, experts, gates, x, fa.MODE_F32)
    dev = torch.from_numpy(plan).to("cuda")
    torch.cuda.synchronize()
    assert eng.sample().hot_allocations == 0
    assert lib.fr_hip_batch_launch(plan.ctypes.data, dev.data_ptr(), None) == fa.OK
    assert lib.fr_hip_batch_output(None, None, 0, None) == fa.OK
    assert eng.sample().hot_allocations == 4
    for _ in range(2):
        run_ok(eng, 0, experts, gates, x)
        assert eng.sample().hot_allocations == 6


@BOTH
@pytest.mark.parametrize("what", ["min", "both"])
def test_prefill_small_down_scales(eng, what, hidden, nblk, tokens, pool, cut):
    """The down of an expert whose fp16 scales are the smallest there are (d and
    dmin 2^-24 to 3 * 2^-24, or d zero and y the min terms alone), on the tokens
    for which it is the only expert with a gate. The main sum has operands of 22
    bits and fp32 sums, the min terms are fp32: at most 2e-6 of a row, as with
    larger scales (operands with f16's absolute floor of 2^-25 would be off by
    2^-13 and more of their largest)."""
    blocks = tuple(range(20 - nblk, 20))
    lay = oracle.layout(hidden, fa.FMT_Q4KT)
    load(eng, hidden, blocks)
    rng = np.random.default_rng(31 + nblk)
    experts, gates, x = chunk(rng, tokens, hidden, rng.choice(512, pool, replace=False))
    chosen = hot_and_cold(experts)
    rows = []
    for e in chosen:
        for t in np.flatnonzero((experts == e).any(axis=1))[:10]:
            if int(t) not in rows:
                gates[t, :10] = np.where(experts[t] == e, gates[t, :10], 0)
                rows.append(int(t))
    assert cut_of(eng, experts, gates, x) == cut
    units = host_units(lay, blocks, 0, chosen)
    try:
        for b in blocks:
            for e in chosen:
                view = slice_view(units[b], lay, 0, e)
                head = view[2 * lay.proj:2 * lay.proj + 32 * lay.down_row].reshape(-1, 144)   # a super-block each
                d = rng.integers(1, 4, (len(head), 2)).astype(np.uint16)                       # fp16 subnormals
                if what == "min":
                    d[:, 0] = 0
                head[:, :4] = d.view(np.uint8).reshape(-1, 4)
                assert eng.refresh(b, units[b], 0, e) == fa.OK
        y = run_ok(eng, 0, experts, gates, x)
        for i in range(0, len(rows), 8):
            part = rows[i:i + 8]
            rc, ref = oracle.ref_run(units, fa.FMT_Q4KT, False, oracle_request(0, experts[part], gates[part], x[part]))
            assert rc == 0
            for j, t in enumerate(part):
                rc, err = oracle.compare(ref[j], y[t])
                assert rc == 0 and err[0] <= 2e-6, (what, t, err)
    finally:
        load(eng, hidden, ())
