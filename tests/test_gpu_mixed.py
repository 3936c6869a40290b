"""All bit-width groups of a bucket in one launch (dq_mixed_*), against the per-group calls they replace
(testbed_evaluation/new_comm_hooks/comm_hooks.py:963-1018 runs the ring once per group) and against the
oracle -- byte for byte."""
import numpy as np
import pytest
import torch

from helpers import BF16, F32, to_bits

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
REC = {8: 274, 4: 146, 2: 82}


def bits_t(t):
    return t.view(torch.int16 if t.element_size() == 2 else torch.int32)


def make_plan(capi, nsc, seed, weights=(1, 1, 1)):
    g = torch.Generator().manual_seed(seed)
    w = torch.tensor(weights, dtype=torch.float)
    q = torch.tensor([8, 4, 2])[torch.multinomial(w, nsc, replacement=True, generator=g)].to(DEV)
    order = torch.full((3 * nsc,), -1, dtype=torch.int32, device=DEV)
    work = torch.zeros(capi.group_plan_work_ints(nsc), dtype=torch.int32, device=DEV)
    capi.group_plan(q, order, work)
    return q, order, work


def segments(counts, chunk, world, nsc):
    """(width, entry of `order` where the run's rows start, row of the random pool of its first record, records, byte
    offset) of ring chunk `chunk`, and the stream size"""
    out, pos, off = [], 0, 0
    for g, (q, n) in enumerate(zip((8, 4, 2), counts)):
        per = -(-n // world)
        begin = min(per * chunk, n)
        cnt = min(per, n - begin)
        out.append((q, g * nsc + begin, pos + begin, cnt, off))
        pos += n
        off += cnt * REC[q]
    return out, off


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("strategy", [2, 3])
@pytest.mark.parametrize("nsc,world,weights", [(1037, 1, (1, 1, 1)), (1037, 3, (1, 2, 3)), (2, 1, (1, 1, 1)),
                                               (515, 4, (1, 0, 1)), (64, 8, (0, 1, 0)), (6403, 8, (1, 6, 2)),
                                               (2051, 7, (1, 3, 1)), (4099, 13, (2, 5, 1))])
def test_mixed_matches_per_group_calls(capi, dt, strategy, nsc, world, weights):
    n_valid = nsc * 256 - 77
    q, order, work = make_plan(capi, nsc, nsc + world, weights)
    counts = work[:3].tolist()
    assert sum(counts) == nsc
    g = torch.Generator().manual_seed(nsc * 3 + strategy)
    full = (torch.randn(nsc * 256, generator=g) * 1e-2).to(dt).to(DEV)
    peer = (torch.randn(nsc * 256, generator=g) * 1e-2).to(dt).to(DEV)
    stats = torch.randn(nsc, 2, generator=g).mul(1e-2).to(torch.bfloat16).to(DEV)
    pool = torch.rand(nsc * 256, generator=g).to(torch.bfloat16 if (dt == torch.bfloat16 or strategy == 2) else dt).to(DEV)
    cap = capi.mixed_required_bytes(nsc, world)
    out = torch.full((n_valid + 300,), 7.0, dtype=dt, device=DEV)
    out_ref = torch.full((n_valid + 300,), 7.0, dtype=dt, device=DEV)
    for chunk in range(world):
        segs, total = segments(counts, chunk, world, nsc)
        assert total <= cap
        enc = torch.full((cap + 16,), 0xAB, dtype=torch.uint8, device=DEV)
        send = torch.full((cap + 16,), 0xCD, dtype=torch.uint8, device=DEV)
        capi.mixed_compress(full, order, work, enc, nsc, strategy, rand_pool=pool, ring_chunk=chunk, ring_world=world)
        peer_before = peer.clone()
        capi.mixed_compress(peer, order, work, send, nsc, strategy, rand_pool=pool, recv=enc, ring_chunk=chunk,
                            ring_world=world)
        assert torch.equal(peer, peer_before)
        capi.mixed_decompress(send, out, order, work, nsc, strategy, stats=stats, n_limit=n_valid, ring_chunk=chunk,
                              ring_world=world)
        assert bool((enc[total:] == 0xAB).all()) and bool((send[total:] == 0xCD).all())    # nothing past the stream
        for width, row0, pos, cnt, off in segs:
            if cnt == 0:
                continue
            rows = order[row0:row0 + cnt]
            rnd = pool[pos * 256:(pos + cnt) * 256]
            nb = cnt * REC[width]
            e = torch.zeros(nb, dtype=torch.uint8, device=DEV)
            s = torch.zeros(nb, dtype=torch.uint8, device=DEV)
            capi.scaling_compress_rows(full, rows, e, rnd, cnt, width, strategy)
            capi.scaling_dec_comp_rows(e, peer, rows, s, rnd, cnt, width, strategy)
            assert torch.equal(enc[off:off + nb], e), (chunk, width)
            assert torch.equal(send[off:off + nb], s), (chunk, width)
            capi.scaling_decompress_rows(s, out_ref, rows, stats, n_valid, cnt, width, strategy)
    assert torch.equal(bits_t(out), bits_t(out_ref))
    assert bool((out[n_valid:] == 7.0).all())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("strategy,world", [(2, 1), (3, 2)])
def test_long_runs_take_the_decoders_of_several_tiles_per_wave(capi, dt, strategy, world):
    """From 262,144 superchunks per ring chunk (or rows of a list) on, the decoders run as waves of four tiles that fetch
    their row-list entries with one load.  Their output must be that of the one-tile kernels, which the same records
    reach here in pieces of 100,000 rows."""
    nsc = 450_001 * world + 5
    n_valid = nsc * 256 - 77
    q, order, work = make_plan(capi, nsc, 11 + world, (1, 6, 2))
    counts = work[:3].tolist()
    g = torch.Generator(device=DEV).manual_seed(5 + strategy)
    full = (torch.randn(nsc * 256, generator=g, device=DEV) * 1e-2).to(dt)
    stats = torch.randn(nsc, 2, generator=g, device=DEV).mul(1e-2).to(torch.bfloat16)
    cap = capi.mixed_required_bytes(nsc, world)
    out = torch.full((n_valid + 300,), 7.0, dtype=dt, device=DEV)
    out_ref = torch.full((n_valid + 300,), 7.0, dtype=dt, device=DEV)
    out_rows = torch.full((n_valid + 300,), 7.0, dtype=dt, device=DEV)
    long_runs = 0
    for chunk in range(world):
        segs, total = segments(counts, chunk, world, nsc)
        enc = torch.zeros(cap, dtype=torch.uint8, device=DEV)
        capi.mixed_compress(full, order, work, enc, nsc, strategy, seed=3, step=chunk, ring_chunk=chunk, ring_world=world)
        capi.mixed_decompress(enc, out, order, work, nsc, strategy, stats=stats, n_limit=n_valid, ring_chunk=chunk,
                              ring_world=world)
        for width, row0, pos, cnt, off in segs:
            rows = order[row0:row0 + cnt]
            for a in range(0, cnt, 100_000):
                b = min(cnt, a + 100_000)
                capi.scaling_decompress_rows(enc[off + a * REC[width]:off + b * REC[width]], out_ref, rows[a:b], stats, n_valid,
                                             b - a, width, strategy)
            capi.scaling_decompress_rows(enc[off:off + cnt * REC[width]], out_rows, rows, stats, n_valid, cnt, width, strategy)
            long_runs += cnt >= 262144
    assert long_runs >= 1                  # the row-list decoder took its long variant as well
    assert torch.equal(bits_t(out), bits_t(out_ref))
    assert torch.equal(bits_t(out_rows), bits_t(out_ref))
    assert bool((out[n_valid:] == 7.0).all()) and bool((out_rows[n_valid:] == 7.0).all())
    # and the decoded values are the source to within the 2-bit step of its widest class
    assert float((out[:n_valid].float() - stats[:, 0].float().repeat_interleave(256)[:n_valid] - full[:n_valid].float()).abs().max()) < 0.1


@pytest.mark.parametrize("dt,odt", [(torch.bfloat16, BF16), (torch.float32, F32)])
@pytest.mark.parametrize("strategy", [2, 3])
def test_mixed_philox_matches_oracle(capi, oracle, dt, odt, strategy):
    """in-kernel rounding stream keyed by the chunk's index in the source vector: every run equals the oracle's
    compress of the gathered superchunks with the gathered uniform values"""
    nsc, seed, step = 333, 2027, 5
    q, order, work = make_plan(capi, nsc, 17)
    counts = work[:3].tolist()
    g = torch.Generator().manual_seed(5)
    full = (torch.randn(nsc * 256, generator=g) * 1e-2).to(dt).to(DEV)
    enc = torch.zeros(capi.mixed_required_bytes(nsc, 1), dtype=torch.uint8, device=DEV)
    capi.mixed_compress(full, order, work, enc, nsc, strategy, seed=seed, step=step)
    uni = oracle.philox_uniform(nsc * 256, seed, step)
    if odt == BF16:
        uni = (uni.view(np.uint32) >> 16).astype(np.uint16)     # k/256 is exact in bf16
    src_h = to_bits(full.cpu())
    ord_h = order.cpu().numpy()
    segs, total = segments(counts, 0, 1, nsc)
    got = enc.cpu().numpy()
    for width, row0, pos, cnt, off in segs:
        rows = ord_h[row0:row0 + cnt]
        gs = src_h.reshape(-1, 256)[rows].reshape(-1).copy()
        gu = uni.reshape(-1, 256)[rows].reshape(-1).copy()
        want = oracle.scaling_compress(gs, gu, cnt * 256, width, 16, strategy, odt)
        assert (got[off:off + cnt * REC[width]] == want).all(), width
    # natural order (rows == identity) of the single-width Philox call uses the same key
    e4 = torch.zeros(capi.required_bytes(nsc * 256, 4, 16, strategy), dtype=torch.uint8, device=DEV)
    capi.scaling_compress_philox(full, e4, nsc * 256, 4, 16, strategy, seed, step)
    want = oracle.scaling_compress(src_h, uni, nsc * 256, 4, 16, strategy, odt)
    assert (e4.cpu().numpy() == want).all()


@pytest.mark.parametrize("dt,odt", [(torch.bfloat16, BF16), (torch.float32, F32)])
@pytest.mark.parametrize("world", [1, 2, 3, 8, 6, 24])
@pytest.mark.parametrize("n", [256 * 40, 256 * 41 - 200, 256 * 41 - 1, 77])
def test_stats_and_centre_on_load(capi, oracle, dt, odt, world, n):
    """superchunk_stats == the oracle's statistics and binary32 means; compress with the centring folded into the
    load == mean_center followed by compress of the residual, with nothing read beyond n"""
    nsc = (n + 255) // 256
    g = torch.Generator().manual_seed(n + world)
    base = torch.randn(n, generator=g) * 1e-2 + 3e-3
    if n >= 1024:
        # superchunks at the bottom of the exponent range: element / world is a denormal binary32 number there, and
        # the centred value must still be the one of the two-step arithmetic
        base[256:512] = torch.randn(256, generator=g) * 1e-39
        base[512:768] = torch.randn(256, generator=g) * 3e-38
        # element / world exactly half-way between two subnormal numbers (m 2^-150, m odd; representable in binary32 for
        # an even world size that is not a power of two), in pairs that cancel in the first step of the mean's tree:
        # the mean is zero and the residual is the rounded quotient itself
        m = torch.randint(0, 500, (128,), generator=g).double() * 2 + 1
        tie = m * world * 2.0 ** -150
        base = base.double()
        base[768:896] = tie
        base[896:1024] = -tie
        base = base.float()
    src = torch.full((n + 64,), float("nan"), dtype=dt, device=DEV)     # a NaN beyond n must never be picked up
    src[:n] = base.to(dt)
    stats = torch.zeros(nsc, 2, dtype=torch.bfloat16, device=DEV)
    mean = torch.zeros(nsc, dtype=torch.float32, device=DEV)
    capi.superchunk_stats(src, stats, mean, n, world)
    st_o, mean_o = oracle.superchunk_stats(to_bits(src[:n].cpu()), n, world, odt)
    assert (to_bits(stats.cpu()).reshape(-1) == st_o).all()
    assert (mean.cpu().numpy().view(np.uint32) == mean_o.view(np.uint32)).all()
    stats2 = torch.zeros_like(stats)
    capi.superchunk_stats(src, stats2, None, n, world)
    assert torch.equal(bits_t(stats), bits_t(stats2))

    residual = torch.zeros(nsc * 256, dtype=dt, device=DEV)
    stats3 = torch.zeros_like(stats)
    capi.superchunk_mean_center(src, residual, stats3, n, world)
    assert torch.equal(bits_t(stats), bits_t(stats3))
    res_o, _ = oracle.superchunk_mean_center(to_bits(src[:n].cpu()), n, world, odt)
    assert (to_bits(residual.cpu()).view(res_o.dtype if odt != F32 else np.uint32) ==
            (res_o if odt != F32 else res_o.view(np.uint32))).all()
    q, order, work = make_plan(capi, nsc, n)
    pool = torch.rand(nsc * 256, generator=g)
    pool[768:1024] = 0.0        # (a random value of 0 turns the lowest bit of a tiny quotient into a code)
    pool = pool.to(dt).to(DEV)
    cap = capi.mixed_required_bytes(nsc, 1)
    for strategy in (2, 3):
        a = torch.zeros(cap, dtype=torch.uint8, device=DEV)
        b = torch.zeros(cap, dtype=torch.uint8, device=DEV)
        capi.mixed_compress(residual, order, work, a, nsc, strategy, rand_pool=pool)
        capi.mixed_compress(src, order, work, b, nsc, strategy, rand_pool=pool, center_mean=mean, center_world=world, n=n)
        assert torch.equal(a, b), strategy
        # the fused step centres its local operand the same way
        a2, b2 = torch.zeros_like(a), torch.zeros_like(a)
        capi.mixed_compress(residual, order, work, a2, nsc, strategy, seed=9, step=1, recv=a)
        capi.mixed_compress(src, order, work, b2, nsc, strategy, seed=9, step=1, recv=a, center_mean=mean,
                            center_world=world, n=n)
        assert torch.equal(a2, b2), strategy


def test_mixed_misaligned_buffers(capi):
    """element buffers that are only element-aligned and streams at odd byte offsets"""
    nsc = 203
    q, order, work = make_plan(capi, nsc, 3)
    g = torch.Generator().manual_seed(1)
    dt = torch.bfloat16
    full_al = (torch.randn(nsc * 256, generator=g) * 1e-2).to(dt).to(DEV)
    pool_al = torch.rand(nsc * 256, generator=g).to(dt).to(DEV)
    full = torch.zeros(nsc * 256 + 8, dtype=dt, device=DEV)[3:3 + nsc * 256].copy_(full_al)
    pool = torch.zeros(nsc * 256 + 8, dtype=dt, device=DEV)[1:1 + nsc * 256].copy_(pool_al)
    cap = capi.mixed_required_bytes(nsc, 1)
    ref = torch.zeros(cap, dtype=torch.uint8, device=DEV)
    capi.mixed_compress(full_al, order, work, ref, nsc, 2, rand_pool=pool_al)
    enc = torch.zeros(cap + 16, dtype=torch.uint8, device=DEV)[5:5 + cap]
    capi.mixed_compress(full, order, work, enc, nsc, 2, rand_pool=pool)
    assert torch.equal(enc, ref)
    out_ref = torch.zeros(nsc * 256, dtype=dt, device=DEV)
    capi.mixed_decompress(ref, out_ref, order, work, nsc, 2)
    out = torch.zeros(nsc * 256 + 8, dtype=dt, device=DEV)[1:1 + nsc * 256]
    capi.mixed_decompress(enc, out, order, work, nsc, 2)
    assert torch.equal(bits_t(out), bits_t(out_ref))


def test_mixed_pipeline_replays_as_graph(capi):
    """stats -> plan -> compress -> decompress of a bucket is a fixed launch sequence with no read-back: captured
    once, replayed on new data, every replay equals the eager result"""
    n = 6553600 // 4
    nsc = n // 256
    g = torch.Generator().manual_seed(11)
    scales = torch.exp(torch.randn(nsc, 1, generator=g) * 6.0) * 1e-3
    src = torch.empty(n, dtype=torch.bfloat16, device=DEV)
    stats = torch.zeros(nsc, 2, dtype=torch.bfloat16, device=DEV)
    mean = torch.zeros(nsc, dtype=torch.float32, device=DEV)
    order = torch.zeros(3 * nsc, dtype=torch.int32, device=DEV)
    work = torch.zeros(capi.group_plan_work_ints(nsc), dtype=torch.int32, device=DEV)
    enc = torch.zeros(capi.mixed_required_bytes(nsc, 1), dtype=torch.uint8, device=DEV)
    out = torch.zeros(n, dtype=torch.bfloat16, device=DEV)
    u = 7.1

    def fill(seed):
        gg = torch.Generator().manual_seed(seed)
        src.copy_((torch.randn(nsc, 256, generator=gg) * scales).reshape(-1).to(torch.bfloat16))

    def pipeline(stream=None):
        capi.superchunk_stats(src, stats, mean, n, 1, stream=stream)
        capi.group_plan_stats(stats, u, None, order, work, stream=stream)
        capi.mixed_compress(src, order, work, enc, nsc, 2, seed=1, step=0, center_mean=mean, center_world=1, n=n,
                            stream=stream)
        capi.mixed_decompress(enc, out, order, work, nsc, 2, stats=stats, n_limit=n, stream=stream)

    fill(0)
    pipeline()
    torch.cuda.synchronize()
    counts0 = work[:3].tolist()
    assert min(counts0) > 0, counts0
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            pipeline(side.cuda_stream)
    for seed in (1, 2, 3):
        fill(seed)
        graph.replay()
        torch.cuda.synchronize()
        got, got_enc, got_counts = out.clone(), enc.clone(), work[:3].tolist()
        out.zero_()
        pipeline()
        torch.cuda.synchronize()
        assert got_counts == work[:3].tolist()
        total = sum(c * REC[w] for c, w in zip(got_counts, (8, 4, 2)))
        assert torch.equal(got_enc[:total], enc[:total])
        assert torch.equal(bits_t(got), bits_t(out))
        err = (out.float() - src.float()).pow(2).sum() / src.float().pow(2).sum()
        assert float(err) < 0.05


@pytest.mark.parametrize("W", [1, 2, 3])
@pytest.mark.parametrize("strategy", [2, 3])
def test_single_pass_pipeline_matches_oracle(capi, oracle, W, strategy):
    """the whole device-resident all-reduce (statistics, widths, partition, ring of mixed launches, mean add) against
    the oracle's functions chained on the host, bit for bit, for every simulated rank"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import dynamic_bitrate_allreduce_single_pass
    n, seed, u = 256 * 301 - 100, 77, 6.0
    nsc = (n + 255) // 256
    g = torch.Generator().manual_seed(W * 10 + strategy)
    scales = torch.exp(torch.randn(nsc, 1, generator=g) * 6.0) * 1e-3
    vecs = [((torch.randn(nsc, 256, generator=g) * scales).reshape(-1)[:n] + 1e-4).to(torch.bfloat16) for _ in range(W)]
    outs, total, counts = dynamic_bitrate_allreduce_single_pass([v.to(DEV) for v in vecs], u, strategy=strategy, seed=seed)
    torch.cuda.synchronize()

    # host chain
    res, stats = [], []
    for v in vecs:
        r, s = oracle.superchunk_mean_center(to_bits(v), n, W, BF16)
        res.append(r.reshape(-1, 256))
        stats.append(torch.from_numpy(s.view(np.int16).copy()).view(torch.bfloat16))
    tot = stats[0].clone()
    for s in stats[1:]:
        tot.add_(s)                                   # bf16 adds, the order of the pipeline
    tot_bits = to_bits(tot)
    assert (to_bits(total.cpu()).reshape(-1) == tot_bits).all()
    qb = oracle.dynamic_bitrate_qbits(tot_bits[1::2].copy(), u)
    cnt = [int((qb == w).sum()) for w in (8, 4, 2)]
    assert counts.tolist() == cnt + [0] and min(cnt) > 0, (counts.tolist(), cnt)
    uni = {}

    def U(rank, step, rows):
        if (rank, step) not in uni:
            x = oracle.philox_uniform(nsc * 256, seed + rank, step)
            uni[(rank, step)] = (x.view(np.uint32) >> 16).astype(np.uint16).reshape(-1, 256)
        return uni[(rank, step)][rows].reshape(-1).copy()

    want = np.zeros((nsc, 256), np.uint16)
    for width in (8, 4, 2):
        rows_g = np.nonzero(qb == width)[0]
        per = -(-rows_g.size // W)
        for c in range(W):
            rows = rows_g[per * c:per * (c + 1)]
            if rows.size == 0:
                continue
            m = rows.size * 256
            stream = oracle.scaling_compress(res[c][rows].reshape(-1).copy(), U(c, 0, rows), m, width, 16, strategy, BF16)
            for s in range(1, W):
                rank = (c + s) % W
                stream = oracle.scaling_dec_comp(stream, res[rank][rows].reshape(-1).copy(), U(rank, s, rows), m, width, 16,
                                                 strategy, BF16)
            dec = np.zeros(m, np.uint16)
            oracle.scaling_decompress(stream, dec, m, width, 16, strategy, BF16)
            want[rows] = dec.reshape(-1, 256)
    final = oracle.superchunk_add_mean_copy(want.reshape(-1), tot_bits, n, BF16)
    for r in range(W):
        assert (to_bits(outs[r].cpu()) == final).all(), r
    exact = torch.stack([v.double() for v in vecs]).sum(0) / W
    err = float((outs[0].cpu().double() - exact).pow(2).sum() / exact.pow(2).sum())
    assert err < 0.02, err


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("strategy", [2, 3])
def test_mixed_special_values(capi, dt, strategy):
    """NaN, infinities, huge, tiny and all-zero superchunks take the guarded path of a wave: the folded calls still equal
    mean_center + the per-width calls, and the random pool may hold values outside [0, 1]"""
    nsc, n = 97, 97 * 256 - 13
    g = torch.Generator().manual_seed(7 + strategy)
    x = torch.randn(n, generator=g) * 1e-2
    x[5] = float("nan"); x[300] = float("inf"); x[301] = float("-inf"); x[1000] = 3e38; x[1001] = -1e-40
    x[256 * 10:256 * 12] = 0.0
    x[256 * 20:256 * 21] = 1e30
    x[256 * 30:256 * 31] = 1e-38
    src = x.to(dt).to(DEV)
    pool = torch.rand(nsc * 256, generator=g)
    pool[77] = 1.5; pool[78] = -0.25; pool[79] = float("nan")
    pool = pool.to(dt).to(DEV)
    q, order, work = make_plan(capi, nsc, 5)
    counts = work[:3].tolist()
    stats = torch.zeros(nsc, 2, dtype=torch.bfloat16, device=DEV)
    mean = torch.zeros(nsc, device=DEV)
    capi.superchunk_stats(src, stats, mean, n, 3)
    residual = torch.zeros(nsc * 256, dtype=dt, device=DEV)
    stats2 = torch.zeros_like(stats)
    capi.superchunk_mean_center(src, residual, stats2, n, 3)
    assert torch.equal(bits_t(stats), bits_t(stats2))
    cap = capi.mixed_required_bytes(nsc, 1)
    enc = torch.zeros(cap, dtype=torch.uint8, device=DEV)
    capi.mixed_compress(src, order, work, enc, nsc, strategy, rand_pool=pool, center_mean=mean, center_world=3, n=n)
    out = torch.full((n,), 7.0, dtype=dt, device=DEV)
    capi.mixed_decompress(enc, out, order, work, nsc, strategy, stats=stats, n_limit=n)
    out_ref = torch.full((n,), 7.0, dtype=dt, device=DEV)
    segs, total = segments(counts, 0, 1, nsc)
    for width, row0, pos, cnt, off in segs:
        rows = order[row0:row0 + cnt]
        e = torch.zeros(cnt * REC[width], dtype=torch.uint8, device=DEV)
        capi.scaling_compress_rows(residual, rows, e, pool[pos * 256:(pos + cnt) * 256], cnt, width, strategy)
        assert torch.equal(enc[off:off + e.numel()], e), width
        capi.scaling_decompress_rows(e, out_ref, rows, stats, n, cnt, width, strategy)
    assert torch.equal(bits_t(out), bits_t(out_ref))


@pytest.mark.parametrize("block", range(6))
def test_mixed_random_shapes(capi, block):
    """seeded random plans, ring splits, element types, random sources and alignments: the one-launch calls against
    the per-width calls on every run of every ring chunk"""
    rng = np.random.default_rng(1000 + block)
    for case in range(12):
        nsc = int(rng.choice([1, 3, 4, 5, 63, 64, 65, 257, 1023, 1500, 4097]))
        world = int(rng.choice([1, 2, 3, 5, 8]))
        weights = tuple(float(w) for w in rng.choice([0.0, 0.2, 1.0, 3.0], size=3))
        if sum(weights) == 0:
            weights = (1.0, 1.0, 1.0)
        dt = [torch.bfloat16, torch.float32][int(rng.integers(2))]
        strategy = int(rng.choice([2, 3]))
        use_philox = bool(rng.integers(2))
        seed = int(rng.integers(1 << 30))
        q, order, work = make_plan(capi, nsc, seed, weights)
        counts = work[:3].tolist()
        g = torch.Generator().manual_seed(seed)
        shift = int(rng.integers(0, 4)) * (8 if dt == torch.bfloat16 else 4) + int(rng.integers(2))   # element offset of the view
        full = torch.zeros(nsc * 256 + 64, dtype=dt, device=DEV)[shift:shift + nsc * 256]
        full.copy_((torch.randn(nsc * 256, generator=g) * float(10.0 ** rng.uniform(-6, 2))).to(dt))
        peer = (torch.randn(nsc * 256, generator=g) * 1e-2).to(dt).to(DEV)
        pool_dt = dt if (dt == torch.bfloat16 or rng.integers(2)) else torch.bfloat16
        pool = torch.rand(nsc * 256, generator=g).to(pool_dt).to(DEV)
        cap = capi.mixed_required_bytes(nsc, world)
        off0 = int(rng.integers(0, 16))
        tag = (block, case, nsc, world, weights, dt, strategy, use_philox, shift, off0)
        for chunk in range(world):
            enc = torch.zeros(cap + 32, dtype=torch.uint8, device=DEV)[off0:off0 + cap]
            send = torch.zeros(cap + 32, dtype=torch.uint8, device=DEV)[off0:off0 + cap]
            kw = dict(seed=seed, step=chunk) if use_philox else dict(rand_pool=pool)
            capi.mixed_compress(full, order, work, enc, nsc, strategy, ring_chunk=chunk, ring_world=world, **kw)
            capi.mixed_compress(peer, order, work, send, nsc, strategy, recv=enc, ring_chunk=chunk, ring_world=world, **kw)
            segs, total = segments(counts, chunk, world, nsc)
            for width, row0, pos, cnt, off in segs:
                if cnt == 0:
                    continue
                rows = order[row0:row0 + cnt]
                nb = cnt * REC[width]
                if use_philox:
                    uni = torch.empty(nsc * 256, dtype=dt, device=DEV)
                    capi.philox_uniform(uni, seed, chunk)
                    rnd = uni.view(-1, 256)[rows.long()].reshape(-1).contiguous()
                else:
                    rnd = pool[pos * 256:(pos + cnt) * 256]
                e = torch.zeros(nb, dtype=torch.uint8, device=DEV)
                s = torch.zeros(nb, dtype=torch.uint8, device=DEV)
                capi.scaling_compress_rows(full, rows, e, rnd, cnt, width, strategy)
                capi.scaling_dec_comp_rows(e, peer, rows, s, rnd, cnt, width, strategy)
                assert torch.equal(enc[off:off + nb], e), tag + (chunk, width)
                assert torch.equal(send[off:off + nb], s), tag + (chunk, width)


def _llama_like(n, seed, dt=torch.bfloat16):
    g = torch.Generator(device=DEV).manual_seed(seed)
    nsc = (n + 255) // 256
    scales = torch.exp(torch.randn(nsc, 1, generator=g, device=DEV) * 6.0) * 1e-3
    return ((torch.randn(nsc, 256, generator=g, device=DEV) * scales).reshape(-1)[:n] + 1e-4).to(dt)


def _four_calls(capi, x, n, u, strategy, seed, step, world=1):
    nsc = (n + 255) // 256
    stats = torch.zeros((nsc, 2), dtype=torch.bfloat16, device=DEV)
    mean = torch.zeros(nsc, dtype=torch.float32, device=DEV)
    order = torch.full((3 * nsc,), -1, dtype=torch.int32, device=DEV)
    work = torch.zeros(capi.group_plan_work_ints(nsc), dtype=torch.int32, device=DEV)
    packed = torch.zeros(capi.mixed_required_bytes(nsc, 1), dtype=torch.uint8, device=DEV)
    out = torch.zeros_like(x)
    capi.superchunk_stats(x, stats, mean, n, world)
    capi.group_plan_stats(stats, u, None, order, work)
    capi.mixed_compress(x, order, work, packed, nsc, strategy, seed=seed, step=step, center_mean=mean, center_world=world, n=n)
    capi.mixed_decompress(packed, out, order, work, nsc, strategy, stats=stats, n_limit=n)
    return stats, mean, order, work, packed, out


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("strategy", [2, 3])
def test_bucket_call_equals_the_four_calls(capi, eden_utils, dt, strategy):
    """dq_dynamic_bitrate_bucket enqueues statistics -> plan -> mixed compress -> mixed decompress with one host call: every
    buffer it writes equals what the four calls write, for all stages at once, for the stages one by one, with u in
    device memory, through ctypes and through the module; step_dev adds to the step of the rounding stream"""
    n, u, seed, step = 256 * 700 - 131, 6.0, 11, 5
    nsc = (n + 255) // 256
    x = _llama_like(n, 3, dt)
    ref = _four_calls(capi, x, n, u, strategy, seed, step)
    assert min(ref[3][:3].tolist()) > 0

    def fresh():
        return (torch.zeros((nsc, 2), dtype=torch.bfloat16, device=DEV), torch.zeros(nsc, dtype=torch.float32, device=DEV),
                torch.full((3 * nsc,), -1, dtype=torch.int32, device=DEV),
                torch.zeros(capi.group_plan_work_ints(nsc), dtype=torch.int32, device=DEV),
                torch.zeros(capi.mixed_required_bytes(nsc, 1), dtype=torch.uint8, device=DEV), torch.zeros_like(x))

    def same(got):
        counts = ref[3][:3].tolist()
        used = sum(c * r for c, r in zip(counts, (274, 146, 82)))
        assert torch.equal(bits_t(got[0]), bits_t(ref[0])) and torch.equal(bits_t(got[1]), bits_t(ref[1]))
        assert got[3][:4].tolist() == ref[3][:4].tolist()
        for g_, c in enumerate(counts):
            assert torch.equal(got[2][g_ * nsc:g_ * nsc + c], ref[2][g_ * nsc:g_ * nsc + c])
        assert torch.equal(got[4][:used], ref[4][:used])
        assert torch.equal(bits_t(got[5]), bits_t(ref[5]))

    # all stages, u a number
    bufs = fresh()
    desc, dev = capi.bucket_descriptor(x, n, *bufs[:5], strategy=strategy, out=bufs[5], u=u, seed=seed, step=step)
    capi.dynamic_bitrate_bucket(desc, dev)
    same(bufs)
    # stage by stage, u and the step offset in device memory
    bufs = fresh()
    u_dev = torch.full((1,), u, dtype=torch.float64, device=DEV)
    step_dev = torch.full((1,), 3, dtype=torch.int64, device=DEV)
    desc, dev = capi.bucket_descriptor(x, n, *bufs[:5], strategy=strategy, out=bufs[5], u=u_dev, seed=seed, step=step - 3,
                                       step_dev=step_dev)
    for stage in (capi.STAGE_STATS, capi.STAGE_PLAN, capi.STAGE_COMPRESS, capi.STAGE_DECOMPRESS):
        capi.dynamic_bitrate_bucket(desc, dev, stages=stage)
    same(bufs)
    # another value of the device-side step: other random values, other bytes
    step_dev.fill_(4)
    capi.dynamic_bitrate_bucket(desc, dev, stages=capi.STAGE_COMPRESS)
    assert not torch.equal(bufs[4], ref[4])
    # the module's twin
    bufs = fresh()
    eden_utils.dynamic_bitrate_bucket(x, n, *bufs[:5], bufs[5], u=u, seed=seed, step=step, strategy=strategy,
                                      stream_p=torch.cuda.current_stream().cuda_stream)
    same(bufs)
    # refusals come before any launch
    with pytest.raises(RuntimeError):
        capi.bucket_descriptor(x, n, bufs[0], bufs[1], bufs[2], bufs[3], bufs[4][:100], strategy=strategy)
    bad, dev = capi.bucket_descriptor(x, n, *bufs[:5], strategy=strategy, out=None, u=u)
    with pytest.raises(RuntimeError):
        capi.dynamic_bitrate_bucket(bad, dev)                     # the decode stage without an output
    torch.cuda.synchronize()


@pytest.mark.parametrize("streams,recorded,whole", [(1, False, False), (2, False, False), (2, True, True), (3, True, False),
                                                    (2, False, True)])
def test_single_pass_buckets_object(capi, streams, recorded, whole):
    """a stream of buckets through the pipeline object -- one host call per bucket or per step, enqueued anew or recorded on the
    second step and replayed -- gives, on every training step, the outputs of the four calls with the rounding stream (seed,
    bucket ordinal * 2^32 + step)"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import SinglePassBuckets
    sizes = [256 * 123, 256 * 300, 256 * 300 - 5, 256 * 300, 256 * 77 + 1]      # (a later, larger bucket makes the scratch grow)
    xs = [_llama_like(n, 40 + k) for k, n in enumerate(sizes)]
    outs = [torch.zeros_like(x) for x in xs]
    seed, u = 9, 6.0
    pipe = SinglePassBuckets(DEV, strategy=2, seed=seed, streams=streams, u=u)
    graph = None

    def enqueue():
        pipe.begin_step()
        if whole:
            pipe.run_all(list(zip(xs, outs)))
        else:
            for x, o in zip(xs, outs):
                pipe.run(x, o)
        pipe.join()

    for step in range(1, 6):
        if recorded and step == 2:
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                enqueue()
        if step == 4:
            u = 7.5
            pipe.set_u(u)
        for x in xs:
            x.mul_(1.25)                      # the sources change between steps; a replay must read the new values
        if graph is None:
            enqueue()
        else:
            pipe.join()
            graph.replay()
        torch.cuda.synchronize()
        for k, (x, o) in enumerate(zip(xs, outs)):
            want = _four_calls(capi, x, x.numel(), u, 2, seed, (k << 32) + step)[5]
            assert torch.equal(bits_t(o), bits_t(want)), (step, k)
            o.zero_()


def test_streams_of_the_pipeline_object_run_side_by_side(capi):
    """dq_streams_overlap: a stream against itself never overlaps; the streams SinglePassBuckets settles on overlap
    with each other and with the caller's stream, also after the process has used up several streams of torch's pool
    (the runtime maps streams onto four hardware queues at their first use, and a queue works in order)"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import SinglePassBuckets
    index = torch.cuda.current_device()
    st = torch.cuda.Stream()
    assert capi.streams_overlap(st.cuda_stream, st.cuda_stream, index) is False
    with pytest.raises(RuntimeError):
        capi._check(capi.lib().dq_streams_overlap(None, None, index, None))
    scratch = torch.zeros(64, device=DEV)
    for used in range(5):
        for streams in (2, 3):
            pipe = SinglePassBuckets(DEV, strategy=2, seed=1, streams=streams, u=6.0)
            assert pipe.side_by_side and len(pipe.streams) == streams
            handles = [torch.cuda.current_stream().cuda_stream] + [s.cuda_stream for s in pipe.streams]
            assert len(set(handles)) == streams + 1
            for i in range(streams + 1):
                for j in range(i + 1, streams + 1):
                    assert capi.streams_overlap(handles[i], handles[j], index), (used, streams, i, j)
        extra = torch.cuda.Stream()              # one more stream of the pool gets its queue
        with torch.cuda.stream(extra):
            scratch.add_(1.0)
        torch.cuda.synchronize()


def test_stream_order_after_orders_two_streams(capi):
    """dq_stream_order_after: work enqueued on the waiting stream afterwards sees what the other stream had been given
    before the call -- also on the 65th and later calls, when the library's ring of events is being reused"""
    index = torch.cuda.current_device()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    big = torch.zeros(1 << 24, device=DEV)
    flag = torch.zeros(8, device=DEV)
    seen = torch.zeros(200, 8, device=DEV)
    torch.cuda.synchronize()
    for k in range(200):
        with torch.cuda.stream(a):
            for _ in range(3):
                big.add_(1.0)                 # something for the flag's writer to queue behind
            flag.fill_(float(k + 1))
        capi.stream_order_after(b, a, index)
        with torch.cuda.stream(b):
            seen[k].copy_(flag)
        capi.stream_order_after(a, b, index)  # the next round's fill must not overtake this copy
    torch.cuda.synchronize()
    assert torch.equal(seen[:, 0].cpu(), torch.arange(1, 201, dtype=torch.float32))
    capi.stream_order_after(a, a, index)      # a stream after itself: nothing to do


@pytest.mark.parametrize("streams", [1, 2, 3])
def test_single_pass_buckets_alternating_between_recorded_and_eager_steps(capi, streams):
    """a step recorded at the start is replayed on a stream of its own, between steps that are enqueued on the caller's as a list or
    bucket by bucket (and a change of u in between): every step gives the outputs of the four calls"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import SinglePassBuckets
    sizes = [256 * 200, 256 * 200, 256 * 120 + 3, 256 * 200, 256 * 64]
    xs = [_llama_like(n, 60 + k) for k, n in enumerate(sizes)]
    outs = [torch.zeros_like(x) for x in xs]
    seed, u = 4, 6.5
    pipe = SinglePassBuckets(DEV, strategy=2, seed=seed, streams=streams, u=u)
    pairs = list(zip(xs, outs))
    main, side = torch.cuda.current_stream(), torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        pipe.begin_step()
        pipe.run_all(pairs)
    modes = ["list", "each", "replay", "replay", "list", "replay", "each", "each", "replay", "list"]
    x_then = [[None] * len(xs) for _ in modes]
    o_then = [[None] * len(xs) for _ in modes]
    us = []
    # no synchronisation between the steps
    for step, mode in enumerate(modes, start=1):
        if step == 5:
            u = 7.25
            pipe.set_u(u)
        us.append(u)
        for k, x in enumerate(xs):
            x.mul_(1.125)
            x_then[step - 1][k] = x.clone()
        if mode == "replay":
            side.wait_stream(main)                # the sources
            with torch.cuda.stream(side):
                pipe.join()
                graph.replay()
        else:
            pipe.begin_step()
            if mode == "list":
                pipe.run_all(pairs)
            else:
                for x, o in pairs:
                    pipe.run(x, o)
        pipe.join()
        for k, o in enumerate(outs):
            o_then[step - 1][k] = o.clone()
    torch.cuda.synchronize()
    for step, mode in enumerate(modes, start=1):
        for k in range(len(xs)):
            x = x_then[step - 1][k]
            want = _four_calls(capi, x, x.numel(), us[step - 1], 2, seed, (k << 32) + step)[5]
            assert torch.equal(bits_t(o_then[step - 1][k]), bits_t(want)), (step, mode, k)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("W,n", [(1, 256), (1, 255), (1, 256 * 9 - 3), (2, 256 * 8), (3, 256 * 37 + 1), (8, 1), (8, 256 * 70 - 255), (16, 256 * 201)])
def test_ranks_in_registers_equal_the_ring_in_steps(capi, W, n, dt):
    """the all-reduce without packed streams at the edges of its tiles, runs and ring chunks, on unaligned vectors too and with
    every guard of the quantiser firing, against one launch per rank and ring step: same bits, same counts, same statistics"""
    from dynamiq_sigcomm_artifact_amd.bitrate import NormHistogram
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import _single_pass_in_steps, dynamic_bitrate_allreduce_single_pass
    nsc = (n + 255) // 256
    for strategy, shift, u in ((2, 0, 6.0), (3, 1, 6.5)):
        g = torch.Generator().manual_seed(n + W + strategy)
        scales = torch.exp(torch.randn(nsc, 1, generator=g) * 6.0) * 1e-3
        vecs = []
        for r in range(W):
            v = torch.zeros(n + shift, dtype=dt, device=DEV)
            v[shift:].copy_(((torch.randn(nsc, 256, generator=g) * scales).reshape(-1)[:n] + 1e-4).to(dt))
            if r == W - 1 and n > 3000:
                v[shift + 5], v[shift + 700], v[shift + 1500:shift + 1756] = float("nan"), float("inf"), 0.0
            vecs.append(v[shift:])
        a, b = NormHistogram(DEV), NormHistogram(DEV)
        outs, total, counts = dynamic_bitrate_allreduce_single_pass(vecs, u, strategy=strategy, seed=11, norm_histogram=a)
        ref, total2, counts2 = _single_pass_in_steps(vecs, u, strategy, 11, None, {}, None, b)
        assert counts.tolist() == counts2.tolist()
        assert torch.equal(bits_t(total), bits_t(total2)) and torch.equal(a.hist, b.hist) and a.count == b.count
        for r in range(W):
            assert torch.equal(bits_t(outs[r]), bits_t(ref[r])), (strategy, r)
        u_dev = torch.full((1,), u, dtype=torch.float64, device=DEV)
        again, _, _ = dynamic_bitrate_allreduce_single_pass(vecs, u_dev, strategy=strategy, seed=11)
        assert all(torch.equal(bits_t(x), bits_t(y)) for x, y in zip(again, ref))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("W,nsc", [(1, 9), (3, 9), (2, 12289)])
def test_ragged_ends_under_a_large_mean(capi, W, nsc, dt):
    """elements behind the vector's end are zeros to the quantiser and not zeros less the mean: one left over would set the scale of a
    chunk and its superchunk a hundred times too large.  The one-rank pass, the rings with and without lists, against one launch per
    rank and ring step"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import _single_pass_in_steps, dynamic_bitrate_allreduce_single_pass
    g = torch.Generator(device=DEV).manual_seed(nsc + W)
    whole = [(1024.0 + 8.0 * torch.randn(nsc * 256, generator=g, device=DEV)).to(dt) for _ in range(W)]
    for left in (1, 2, 3, 7, 15, 16, 17, 30, 130, 255) if nsc < 100 else (3, 130):
        vecs = [v[:nsc * 256 - 256 + left].clone() for v in whole]
        for strategy, u in ((2, 60.0), (3, 6.0), (2, -60.0)):
            outs, _, _ = dynamic_bitrate_allreduce_single_pass(vecs, u, strategy=strategy, seed=11)
            ref, _, _ = _single_pass_in_steps(vecs, u, strategy, 11, None, {}, None, None)
            assert all(torch.equal(bits_t(x), bits_t(y)) for x, y in zip(outs, ref)), (left, strategy, u)
            # 8 bits: steps of the residuals' largest, at most 50, / 127 (AEE), and the binary16-wide mean's rounding
            if u > 50.0:
                assert float((outs[0].float() - 1024.0).abs().max()) < 64.0, left


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("strategy", [2, 3])
@pytest.mark.parametrize("W,nsc", [(1, 510), (2, 510), (2, 8704)])
def test_chunk_scales_on_whole_ratios(capi, W, nsc, strategy, dt):
    """chunks whose scale is k / 255 of their superchunk's, and a few float32 steps beside it: the scale byte is the ceiling of a number
    on, just below or just above an integer, which the levels in registers estimate and the packed streams divide out"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import _single_pass_in_steps, dynamic_bitrate_allreduce_single_pass
    rng = np.random.default_rng(nsc + strategy)
    top = np.exp(rng.uniform(np.log(1e-3), np.log(1e3), (nsc, 1)))
    r = np.array([127.0, 7.0, 1.0])[np.arange(nsc) % 3][:, None]
    k = rng.integers(1, 256, (nsc, 16)).astype(np.float64)
    k[:, 0] = 255.0
    a = np.maximum((k / 255.0 * (top * W / r + 1e-7) - 1e-7) * r, 0.0).astype(np.float32)
    steps = rng.integers(-3, 4, (nsc, 16))
    steps[:, 0] = 0
    for _ in range(3):
        a = np.where(steps > 0, np.nextafter(a, np.float32(np.inf)), np.where(steps < 0, np.nextafter(a, np.float32(0.0)), a))
        steps = steps - np.sign(steps)
    # (every value with its negative: the means are zero and the centring changes nothing)
    body = a[:, :, None] * rng.uniform(0.0, 1.0, (nsc, 16, 8)).astype(np.float32)
    body[:, :, 3] = a
    x = torch.from_numpy(np.concatenate([body, -body], axis=2).reshape(-1)).to(DEV).to(dt)
    vecs = [x] + [torch.zeros_like(x) for _ in range(W - 1)]
    outs, _, counts = dynamic_bitrate_allreduce_single_pass(vecs, 6.0, strategy=strategy, seed=11)
    ref, _, counts2 = _single_pass_in_steps(vecs, 6.0, strategy, 11, None, {}, None, None)
    assert counts.tolist() == counts2.tolist()
    assert all(torch.equal(bits_t(p), bits_t(q)) for p, q in zip(outs, ref))


@pytest.mark.parametrize("W,n,dt", [
    (8, 1, torch.bfloat16), (2, 256 * 3, torch.float32), (3, 256 * 4 + 1, torch.bfloat16), (16, 256 * 5, torch.bfloat16),
    (2, 256 * 4096, torch.bfloat16), (5, 256 * 4097, torch.bfloat16),          # as many words as a trip takes, one more
    (2, 256 * 12288, torch.bfloat16), (3, 256 * 12288 - 255, torch.float32),   # the last length of two and three fp32 ranks
    (2, 256 * 12288 + 1, torch.bfloat16)])
def test_rings_without_lists(capi, W, n, dt):
    """short rings find their groups from the counts per four superchunks: widths that change from one superchunk to the next, and all
    of one width, against one launch per rank and ring step, which has its lists from the plan"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import _single_pass_in_steps, dynamic_bitrate_allreduce_single_pass
    g = torch.Generator(device=DEV).manual_seed(n + W)
    nsc = (n + 255) // 256
    scales = torch.exp(torch.randn(nsc, 1, generator=g, device=DEV) * 6.0) * 1e-3
    vecs = [(torch.randn(nsc, 256, generator=g, device=DEV) * scales).reshape(-1)[:n].to(dt).contiguous() for _ in range(W)]
    seen = set()
    for strategy, u in ((2, 6.0), (3, 6.5), (2, -40.0), (2, 60.0), (3, float("nan"))):
        u_dev = torch.full((1,), u, dtype=torch.float64, device=DEV)
        ref, total2, counts2 = _single_pass_in_steps(vecs, u_dev, strategy, 11, None, {}, None, None)
        for offset in (u_dev, u) if u == u else (u_dev,):
            outs, total, counts = dynamic_bitrate_allreduce_single_pass(vecs, offset, strategy=strategy, seed=11)
            assert counts.tolist() == counts2.tolist() and torch.equal(bits_t(total), bits_t(total2))
            assert all(torch.equal(bits_t(x), bits_t(y)) for x, y in zip(outs, ref)), (strategy, u)
        seen.add(tuple(c > 0 for c in counts.tolist()))
    assert len(seen) > 1


@pytest.mark.parametrize("shift", [1, 2, 3])
def test_rings_without_lists_with_counts_off_the_16_bytes(capi, shift):
    """group sizes and lists aligned to their 32-bit numbers alone, with the offset a number and in device memory"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import dynamic_bitrate_allreduce_single_pass
    W, n, dt = 3, 256 * 301 - 7, torch.bfloat16
    nsc = (n + 255) // 256
    g = torch.Generator(device=DEV).manual_seed(n)
    scales = torch.exp(torch.randn(nsc, 1, generator=g, device=DEV) * 6.0) * 1e-3
    vecs = [(torch.randn(nsc, 256, generator=g, device=DEV) * scales).reshape(-1)[:n].to(dt).contiguous() for _ in range(W)]
    want, total, counts = dynamic_bitrate_allreduce_single_pass(vecs, 6.0, seed=11)
    ints = lambda m: torch.zeros(m + 4, dtype=torch.int32, device=DEV)[shift:shift + m]
    work = {"key": ("single_pass", nsc, dt, W), "total": torch.empty((nsc, 2), dtype=torch.bfloat16, device=DEV),
            "mean": torch.empty(W * nsc, dtype=torch.float32, device=DEV), "plan": ints(capi.group_plan_work_ints(nsc)), "order": ints(3 * nsc)}
    work["counts"] = work["plan"][:4]
    assert work["counts"].data_ptr() % 16 == 4 * shift
    for u in (6.0, torch.full((1,), 6.0, dtype=torch.float64, device=DEV)):
        outs, total2, counts2 = dynamic_bitrate_allreduce_single_pass(vecs, u, seed=11, work=work)
        assert counts2.data_ptr() == work["counts"].data_ptr() and counts2.tolist() == counts.tolist()
        assert torch.equal(bits_t(total), bits_t(total2)) and all(torch.equal(bits_t(x), bits_t(y)) for x, y in zip(outs, want))
        work["counts"].fill_(-1)


@pytest.mark.parametrize("W,n,dt", [(8, 256 * 12288, torch.bfloat16), (16, 256 * 8705 - 3, torch.float32)])
def test_rings_without_lists_behind_several_tiles_per_wave(capi, W, n, dt):
    """so many ranks that the statistics take four tiles per wave while the ring still goes by their counts"""
    test_rings_without_lists(capi, W, n, dt)


@pytest.mark.parametrize("W,n", [(2, 256 * 8192), (3, 256 * 8192 + 1), (5, 256 * 8195)])
def test_ranks_on_either_side_of_a_superchunk_per_wave(capi, W, n):
    """bf16 beyond the last length of four elements per lane: two superchunks per wave, the last wave with one of them, with lists and
    without"""
    test_ranks_in_registers_equal_the_ring_in_steps(capi, W, n, torch.bfloat16)


@pytest.mark.parametrize("W,n,dt", [
    (2, 256 * 5120, torch.bfloat16), (2, 256 * 5120 + 1, torch.bfloat16), (5, 256 * 5120 + 1, torch.bfloat16),
    (6, 256 * 5120 + 1, torch.bfloat16), (6, 256 * 8192 + 1, torch.bfloat16),
    (2, 256 * 5120, torch.float32), (2, 256 * 5120 + 1, torch.float32), (3, 256 * 8192, torch.float32), (3, 256 * 8192 + 1, torch.float32)])
def test_ranks_on_either_side_of_the_lines_of_a_superchunk_per_wave(capi, W, n, dt):
    """with lists and the values drawn: two bf16 ranks take a superchunk per wave to 5,120 superchunks and two per wave beyond, more of them
    to 7,168; fp32 a superchunk per wave to 8,192, two ranks in AEE to 5,120, and four per wave beyond"""
    test_ranks_in_registers_equal_the_ring_in_steps(capi, W, n, dt)


@pytest.mark.parametrize("W,n,dt", [
    (2, 256 * 5121 - 255, torch.bfloat16), (3, 256 * 5122 - 250, torch.bfloat16), (4, 256 * 5123 - 247, torch.bfloat16),
    (7, 256 * 5127 - 5, torch.bfloat16), (2, 256 * 12288 - 1, torch.bfloat16), (3, 256 * 12289, torch.bfloat16),
    (4, 256 * 20480 - 13, torch.bfloat16), (5, 256 * 20481 - 13, torch.bfloat16)])
def test_rings_of_eight_elements_per_lane(capi, W, n, dt):
    """bf16 with the values drawn, from 5,121 superchunks on (few ranks): two superchunks of different widths and first ranks per wave, the
    last wave with one or both of them, the vector's end at places all over a lane's eight; lists to 12,288 or 20,480 superchunks"""
    test_ranks_in_registers_equal_the_ring_in_steps(capi, W, n, dt)


@pytest.mark.parametrize("W,n,dt", [
    (2, 256 * 5120 - 254, torch.bfloat16), (2, 256 * 5121 - 6, torch.bfloat16), (2, 256 * 20480 - 3, torch.bfloat16),
    (2, 256 * 20480 + 1, torch.bfloat16), (3, 256 * 12288 + 3, torch.float32), (4, 256 * 16384 - 2, torch.float32), (4, 256 * 16384 + 1, torch.float32)])
def test_lines_of_the_rings_without_lists(capi, W, n, dt):
    test_rings_without_lists(capi, W, n, dt)


@pytest.mark.parametrize("W,n", [(3, 256 * 7168), (3, 256 * 7169 - 250), (4, 256 * 7168 - 3), (4, 256 * 7169), (5, 256 * 7168 - 1), (5, 256 * 7169 - 7),
                                 (8, 256 * 7169)])
def test_rings_on_either_side_of_eight_elements_per_lane(capi, W, n):
    """bf16: three and more ranks with lists, five and more without, take four elements per lane to 7,168 superchunks"""
    test_ranks_in_registers_equal_the_ring_in_steps(capi, W, n, torch.bfloat16)
    test_rings_without_lists(capi, W, n, torch.bfloat16)


@pytest.mark.parametrize("W,nsc", [(2, 5121), (3, 12288), (5, 12289), (4, 20480)])
@pytest.mark.parametrize("off_in,off_out", [(1, 3), (0, 1), (2, 0)])
def test_rings_off_the_16_bytes(capi, W, nsc, off_in, off_out):
    """bf16 vectors or outputs (or both) off the 16 bytes; outputs off them take four elements per lane where aligned ones take eight, with
    lists and without"""
    from dynamiq_sigcomm_artifact_amd.bitrate import NormHistogram
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import _single_pass_in_steps, dynamic_bitrate_allreduce_single_pass
    n = nsc * 256 - 3
    g = torch.Generator(device=DEV).manual_seed(nsc + W)
    scales = torch.exp(torch.randn(nsc, 1, generator=g, device=DEV) * 6.0) * 1e-3
    vecs = []
    for _ in range(W):
        v = torch.zeros(n + 8, dtype=torch.bfloat16, device=DEV)
        vecs.append(v[off_in:off_in + n].copy_((torch.randn(nsc, 256, generator=g, device=DEV) * scales).reshape(-1)[:n]))
    for strategy, u in ((2, 6.0), (3, 6.5)):
        ref, _, _ = _single_pass_in_steps(vecs, u, strategy, 11, None, {}, None, None)
        for hist in (None, NormHistogram(DEV)):
            rooms = [torch.full((n + 8,), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(W)]
            outs = [r[off_out:off_out + n] for r in rooms]
            dynamic_bitrate_allreduce_single_pass(vecs, u, strategy=strategy, seed=11, out=outs, norm_histogram=hist)
            assert all(torch.equal(bits_t(x), bits_t(y)) for x, y in zip(outs, ref)), (strategy, hist is None)
            assert all(bool((r[:off_out] == 7.0).all()) and bool((r[off_out + n:] == 7.0).all()) for r in rooms)


@pytest.mark.parametrize("dt,off", [(torch.bfloat16, k) for k in range(1, 8)] + [(torch.float32, k) for k in (1, 2, 3)])
def test_short_rings_at_every_offset_from_the_16_bytes(capi, dt, off):
    """a lane's elements in one piece from any element on, with ends at every place in the last lane and vectors shorter than a lane's
    share; eight elements per lane at the last length"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import _single_pass_in_steps, dynamic_bitrate_allreduce_single_pass
    g = torch.Generator(device=DEV).manual_seed(off)
    whole = [torch.full((256 * 5200 + 16,), 3.0, device=DEV).to(dt) for _ in range(2)]
    for n in (1, 2, 3, 4, 5, 7, 8, 9, 255, 256, 257, 764, 768 + off, 256 * 5122 - off):
        vecs = [w[off:off + n].copy_(torch.randn(n, generator=g, device=DEV)) for w in whole]
        outs, _, _ = dynamic_bitrate_allreduce_single_pass(vecs, 6.0, strategy=2, seed=11)
        ref, _, _ = _single_pass_in_steps(vecs, 6.0, 2, 11, None, {}, None, None)
        assert all(torch.equal(bits_t(x), bits_t(y)) for x, y in zip(outs, ref)), n


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_ends_inside_a_lane_of_a_short_ring(capi, dt):
    """vectors of one to nine elements, and every end in the last superchunk's first and last lanes"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import _single_pass_in_steps, dynamic_bitrate_allreduce_single_pass
    g = torch.Generator(device=DEV).manual_seed(17)
    whole = [torch.randn(256 * 3, generator=g, device=DEV).to(dt) for _ in range(3)]
    for n in list(range(1, 10)) + [256 + k for k in range(1, 10)] + [768 - k for k in range(10)]:
        vecs = [v[:n].clone() for v in whole]
        outs, _, _ = dynamic_bitrate_allreduce_single_pass(vecs, 6.0, strategy=2, seed=11)
        ref, _, _ = _single_pass_in_steps(vecs, 6.0, 2, 11, None, {}, None, None)
        assert all(torch.equal(bits_t(x), bits_t(y)) for x, y in zip(outs, ref)), n


@pytest.mark.parametrize("W,n,dt,offset", [
    (8, 1024 * 2048, torch.bfloat16, 0),           # a tile per wave of the statistics
    (8, 1024 * 2048 + 1, torch.bfloat16, 0),
    (8, 1024 * 2432, torch.bfloat16, 0),           # the last length with a tile per wave
    (8, 1024 * 2432 + 1, torch.bfloat16, 0),       # four tiles per wave; one element in the last of them
    (3, 1024 * 6486 - 255, torch.float32, 0),
    (3, 1024 * 5464 - 255, torch.float32, 0),
    (3, 1024 * 5465, torch.bfloat16, 1),           # vectors off the 16 bytes
    (9, 1024 * 4 * 500 + 256 * 7, torch.bfloat16, 0),
    (8, 300 << 16, torch.bfloat16, 0),             # the last one that the cache is to keep
    (8, (300 << 16) + 1024 * 9 + 300, torch.bfloat16, 0),
    (4, (300 << 16) + 1024 * 3, torch.float32, 1),
])
def test_statistics_of_long_vectors(capi, W, n, dt, offset):
    """the reduced statistics against the sums of the ranks' own in the element type, and the all-reduce behind them against the
    ring in steps, which has its statistics from other kernels"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import _single_pass_in_steps, dynamic_bitrate_allreduce_single_pass
    g = torch.Generator(device=DEV).manual_seed(n + W)
    vecs = []
    for r in range(W):
        x = torch.randn(n + offset, generator=g, device=DEV)
        x.view(-1)[:n // 4096 * 4096].view(-1, 4096).mul_(torch.exp2(torch.randint(-9, 3, (n // 4096, 1), generator=g, device=DEV).float()))
        vecs.append(x.to(dt)[offset:])
        del x
    outs, total, _ = dynamic_bitrate_allreduce_single_pass(vecs, 6.0, strategy=2, seed=3)
    want = None
    for v in vecs:
        stats = torch.empty_like(total)
        capi.superchunk_stats(v, stats, None, n, W)
        want = stats if want is None else want + stats
    assert torch.equal(bits_t(total), bits_t(want))
    ref, _, _ = _single_pass_in_steps(vecs, 6.0, 2, 3, None, {}, None, None)
    assert all(torch.equal(bits_t(x), bits_t(y)) for x, y in zip(outs, ref))


@pytest.mark.parametrize("W", [1, 3])
@pytest.mark.parametrize("elsewhere", [False, pytest.param(True, marks=pytest.mark.skipif(
    not torch.cuda.is_available() or torch.cuda.device_count() < 2, reason="needs a second GPU"))])
def test_all_reduce_runs_on_the_current_stream_of_the_vectors(capi, W, elsewhere):
    """without a stream of the caller's the launches go to the current stream of the vectors' device, behind what is on it, also
    where another device is the current one"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import dynamic_bitrate_allreduce_single_pass
    device = torch.device("cuda", 1 if elsewhere else 0)
    vecs = [_llama_like(256 * 50 - 3, r).to(device) for r in range(W)]
    want, _, _ = dynamic_bitrate_allreduce_single_pass([v * 2 for v in vecs], 6.0, seed=3, stream=torch.cuda.default_stream(device))
    busy = torch.zeros(1 << 25, device=device)
    side = torch.cuda.Stream(device=device)
    torch.cuda.synchronize(device)
    with torch.cuda.stream(side):                  # (makes the vectors' device current)
        for _ in range(8):
            busy.add_(1.0)
        for v in vecs:
            v.mul_(2)
        with torch.cuda.device(0):
            outs, _, _ = dynamic_bitrate_allreduce_single_pass(vecs, 6.0, seed=3)
    torch.cuda.synchronize(device)
    assert all(torch.equal(bits_t(x), bits_t(y)) for x, y in zip(outs, want))


@pytest.mark.parametrize("u", [-4.0, 0.0, 3.984375, 6.0, 8.0, 15.5])
def test_widths_of_every_norm_in_the_one_rank_pass(capi, u):
    """the width that the one-rank pass picks by its quick score equals the width rule's for every bf16 norm from 2^-63 to 2^62 --
    each fills one wave (four superchunks), so that no other norm sends the wave to the rule itself"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import SinglePassBuckets
    norms = torch.arange(64 << 7, (189 << 7) + 1, dtype=torch.int16, device=DEV).view(torch.bfloat16).float()
    norms = torch.cat([norms.repeat_interleave(4), torch.tensor([0.0, float("inf")], device=DEV).repeat_interleave(4)])
    signs = torch.tensor([1.0, -1.0], device=DEV).repeat(128)
    x = (norms[:, None] / 16 * signs).reshape(-1).contiguous()      # 256 elements of +-norm / 16: mean zero
    out = torch.zeros_like(x)
    pipe = SinglePassBuckets(DEV, strategy=2, seed=5, streams=1, u=u)
    pipe.begin_step()
    pipe.run(x, out)
    pipe.join()
    torch.cuda.synchronize()
    work, _, want = _four_calls(capi, x, x.numel(), u, 2, 5, 1)[3:]
    assert torch.equal(bits_t(out), bits_t(want))
    assert pipe.counts(0)[:3].tolist() == work[:3].tolist()


@pytest.mark.parametrize("bits,u", [(8, 60.0), (2, -60.0)])
def test_estimates_just_below_zero_round_down(capi, bits, u):
    """elements whose rounding estimate falls a few 2^-25 around zero, where the fraction of a negative number rounds up to one:
    the one-rank pass against the four calls"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import SinglePassBuckets
    nsc, top = 4096, float(2 ** (bits - 1) - 1)
    rnd = torch.empty(nsc * 256, dtype=torch.float32, device=DEV)
    capi.philox_uniform(rnd, 5, 1)
    step = 255 * torch.tensor((1.0 + 1e-7) / 255).to(torch.bfloat16).double().item()      # of a chunk with maximum `top`
    jitter = 1 + (torch.arange(nsc * 256, device=DEV) // 2 % 13 - 6).double() * 2.0 ** -24
    x = (step * (rnd.double() - 1 - 2.0 ** (bits - 21)) * jitter).float().view(-1, 16)
    x[:, 0] = top
    x[:, 1::2] = -x[:, 0::2]                                        # pairs: mean zero
    x = x.reshape(-1).contiguous()
    out = torch.zeros_like(x)
    pipe = SinglePassBuckets(DEV, strategy=2, seed=5, streams=1, u=u)
    pipe.begin_step()
    pipe.run(x, out)
    pipe.join()
    torch.cuda.synchronize()
    assert pipe.counts(0).tolist() == [nsc if bits == w else 0 for w in (8, 4, 2)] + [0]
    assert torch.equal(out, _four_calls(capi, x, x.numel(), u, 2, 5, 1)[5])


@pytest.mark.parametrize("inside", [False, True])
def test_recorded_step_draws_fresh_values(capi, inside):
    """a step recorded after eager ones on another stream, with begin_step() inside the recording or before every replay, against
    the four calls with the counter where it stands; eager steps between the replays go on from there"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import SinglePassBuckets
    u, seed = 6.0, 7
    xs = [_llama_like(n, n, torch.bfloat16) for n in (256 * 40 - 9, 256 * 21)]
    outs = [torch.zeros_like(x) for x in xs]
    pairs = list(zip(xs, outs))
    pipe = SinglePassBuckets(DEV, strategy=2, seed=seed, u=u)

    def expect(step):
        torch.cuda.synchronize()
        for k, (x, o) in enumerate(pairs):
            assert torch.equal(bits_t(o), bits_t(_four_calls(capi, x, x.numel(), u, 2, seed, (k << 32) + step)[5])), (step, k)
            o.zero_()

    step = 0
    for _ in range(2):
        pipe.begin_step()
        step += 1
        pipe.run_all(pairs)
        pipe.join()
        expect(step)
    if not inside:
        pipe.begin_step()
        step += 1
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        if inside:
            pipe.begin_step()
        pipe.run_all(pairs)
        pipe.join()
    for k in range(4):
        if inside:
            step += 1
        elif k > 0:
            pipe.begin_step()
            step += 1
        graph.replay()
        expect(step)
        if k == 1:
            pipe.begin_step()
            step += 1
            pipe.run_all(pairs)
            pipe.join()
            expect(step)


@pytest.mark.parametrize("streams", [1, 2])
def test_recorded_step_outlives_its_scratch(capi, streams):
    """a step recorded before a larger bucket and a longer list have replaced the object's scratch: its replays write outputs and
    counts of their own, and nothing into memory that the allocator has handed out since"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import SinglePassBuckets
    u, seed = 6.0, 13
    pairs = [(x, torch.zeros_like(x)) for x in (_llama_like(n, n) for n in (256 * 50 - 7, 256 * 30, 256 * 41))]
    pipe = SinglePassBuckets(DEV, strategy=2, seed=seed, streams=streams, u=u)
    pipe.begin_step()
    pipe.run_all(pairs)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        pipe.begin_step()
        pipe.run_all(pairs)
    room = pipe._room
    more = [(x, torch.zeros_like(x)) for x in (_llama_like(n, n) for n in (256 * 4000, 256 * 3, 256 * 5, 256, 256 * 2))]
    pipe.begin_step()
    pipe.run_all(more)                                     # (step 2: the recording itself has run nothing)
    assert pipe._room[0] > room[0] and pipe._room[1] > room[1]
    torch.cuda.synchronize()
    # whatever the allocator has to give of these sizes
    canaries = [torch.full((room[0] * 2,), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(64)]
    canaries += [torch.full((max(1, room[1]) * 4,), 7, dtype=torch.int32, device=DEV) for _ in range(64)]
    for step in (3, 4, 5):
        graph.replay()
        torch.cuda.synchronize()
        for k, (x, o) in enumerate(pairs):
            want = _four_calls(capi, x, x.numel(), u, 2, seed, (k << 32) + step)
            assert torch.equal(bits_t(o), bits_t(want[5])), (step, k)
            if k + streams >= len(pairs):                  # the last bucket of its slot
                assert pipe.counts(k % streams).tolist() == want[3][:4].tolist(), (step, k)
            o.zero_()
        assert all(bool((c == 7).all()) for c in canaries)


@pytest.mark.parametrize("recorded", [False, True])
def test_first_use_on_another_stream(capi, recorded):
    """an object made on one stream, behind work that keeps it busy, and used on another without a word from the caller: its step
    counter and u are there when the first launch reads them, likewise after set_u; eager, and made and used in one recording"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import SinglePassBuckets
    x = _llama_like(256 * 33, 3)
    out, second = torch.zeros_like(x), torch.zeros_like(x)
    maker, user, third = torch.cuda.Stream(), torch.cuda.Stream(), torch.cuda.Stream()
    busy = torch.zeros(1 << 26, device=DEV)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()

    def whole():
        if recorded:
            for s in (user, third):
                s.wait_stream(maker)
        for _ in range(8):
            busy.add_(1.0)
        pipe = SinglePassBuckets(DEV, strategy=2, seed=2, u=6.0)
        with torch.cuda.stream(user):
            pipe.begin_step()
            pipe.run(x, out)
            pipe.join()
            pipe.set_u(8.5)
        with torch.cuda.stream(third):
            pipe.run(x, second)
        pipe.join()
        return pipe

    with torch.cuda.stream(maker):
        if recorded:
            with torch.cuda.graph(graph, stream=maker):
                pipe = whole()
        else:
            pipe = whole()
    for _ in range(3 if recorded else 1):
        if recorded:
            out.zero_()
            second.zero_()
            torch.cuda.synchronize()
            graph.replay()
        torch.cuda.synchronize()
        for o, u in ((out, 6.0), (second, 8.5)):
            assert torch.equal(bits_t(o), bits_t(_four_calls(capi, x, x.numel(), u, 2, 2, 1)[5])), u
    del pipe


@pytest.mark.parametrize("inside", [False, True])
def test_replays_in_order_with_eager_steps_on_another_stream(capi, inside):
    """join() (begin_step() where it is not part of the recording) on the stream of a replay puts the replay into the object's order:
    eager steps on another stream before and after it, no other wait between them"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import SinglePassBuckets
    u, seed = 6.0, 17
    xs = [_llama_like(n, n) for n in (256 * 3000, 256 * 41 - 3)]
    pairs = [(x, torch.zeros_like(x)) for x in xs]
    other = [(x, torch.zeros_like(x)) for x in xs]
    pipe = SinglePassBuckets(DEV, strategy=2, seed=seed, u=u)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    busy = torch.zeros(1 << 24, device=DEV)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=a):
        if inside:
            pipe.begin_step()
        pipe.run_all(pairs)
    seen, step = [], 0
    for _ in range(6):
        with torch.cuda.stream(a):
            busy.add_(1.0)                       # the replay starts late
            pipe.join() if inside else pipe.begin_step()
            graph.replay()
            step += 1
            seen.append((step, [o.clone() for _, o in pairs]))
        with torch.cuda.stream(b):
            pipe.begin_step()
            step += 1
            pipe.run_all(other)
            seen.append((step, [o.clone() for _, o in other]))
    torch.cuda.synchronize()
    for step, outs in seen:
        for k, (x, o) in enumerate(zip(xs, outs)):
            assert torch.equal(bits_t(o), bits_t(_four_calls(capi, x, x.numel(), u, 2, seed, (k << 32) + step)[5])), (step, k)


def test_threads_share_an_object(capi):
    """threads that enqueue buckets of one step, each on a stream of its own, with scratch that grows on the way: the step counter
    advances once a step, and every bucket draws that step's values"""
    import threading
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import SinglePassBuckets
    u, seed, steps, count = 6.0, 23, 6, 4
    pipe = SinglePassBuckets(DEV, strategy=2, seed=seed, u=u)
    xs = [[_llama_like(256 * (40 + 500 * t + 7 * k), 10 * t + k) for k in range(3)] for t in range(count)]
    outs = [[[torch.zeros_like(x) for x in mine] for mine in xs] for _ in range(steps)]
    for mine in xs:
        for x in mine:
            pipe.ordinals[(x.data_ptr(), x.numel())] = len(pipe.ordinals)     # whichever thread comes first
    torch.cuda.synchronize()
    failed = []

    def work(t, step):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for x, o in zip(xs[t], outs[step][t]):
                    pipe.run(x, o)
                pipe.run_all(list(zip(xs[t], outs[step][t])))
        except Exception as exc:      # noqa: BLE001 (shown by the assertion below)
            failed.append(exc)

    for step in range(steps):
        pipe.begin_step()
        threads = [threading.Thread(target=work, args=(t, step)) for t in range(count)]
        for t in threads:
            t.start()
        for t in threads:
            t.join(60)
    torch.cuda.synchronize()
    assert not failed and int(pipe.step_dev) == steps
    for step in range(steps):
        for t in range(count):
            for k, (x, o) in enumerate(zip(xs[t], outs[step][t])):
                want = _four_calls(capi, x, x.numel(), u, 2, seed, ((3 * t + k) << 32) + step + 1)[5]
                assert torch.equal(bits_t(o), bits_t(want)), (step, t, k)


@pytest.mark.parametrize("kinds", ["bf", "fbb", "bfbfb", "b" * 33 + "f" * 34 + "b"])
def test_list_of_buckets_of_two_types(capi, kinds):
    """bf16 and fp32 buckets in one list, one step counter for all of them: against the four calls bucket by bucket; the list is
    recognised on later steps, and is not taken for one of another order of types"""
    from dynamiq_sigcomm_artifact_amd.bitrate import NormHistogram
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import SinglePassBuckets
    types = {"b": torch.bfloat16, "f": torch.float32}
    u, seed = 6.0, 19
    xs = [_llama_like(256 * (3 + k % 5) - k % 3, 70 + k, types[t]) for k, t in enumerate(kinds)]
    pairs = [(x, torch.zeros_like(x)) for x in xs]
    hist = NormHistogram(DEV)
    pipe = SinglePassBuckets(DEV, strategy=2, seed=seed, u=u, norm_histogram=hist)
    for step in range(1, 4):
        pipe.begin_step()
        pipe.run_all(pairs)
        torch.cuda.synchronize()
        for k, (x, o) in enumerate(pairs):
            want = _four_calls(capi, x, x.numel(), u, 2, seed, (k << 32) + step)
            assert torch.equal(bits_t(o), bits_t(want[5])), (step, k)
            o.zero_()
        assert pipe.counts((len(pairs) - 1) % 2).tolist() == want[3][:4].tolist()
    assert int(pipe.step_dev) == 3 and len(pipe.cache) == 1
    nsc = sum((x.numel() + 255) // 256 for x in xs)
    assert hist.count == 3 * nsc and int(hist.hist.sum()) == 3 * nsc
    assert not pipe._last[0].matches(pairs[::-1])


@pytest.mark.parametrize("kinds", ["b" * 12, "b" * 13, "f" * 12 + "b" * 13 + "f"])
def test_lists_on_either_side_of_a_launchs_room(capi, kinds):
    """a launch has room for one, twelve or 32 buckets"""
    test_list_of_buckets_of_two_types(capi, kinds)


@pytest.mark.parametrize("shape", ["chain", "rewrite", "reuse", "overlap", "in place", "shared source", "views"])
def test_list_of_buckets_that_share_memory(capi, shape):
    """buckets of one list that read or write what another of the list writes give the results of one bucket after the other, and
    those that share nothing (or a source) stay in one run of launches"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import SinglePassBuckets
    n, u, seed = 256 * 1024, 6.0, 29
    base = _llama_like(6 * n, 31)
    t = [base[k * n:(k + 1) * n] for k in range(6)]
    pairs = {"chain": [(t[0], t[1]), (t[1], t[2]), (t[2], t[3])],
             "rewrite": [(t[0], t[3]), (t[1], t[3]), (t[2], t[4])],
             "reuse": [(t[0], t[2]), (t[1], t[0]), (t[0], t[4])],
             "overlap": [(t[0], base[2 * n - 256:3 * n - 256]), (t[1], t[4]), (base[2 * n + 77:3 * n + 77], t[5])],
             "in place": [(t[0], t[0]), (t[1], t[1]), (t[2], t[2])],
             "shared source": [(t[0], t[2]), (t[0], t[3]), (t[1], t[4])],
             "views": [(base[:n - 3], base[2 * n:3 * n - 3]), (base[n - 3:n], base[3 * n:3 * n + 3]), (t[1], t[4])]}[shape]
    begin = base.clone()
    want = begin.clone()

    def of(copy, view):
        at = (view.data_ptr() - base.data_ptr()) // base.element_size()
        return copy[at:at + view.numel()]

    pipe = SinglePassBuckets(DEV, strategy=2, seed=seed, u=u)
    order = [pipe.ordinals.setdefault((x.data_ptr(), x.numel()), len(pipe.ordinals)) for x, _ in pairs]
    for step in range(1, 4):
        for (x, o), ordinal in zip(pairs, order):
            of(want, o).copy_(_four_calls(capi, of(want, x).clone(), x.numel(), u, 2, seed, (ordinal << 32) + step)[5])
        pipe.begin_step()
        pipe.run_all(pairs)
        torch.cuda.synchronize()
        assert torch.equal(bits_t(base), bits_t(want)), step
        assert pipe._last[0].runs == {"chain": [1, 1, 1], "rewrite": [1, 2], "reuse": [1, 1, 1], "overlap": [1, 2]}.get(shape, [3])


@pytest.mark.parametrize("streams", [1, 3])
def test_state_of_the_pipeline_object(capi, streams):
    """step_devs, pending and scratch: the steps begun so far, what join() would wait for, room and counts per slot; a counter that
    the caller sets is the one that the next bucket draws from"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import SinglePassBuckets
    x = _llama_like(256 * 20, 4)
    out = torch.zeros_like(x)
    pipe = SinglePassBuckets(DEV, strategy=2, seed=5, streams=streams, u=6.0)
    assert pipe.scratch == [{}] * streams and pipe.pending == [False] * streams
    pipe.begin_step()
    pipe.begin_step()
    assert [int(s) for s in pipe.step_devs] == [2] * streams
    for s in pipe.step_devs:
        s.fill_(40)
    pipe.begin_step()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        k = pipe.run(x, out)
        assert pipe.pending == [False] * streams
    assert pipe.pending == [True] * streams
    pipe.join()
    assert pipe.pending == [False] * streams
    torch.cuda.synchronize()
    want = _four_calls(capi, x, x.numel(), 6.0, 2, 5, 41)
    assert torch.equal(bits_t(out), bits_t(want[5])) and int(pipe.step_dev) == 41
    assert pipe.scratch[k]["nsc"] == 20 and pipe.scratch[k]["work"][:4].tolist() == want[3][:4].tolist() == pipe.counts(k).tolist()


@pytest.mark.parametrize("form", [list, tuple, lambda p: [list(q) for q in p], lambda p: dict(p).items(), lambda p: ([x, o] for x, o in p)],
                         ids=["list", "tuple", "lists", "items", "generator"])
def test_whatever_holds_the_buckets(capi, form):
    """a step's buckets as a list of pairs, a tuple, a list of lists, a dictionary's items, a generator; and none at all"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import SinglePassBuckets
    xs = [_llama_like(256 * 5 - k, 90 + k) for k in range(3)]
    pairs = [(x, torch.zeros_like(x)) for x in xs]
    pipe = SinglePassBuckets(DEV, strategy=2, seed=5, u=6.0)
    pipe.run_all(form([]))
    for step in range(1, 4):
        pipe.begin_step()
        pipe.run_all(form(pairs))
        pipe.run_all(form([]))
        torch.cuda.synchronize()
        for k, (x, o) in enumerate(pairs):
            assert torch.equal(bits_t(o), bits_t(_four_calls(capi, x, x.numel(), 6.0, 2, 5, (k << 32) + step)[5])), (step, k)
            o.zero_()
    assert len(pipe.cache) == 1


@pytest.mark.parametrize("shift", [-256, 1, 8 * 256])
@pytest.mark.parametrize("path", ["buckets", "lists", "all-reduce", "grouped", "fixed"])
def test_outputs_across_their_sources(capi, path, shift):
    """an output that lies across its source at another address, as every call took it when there were buffers between the two:
    the results are those with an output elsewhere"""
    from dynamiq_sigcomm_artifact_amd import dynamiq_pipeline as P
    from dynamiq_sigcomm_artifact_amd.compressors import Aee_Dynamic_Range_GPU_kern
    n, u = 256 * 600 - 5, 6.0
    for W in (1, 3):
        codecs = lambda: {q: [Aee_Dynamic_Range_GPU_kern(q, 16, {"d": {0: 256 * 1200}, "world_size": 1}, device=DEV,
                                                         generator=torch.Generator(device=DEV).manual_seed(q + r)) for r in range(W)]
                          for q in (8, 4, 2)}
        calls = {"all-reduce": lambda v, o, c: P.dynamic_bitrate_allreduce_single_pass(v, u, seed=4, out=o)[0],
                 "grouped": lambda v, o, c: P.dynamic_bitrate_allreduce_grouped(v, u, c, out=o)[0],
                 "fixed": lambda v, o, c: P.fixed_proportion_allreduce_grouped(v, {8: 0.2, 4: 0.5, 2: 0.3}, c, out=o)[0]}
        data = [_llama_like(n, 50 + r) for r in range(W)]
        rooms = [torch.zeros(n + 8 * 256 + 512, dtype=torch.bfloat16, device=DEV) for _ in range(W)]
        vecs = [room[256:256 + n] for room in rooms]
        outs = [room[256 + shift:256 + shift + n] for room in rooms]
        pipe = P.SinglePassBuckets(DEV, strategy=2, seed=5, u=u)
        for step in range(1, 3):
            for v, d in zip(vecs, data):
                v.copy_(d)
            if path in calls:
                want = calls[path](data, [torch.zeros_like(d) for d in data], codecs())
                got = calls[path](vecs, outs, codecs())
            else:
                pipe.begin_step()
                if path == "lists":
                    pipe.run_all(list(zip(vecs, outs)))
                else:
                    for v, o in zip(vecs, outs):
                        pipe.run(v, o)
                got = outs
                want = [_four_calls(capi, d, n, u, 2, 5, (r << 32) + step)[5] for r, d in enumerate(data)]
            torch.cuda.synchronize()
            assert all(torch.equal(bits_t(x), bits_t(y)) for x, y in zip(got, want)), (W, step)


def test_bucket_seen_before_is_checked_again(capi):
    """an output at a known address that has become too short is refused, not written beyond its end; scratch in use on two streams
    grows without disturbing either"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import SinglePassBuckets
    x = _llama_like(256 * 64, 5, torch.bfloat16)
    out = torch.zeros_like(x)
    pipe = SinglePassBuckets(DEV, strategy=2, seed=3, u=6.0)
    pipe.begin_step()
    pipe.run(x, out)
    pipe.run_all([(x, out)])
    with pytest.raises(RuntimeError, match="output"):
        pipe.run(x, out[:-256])
    with pytest.raises(RuntimeError, match="output"):
        pipe.run_all([(x, out[:-256])])
    big = _llama_like(256 * 300 + 1, 6, torch.bfloat16)
    result = torch.zeros_like(big)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        pipe.run(x, out)
    pipe.run(big, result)
    torch.cuda.synchronize()
    for k, (v, o) in enumerate(((x, out), (big, result))):
        assert torch.equal(bits_t(o), bits_t(_four_calls(capi, v, v.numel(), 6.0, 2, 3, (k << 32) + 1)[5]))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("W,tiles,less", [(8, 1 << 14, 0), (8, (1 << 14) + 1, 300), (8, (1 << 14) - 1, 0), (9, 14564, 767), (2, 1 << 16, 1)])
def test_statistics_of_two_tiles_per_wave(capi, W, tiles, less, dt):
    """around 2^17 tiles of all ranks, where a wave of the statistics takes two of them: an odd number of tiles, a ragged last one,
    more ranks than a workgroup has waves; against the statistics rank by rank and their bf16 sums in rank order"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import dynamic_bitrate_allreduce_single_pass
    n = 1024 * tiles - less
    nsc = (n + 255) // 256
    g = torch.Generator(device=DEV).manual_seed(W + less)
    vecs = [torch.randn(n, generator=g, device=DEV).add_(0.1 * r).to(dt) for r in range(W)]
    work = {}
    _, total, _ = dynamic_bitrate_allreduce_single_pass(vecs, 6.0, seed=1, work=work)
    stats, mean = torch.empty((nsc, 2), dtype=torch.bfloat16, device=DEV), torch.empty(nsc, device=DEV)
    want = None
    for r, v in enumerate(vecs):
        capi.superchunk_stats(v, stats, mean, n, W)
        want = stats.clone() if want is None else want.add_(stats)
        assert torch.equal(mean, work["mean"][r * nsc:(r + 1) * nsc]), r
    assert torch.equal(bits_t(total), bits_t(want))
