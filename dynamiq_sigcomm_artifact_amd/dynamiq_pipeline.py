"""One bucket partition of DynamiQ's dynamic-bitrate all-reduce, with the W ranks
simulated in one GPU's HBM -- the host-side mirror of
``compress_and_reduce_and_decompress`` in
testbed_evaluation/new_comm_hooks/comm_hooks.py:932-1024:

  superchunk_mean_center -> (stats all-reduce) -> per-superchunk q in {2,4,8} ->
  per bit width: gather the superchunks of that width, compressed ring
  all-reduce, scatter back -> superchunk_add_mean_copy.

The stats all-reduce, a collective in the reference, is a sequential bf16 sum
over the simulated ranks here; with one rank the ring degenerates to
compress -> decompress of the rank's own chunk (ring_rdma.py:606-621 with
size == 1).
"""
import threading

import torch

from . import bitrate
from .compressors import (Aee_Dynamic_Range_GPU_kern, Mee_Dynamic_Range_GPU_kern, superchunk_add_mean_copy,
                          superchunk_mean_center)
from . import load_eden_utils
from .ring_sim import ring_allreduce, ring_allreduce_rows

SUPERCHUNK = 256
_U64 = 0xFFFFFFFFFFFFFFFF


def dynamic_bitrate_allreduce(rank_vecs, u, compressors, out=None):
    """rank_vecs: list of W equal-length 1-D tensors (fp16/bf16).  compressors:
    {2: [c_rank0, ...], 4: [...], 8: [...]}.  Returns (result tensors per rank,
    reduced stats, qbits)."""
    W = len(rank_vecs)
    n = rank_vecs[0].numel()
    nsc = (n + SUPERCHUNK - 1) // SUPERCHUNK
    dev, dt = rank_vecs[0].device, rank_vecs[0].dtype
    residuals = [torch.empty(nsc * SUPERCHUNK, dtype=dt, device=dev) for _ in range(W)]
    stats = [torch.empty((nsc, 2), dtype=torch.bfloat16, device=dev) for _ in range(W)]
    for r in range(W):
        superchunk_mean_center(rank_vecs[r], residuals[r], stats[r], n, W, SUPERCHUNK)
    total = stats[0].clone()
    for r in range(1, W):
        total.add_(stats[r])
    norms = total[:, 1]
    qbits = bitrate.dynamic_bitrate_qbits(norms, u)

    res2d = [res.view(-1, SUPERCHUNK) for res in residuals]
    for q in (8, 4, 2):
        idx = torch.nonzero(qbits == q, as_tuple=False).view(-1)
        if idx.numel() == 0:
            continue
        groups = [torch.index_select(res2d[r], 0, idx).reshape(-1) for r in range(W)]
        comps = compressors[q]
        if W == 1:
            c = comps[0]
            send = c.create_tensor(groups[0], torch.uint8)
            c.compression(groups[0], send)
            c.decompression(send, groups[0])
        else:
            ring_allreduce(groups, comps, align=SUPERCHUNK)
        for r in range(W):
            res2d[r].index_copy_(0, idx, groups[r].view(-1, SUPERCHUNK))

    outs = out if out is not None else [torch.empty(n, dtype=dt, device=dev) for _ in range(W)]
    for r in range(W):
        superchunk_add_mean_copy(residuals[r], outs[r], total, n, SUPERCHUNK)
    return outs, total, qbits


_RANKS_STATS, _RANKS_RING = 1, 4


def _across(out, x):
    """does `out` lie across the vector `x` at another address?  The passes that have no buffer between the two cannot do that."""
    a, b, size = out.data_ptr(), x.data_ptr(), x.numel() * x.element_size()
    return a != b and a < b + size and b < a + size


def _pooled_codecs(rank_vecs, compressors):
    """the native objects of the compressors, one list per width (8, 4, 2 bits), when the whole all-reduce can run without
    packed streams (csrc/dq_single_pass.hip): the package's own pooled compressors of one strategy, bf16 vectors and no
    more ranks than the arguments of one launch hold.  Else None: the ring then runs call by call."""
    from . import capi
    W = len(rank_vecs)
    if W > capi.ranks_max(True) or rank_vecs[0].dtype != torch.bfloat16:
        return None
    native, strategy = [], None
    for q in (8, 4, 2):
        of_width = compressors.get(q, ())
        if len(of_width) < W:
            return None
        native.append([])
        for c in of_width:
            if type(c) is not Aee_Dynamic_Range_GPU_kern and type(c) is not Mee_Dynamic_Range_GPU_kern:
                return None
            codec = c._codec
            if strategy is None:
                strategy = c.strategy
            if codec.philox or c._picks_rows or c.chunk_size != 16 or c.nbits != q or c.strategy != strategy:
                return None
            native[-1].append(codec)
    return native


def dynamic_bitrate_allreduce_grouped(rank_vecs, u, compressors, out=None, work=None, device_qbits=False):
    """Same inputs, same results (bit for bit) as dynamic_bitrate_allreduce, with the gather, the scatter
    and the final mean add folded into the codec kernels: one device-side partition of the superchunk
    indices by width (a single 16-byte read-back for the three group sizes, in place of three
    torch.nonzero), no group tensors, no index_select / index_copy_ / superchunk_add_mean_copy passes.
    With the package's pooled compressors the ring itself is one launch for all ranks, steps and widths.

    device_qbits=True also computes the bit widths inside the partition call (the rule of
    bitrate.dynamic_bitrate_qbits with the library's fixed-polynomial log2 in place of torch.log2; the two
    agree except where a log2 value lies within a few binary32 ulps of a bf16 rounding boundary)."""
    from . import capi
    eu = load_eden_utils()
    W = len(rank_vecs)
    n = rank_vecs[0].numel()
    nsc = (n + SUPERCHUNK - 1) // SUPERCHUNK
    dev, dt = rank_vecs[0].device, rank_vecs[0].dtype
    if work is None:
        work = {}
    codecs = _pooled_codecs(rank_vecs, compressors)
    if codecs and out is not None and any(_across(o, v) for o in out for v in rank_vecs):
        codecs = None
    key = (nsc, dt, W, codecs is None)
    if work.get("key") != key:
        work["key"] = key
        work["residuals"] = [] if codecs else [torch.empty(nsc * SUPERCHUNK, dtype=dt, device=dev) for _ in range(W)]
        work["stats"] = [] if codecs else [torch.empty((nsc, 2), dtype=torch.bfloat16, device=dev) for _ in range(W)]
        work["order"] = torch.empty(3 * nsc, dtype=torch.int32, device=dev)
        work["mean"] = torch.empty(W * nsc, dtype=torch.float32, device=dev) if codecs else None
    residuals, stats, order = work["residuals"], work["stats"], work["order"]
    stream = torch.cuda.current_stream().cuda_stream
    outs = out if out is not None else [torch.empty(n, dtype=dt, device=dev) for _ in range(W)]
    if codecs:
        # all ranks' statistics and their sum in one launch; nothing is centred yet
        total = torch.empty((nsc, 2), dtype=torch.bfloat16, device=dev)
        capi.host().ranks_pooled(rank_vecs, outs, n, total, work["mean"], order, order, codecs, (0, 0, 0), _RANKS_STATS,
                                 compressors[8][0].strategy)
    else:
        for r in range(W):
            superchunk_mean_center(rank_vecs[r], residuals[r], stats[r], n, W, SUPERCHUNK)
        total = stats[0] if W == 1 else stats[0].clone()
        for r in range(1, W):
            total.add_(stats[r])
    if device_qbits:
        qbits = work.get("qbits")
        if qbits is None or qbits.numel() != nsc:
            qbits = work["qbits"] = torch.empty(nsc, dtype=torch.int64, device=dev)
        sizes = eu.group_plan_stats(total, float(u), order, qbits, stream)
    else:
        qbits = bitrate.dynamic_bitrate_qbits(total[:, 1], u)
        sizes = eu.group_plan(qbits, order, stream)
    counts = sizes.tolist()
    assert counts[3] == 0, "bit widths outside {2, 4, 8}"

    if codecs:
        capi.host().ranks_pooled(rank_vecs, outs, n, total, work["mean"], order, sizes, codecs, counts[:3], _RANKS_RING,
                                 compressors[8][0].strategy)
        return outs, total, qbits
    for g, (q, cnt) in enumerate(zip((8, 4, 2), counts[:3])):
        if cnt == 0:
            continue
        rows = order[g * nsc:g * nsc + cnt]          # every width has a region of nsc entries
        comps = compressors[q]
        if W == 1:
            c = comps[0]
            send = work.get(("send", q))
            need = c.compressed_numel(cnt * SUPERCHUNK)
            if send is None or send.numel() < need:
                send = work[("send", q)] = torch.empty(need, dtype=torch.uint8, device=dev)
            c.compression_rows(residuals[0], rows, send)
            c.decompression_rows(send, outs[0], rows, total, n)
        else:
            ring_allreduce_rows(residuals, rows, comps, outs, total, n)
    return outs, total, qbits


def fixed_proportion_allreduce(rank_vecs, thresholds, compressors, out=None, fixed_4bit_only=False):
    """One bucket partition of the non-dynamic hook, ``P2P_dynamiQ_hook``'s ``compress_and_reduce_and_decompress``
    (comm_hooks.py:682-786), as the reference's op sequence: mean-centre, reduce the statistics, sort the norms
    (stable, descending), gather the first / middle / last share as the 8- / 4- / 2-bit groups **in sorted order**, one
    compressed ring per group, scatter back, add the means.  ``fixed_4bit_only`` is the "fixed" method: only the 4-bit
    group (everything, thresholds {4: 1, 8: 0, 2: 0}) is communicated (:768-772)."""
    W = len(rank_vecs)
    n = rank_vecs[0].numel()
    nsc = (n + SUPERCHUNK - 1) // SUPERCHUNK
    dev, dt = rank_vecs[0].device, rank_vecs[0].dtype
    residuals = [torch.empty(nsc * SUPERCHUNK, dtype=dt, device=dev) for _ in range(W)]
    stats = [torch.empty((nsc, 2), dtype=torch.bfloat16, device=dev) for _ in range(W)]
    for r in range(W):
        superchunk_mean_center(rank_vecs[r], residuals[r], stats[r], n, W, SUPERCHUNK)
    total = stats[0].clone()
    for r in range(1, W):
        total.add_(stats[r])
    groups_idx = bitrate.fixed_proportion_groups(total[:, 1], thresholds)
    res2d = [res.view(-1, SUPERCHUNK) for res in residuals]
    for q, idx in zip((8, 4, 2), groups_idx):
        if idx.numel() == 0 or (fixed_4bit_only and q != 4):
            continue
        groups = [torch.index_select(res2d[r], 0, idx).reshape(-1) for r in range(W)]
        comps = compressors[q]
        if W == 1:
            c = comps[0]
            send = c.create_tensor(groups[0], torch.uint8)
            c.compression(groups[0], send)
            c.decompression(send, groups[0])
        else:
            ring_allreduce(groups, comps, align=SUPERCHUNK)
        for r in range(W):
            res2d[r].index_copy_(0, idx, groups[r].view(-1, SUPERCHUNK))
    outs = out if out is not None else [torch.empty(n, dtype=dt, device=dev) for _ in range(W)]
    for r in range(W):
        superchunk_add_mean_copy(residuals[r], outs[r], total, n, SUPERCHUNK)
    return outs, total, groups_idx


def fixed_proportion_allreduce_grouped(rank_vecs, thresholds, compressors, out=None, fixed_4bit_only=False):
    """The same all-reduce, bit for bit, with the sort, the slices, the gathers, the scatters and the final mean add
    replaced by one launch of the device plan (group_plan_sorted) and, with the package's pooled compressors, one launch of
    the whole ring (else the row-list codec calls); the group sizes follow from the fractions on the host, so nothing is
    read back."""
    from . import capi
    W = len(rank_vecs)
    n = rank_vecs[0].numel()
    nsc = (n + SUPERCHUNK - 1) // SUPERCHUNK
    dev, dt = rank_vecs[0].device, rank_vecs[0].dtype
    counts = bitrate.fixed_proportion_counts(nsc, thresholds)
    codecs = _pooled_codecs(rank_vecs, compressors)
    if codecs and not (fixed_4bit_only and counts[1] != nsc):
        # three launches for all ranks, steps and widths: statistics, sorted plan, ring
        outs = out if out is not None else [torch.empty(n, dtype=dt, device=dev) for _ in range(W)]
        done = capi.host().ranks_fixed(rank_vecs, outs, n, codecs, *counts, compressors[8][0].strategy)
        if done is not None:
            return outs, done[0], done[1], counts
    eu = load_eden_utils()
    residuals = [torch.empty(nsc * SUPERCHUNK, dtype=dt, device=dev) for _ in range(W)]
    stats = [torch.empty((nsc, 2), dtype=torch.bfloat16, device=dev) for _ in range(W)]
    for r in range(W):
        superchunk_mean_center(rank_vecs[r], residuals[r], stats[r], n, W, SUPERCHUNK)
    total = stats[0] if W == 1 else stats[0].clone()
    for r in range(1, W):
        total.add_(stats[r])
    order = torch.empty(3 * nsc, dtype=torch.int32, device=dev)
    eu.group_plan_sorted(total, counts[0], counts[2], order, None, torch.cuda.current_stream().cuda_stream)
    outs = out if out is not None else [torch.empty(n, dtype=dt, device=dev) for _ in range(W)]
    if fixed_4bit_only:
        # the groups that are not communicated keep their local residual: copy it through first
        for r in range(W):
            superchunk_add_mean_copy(residuals[r], outs[r], total, n, SUPERCHUNK)
    for g, (q, cnt) in enumerate(zip((8, 4, 2), counts)):
        if cnt == 0 or (fixed_4bit_only and q != 4):
            continue
        rows = order[g * nsc:g * nsc + cnt]
        comps = compressors[q]
        if W == 1:
            c = comps[0]
            send = torch.empty(c.compressed_numel(cnt * SUPERCHUNK), dtype=torch.uint8, device=dev)
            c.compression_rows(residuals[0], rows, send)
            c.decompression_rows(send, outs[0], rows, total, n)
        else:
            ring_allreduce_rows(residuals, rows, comps, outs, total, n)
    return outs, total, order, counts


def dynamic_bitrate_allreduce_single_pass(rank_vecs, u, strategy=2, seed=0, out=None, work=None, stream=None,
                                          norm_histogram=None):
    """The same all-reduce with every stage kept on the device and without packed streams: the records of a ring step
    between ranks that share this GPU's memory are read by the next step only, so a superchunk goes through the whole
    ring in registers (csrc/dq_single_pass.hip).  Three launches per bucket (statistics of all ranks, plan, ring) -- two on
    short vectors, whose ring plans itself, and with one rank, where nothing depends on another superchunk -- whatever
    the number of ranks; nothing is read back, and the launches can be captured once and replayed as a graph.

    The bit widths follow the device rule of group_plan_stats; the rounding randomness is the in-kernel stream keyed by
    (seed + rank, ring step, index of the chunk in the vector), so results are reproducible but not those of
    dynamic_bitrate_allreduce, whose random values come from the pool.

    u: the offset of the width rule, a number or a float64 device tensor (e.g. result[0:1] of the offset search: then
    nothing of the step is read back).
    stream: a torch stream or a raw handle; None: the current stream of the vectors' device.
    norm_histogram: a bitrate.NormHistogram that collects the reduced norms of the step's buckets for the search of
    the next step's u (comm_hooks.py:962, 904-931).

    Returns (result tensors per rank, reduced stats, device int32 tensor [n8, n4, n2, other])."""
    from . import capi
    W = len(rank_vecs)
    n = rank_vecs[0].numel()
    dev, dt = rank_vecs[0].device, rank_vecs[0].dtype
    if work is None:
        work = {}
    if W > capi.ranks_max():
        return _single_pass_in_steps(rank_vecs, u, strategy, seed, out, work, stream, norm_histogram)
    nsc = (n + SUPERCHUNK - 1) // SUPERCHUNK
    key = ("single_pass", nsc, dt, W)
    if work.get("key") != key:
        work.clear()
        work["key"] = key
        work["total"] = torch.empty((nsc, 2), dtype=torch.bfloat16, device=dev)
        work["plan"] = torch.zeros(capi.group_plan_work_ints(nsc) if W > 1 else 4, dtype=torch.int32, device=dev)
        work["counts"] = work["plan"][:4]
        if W > 1:
            work["mean"] = torch.empty(W * nsc, dtype=torch.float32, device=dev)
            work["order"] = torch.empty(3 * nsc, dtype=torch.int32, device=dev)
    outs = out if out is not None else [torch.empty(n, dtype=dt, device=dev) for _ in range(W)]
    hist = None if norm_histogram is None else norm_histogram.hist
    total = work["total"]
    if W == 1:
        done = capi.host().roundtrip(rank_vecs[0], outs[0], n, total, work["counts"], u, hist, seed & _U64, strategy, stream)
    else:
        done = capi.host().ranks_dynamic(rank_vecs, outs, n, total, work["mean"], work["order"], work["plan"], u, hist, seed & _U64,
                                         strategy, stream)
    if not done:        # an output lies across a vector at another address
        return _single_pass_in_steps(rank_vecs, u, strategy, seed, out, work, stream, norm_histogram)
    if norm_histogram is not None:
        norm_histogram.count += nsc
    return outs, total, work["counts"]


def _single_pass_in_steps(rank_vecs, u, strategy, seed, out, work, stream, norm_histogram):
    """the same with one launch per rank and ring step and the packed streams in memory: for more simulated ranks than the
    arguments of one launch hold, and for outputs that lie across the vectors"""
    from . import capi
    W = len(rank_vecs)
    n = rank_vecs[0].numel()
    nsc = (n + SUPERCHUNK - 1) // SUPERCHUNK
    dev, dt = rank_vecs[0].device, rank_vecs[0].dtype
    key = ("single_pass in steps", nsc, dt, W)
    if work.get("key") != key:
        work.clear()
        work["key"] = key
        cap = capi.mixed_required_bytes(nsc, W)
        work["stats"] = [torch.empty((nsc, 2), dtype=torch.bfloat16, device=dev) for _ in range(W)]
        work["mean"] = [torch.empty(nsc, dtype=torch.float32, device=dev) for _ in range(W)]
        work["total"] = torch.empty((nsc, 2), dtype=torch.bfloat16, device=dev)
        work["order"] = torch.empty(3 * nsc, dtype=torch.int32, device=dev)
        work["plan"] = torch.zeros(capi.group_plan_work_ints(nsc), dtype=torch.int32, device=dev)
        work["send"] = [torch.zeros(cap, dtype=torch.uint8, device=dev) for _ in range(W)]
        work["recv"] = [torch.zeros(cap, dtype=torch.uint8, device=dev) for _ in range(W)]
    stats, mean, order, plan = work["stats"], work["mean"], work["order"], work["plan"]
    send, recv = work["send"], work["recv"]
    # one stream for the kernels and for the torch ops between them (the statistics sum, the exchange copies):
    # resolved once per bucket, not once per launch
    torch_stream = capi.torch_stream(stream, dev)
    stream = torch_stream.cuda_stream
    for r in range(W):
        capi.superchunk_stats(rank_vecs[r], stats[r], mean[r], n, W, stream=stream)
    total = work["total"]
    with torch.cuda.stream(torch_stream):
        total.copy_(stats[0])
        for r in range(1, W):
            total.add_(stats[r])
    # with u on the device the histogram is filled by a few more workgroups of the plan launch, otherwise by a launch of its own
    capi.group_plan_stats(total, u if isinstance(u, torch.Tensor) else float(u), None, order, plan, stream=stream,
                          hist=None if norm_histogram is None else norm_histogram.hist)
    if norm_histogram is not None:
        norm_histogram.count += nsc
    outs = out if out is not None else [torch.empty(n, dtype=dt, device=dev) for _ in range(W)]

    def encode(r, chunk, step, received=None):
        capi.mixed_compress(rank_vecs[r], order, plan, send[r], nsc, strategy, seed=seed + r, step=step, recv=received,
                            center_mean=mean[r], center_world=W, n=n, ring_chunk=chunk, ring_world=W, stream=stream)

    def decode(r, packed, chunk):
        capi.mixed_decompress(packed, outs[r], order, plan, nsc, strategy, stats=total, n_limit=n, ring_chunk=chunk,
                              ring_world=W, stream=stream)

    def exchange(src_bufs, dst_bufs):
        with torch.cuda.stream(torch_stream):
            for r in range(W):
                dst_bufs[(r + 1) % W].copy_(src_bufs[r])

    # reduce-scatter: W - 1 steps, then the owner's step; all-gather of the owners' streams
    for step in range(W - 1):
        for r in range(W):
            encode(r, (r - step + W) % W, step, None if step == 0 else recv[r])
        exchange(send, recv)
    for r in range(W):
        encode(r, (r + 1) % W, W - 1, recv[r] if W > 1 else None)
        decode(r, send[r], (r + 1) % W)
    bufs = [send, recv]
    for step in range(W - 1):
        exchange(bufs[step & 1], bufs[(step ^ 1) & 1])
        for r in range(W):
            decode(r, bufs[(step ^ 1) & 1][r], (r - step + W) % W)
    return outs, total, plan[:4]


def pick_streams(device, want, tries=16):
    """`want` streams that run side by side with each other and with the caller's current stream; returns (streams, ok).
    The runtime maps the streams of a process onto a few hardware queues when they are first used, and a queue works
    through what it is given in order, whichever stream it came from.  Two streams on one queue take turns; and with the
    caller's stream on the queue of one of them, an event that orders the *next* piece of work after the caller's
    (recorded on the caller's stream) completes only after the piece enqueued just before it -- either way two buckets
    "in flight" run as slowly as on one stream (measured: 31 against 18.5 us per 25 MB bucket).  Which streams share a
    queue depends on what else the process has used, so candidates are taken from torch's pool until `want` of them
    overlap with each other and with the current stream (capi.streams_overlap, about a millisecond per pair); if the
    pool does not yield that many, the set is filled up and ok is False."""
    from . import capi
    device = torch.device(device)
    index = device.index if device.index is not None else torch.cuda.current_device()
    apart = [torch.cuda.current_stream(device).cuda_stream]
    chosen = []
    while len(chosen) < want and tries > 0:
        tries -= 1
        cand = torch.cuda.Stream(device=device)
        if cand.cuda_stream not in apart and all(capi.streams_overlap(h, cand.cuda_stream, index) for h in apart):
            chosen.append(cand)
            apart.append(cand.cuda_stream)
    ok = len(chosen) == want
    while len(chosen) < want:
        chosen.append(torch.cuda.Stream(device=device))
    return chosen, ok


class SinglePassBuckets(object):
    """The single-pass dynamic-bitrate path for a stream of buckets on one rank (a ring of one: statistics, widths,
    encode, decode, mean add -- what dynamic_bitrate_allreduce_single_pass does for W = 1).  A superchunk's result depends
    on no other superchunk, so one launch makes one pass over the bucket, and over as many buckets as are at hand:

      * ``run(x, out)`` enqueues one bucket: two launches, the pass and the tally of its widths (and norms);
      * ``run_all`` enqueues a whole step's buckets, two launches for every 32 of them.  The results are those of run() on one
        bucket after the other: where the element type changes along the list, or a bucket's memory is one that an earlier
        one writes (or its output one that an earlier one reads), it starts launches of its own.  DDP hands the hook the same
        bucket views on every step: the list is laid out once and recognised afterwards.

    Everything runs on the caller's current stream: a launch that fills the GPU gains nothing from a second stream beside
    it, and handing a bucket to another stream costs the host more than enqueueing it.  ``streams`` says how many slots
    run() deals the buckets out to (the index it returns, and counts() takes); the streams of that many slots
    (``pipe.streams``, found on first use to run side by side with the caller's, see pick_streams) are at the caller's
    disposal.  ``graphs`` and ``inline_first`` are accepted and change nothing: there is no longer a host cost per bucket
    that a recorded graph would save.

    The offset u of the width rule is read from device memory when a launch runs (``set_u`` or a float64 tensor of the
    caller's, e.g. the result of the offset search), and the rounding stream of the encoder is (seed, bucket ordinal *
    2^32 + the step counter in device memory): ``begin_step`` once per training step advances the counter, with the next
    launch or, once launches of the object have been recorded into a graph, at once -- a replay draws fresh random values
    if begin_step was recorded with it or is called before it.

    run(x, out) enqueues a bucket and returns at once; join() makes the caller's current stream wait for everything
    the object has enqueued so far.  The caller must not overwrite x or read out before join().

    A graph that the caller records is replayed without the object knowing: it uses the object's memory (and is not replayed
    any more once the object is gone), and ``superchunks`` and the histogram's ``count`` count its buckets once, at the
    recording.  Replays and the object's own launches share the step counter and the statistics, so they have to follow one
    another.  ``join()`` (or ``begin_step()``) on the stream of the replay just before it does that: the replay waits for
    what the object has enqueued, and what the object enqueues afterwards, on whichever stream, waits for the replay.
    Without it, and between replays on different streams, the order is the caller's to see to.

    Threads may share an object: its calls take turns (the steps that a launch takes along, the order of the launches and the
    scratch belong together)."""

    def __init__(self, device, strategy=2, seed=0, streams=2, graphs=True, u=None, norm_histogram=None, inline_first=True):
        from . import capi
        self.capi = capi
        self.device = torch.device(device)
        self.strategy, self.seed, self.graphs, self.inline_first = strategy, int(seed), graphs, bool(inline_first)
        self.slots = max(1, int(streams))
        self._step = torch.zeros(1, dtype=torch.int64, device=self.device)
        self.u_dev = u if isinstance(u, torch.Tensor) else torch.full((1,), 60.0 if u is None else float(u), dtype=torch.float64,
                                                                     device=self.device)
        self.hist = norm_histogram
        self._host = capi.host()
        self._turn = threading.RLock()
        self._counts = torch.zeros((self.slots, 4), dtype=torch.int32, device=self.device)
        self._buckets = self._host.Buckets(strategy, self.seed & _U64, self._step, self.u_dev,
                                           None if norm_histogram is None else norm_histogram.hist, self._counts)
        self._room = (0, 0)      # superchunks and buckets that the scratch holds
        self._scratch = None     # statistics; counts of the buckets that are not the last of their slot
        self._replaced = []      # scratch that a recorded graph may still write to
        self._last = None        # the list run_all saw last: (batch, superchunks)
        self.cache = {}          # addresses and sizes of a list of buckets -> (batch, superchunks, slots)
        self.ordinals = {}       # (x.data_ptr(), n) -> ordinal of the bucket in the random stream
        self.superchunks = 0

    def _pick(self):
        if "_streams" not in self.__dict__:
            self._streams, self._side_by_side = pick_streams(self.device, self.slots)

    @property
    def streams(self):
        self._pick()
        return self._streams

    @property
    def side_by_side(self):
        self._pick()
        return self._side_by_side

    # ---- state ----------------------------------------------------------------------------------------------
    @property
    def step_dev(self):
        """the step counter in device memory, int64 [1], with the steps begun so far"""
        with self._turn:
            self._buckets.settle()
        return self._step

    @property
    def step_devs(self):
        """the same per slot: all slots have one counter"""
        return [self.step_dev] * self.slots

    @property
    def pending(self):
        """per slot: is there work that the caller's current stream has not been ordered behind (what join() does)?"""
        with self._turn:
            return [self._buckets.behind()] * self.slots

    @property
    def scratch(self):
        """per slot, once there has been a bucket: the superchunks that the statistics shared by all slots have room for, and the
        counts of the slot's last bucket (means, row lists and a packed stream are not made)"""
        with self._turn:
            return [{"nsc": self._room[0], "work": self._counts[k]} if self._scratch else {} for k in range(self.slots)]

    # ---- once per training step ----------------------------------------------------------------------------
    def set_u(self, u):
        """the offset of the width rule for the buckets enqueued from now on (a number; a tensor was given at construction)"""
        with self._turn:
            self.join()
            self.u_dev.fill_(float(u))

    def begin_step(self):
        """advance the step counter of the rounding stream: the next launch does it on its way"""
        with self._turn:
            self._buckets.begin_step()

    # ---- per bucket ---------------------------------------------------------------------------------------------
    def _grow(self, superchunks, buckets):
        """scratch for so many superchunks and buckets.  A recorded graph goes on writing to the scratch of its day: from the
        first recording on, replaced scratch is kept as long as the object, and grows to at least twice, so that all of the
        replaced together stay below the present."""
        self.join()
        factor = 1
        if self._buckets.recorded and self._scratch is not None:
            factor = 2
            self._replaced.append(self._scratch)
        self._room = (max(superchunks, factor * self._room[0]), max(buckets, factor * self._room[1]))
        self._scratch = (torch.empty((self._room[0], 2), dtype=torch.bfloat16, device=self.device),
                         torch.empty((self._room[1], 4), dtype=torch.int32, device=self.device))
        self._buckets.scratch(*self._scratch)
        self.cache.clear()       # what was laid out over the old buffers
        self._last = None

    def _batch(self, pairs, key, given=None):
        """lays out a list of buckets seen for the first time (or again after the scratch grew); given: what the caller has,
        where the sources are copies of it for one launch"""
        total = sum((x.numel() + SUPERCHUNK - 1) // SUPERCHUNK for x, _ in pairs)
        # a source keeps its ordinal, and with it its random stream and its slot, from step to step
        ordinals = [self.ordinals.setdefault((x.data_ptr(), x.numel()), len(self.ordinals)) for x, _ in given or pairs]
        slots = [o % self.slots for o in ordinals]
        # the counts of a slot are those of its last bucket
        last = {slot: k for k, slot in enumerate(slots)}
        rows = [slot if last[slot] == k else self.slots + k for k, slot in enumerate(slots)]
        spare = max(rows) + 1 - self.slots
        if total > self._room[0] or spare > self._room[1]:
            self._grow(total, max(0, spare))
        batch = self._host.Batch(self._buckets, pairs, [(o << 32) & _U64 for o in ordinals], rows)
        entry = (batch, total, slots[0])
        if given is None:
            self.cache[key] = entry
        return entry

    def _enqueue(self, entry):
        batch, superchunks, _ = entry
        batch.launch(self._buckets)
        if self.hist is not None:
            self.hist.count += superchunks
        self.superchunks += superchunks

    def run(self, x, out):
        """enqueue one bucket: out = decode(encode(x)) with the widths of its reduced norms; returns its slot"""
        key = (x.data_ptr(), out.data_ptr(), x.numel(), x.dtype)
        with self._turn:
            entry = self.cache.get(key)
            if entry is None or not entry[0].matches([(x, out)]):
                if _across(out, x):
                    self.join()
                    copy = x.clone()
                    entry = self._batch([(copy, out)], key, [(x, out)])
                else:
                    entry = self._batch([(x, out)], key)
            self._enqueue(entry)
        return entry[2]

    def run_all(self, pairs):
        """enqueue a whole step's buckets, [(x, out), ...]"""
        with self._turn:
            last = self._last
            if last is None or not last[0].matches(pairs):
                pairs = [(x, o) for x, o in pairs]      # whatever holds them
                if not pairs:
                    return
                if any(_across(o, x) for x, o in pairs):
                    for x, o in pairs:
                        self.run(x, o)
                    return
                key = tuple((x.data_ptr(), o.data_ptr(), x.numel(), x.dtype) for x, o in pairs)
                last = self.cache.get(key)
                if last is None or not last[0].matches(pairs):
                    last = self._batch(pairs, key)
                self._last = last
            self._enqueue(last)

    def counts(self, k):
        """device int32 tensor [n8, n4, n2, other] of the last bucket of slot k"""
        return self._counts[k]

    def join(self):
        """the caller's current stream waits for everything that the object has enqueued so far, and the object's next launch
        for what is on that stream by then (a graph replayed there, for instance)"""
        with self._turn:
            self._buckets.join()
