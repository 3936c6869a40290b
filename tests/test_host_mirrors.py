"""Host-side mirrors of the reference's Python callers: bit-width allocation (CPU),
compressor objects and the simulated ring (GPU)."""
import types

import numpy as np
import pytest
import torch

from helpers import BF16, bits_to_f32, to_bits

DEV = "cuda:0"


# ---- bit-width allocation (torch ops, runs anywhere) ------------------------------------------

def test_bitrate_search_hits_target():
    from dynamiq_sigcomm_artifact_amd import bitrate as B
    g = torch.Generator().manual_seed(0)
    norms = [torch.exp(torch.randn(5000, generator=g) * 5 - 6).to(torch.bfloat16) for _ in range(3)]
    assert B.dynamic_bitrate_target_bitrate("dynamiQ_mee_5bit_dynamic_bitrate") == 5.0
    assert B.dynamic_bitrate_target_bitrate("dynamiq_aee_dynamic_bitrate") == 5.0
    assert B.dynamic_bitrate_target_bitrate("x_3bit") == 3.0
    target = 5.0 - B.DYNAMIC_BITRATE_HEADROOM
    u, avg, delta = B.dynamic_bitrate_binary_search_u(norms, target)
    assert B.DYNAMIC_BITRATE_U_MIN <= u <= B.DYNAMIC_BITRATE_U_MAX
    assert abs(avg - target) <= B.DYNAMIC_BITRATE_TOL and abs(delta - (target - avg)) < 1e-12
    # extremes of u (comm_hooks.py:1087: the first compressed round starts at u = 60 -> all 8-bit)
    assert B.dynamic_bitrate_average_bits(norms, 60.0) == 8.0
    assert B.dynamic_bitrate_average_bits(norms, -10.0) == 2.0
    # the incremental rule keeps a converged u and walks back from a bad one
    u2, avg2, d2 = B.dynamic_bitrate_adjust_u(norms, u, target)
    assert u2 == u and abs(d2) <= B.DYNAMIC_BITRATE_TOL
    u3, avg3, d3 = B.dynamic_bitrate_adjust_u(norms, u + 6.0, target)
    assert abs(d3) < abs(B.dynamic_bitrate_avg_delta(norms, u + 6.0, target)[1])
    # qbits values and monotonicity in the norm
    q = B.dynamic_bitrate_qbits(torch.sort(norms[0].float())[0], u)
    assert set(q.unique().tolist()) <= {2, 4, 8} and bool((q[1:] >= q[:-1]).all())
    assert B.dynamic_bitrate_average_bits([], 0.0) == 0.0


# ---- compressor objects -------------------------------------------------------------------------

def _params(d, world, method="dynamiQ_aee_5bit"):
    return {"d": {(0, 0): d}, "world_size": world, "rank": 0,
            "args": types.SimpleNamespace(aggregation_method=method)}


@pytest.mark.gpu
def test_compressor_object_matches_reference_bookkeeping(eden_utils, oracle):
    from dynamiq_sigcomm_artifact_amd.compressors import Aee_Dynamic_Range_GPU_kern, Mee_Dynamic_Range_GPU_kern
    d, W = 256 * 40, 4
    for cls, strategy in ((Aee_Dynamic_Range_GPU_kern, 2), (Mee_Dynamic_Range_GPU_kern, 3)):
        c = cls(4, 16, _params(d, W))
        assert c.strategy == strategy and c.supergroup == 16 and c.range == 7
        # utils_aggregation.py:380-389: pool rows = 3 * ((d + C) // C) // W
        assert tuple(c.randomized_vec_pool.shape) == (3 * ((d + 16) // 16) // W, 16)
        assert c.randomized_vec_pool.dtype == torch.bfloat16
        assert c.compressed_numel(1000) == 4 * 146 and c.padded_n(1000) == 1024
        assert c.create_tensor(torch.zeros(1000), torch.uint8).numel() == 4 * 146
        # LCG of the row offsets (:391,395-397,409-420)
        seed = (4 * 998244353) & 0xFFFFFFFF
        n = 256 * 8
        x = (torch.randn(n, device=DEV) * 1e-3).to(torch.bfloat16)
        send = c.create_tensor(x, torch.uint8)
        rows = c.randomized_vec_pool.shape[0]
        for _ in range(3):
            seed = (seed * 671431 + 1000000007) & 0xFFFFFFFF
            randl = seed % (rows - n // 16 - 1)
            c.compression(x, send)
            rnd = c.randomized_vec_pool[randl:randl + n // 16, :].reshape(-1)
            want = oracle.scaling_compress(to_bits(x), to_bits(rnd), n, 4, 16, strategy, BF16)
            assert (send.cpu().numpy() == want).all()
        out = torch.zeros_like(x)
        c.decompression(send, out)
        dec = np.zeros(n, np.uint16)
        oracle.scaling_decompress(want, dec, n, 4, 16, strategy, BF16)
        assert (to_bits(out) == dec).all()
        c.decompression_add(send, out)
        oracle.scaling_decompress(want, dec, n, 4, 16, strategy, BF16, add=True)
        assert (to_bits(out) == dec).all()


@pytest.mark.gpu
def test_loaded_random_pool_keeps_the_dtype_the_reference_keeps(eden_utils, oracle):
    """the "correlated" mode loads its pool from a file: the AEE class keeps the file's dtype (utils_aggregation.py:389),
    the MEE class casts it to float16 (:488), so a bfloat16 call of the MEE class rounds every value twice"""
    from dynamiq_sigcomm_artifact_amd.compressors import Aee_Dynamic_Range_GPU_kern, Mee_Dynamic_Range_GPU_kern
    d, W, n = 256 * 40, 2, 256 * 6
    g = torch.Generator().manual_seed(8)
    loaded = torch.rand(3 * ((d + 16) // 16) // W * 16 + 100, generator=g)
    x = (torch.randn(n, generator=g) * 1e-3).to(torch.bfloat16)
    twice = loaded.to(torch.float16).to(torch.bfloat16)
    once = loaded.to(torch.bfloat16)
    assert not torch.equal(twice, once)
    for cls, strategy, seen, kept in ((Aee_Dynamic_Range_GPU_kern, 2, once, torch.float32),
                                      (Mee_Dynamic_Range_GPU_kern, 3, twice, torch.float16)):
        c = cls(4, 16, dict(_params(d, W), rand_pool_tensor=loaded))
        assert c.randomized_vec_pool.dtype == kept
        rows = c.randomized_vec_pool.shape[0]
        assert rows == 3 * ((d + 16) // 16) // W
        send = c.create_tensor(x, torch.uint8)
        c.compression(x.to(DEV), send)
        seed = ((4 * 998244353) & 0xFFFFFFFF) * 671431 + 1000000007 & 0xFFFFFFFF
        randl = seed % (rows - n // 16 - 1)
        rnd = seen[randl * 16:randl * 16 + n]
        want = oracle.scaling_compress(to_bits(x), to_bits(rnd), n, 4, 16, strategy, BF16)
        assert (send.cpu().numpy() == want).all()


def _own_rows(how, made):
    """a compressor class, or object, that picks its rows of the pool itself"""
    from dynamiq_sigcomm_artifact_amd.compressors import Aee_Dynamic_Range_GPU_kern as Base

    class Rows(Base):
        def rand_pool(self, n, dtype):
            made.append(self.randomized_vec_pool.to(dtype)[3:3 + n // self.chunk_size])
            return made[-1]

    class Next(Base):
        def gen_next_rand(self):
            made.append(5)
            return 5

    def one(params, **kw):
        c = Base(4, 16, params, **kw)
        c.gen_next_rand = lambda: made.append(5) or 5
        return c

    return {"rows": lambda params, **kw: Rows(4, 16, params, **kw), "next": lambda params, **kw: Next(4, 16, params, **kw), "object": one}[how]


@pytest.mark.parametrize("how", ["rows", "next", "object"])
def test_own_choice_of_rows_is_asked_for(how):
    """a subclass (or an object) with a rand_pool or gen_next_rand of its own is called for every encoding call, and the module gets
    the rows that it picked; an all-reduce with such compressors goes call by call"""
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import _pooled_codecs
    made, given = [], []
    c = _own_rows(how, made)(_params(256 * 40, 1), device="cpu")

    def note(*args):
        given.append(args)

    c.eden_utils = types.SimpleNamespace(scaling_compress=note, scaling_dec_comp=note)
    c._stream = lambda: 0
    x, y = torch.ones(512, dtype=torch.bfloat16), torch.zeros(292, dtype=torch.uint8)
    c.compression(x, y)
    c.dec_compression(y, x, y)
    c.compression(x[:0], y)
    first = 3 if how == "rows" else 5
    want = c.randomized_vec_pool.to(torch.bfloat16)[first:first + 32]
    assert len(given) == 2 and len(made) == 2
    assert all(torch.equal(rows, want) for rows in (given[0][2], given[1][3]))
    assert [g[-5:] for g in given] == [(512, 4, 16, 0, 2)] * 2
    vec = types.SimpleNamespace(dtype=torch.bfloat16)
    assert _pooled_codecs([vec], {q: [c] for q in (8, 4, 2)}) is None


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["rows", "next", "object"])
def test_own_choice_of_rows_on_the_gpu(capi, how):
    made = []
    c = _own_rows(how, made)(_params(256 * 40, 1), device=DEV)
    x = (torch.randn(256 * 6, device=DEV) * 1e-3).to(torch.bfloat16)
    send, want = c.create_tensor(x, torch.uint8), c.create_tensor(x, torch.uint8)
    c.compression(x, send)
    first = 3 if how == "rows" else 5
    pool = c.randomized_vec_pool.to(torch.bfloat16)[first:first + 96].reshape(-1).contiguous()
    capi.scaling_compress(x, want, pool, x.numel(), 4, 16, 2)
    assert torch.equal(send, want) and len(made) == 1
    again = torch.zeros_like(send)
    c.dec_compression(send, x, again)
    capi.scaling_dec_comp(want, x, send, pool, x.numel(), 4, 16, 2)
    assert torch.equal(again, send) and len(made) == 2


@pytest.mark.gpu
def test_replaced_pool_is_checked(capi):
    """a pool that a caller has put in the place of the object's: refused where a call would read beyond its rows or take them for
    another type; rows that are wider than a chunk are read from their starts, as slices of such a pool are"""
    from dynamiq_sigcomm_artifact_amd.compressors import Aee_Dynamic_Range_GPU_kern
    from dynamiq_sigcomm_artifact_amd.dynamiq_pipeline import fixed_proportion_allreduce_grouped
    c = Aee_Dynamic_Range_GPU_kern(4, 16, _params(256 * 40, 1), device=DEV)
    x = (torch.randn(256 * 6, device=DEV) * 1e-3).to(torch.bfloat16)
    send, want = c.create_tensor(x, torch.uint8), c.create_tensor(x, torch.uint8)
    good = c.randomized_vec_pool
    thresholds = {8: 0.2, 4: 0.5, 2: 0.3}
    shared = {q: [Aee_Dynamic_Range_GPU_kern(q, 16, _params(256 * 40, 1), device=DEV)] for q in (8, 4, 2)}
    for bad, text in ((good.to(torch.float16), "dtype"), (good[:, :8].contiguous(), "too small|16 values"), (good.reshape(-1), "rows"),
                      (good.cpu(), "CUDA|contiguous tensor"), (good[:, ::2], "contiguous")):
        for owner in (c, shared[4][0]):
            owner.randomized_vec_pools[torch.bfloat16] = bad
        with pytest.raises(RuntimeError, match=text):
            c.compression(x, send)
        with pytest.raises(RuntimeError, match=text):
            c.dec_compression(send, x, want)
        with pytest.raises(RuntimeError, match=text):
            fixed_proportion_allreduce_grouped([x], thresholds, shared)
    wide = torch.rand((500, 48), device=DEV).to(torch.bfloat16)
    c.randomized_vec_pools[torch.bfloat16] = wide
    seed = (c.rand_seed * 671431 + 1000000007) & 0xFFFFFFFF
    c.compression(x, send)
    first = seed % (500 - 96 - 1)
    capi.scaling_compress(x, want, wide[first:first + 96].reshape(-1), x.numel(), 4, 16, 2)
    assert torch.equal(send, want)


@pytest.mark.gpu
def test_attributes_of_a_compressor_apply_to_the_next_call(capi):
    """width, chunk size, strategy, seed of the rounding stream and the pools, set after construction, are what the next call uses;
    without a seed the pool is"""
    from dynamiq_sigcomm_artifact_amd.compressors import Aee_Dynamic_Range_GPU_kern
    n = 256 * 6
    c = Aee_Dynamic_Range_GPU_kern(4, 16, _params(256 * 40, 1), device=DEV)
    x = (torch.randn(n, device=DEV) * 1e-3).to(torch.bfloat16)
    send = torch.zeros(capi.required_bytes(n, 8, 8, 3), dtype=torch.uint8, device=DEV)
    want = torch.zeros_like(send)
    c.nbits, c.strategy, c.philox_seed, c.philox_step = 8, 3, 77, 10
    c.compression(x, send)
    capi.scaling_compress_philox(x, want, n, 8, 16, 3, 77, 11)
    assert torch.equal(send, want) and c.philox_step == 11
    c.chunk_size, c.philox_seed, c.randomized_vec_pools = 8, None, {}
    c.randomized_vec_pool = torch.rand((600, 8), device=DEV).to(torch.bfloat16)
    first = ((c.rand_seed * 671431 + 1000000007) & 0xFFFFFFFF) % (600 - n // 8 - 1)
    c.compression(x, send)
    pool = c.randomized_vec_pool[first:first + n // 8].reshape(-1)
    capi.scaling_compress(x, want, pool, n, 8, 8, 3)
    assert torch.equal(send, want) and c.philox_seed is None
    out, back = torch.zeros_like(x), torch.zeros_like(x)
    c.decompression(send, out)
    capi.scaling_decompress(want, back, n, 8, 8, 3)
    assert torch.equal(out, back)
    c.chunk_size = 0
    with pytest.raises(RuntimeError, match="positive"):
        c.compression(x, send)


def test_attributes_of_a_compressor_on_the_cpu():
    from dynamiq_sigcomm_artifact_amd.compressors import Mee_Dynamic_Range_GPU_kern
    c = Mee_Dynamic_Range_GPU_kern(5, 16, dict(_params(256 * 40, 2), philox_seed=3, rank=1), device="cpu")
    assert c.philox_seed == 3 + 0x9E3779B97F4A7C15 and c.philox_step == 5 << 32 and c.randomized_vec_pool is None
    c.philox_seed = None
    assert c.philox_seed is None and not c._codec.philox
    c.philox_seed = -1
    assert c.philox_seed == 2 ** 64 - 1 and c._codec.philox
    c.strategy, c.nbits, c.chunk_size = 2, 4, 32
    assert (c._codec.strategy, c._codec.nbits, c._codec.chunk) == (2, 4, 32)
    c.randomized_vec_pools = pools = {}
    assert c.randomized_vec_pools is pools


def test_empty_vectors_are_nothing_to_do():
    """an empty chunk of a ring returns before anything is checked or drawn, wherever it lives"""
    from dynamiq_sigcomm_artifact_amd.compressors import Aee_Dynamic_Range_GPU_kern
    c = Aee_Dynamic_Range_GPU_kern(4, 16, _params(256 * 40, 1), device="cpu")
    seed = c.rand_seed
    none, stream = torch.zeros(0, dtype=torch.bfloat16), torch.zeros(0, dtype=torch.uint8)
    c.compression(none, stream)
    c.dec_compression(stream, none, stream)
    c.decompression(stream, none)
    c.decompression_add(stream, none)
    assert c.rand_seed == seed
    with pytest.raises(RuntimeError, match="CUDA"):
        c.compression(torch.zeros(256, dtype=torch.bfloat16), stream)


def _oracle_ring(oracle, vecs_bits, pools, nbits, strategy, W):
    """the same schedule on the CPU with oracle calls (ring_rdma.py:590-631)"""
    n = vecs_bits[0].size
    csize = ((n + W - 1) // W + 255) // 256 * 256
    bounds = [(csize * i, min(csize * (i + 1), n)) for i in range(W)]
    seeds = [(nbits * 998244353) & 0xFFFFFFFF for _ in range(W)]
    send = [None] * W
    recv = [None] * W

    def rand_for(r, cnt):
        seeds[r] = (seeds[r] * 671431 + 1000000007) & 0xFFFFFFFF
        rows = pools[r].size // 16
        randl = seeds[r] % (rows - cnt // 16 - 1)
        return np.ascontiguousarray(pools[r][randl * 16: randl * 16 + cnt])

    def chunk(r, i):
        lo, hi = bounds[i]
        return vecs_bits[r][lo:hi]

    def exch(src):
        return [src[(r - 1) % W] for r in range(W)]

    for step in range(W - 1):
        for r in range(W):
            if step == 0:
                c = np.ascontiguousarray(chunk(r, r))
                send[r] = oracle.scaling_compress(c, rand_for(r, c.size), c.size, nbits, 16, strategy, BF16)
            else:
                c = np.ascontiguousarray(chunk(r, (r - step) % W))
                send[r] = oracle.scaling_dec_comp(recv[r], c, rand_for(r, c.size), c.size, nbits, 16, strategy, BF16)
        recv = exch(send)
    for r in range(W):
        lo, hi = bounds[(r + 1) % W]
        c = np.ascontiguousarray(vecs_bits[r][lo:hi])
        send[r] = oracle.scaling_dec_comp(recv[r], c, rand_for(r, c.size), c.size, nbits, 16, strategy, BF16)
        oracle.scaling_decompress(send[r], c, c.size, nbits, 16, strategy, BF16)
        vecs_bits[r][lo:hi] = c
    bufs = [send, recv]
    for step in range(W - 1):
        bufs[(step ^ 1) & 1] = exch(bufs[step & 1])
        for r in range(W):
            lo, hi = bounds[(r - step) % W]
            c = np.zeros(hi - lo, np.uint16)
            oracle.scaling_decompress(bufs[(step ^ 1) & 1][r], c, c.size, nbits, 16, strategy, BF16)
            vecs_bits[r][lo:hi] = c
    return vecs_bits


@pytest.mark.gpu
@pytest.mark.parametrize("W,nbits,strategy", [(4, 4, 2), (8, 8, 2), (3, 4, 3), (8, 2, 2)])
def test_simulated_ring_matches_oracle_schedule(eden_utils, oracle, W, nbits, strategy):
    from dynamiq_sigcomm_artifact_amd import compressors as CP
    from dynamiq_sigcomm_artifact_amd.ring_sim import ring_allreduce
    n = 256 * 37   # ragged: the last ring chunk is shorter than the others
    g = torch.Generator().manual_seed(W * 10 + nbits)
    sig = torch.exp(torch.rand(W, generator=g) * 4.6 - 9.2)          # log-uniform in [1e-4, 1e-2]
    grads = [(torch.randn(n, generator=g) * sig[r]).to(torch.bfloat16) for r in range(W)]
    exact = torch.stack([x.double() for x in grads]).sum(0)
    cls = CP.Aee_Dynamic_Range_GPU_kern if strategy == 2 else CP.Mee_Dynamic_Range_GPU_kern
    gen = torch.Generator(device=DEV).manual_seed(99)
    comps = [cls(nbits, 16, dict(_params(n, W), rank=r), generator=gen) for r in range(W)]
    vecs = [x.to(DEV) for x in grads]
    ring_allreduce(vecs, comps)
    torch.cuda.synchronize()
    # every rank holds the same bytes
    for r in range(1, W):
        assert torch.equal(vecs[r], vecs[0])
    # and they are the bytes the oracle produces for the same schedule and random offsets
    pools = [to_bits(c.randomized_vec_pool.reshape(-1)) for c in comps]
    want = _oracle_ring(oracle, [to_bits(x) for x in grads], pools, nbits, strategy, W)
    assert (to_bits(vecs[0]) == want[0]).all()
    nmse = float(((vecs[0].double().cpu() - exact) ** 2).sum() / (exact ** 2).sum())
    assert nmse < {2: 4.0, 4: 0.12, 8: 6e-4}[nbits], nmse


def test_bench_refuses_more_than_one_gpu():
    """no multi-GPU figure is produced: bench.py --gpus 2 exits with a message before touching a device"""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, os.path.join(root, "bench.py"), "--gpus", "2"], capture_output=True, text=True)
    assert r.returncode == 2 and "--gpus must be 1" in r.stderr and r.stdout.strip() == ""


def test_bench_line_stays_short():
    """the cells of the other configurations go into the line as one entry per configuration: 49 cells were 30 KB, of which
    a reader who keeps the last 8 KB of the output had no line left"""
    import importlib.util
    import json
    import os
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    spec = importlib.util.spec_from_file_location("bench_program", os.path.join(root, "bench.py"))
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    cells = [{"workload": "config %s: cell %d of many, with a long description of what it is" % (name, k), "compress_us": 10.0 + k,
              "compress_frac": 0.5 + 0.001 * k, "decompress_frac": 0.6, "fused_frac": 0.7 if k else None, "GBps_fp32_in": 1500.0 + k,
              "nmse": 0.01, "bit_exact_vs_oracle": True}
             for name, count in (("2", 8), ("3", 4), ("4", 3), ("5", 28), ("ref", 6)) for k in range(count)]
    out = bench.summary(cells)
    assert {k: v["cells"] for k, v in out.items()} == {"config 2": 8, "config 3": 4, "config 4": 3, "config 5": 28, "config ref": 6}
    assert out["config 5"]["compress_frac"] == [0.5, 0.527] and out["config 3"]["GBps_fp32_in"] == [1500.0, 1503.0]
    assert out["config 2"]["fused_frac"] == [0.7, 0.7] and "nmse" not in out["config 2"]
    assert all(v["bit_exact_vs_oracle"] is True for v in out.values())
    cells[3]["bit_exact_vs_oracle"] = False
    cells[9]["bit_exact_vs_oracle"] = None
    out = bench.summary(cells)
    assert out["config 2"]["bit_exact_vs_oracle"] is False and out["config 3"]["bit_exact_vs_oracle"] is None
    assert len(json.dumps(out)) < 2000
    assert bench.summary([]) == {}


def test_division_by_the_world_size_as_a_multiplication():
    """The mixed kernels split a group of n superchunks over the ring as ceil(n / world) per rank and compute the
    quotient as (x * ceil(2^40 / world)) >> 40 for x < 2^24 and world <= 2^16 (dq_scaling_mixed.hip: divide_by_world).
    Brute force over every world size and the operands where such a reciprocal goes wrong first: multiples of the
    divisor minus one, the largest operands, and a random sample."""
    import numpy as np
    rng = np.random.default_rng(5)
    top = (1 << 24) - 1
    for d in range(2, 65537):
        m = ((1 << 40) + d - 1) // d
        k = np.concatenate([np.arange(1, 6, dtype=np.uint64), np.uint64(top // d) - np.arange(0, 4, dtype=np.uint64)])
        x = np.concatenate([k * np.uint64(d) - np.uint64(1), k * np.uint64(d), np.array([top, top - 1, 0, 1], np.uint64),
                            rng.integers(0, top + 1, 24, dtype=np.uint64)])
        x = x[x <= top]
        assert ((x * np.uint64(m)) >> np.uint64(40) == x // np.uint64(d)).all(), d


def test_uniform_values_are_drawn_only_beside_a_known_torch():
    """the kernel restates which element of uniform_ comes from where in the generator's stream, as the releases below do it; with
    any other torch compress leaves the drawing to uniform_"""
    from dynamiq_sigcomm_artifact_amd import thc
    for version in ("2.10.0", "2.10.0+rocm7.0", "2.10.1a0"):
        assert thc._drawn_dimensions(version) == (1 << 19, 1 << 25)
    for version in ("2.9.1", "2.11.0+rocm7.1", "2.1.0", "3.10.0"):
        least, greatest = thc._drawn_dimensions(version)
        assert least > greatest
    assert thc._DRAWN == thc._drawn_dimensions(torch.__version__)
