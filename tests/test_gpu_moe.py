"""GPU parity of the MoE half (cpg_moe_forward) and its building blocks, through the C ABI.

Bars (from the path's contract): dequantised weights, xn, router logits, top-K indices and
renormalised weights bit-exact; MoE output within 1e-3 max relative error, measured as
max|gpu - ref| / max|ref| over the output, against the reference engine at both of its
Q4 numerics (CP_THREADS=1 scalar, CP_THREADS=8 AVX2).
"""
import ctypes
import os
import sys

import numpy as np
import pytest

from tests.conftest import golden
from tests.gpu_helpers import DeviceMoE, rel_err, bits, route_mode, expert_mode, fused_mode

pytestmark = pytest.mark.gpu

MOE_TOL = 1e-3
# the MFMA paths' own bar: measured at most 1.5e-6; an activation split whose lo half misses
# its hi half (an f16 unit lost) shows as ~3e-5
SPLIT_TOL = 1e-5
WT_TOL = 1e-5     # certified routing: renormalised weights from the certified logits


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def test_device(cpg):
    name = cpg.device_name()
    say("device:", name)
    assert "gfx950" in name


# ------------------------------------------------------------------ expf, dequant, generator

def _chunks(cpg, op, check, nchunks=32):
    """Run device math op over every float32 bit pattern in nchunks chunks; check(start,
    x, y) must return a falsy value or a message."""
    chunk = (1 << 32) // nchunks
    xb, yb = cpg.DeviceBuffer(chunk * 4), cpg.DeviceBuffer(chunk * 4)
    for c in range(nchunks):
        start = c * chunk
        xbits = np.arange(start, start + chunk, dtype=np.uint64).astype(np.uint32)
        xb.upload(xbits)
        cpg.check(cpg.lib().cpg_math_dev(op, xb.ptr, None, yb.ptr, chunk), "cpg_math_dev")
        msg = check(start, xbits.view(np.float32), yb.download(np.float32, chunk))
        assert not msg, f"chunk {c}: {msg}"


def test_expf_exhaustive(cpg, oracle):
    """The device expf against the oracle's (itself equal to glibc on all inputs), every
    float32 bit pattern."""
    fn = oracle.L.or_expf_check
    fn.restype = ctypes.c_long
    fn.argtypes = [ctypes.c_uint64, ctypes.c_uint64, ctypes.c_void_p, ctypes.c_int,
                   ctypes.POINTER(ctypes.c_uint64)]
    threads = min(16, os.cpu_count() or 1)

    def check(start, x, y):
        fb = ctypes.c_uint64(0)
        bad = fn(start, y.size, y.ctypes.data, threads, ctypes.byref(fb))
        return bad and f"{bad} mismatches, first at {fb.value:#010x}"
    _chunks(cpg, cpg.MATH_EXPF, check)
    say("expf: all 2^32 inputs identical")


def test_sqrt_exhaustive(cpg):
    """The RMSNorm's sqrt is correctly rounded (as glibc sqrtf) on every float32 input."""
    def check(start, x, y):
        with np.errstate(invalid="ignore"):
            want = np.sqrt(x)
        same = (y.view(np.uint32) == want.view(np.uint32)) | (np.isnan(y) & np.isnan(want))
        return (not same.all()) and f"{(~same).sum()} mismatches at {x[~same][:4]}"
    _chunks(cpg, cpg.MATH_SQRT, check)
    say("sqrt: all 2^32 inputs correctly rounded")


def test_div_and_silu(cpg, oracle):
    """Division is correctly rounded (random pairs over all exponents + edge cases); SiLU
    follows kernels.c:416 with the glibc-identical expf."""
    rng = np.random.default_rng(11)
    n = 1 << 24
    a = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32).view(np.float32)
    b = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32).view(np.float32)
    edge = np.array([0.0, -0.0, 1.0, 3.0, 1e-45, 1e-38, 3.4e38, np.inf, -np.inf], np.float32)
    a = np.concatenate([a, np.repeat(edge, edge.size)])
    b = np.concatenate([b, np.tile(edge, edge.size)])
    xa, xb, out = cpg.to_device(a), cpg.to_device(b), cpg.DeviceBuffer(a.nbytes)
    cpg.check(cpg.lib().cpg_math_dev(cpg.MATH_DIV, xa.ptr, xb.ptr, out.ptr, a.size), "div")
    got = out.download(np.float32, a.size)
    with np.errstate(all="ignore"):
        want = a / b
    same = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
    assert same.all(), (a[~same][:4], b[~same][:4])
    x = rng.normal(0, 6, 1 << 16).astype(np.float32)
    xd = cpg.to_device(x)
    cpg.check(cpg.lib().cpg_math_dev(cpg.MATH_SILU, xd.ptr, None, out.ptr, x.size), "silu")
    got = out.download(np.float32, x.size)
    want = np.array([oracle.L.or_silu(float(v)) for v in x], np.float32)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def test_f16_scale_conversion_exhaustive(cpg, oracle):
    """The hardware fp16 -> fp32 conversion the one-token GEMVs apply to block scales equals
    the reference's f16_to_f32 (engine/kernels/kernels.c:109-130, restated by the oracle) on all
    65,536 bit patterns: bit for bit, NaNs as NaNs."""
    h = np.arange(1 << 16, dtype=np.uint32)
    x, out = cpg.to_device(h.view(np.float32)), cpg.DeviceBuffer(h.size * 4)
    cpg.check(cpg.lib().cpg_math_dev(cpg.MATH_F16, x.ptr, None, out.ptr, h.size), "f16")
    got = out.download(np.float32, h.size)
    want = np.array([oracle.L.or_f16_to_f32(int(v)) for v in h], np.float32)
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))


@pytest.mark.parametrize("enc", [4, 8])
def test_dequant_exhaustive(cpg, oracle, enc):
    """All 65,536 fp16 scales x every nibble / int8 value: v4 rows and the row-tiled layout
    (after cpg_repack) against the oracle, bit for bit."""
    from tests.test_oracle import all_scale_blocks_q4, all_scale_blocks_q8
    blk = all_scale_blocks_q4() if enc == 4 else all_scale_blocks_q8()
    rows, cols = (2048, 1024) if enc == 4 else (4096, 4096)
    n = rows * cols
    want = oracle.dequant_row(enc, blk, n)
    src = cpg.to_device(blk)
    out = cpg.DeviceBuffer(n * 4)
    cpg.check(cpg.lib().cpg_dequant_rows(enc, src.ptr, rows, cols, out.ptr), "dequant_rows")
    got = out.download(np.float32, n)
    assert np.array_equal(bits(got), bits(want))
    tiled = cpg.DeviceBuffer(cpg.lib().cpg_matrix_bytes(enc, rows, cols))
    cpg.check(cpg.lib().cpg_repack(enc, tiled.ptr, src.ptr, rows, cols), "repack")
    cpg.check(cpg.lib().cpg_dequant_tiled(enc, tiled.ptr, rows, cols, 0, rows, out.ptr), "tiled")
    got = out.download(np.float32, n)
    assert np.array_equal(bits(got), bits(want))


@pytest.mark.parametrize("enc", [4, 8])
def test_generator_device_equals_host(cpg, enc):
    L = cpg.lib()
    for stream in (cpg.stream_id(0, cpg.K_WG, 5), cpg.stream_id(47, cpg.K_WD, 127)):
        rows, cols = 768, 2048
        host = cpg.gen_blocks(enc, 20261017, stream, rows * cols, 0.02)
        dev = cpg.DeviceBuffer(host.nbytes)
        cpg.check(L.cpg_gen_blocks(enc, 20261017, stream, rows, cols, 0.02, dev.ptr), "gen")
        assert np.array_equal(dev.download(np.uint8, host.nbytes), host)
    # whole experts straight into the tiled layout == host blocks repacked
    D, F, E = 256, 128, 2
    eb = L.cpg_expert_bytes(enc, D, F)
    a, b = cpg.DeviceBuffer(E * eb), cpg.DeviceBuffer(E * eb)
    a.zero(); b.zero()
    cpg.check(L.cpg_gen_experts(enc, 99, 3, D, E, F, a.ptr), "gen_experts")
    mg = L.cpg_matrix_bytes(enc, F, D)
    for e in range(E):
        for kind, k in enumerate((cpg.K_WG, cpg.K_WU, cpg.K_WD)):
            rows, cols = (F, D) if kind < 2 else (D, F)
            blk = cpg.gen_blocks(enc, 99, cpg.stream_id(3, k, e), rows * cols, 0.02)
            cpg.check(L.cpg_upload_matrix(enc, b.ptr + e * eb + kind * mg, blk.ctypes.data,
                                          rows, cols), "upload")
    cpg.sync()
    assert np.array_equal(a.download(np.uint8, E * eb), b.download(np.uint8, E * eb))


# ------------------------------------------------------------------ MoE, small geometry vs oracle

@pytest.fixture(scope="module", params=["small_q4", "small_q8"])
def small(request, cpg):
    from cachepotato_amd import synth
    spec = synth.SMALL[request.param]
    m = DeviceMoE(spec, max_T=128)
    yield m
    m.close()


@pytest.mark.parametrize("T", [1, 2, 5, 16, 17, 64, 100])
def test_moe_small_vs_oracle(cpg, oracle, small, T):
    from cachepotato_amd import synth
    spec = small.spec
    x = synth.inputs(spec, 1000 + T, T)
    got = small.forward(x)
    for threads in (1, 8):
        want = oracle.moe(spec, small.wgate_host, synth.ln2(spec), small.host_mats, x,
                          threads=threads)
        for k in ("xn", "router", "wt"):
            assert np.array_equal(bits(got[k]), bits(want[k])), (k, threads)
        assert np.array_equal(got["topk"], want["topk"])
        e = rel_err(got["mlp"], want["mlp"])
        say(f"{spec.enc} T={T} threads={threads}: mlp rel err {e:.2e}")
        assert e <= MOE_TOL


ROUTE_MODES = {"auto": 0, "fallback": 2, "refine": 3}   # cachepotato_amd.ROUTE_*


@pytest.mark.parametrize("mode", ["auto", "fallback", "refine"])
@pytest.mark.parametrize("T", [1, 2, 5, 16])
def test_moe_small_certified(cpg, oracle, small, T, mode):
    """Certified routing (neither logits nor xn asked for, T <= 16): top-K identical to the
    reference; weights within WT_TOL; MoE output within 1e-3. The fallback mode fails every
    certificate and skips the refined step, so the exact chains run for every token and the
    weights are bit-identical; the refine mode fails every certificate, so the refined step
    (exact chains of the candidates only) runs for every token."""
    from cachepotato_amd import synth
    spec = small.spec
    x = synth.inputs(spec, 3000 + T, T)
    f0, x0 = small.fallbacks(), small.exact_routings()
    with route_mode(ROUTE_MODES[mode]):
        got = small.forward(x, outputs=False)
    nfb, nex = small.fallbacks() - f0, small.exact_routings() - x0
    if mode != "auto":
        assert nfb == T
    if mode == "fallback":
        assert nex == T
    for threads in (1, 8):
        want = oracle.moe(spec, small.wgate_host, synth.ln2(spec), small.host_mats, x,
                          threads=threads)
        assert np.array_equal(got["topk"], want["topk"])
        if mode == "fallback":
            assert np.array_equal(bits(got["wt"]), bits(want["wt"]))
        assert rel_err(got["wt"], want["wt"]) <= WT_TOL
        e = rel_err(got["mlp"], want["mlp"])
        assert e <= MOE_TOL
    say(f"certified {spec.enc} T={T} {mode}: {nfb} fallbacks ({nex} with every chain exact), "
        f"mlp rel err {e:.2e}")


@pytest.mark.parametrize("F", [128, 192])
@pytest.mark.parametrize("mode", ["auto", "fallback"])
def test_moe_one_token_gateup_rows(cpg, oracle, F, mode):
    """The one-token gate/up kernel at D = 2048 with 32 rows of each matrix per workgroup
    (F = 128: F not a multiple of 24) and with 24 (F = 192), certified and on the exact
    fallback (which loads the exact expert's rows again): top-K identical to the reference,
    MoE output within MOE_TOL, at both reference numerics."""
    from cachepotato_amd import synth
    spec = synth.MoESpec(D=2048, E=16, K=8, F=F, enc=synth.ENC_Q4)
    m = DeviceMoE(spec, max_T=1)
    try:
        for i in range(4):
            x = synth.inputs(spec, 500 + i, 1)
            with route_mode(ROUTE_MODES[mode]):
                got = m.forward(x, outputs=False)
            for threads in (1, 8):
                want = oracle.moe(spec, m.wgate_host, synth.ln2(spec), m.host_mats, x,
                                  threads=threads)
                assert np.array_equal(got["topk"], want["topk"]), (F, mode, i, threads)
                e = rel_err(got["mlp"], want["mlp"])
                assert e <= MOE_TOL, (F, mode, i, threads, e)
        say(f"one-token gate/up F={F} {mode}: mlp rel err {e:.2e}")
    finally:
        m.close()


@pytest.mark.parametrize("T", [1, 5])
@pytest.mark.parametrize("mode", ["auto", "fallback"])
def test_moe_many_experts_certified(cpg, oracle, T, mode):
    """160 experts (more than four ranking threads per expert fit a routing workgroup of 512
    threads, so each token's last routing workgroup ranks with the general form, and one token
    takes the routing path of several): top-K identical to the reference, MoE output within
    MOE_TOL, certified and on the exact fallback."""
    from cachepotato_amd import synth
    spec = synth.MoESpec(D=256, E=160, K=4, F=128, enc=synth.ENC_Q4)
    m = DeviceMoE(spec, max_T=T)
    try:
        x = synth.inputs(spec, 700 + T, T)
        with route_mode(ROUTE_MODES[mode]):
            got = m.forward(x, outputs=False)
        for threads in (1, 8):
            want = oracle.moe(spec, m.wgate_host, synth.ln2(spec), m.host_mats, x,
                              threads=threads)
            assert np.array_equal(got["topk"], want["topk"]), (T, mode, threads)
            if mode == "fallback":
                assert np.array_equal(bits(got["wt"]), bits(want["wt"]))
            assert rel_err(got["wt"], want["wt"]) <= WT_TOL
            e = rel_err(got["mlp"], want["mlp"])
            assert e <= MOE_TOL, (T, mode, threads, e)
        say(f"E=160 T={T} {mode}: mlp rel err {e:.2e}")
    finally:
        m.close()


def test_moe_small_attn_and_accumulate(cpg, oracle, small):
    """hh = x + attn feeds the router (qwen3_moe.c:178); mlp is accumulated into."""
    from cachepotato_amd import synth
    spec = small.spec
    x = synth.inputs(spec, 77, 9)
    attn = synth.inputs(spec, 177, 9) * np.float32(0.5)
    mlp0 = synth.inputs(spec, 277, 9)
    got = small.forward(x, mlp_in=mlp0, attn=attn)
    want = oracle.moe(spec, small.wgate_host, synth.ln2(spec), small.host_mats, x, attn=attn)
    assert np.array_equal(bits(got["router"]), bits(want["router"]))
    assert np.array_equal(got["topk"], want["topk"])
    assert rel_err(got["mlp"] - mlp0, want["mlp"]) <= MOE_TOL


def test_moe_small_ties(cpg, oracle):
    """Identical router rows: the lower expert id wins every tie, as in the reference
    (qwen3_moe.c:184-194). With positive inputs the logits are 0.01*sum(xn) for experts
    2, 7, 11, 0.005*sum(xn) for 4, 5 and 0 for the rest, so top-4 is [2, 7, 11, 4]."""
    from cachepotato_amd import synth
    from cachepotato_amd.synth import MoESpec
    spec = MoESpec(D=256, E=16, K=4, F=128, enc=4)
    m = DeviceMoE(spec, max_T=4)
    w = np.zeros((16, 256), np.float32)
    w[[2, 7, 11], :] = 0.01
    w[[4, 5], :] = 0.005
    m.wgate.upload(w)
    x = np.abs(synth.inputs(spec, 5, 3))
    got = m.forward(x)
    f0 = m.fallbacks()
    cert = m.forward(x, outputs=False)          # exact ties cannot be certified: fallback
    nfb = m.fallbacks() - f0
    want = oracle.moe(spec, w, synth.ln2(spec), m.host_mats, x)
    m.close()
    assert nfb == 3
    for r in (got, cert):
        assert r["topk"].tolist() == [[2, 7, 11, 4]] * 3
        assert np.array_equal(r["topk"], want["topk"])
        assert np.array_equal(bits(r["wt"]), bits(want["wt"]))


# ------------------------------------------------------------------ MoE, full size vs reference fixtures

@pytest.fixture(scope="module")
def full_q4(cpg):
    from cachepotato_amd import synth
    z = golden("moe_q4_b1_t1.npz")
    m = DeviceMoE(synth.CONFIGS["q4_b1"], max_T=512, device_gen=True, check_sha=True)
    assert m.sha_experts == str(z["sha_experts"]), "device-generated weights differ from the fixture's"
    yield m
    m.close()


def _oracle_mlp_1000(m):
    """The oracle's MoE output for all 1000 input vectors of m's workload (the reference's
    scalar Q4 numerics), computed once per layer object: one or_moe call per vector on a thread
    pool (the C calls release the GIL)."""
    if getattr(m, "_oracle_mlp", None) is None:
        from concurrent.futures import ThreadPoolExecutor
        from cachepotato_amd import synth
        from oracle.bindings import Oracle
        orc, spec = Oracle(), m.spec
        mats = m.host_mats if getattr(m, "host_mats", None) is not None else synth.experts_v4(spec)
        wg, ln2 = m.wgate_host, synth.ln2(spec)
        X = synth.inputs(spec, 0, 1000)
        with ThreadPoolExecutor(max_workers=min(16, os.cpu_count() or 1)) as ex:
            outs = list(ex.map(lambda v: orc.moe(spec, wg, ln2, mats, X[v:v + 1], threads=1)["mlp"][0],
                               range(1000)))
        m._oracle_mlp = np.stack(outs)
    return m._oracle_mlp


def _oracle_mlp_rows(m, X, threads):
    """The oracle's MoE output for every row of X (one or_moe call per token on a thread
    pool; a token's output does not depend on the other tokens of its call) at the reference's
    scalar (threads=1) or AVX2 (threads=8) Q4 numerics, cached on m per numerics."""
    cache = m.__dict__.setdefault("_oracle_rows", {})
    if threads not in cache:
        from concurrent.futures import ThreadPoolExecutor
        from cachepotato_amd import synth
        from oracle.bindings import Oracle
        orc, spec = Oracle(), m.spec
        mats = m.host_mats if getattr(m, "host_mats", None) is not None else synth.experts_v4(spec)
        wg, ln2 = m.wgate_host, synth.ln2(spec)
        with ThreadPoolExecutor(max_workers=min(16, os.cpu_count() or 1)) as ex:
            outs = list(ex.map(lambda v: orc.moe(spec, wg, ln2, mats, X[v:v + 1],
                                                 threads=threads)["mlp"][0], range(len(X))))
        cache[threads] = np.stack(outs)
    return cache[threads]


def _check_all_mlp(m, mlps, name):
    """Every vector's MoE output element by element against the oracle (the bar: normwise
    relative error per vector within MOE_TOL)."""
    want = _oracle_mlp_1000(m)
    errs = [rel_err(mlps[v], want[v]) for v in range(1000)]
    say(f"{name}: all 1000 outputs elementwise, worst rel err {max(errs):.2e}")
    assert max(errs) <= MOE_TOL


def _check_b1(m, name):
    from cachepotato_amd import synth
    from tests.golden.make_golden import sha
    z1, z8 = golden(f"moe_{name}_t1.npz"), golden(f"moe_{name}_t8.npz")
    assert sha(m.wgate_host) == str(z1["sha_wgate"])
    X = synth.inputs(m.spec, 0, 1000)
    topk, router, worst, mlps = [], [], 0.0, []
    for v in range(1000):
        r = m.forward(X[v:v + 1])
        topk.append(r["topk"][0])
        router.append(r["router"][0])
        mlps.append(r["mlp"][0])
        if v < 8:
            assert np.array_equal(bits(r["router"][0]), bits(z1["full_router"][v]))
            for z in (z1, z8):
                worst = max(worst, rel_err(r["mlp"][0], z["full_mlp"][v]))
        for z in (z1, z8):
            assert rel_err(np.sqrt((r["mlp"][0].astype(np.float64) ** 2).sum()),
                           z["mlp_norm"][v]) <= MOE_TOL
    assert np.array_equal(np.array(topk), z1["topk"]) and np.array_equal(z1["topk"], z8["topk"])
    assert sha(np.array(router)) == str(z1["sha_router"])
    say(f"{name}: 1000 vectors, routing bit-exact, worst mlp rel err {worst:.2e}")
    assert worst <= MOE_TOL
    _check_all_mlp(m, mlps, name)


def test_moe_q4_b1_golden(full_q4):
    _check_b1(full_q4, "q4_b1")


def _check_b1_certified(m, name):
    """The decode path as served (no logits asked for): top-8 of all 1000 vectors identical
    to the reference engine's, MoE outputs within 1e-3."""
    from cachepotato_amd import synth
    z1, z8 = golden(f"moe_{name}_t1.npz"), golden(f"moe_{name}_t8.npz")
    X = synth.inputs(m.spec, 0, 1000)
    f0 = m.fallbacks()
    topk, worst, mlps = [], 0.0, []
    for v in range(1000):
        r = m.forward(X[v:v + 1], outputs=False)
        topk.append(r["topk"][0])
        mlps.append(r["mlp"][0])
        if v < 8:
            for z in (z1, z8):
                worst = max(worst, rel_err(r["mlp"][0], z["full_mlp"][v]))
        for z in (z1, z8):
            assert rel_err(np.sqrt((r["mlp"][0].astype(np.float64) ** 2).sum()),
                           z["mlp_norm"][v]) <= MOE_TOL
    nfb = m.fallbacks() - f0
    assert np.array_equal(np.array(topk), z1["topk"])
    say(f"{name} certified: 1000 vectors, top-8 bit-exact, {nfb} fallbacks, "
        f"worst mlp rel err {worst:.2e}")
    assert worst <= MOE_TOL
    _check_all_mlp(m, mlps, name + " certified")


def test_moe_q4_b1_golden_certified(full_q4):
    _check_b1_certified(full_q4, "q4_b1")


def test_moe_q4_b1_golden_refined(full_q4):
    """Every certificate failed on purpose, so each token takes the refined step (the exact
    chains of the experts whose bounds reach the top 8, then the order certified again): top-8
    of 300 vectors identical to the reference engine's, outputs within 1e-3. The step must settle nearly every token without the exact chains of all rows."""
    from cachepotato_amd import synth
    z1, z8 = golden("moe_q4_b1_t1.npz"), golden("moe_q4_b1_t8.npz")
    m = full_q4
    X = synth.inputs(m.spec, 0, 300)
    f0, x0 = m.fallbacks(), m.exact_routings()
    topk, worst = [], 0.0
    with route_mode(ROUTE_MODES["refine"]):
        for v in range(300):
            r = m.forward(X[v:v + 1], outputs=False)
            topk.append(r["topk"][0])
            if v < 8:
                for z in (z1, z8):
                    worst = max(worst, rel_err(r["mlp"][0], z["full_mlp"][v]))
    nfb, nex = m.fallbacks() - f0, m.exact_routings() - x0
    assert nfb == 300
    assert np.array_equal(np.array(topk), z1["topk"][:300])
    say(f"q4_b1 refined: 300 vectors, top-8 bit-exact, {nex} needed every chain exact, "
        f"worst mlp rel err {worst:.2e}")
    assert worst <= MOE_TOL
    assert nex <= 15


def test_moe_q8_b1_golden(cpg):
    from cachepotato_amd import synth
    z = golden("moe_q8_b1_t1.npz")
    m = DeviceMoE(synth.CONFIGS["q8_b1"], max_T=1, device_gen=True, check_sha=True)
    assert m.sha_experts == str(z["sha_experts"])
    try:
        _check_b1(m, "q8_b1")
        _check_b1_certified(m, "q8_b1")
    finally:
        m.close()


def _check_batched(m, name, tight=None):
    from cachepotato_amd import synth
    from tests.golden.make_golden import sha, PREFILL_KEEP
    z1, z8 = golden(f"moe_{name}_t1.npz"), golden(f"moe_{name}_t8.npz")
    assert sha(m.wgate_host) == str(z1["sha_wgate"])
    calls = z1["calls"]
    X = synth.inputs(m.spec, 0, int(calls.max()) + 1)
    topk, router, norms, worst, mlps = [], [], [], 0.0, []
    for ci, call in enumerate(calls):
        r = m.forward(X[call])
        topk.append(r["topk"])
        router.append(r["router"])
        mlps.append(r["mlp"])
        norms.append(np.sqrt((r["mlp"].astype(np.float64) ** 2).sum(1)))
        if ci == 0:
            keep = PREFILL_KEEP if name == "q4_prefill512" else list(range(len(call)))
            assert np.array_equal(r["topk"][keep], z1["full_topk"])
            assert np.array_equal(bits(r["router"][keep]), bits(z1["full_router"]))
            for z in (z1, z8):
                worst = max(worst, rel_err(r["mlp"][keep], z["full_mlp"]))
        say(f"{name} call {ci}: {len(call)} tokens, {m.distinct()} distinct experts")
    assert np.array_equal(np.concatenate(topk), z1["topk"])
    assert sha(np.concatenate(router)) == str(z1["sha_router"])
    for z in (z1, z8):
        assert rel_err(np.concatenate(norms), z["mlp_norm"]) <= MOE_TOL
    say(f"{name}: routing bit-exact, worst mlp rel err {worst:.2e}")
    assert worst <= (MOE_TOL if tight is None else tight)
    _check_rows_elementwise(m, X, calls, mlps, name, tight)


def _check_rows_elementwise(m, X, calls, mlps, name, tight=None):
    """Every token of every call element by element against the oracle at both reference
    numerics: per token, max|gpu - ref| / max|ref| within the bar."""
    rows = np.concatenate([np.asarray(c) for c in calls])
    got = np.concatenate(mlps)
    bar = MOE_TOL if tight is None else tight
    for threads in (1, 8):
        want = _oracle_mlp_rows(m, X, threads)[rows]
        errs = np.array([rel_err(got[i], want[i]) for i in range(len(rows))])
        say(f"{name}: all {len(rows)} tokens elementwise (threads={threads}), worst rel err "
            f"{errs.max():.2e} at token {int(rows[errs.argmax()])}")
        assert errs.max() <= bar, (threads, int(rows[errs.argmax()]))


def test_moe_q4_b16_zipf_golden(cpg):
    from cachepotato_amd import synth
    m = DeviceMoE(synth.CONFIGS["q4_b16_zipf"], max_T=16, device_gen=True)
    try:
        _check_batched(m, "q4_b16_zipf")
        # the same batches through certified routing
        z1, z8 = golden("moe_q4_b16_zipf_t1.npz"), golden("moe_q4_b16_zipf_t8.npz")
        X = synth.inputs(m.spec, 0, int(z1["calls"].max()) + 1)
        f0 = m.fallbacks()
        topk, norms, mlps = [], [], []
        for call in z1["calls"]:
            r = m.forward(X[call], outputs=False)
            topk.append(r["topk"])
            mlps.append(r["mlp"])
            norms.append(np.sqrt((r["mlp"].astype(np.float64) ** 2).sum(1)))
        assert np.array_equal(np.concatenate(topk), z1["topk"])
        for z in (z1, z8):
            assert rel_err(np.concatenate(norms), z["mlp_norm"]) <= MOE_TOL
        say(f"q4_b16_zipf certified: top-8 bit-exact, {m.fallbacks() - f0} exact fallbacks")
        _check_rows_elementwise(m, X, z1["calls"], mlps, "q4_b16_zipf certified")
    finally:
        m.close()


@pytest.mark.parametrize("experts", ["mfma", "gemv"])
def test_moe_q4_prefill512_golden(cpg, experts):
    """The 512-token prefill chunk against the reference engine's goldens through both expert
    paths: the MFMA grouped GEMMs (the default from 64 tokens) and the grouped GEMVs."""
    import cachepotato_amd as C
    from cachepotato_amd import synth
    m = DeviceMoE(synth.CONFIGS["q4_prefill512"], max_T=512, device_gen=True)
    try:
        with expert_mode(C.EXPERTS_MFMA if experts == "mfma" else C.EXPERTS_GEMV):
            _check_batched(m, "q4_prefill512", tight=SPLIT_TOL)
    finally:
        m.close()


@pytest.mark.parametrize("T", [8, 16, 17, 64, 100])
def test_moe_small_mfma_vs_oracle(cpg, oracle, small, T):
    """The MFMA grouped GEMMs forced at small token counts (chunks of 1..64 tokens, Q4 and
    Q8 weights) against the oracle at both reference numerics; up to 16 tokens they run the
    one-tile kernels (64 gate/up rows per workgroup; at top-4 up to 64 pairs, so in two groups of
    wavefronts)."""
    import cachepotato_amd as C
    from cachepotato_amd import synth
    spec = small.spec
    x = synth.inputs(spec, 5000 + T, T)
    with expert_mode(C.EXPERTS_MFMA):
        got = small.forward(x)
    with expert_mode(C.EXPERTS_GEMV):
        gemv = small.forward(x)
    assert np.array_equal(got["topk"], gemv["topk"])
    for threads in (1, 8):
        want = oracle.moe(spec, small.wgate_host, synth.ln2(spec), small.host_mats, x,
                          threads=threads)
        assert np.array_equal(got["topk"], want["topk"])
        e, eg = rel_err(got["mlp"], want["mlp"]), rel_err(gemv["mlp"], want["mlp"])
        say(f"{spec.enc} T={T} threads={threads}: mfma mlp rel err {e:.2e} (gemv {eg:.2e})")
        assert e <= SPLIT_TOL


@pytest.mark.parametrize("T", [2, 7, 16])
def test_moe_small_certified_batch_invariance(small, T):
    """Certified calls of 2 to 16 tokens (the one-tile GEMMs, reading the selections): a token's
    outputs do not depend on the batch it is in, bit for bit, and agree with the grouped GEMVs
    within rounding."""
    import cachepotato_amd as C
    from cachepotato_amd import synth
    x = synth.inputs(small.spec, 7000, 16)
    ref = small.forward(x, outputs=False)
    got = small.forward(x[16 - T:], outputs=False)
    for k in ("topk", "wt", "mlp"):
        assert np.array_equal(got[k].view(np.uint32), ref[k][16 - T:].view(np.uint32)), k
    with expert_mode(C.EXPERTS_GEMV):
        gemv = small.forward(x[16 - T:], outputs=False)
    assert np.array_equal(got["topk"], gemv["topk"])
    assert rel_err(got["mlp"], gemv["mlp"]) <= SPLIT_TOL


@pytest.mark.parametrize("enc", [4, 8])
def test_moe_certified_batches_full_width(cpg, oracle, enc):
    """Certified calls of 2 to 16 tokens at the model's width (D = 2048, F = 768, top-8: 16 and 6 or
    32 and 12 stages of the one-tile GEMMs, past every ring's depth) against the oracle. A token's
    outputs do not depend on the batch it is in, bit for bit: up to 8 tokens (64 pairs) two groups
    of wavefronts sum its blocks, from 9 on one group in their order."""
    from cachepotato_amd import synth
    spec = synth.MoESpec(D=2048, E=16, K=8, F=768, enc=enc)
    m = DeviceMoE(spec, max_T=16)
    try:
        x = synth.inputs(spec, 7300, 16)
        want = oracle.moe(spec, m.wgate_host, synth.ln2(spec), m.host_mats, x, threads=8)
        got = {T: m.forward(x[:T], outputs=False) for T in (2, 3, 7, 8, 9, 13, 16)}
        for T, g in got.items():
            assert np.array_equal(g["topk"], want["topk"][:T]), T
            e = max(rel_err(g["mlp"][t], want["mlp"][t]) for t in range(T))
            say(f"certified enc={enc} T={T}: worst token {e:.2e}")
            assert e <= SPLIT_TOL, T
            for k in ("topk", "wt", "mlp"):
                assert np.array_equal(g[k].view(np.uint32), got[16][k][:T].view(np.uint32)), (T, k)
    finally:
        m.close()


@pytest.mark.parametrize("T", [17, 32, 44, 45])
def test_moe_small_crowded_experts_vs_oracle(cpg, oracle, small, T):
    """Every token takes the same experts, so each has T tokens: chunks of 16 (17 = one row past a
    chunk, 32 = two whole ones, 44 = the last call with them at 16 experts, top-4) and a chunk of
    64 (45), against the oracle."""
    from cachepotato_amd import synth
    spec = small.spec
    x = np.repeat(synth.inputs(spec, 7100, 1), T, 0)
    x = (x + 1e-3 * synth.inputs(spec, 7200, T)).astype(np.float32)
    got = small.forward(x)
    want = oracle.moe(spec, small.wgate_host, synth.ln2(spec), small.host_mats, x, threads=8)
    assert np.array_equal(got["topk"], want["topk"])
    assert np.bincount(got["topk"].ravel()).max() > 16
    for t in range(T):
        assert rel_err(got["mlp"][t], want["mlp"][t]) <= SPLIT_TOL, t


# ------------------------------------------------------------------ full-size properties

def test_moe_batch_invariance_and_determinism(full_q4):
    """Below 8 tokens (the grouped GEMVs) a token's outputs do not depend on the batch it is
    in, bit for bit; from 8 tokens the experts run as MFMA GEMMs on hi/lo halves of xn, whose
    outputs agree with the one-token path within 1e-5 while the routing stays bit-identical.
    Reruns are identical (no atomics in any sum)."""
    from cachepotato_amd import synth
    X = synth.inputs(full_q4.spec, 4000, 40)
    for T in (7, 40):
        batch = full_q4.forward(X[:T])
        again = full_q4.forward(X[:T])
        for k in batch:
            assert np.array_equal(batch[k].view(np.uint32), again[k].view(np.uint32)), (T, k)
        for t in (0, T // 2, T - 1):
            one = full_q4.forward(X[t:t + 1])
            for k in one:
                if T < 8 or k != "mlp":
                    assert np.array_equal(one[k][0].view(np.uint32),
                                          batch[k][t].view(np.uint32)), (T, k, t)
                else:
                    assert rel_err(batch[k][t], one[k][0]) <= 1e-5, (T, k, t)


def test_moe_rejects_bad_shapes(cpg):
    import cachepotato_amd as C
    L = C.lib()
    assert not L.cpg_moe_ws_create(2048, 300, 8, 768, 4)      # E > 256
    assert not L.cpg_moe_ws_create(2048, 128, 0, 768, 4)      # K = 0
    assert L.cpg_repack(4, None, None, 100, 64) == -1          # rows not a multiple of 64


# ------------------------------------------------------------------ qwen3_mm: one matrix

@pytest.mark.parametrize("enc,n_in,n_out", [(0, 2048, 128), (0, 96, 7), (4, 2048, 768),
                                            (4, 768, 2048), (8, 2048, 768), (8, 4096, 100)])
def test_mm(cpg, oracle, enc, n_in, n_out):
    """cpg_mm against matmul_wx / matmul_wx_q4 / matmul_wx_q8 (kernels.c:84-95, :514-540,
    :368-396) on v4-layout weights: f32 bit-exact (the same serial chain), Q4/Q8 within
    fp32 accumulation error of both of the reference's Q4 numerics."""
    from cachepotato_amd import synth
    rng = np.random.default_rng(n_in * 31 + n_out + enc)
    x = rng.standard_normal(n_in).astype(np.float32)
    if enc == 0:
        w = (rng.standard_normal((n_out, n_in)) * 0.02).astype(np.float32)
    else:
        w = oracle.encode(enc, (rng.standard_normal(n_out * n_in) * 0.02).astype(np.float32))
    wd, xd, od = cpg.to_device(w), cpg.to_device(x), cpg.DeviceBuffer(n_out * 4)
    cpg.check(cpg.lib().cpg_mm(enc, wd.ptr, xd.ptr, n_in, n_out, od.ptr), "cpg_mm")
    got = od.download(np.float32, n_out)
    if enc == 0:
        want = oracle.matmul(0, w, x, n_in, n_out)
        assert np.array_equal(bits(got), bits(want))
    else:
        for threads in (1, 8):
            want = oracle.matmul(enc, w, x, n_in, n_out, threads=threads)
            e = rel_err(got, want)
            assert e <= 1e-5, (threads, e)
    say(f"mm enc={enc} {n_out}x{n_in}: ok")


@pytest.mark.parametrize("name,T", [("small_q4", 1), ("small_q4", 5), ("small_q8", 1),
                                    ("q4_b1", 1)])
def test_moe_forward_res_equals_forward_plus_residual(cpg, name, T):
    """cpg_moe_forward_res (the residual folded into the down projection for one token, a
    separate residual kernel otherwise) gives x + (attn + mlp) with exactly the bits of
    cpg_moe_forward followed by that sum, and leaves the mlp scratch at zero."""
    from cachepotato_amd import synth
    spec = synth.CONFIGS[name] if name in synth.CONFIGS else synth.SMALL[name]
    m = DeviceMoE(spec, max_T=max(T, 1), device_gen=name == "q4_b1")
    try:
        x = synth.inputs(spec, 0, T)
        attn = (synth.inputs(spec, 1, T) * 0.1).astype(np.float32)
        ref = m.forward(x, attn=attn, outputs=False)
        want = (x + (attn + ref["mlp"])).astype(np.float32)
        got, tk, mlp_after = m.forward_res(x, attn)
        assert np.array_equal(tk, ref["topk"])
        assert np.array_equal(bits(got), bits(want))
        assert not mlp_after.any()
    finally:
        m.close()


@pytest.mark.parametrize("name", ["q4_b1", "q8_b1"])
@pytest.mark.parametrize("mode", ["auto", "fallback"])
def test_moe_fused_equals_separate_kernels(cpg, name, mode):
    """One token through the fused kernel (routing, experts and combine in one launch, the
    phases handing over through tagged data) gives the bits of the three separate kernels:
    top-K, weights, mlp, and with the residual folded in; with every certification forced to
    fail it takes the exact fallback and still agrees. No wait may time out."""
    import cachepotato_amd as C
    from cachepotato_amd import synth
    spec = synth.CONFIGS[name]
    m = DeviceMoE(spec, max_T=1, device_gen=True)
    try:
        X = synth.inputs(spec, 7000, 48)
        A = (synth.inputs(spec, 8000, 48) * 0.05).astype(np.float32)
        f0 = m.fallbacks()
        with route_mode(C.ROUTE_FORCE_FALLBACK if mode == "fallback" else C.ROUTE_AUTO):
            for i in range(len(X)):
                with fused_mode(False):
                    sep = m.forward(X[i:i + 1], attn=A[i:i + 1], outputs=False)
                    sep_res = m.forward_res(X[i:i + 1], A[i:i + 1])
                with fused_mode(True):
                    fus = m.forward(X[i:i + 1], attn=A[i:i + 1], outputs=False)
                    fus_res = m.forward_res(X[i:i + 1], A[i:i + 1])
                for k in ("topk", "wt", "mlp"):
                    assert np.array_equal(bits(fus[k]), bits(sep[k])), (i, k)
                assert np.array_equal(bits(fus_res[0]), bits(sep_res[0])), i
                assert np.array_equal(fus_res[1], sep_res[1]), i
        nfb = m.fallbacks() - f0
        say(f"{name} {mode}: 48 tokens fused == separate, {nfb} exact fallbacks")
        if mode == "fallback":
            assert nfb == 4 * 48          # every call of both paths, with and without residual
        assert m.status() == 0
    finally:
        m.close()
