"""The work this framework is timed on, through the C ABI of include/cpg.h.

Three kinds of case, all at the geometry the framework is built for (hidden 2048, 32 query and
4 key/value heads of 128, 128 experts top-8 of 768, vocabulary 151936, Q4_0 or Q8_0 weights):

  moe     the MoE half of a layer for T tokens (cpg_moe_forward), over L layers of their own
          weights: T = 1 is a decode step, 2..16 a decode batch, 17..512 a prompt's chunk;
  attn    the attention half for T tokens at position pos of a cache that earlier tokens have
          filled (cpg_attn_forward), over L layers: T = 1 is a decode step, more is a prompt
          or a chat turn appended to its conversation;
  model   embedding, L layers (cpg_attn_forward, cpg_moe_forward_res) and the head
          (cpg_head_next): one decode step replayed as a graph (T = 1), as a decoding program
          runs it, or one prompt's prefill.

Several layers in a case keep a pass's weights out of the caches, where a model of 48 layers
would not find them either. Prompts run in chunks of at most 512 tokens and positions go up to
8191, the limits of cp_open. Weights are Gaussian, encoded as the model's file holds them and
brought into the device layout by cpg_repack, as the loader does.
"""
import ctypes
import math

import torch

import cachepotato_amd as C

D, H, KV, HD, E, K, F, V = 2048, 32, 4, 128, 128, 8, 768, 151936
NQKV = (H + 2 * KV) * HD
EPS, THETA, SIGMA = 1e-6, 1e6, 0.02
MAX_POS = 8192            # positions a model can be opened with
EMB_ROWS = 4096           # rows of the embedding table a case draws its ids from
Q4, Q8 = C.ENC_Q4, C.ENC_Q8
BITS = {Q4: 4.5, Q8: 8.5}                       # per weight, block scales included


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # one step of greedy decoding early in a conversation: what a chat spends most time on
        {"name": "decode_q4_p200", "kind": "model", "T": 1, "pos": 200, "enc": Q4, "L": 12},
        # the same with an all-Q8_0 file, near the end of the default context of 2048
        {"name": "decode_q8_p1900", "kind": "model", "T": 1, "pos": 1900, "enc": Q8, "L": 6},
        # an ordinary prompt, up to its first logits
        {"name": "prefill_q4_t96", "kind": "model", "T": 96, "pos": 0, "enc": Q4, "L": 4},
        # the MoE half of a decode step, Q8_0 experts
        {"name": "moe_q8_t1", "kind": "moe", "T": 1, "enc": Q8, "skew": False, "L": 8},
        # a few sequences decoded together, or the tokens of a drafted continuation
        {"name": "moe_q4_t4", "kind": "moe", "T": 4, "enc": Q4, "skew": False, "L": 4},
        # a full decode batch whose tokens favour the same experts (Zipf)
        {"name": "moe_q4_t16_skew", "kind": "moe", "T": 16, "enc": Q4, "skew": True, "L": 3},
        # a short question
        {"name": "moe_q4_t45", "kind": "moe", "T": 45, "enc": Q4, "skew": False, "L": 2},
        # a longer prompt, Q8_0 experts
        {"name": "moe_q8_t160", "kind": "moe", "T": 160, "enc": Q8, "skew": False, "L": 1},
        # a whole chunk of a long prompt
        {"name": "moe_q4_t512", "kind": "moe", "T": 512, "enc": Q4, "skew": False, "L": 1},
        # one token far into a long conversation
        {"name": "attn_q4_t1_p6000", "kind": "attn", "T": 1, "pos": 6000, "enc": Q4, "L": 8},
        # a short chat turn appended to its conversation
        {"name": "attn_q8_t21_p700", "kind": "attn", "T": 21, "pos": 700, "enc": Q8, "L": 4},
        # the last chunk of a prompt of 4096 tokens
        {"name": "attn_q4_t512_p3584", "kind": "attn", "T": 512, "pos": 3584, "enc": Q4, "L": 1},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _moe_layers(T):
    return 8 if T == 1 else 4 if T < 12 else 2 if T < 64 else 1


def draw(rng):
    enc = rng.choice([Q4, Q4, Q8])
    kind = rng.choice(["moe", "moe", "moe", "attn", "attn", "model"])
    if kind == "moe":
        T = _log_int(rng, 1, 512)
        return {"kind": kind, "T": T, "enc": enc, "skew": rng.random() < 0.4,
                "L": _moe_layers(T)}
    # T * pos is kept to what the largest listed chunk has
    decode = rng.random() < 0.4
    T = 1 if decode else _log_int(rng, 2, 512 if kind == "attn" else 128)
    if not decode and rng.random() < 0.5:
        pos = 0
    else:
        pos = _log_int(rng, 1, min(MAX_POS - T, 3584 * 512 // T))
    if kind == "attn":
        return {"kind": kind, "T": T, "pos": pos, "enc": enc, "L": 8 if T == 1 else 4 if T < 64 else 1}
    return {"kind": kind, "T": T, "pos": min(pos, 4000), "enc": enc, "L": 6 if T == 1 else 3}


# ---------------------------------------------------------------- inputs

def _gen(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000003 + stream * 7919 + 17)
    return g


def _normal(seed, stream, *shape, sigma=1.0):
    return torch.randn(*shape, generator=_gen(seed, stream), device="cuda") * sigma


def _blocks(enc, w):
    """float values (n, 32) as Q4_0 / Q8_0 blocks of the file format: (n, 18 or 34) bytes."""
    d = (w.abs().amax(1, keepdim=True) / (8.0 if enc == Q4 else 127.0)).to(torch.float16)
    df = d.float()
    q = w * torch.where(df != 0, 1.0 / df, torch.zeros_like(df))
    scale = d.view(torch.uint8).reshape(-1, 2)
    if enc == Q8:
        return torch.cat([scale, q.round().clamp_(-127, 127).to(torch.int8).view(torch.uint8)], 1)
    q = q.round().clamp_(-8, 7).to(torch.int32) & 15
    return torch.cat([scale, (q[:, :16] | q[:, 16:] << 4).to(torch.uint8)], 1)


def _values(enc, b):
    """the blocks' values in 64 bits, (n, 32)"""
    d = b[:, :2].contiguous().view(torch.float16).double()
    if enc == Q8:
        return d * b[:, 2:].contiguous().view(torch.int8).double()
    n = b[:, 2:].int()
    q = torch.cat([n & 15, n >> 4], 1)
    return d * torch.where(q > 7, q - 16, q).double()


def _matrix(enc, seed, stream, rows, cols, sigma):
    """a random matrix in the file's layout: (rows * cols / 32, 18 or 34) bytes"""
    return _blocks(enc, _normal(seed, stream, rows * cols // 32, 32, sigma=sigma))


def _repack(enc, mats, dst, offset=0):
    """(blocks, rows, cols) one after another into the device layout at dst + offset"""
    torch.cuda.synchronize()                     # the library runs on a stream of its own
    for b, rows, cols in mats:
        C.check(C.lib().cpg_repack(enc, dst.data_ptr() + offset, b.data_ptr(), rows, cols), "repack")
        offset += C.lib().cpg_matrix_bytes(enc, rows, cols)
    C.sync()


def _gain(seed, stream, n):
    return 1.0 + _normal(seed, stream, n, sigma=0.1)


ZIPF = [r ** -1.1 for r in range(1, E + 1)]
ZIPF = [p / sum(ZIPF) for p in ZIPF]
SKEW, SHIFT = 0.011, 1.0                        # of the router rows, of the inputs


def _direction(seed):
    c = _normal(seed, 3, D).double()
    return c / c.norm()


def _moe_weights(enc, seed, layer, skew, out_sigma):
    """one layer's router, norm gain and experts, as the file holds them"""
    s = 100 * (layer + 1)
    wgate = _normal(seed, s, E, D, sigma=SIGMA)
    if skew:
        # inputs shifted along c then add a Zipf-like bias to the logits, the layer's own order
        c = _direction(seed)
        order = torch.randperm(E, generator=_gen(seed, s + 1), device="cuda")
        bias = SKEW * torch.tensor(ZIPF, device="cuda").double().log()[order]
        w = wgate.double()
        wgate = (w + (bias - w @ c)[:, None] * c).float()
    return dict(wgate=wgate.contiguous(), ln2=_gain(seed, s + 2, D),
                gate=_matrix(enc, seed, s + 3, E * F, D, SIGMA),
                up=_matrix(enc, seed, s + 4, E * F, D, SIGMA),
                down=_matrix(enc, seed, s + 5, E * D, F, out_sigma))


def _attn_weights(enc, seed, layer, out_sigma):
    s = 100 * (layer + 1) + 50
    return dict(ln1=_gain(seed, s, D), qn=_gain(seed, s + 1, HD), kn=_gain(seed, s + 2, HD),
                wqkv=_matrix(enc, seed, s + 3, NQKV, D, SIGMA),
                wo=_matrix(enc, seed, s + 4, D, H * HD, out_sigma))


def _cache(seed, layer, pos):
    """keys and values of `pos` earlier tokens, of the size normed keys and values have"""
    s = 100 * (layer + 1) + 60
    return _normal(seed, s, pos, KV * HD), _normal(seed, s + 1, pos, KV * HD, sigma=0.9)


def _tokens(case, seed):
    """the T tokens' residual stream and the attention's contribution to it"""
    T = case["T"]
    x, attn = _normal(seed, 1, T, D), _normal(seed, 2, T, D, sigma=0.2)
    if case.get("skew"):
        x = (x.double() + SHIFT * math.sqrt(D) * _direction(seed)).float()
    return x, attn


def _model_ids(case, seed):
    return torch.randint(EMB_ROWS, (case["T"],), generator=_gen(seed, 4), device="cuda",
                         dtype=torch.int32)


def _out_sigma(case):
    """the matrices that write into the residual stream of a 48-layer model are smaller"""
    return SIGMA / math.sqrt(96) if case["kind"] == "model" else SIGMA


# ---------------------------------------------------------------- what a program keeps

_rope = {}


def _rope_table(n):
    """the rotation pairs of positions 0..n-1, computed once for the longest asked for"""
    if _rope.get("n", 0) < n:
        t = torch.empty(n * HD)
        C.check(C.lib().cpg_rope_table(THETA, HD, n, t.data_ptr()), "rope")
        _rope.update(n=n, t=t.cuda())
    return _rope["t"]


class _State:
    """Buffers, layers and workspaces of one case; closed when the program drops it."""

    def __init__(self, case):
        C.init(0)
        self.case, self.keep, self.moe_ws, self.attn_ws, self.graph = case, [], None, None, None

    def hold(self, *t):
        self.keep.extend(t)
        return t[0]

    def moe_layer(self, enc, w):
        lib = C.lib()
        per, mg = lib.cpg_expert_bytes(enc, D, F), lib.cpg_matrix_bytes(enc, F, D)
        md = lib.cpg_matrix_bytes(enc, D, F)
        ex = self.hold(torch.empty(E * per, dtype=torch.uint8, device="cuda"))
        parts = [w[k].view(E, -1, w[k].shape[1]) for k in ("gate", "up", "down")]
        torch.cuda.synchronize()
        for e in range(E):
            base = ex.data_ptr() + e * per
            for p, off, rows, cols in zip(parts, (0, mg, 2 * mg), (F, F, D), (D, D, F)):
                C.check(lib.cpg_repack(enc, base + off, p[e].data_ptr(), rows, cols), "repack")
        C.sync()
        assert 2 * mg + md == per
        self.hold(w["wgate"], w["ln2"])
        return C.MoELayer(D, E, K, F, enc, EPS, w["ln2"].data_ptr(), w["wgate"].data_ptr(),
                          ex.data_ptr())

    def attn_layer(self, enc, w, n):
        lib = C.lib()
        qkv = self.hold(torch.empty(lib.cpg_matrix_bytes(enc, NQKV, D), dtype=torch.uint8, device="cuda"))
        wo = self.hold(torch.empty(lib.cpg_matrix_bytes(enc, D, H * HD), dtype=torch.uint8, device="cuda"))
        _repack(enc, [(w["wqkv"], NQKV, D)], qkv)
        _repack(enc, [(w["wo"], D, H * HD)], wo)
        rope = self.hold(_rope_table(n))
        self.hold(w["ln1"], w["qn"], w["kn"])
        return C.AttnLayer(D, H, KV, HD, THETA, EPS, enc, w["ln1"].data_ptr(), w["qn"].data_ptr(),
                           w["kn"].data_ptr(), qkv.data_ptr(), wo.data_ptr(), rope.data_ptr(), n)

    def caches(self, case, seed):
        """per layer a key and a value cache, with room for the tokens decoded next"""
        T, pos, L = case["T"], case["pos"], case["L"]
        self.cap = min(MAX_POS, pos + T + 128)
        self.kc = torch.zeros(L, self.cap, KV * HD, device="cuda")
        self.vc = torch.zeros(L, self.cap, KV * HD, device="cuda")
        for l in range(L):
            self.kc[l, :pos], self.vc[l, :pos] = _cache(seed, l, pos)

    def __del__(self):
        lib = C.lib()
        C.sync()
        if self.graph:
            lib.cpg_graph_destroy(self.graph)
        if self.moe_ws:
            lib.cpg_moe_ws_destroy(self.moe_ws)
        if self.attn_ws:
            lib.cpg_attn_ws_destroy(self.attn_ws)


def _made(ptr):
    if not ptr:
        raise C.CPGError(C.last_error())
    return ptr


def prepare(case, seed):
    s, kind, T, L, enc = _State(case), case["kind"], case["T"], case["L"], case["enc"]
    lib = C.lib()
    if kind != "attn":
        s.moe_ws = _made(lib.cpg_moe_ws_create(D, E, K, F, T))
        s.moe = [s.moe_layer(enc, _moe_weights(enc, seed, l, case.get("skew"), _out_sigma(case)))
                 for l in range(L)]
        s.topk = torch.empty(L, T, K, dtype=torch.int32, device="cuda")
    if kind != "moe":
        s.attn_ws = _made(lib.cpg_attn_ws_create(D, H, KV, HD, T))
        s.caches(case, seed)
        s.att = [s.attn_layer(enc, _attn_weights(enc, seed, l, _out_sigma(case)), s.cap) for l in range(L)]
    if kind == "moe":
        s.x, s.attn = _tokens(case, seed)
        s.wt = torch.empty(L, T, K, device="cuda")
        s.mlp = torch.empty(L, T, D, device="cuda")
    elif kind == "attn":
        s.x = _normal(seed, 1, T, D)
        s.out = torch.empty(L, T, D, device="cuda")
    else:
        s.ids = _model_ids(case, seed)
        s.embed = _matrix(Q8, seed, 5, EMB_ROWS, D, 1.0)
        s.head = torch.empty(lib.cpg_matrix_bytes(Q8, V, D), dtype=torch.uint8, device="cuda")
        _repack(Q8, [(_matrix(Q8, seed, 6, V, D, SIGMA), V, D)], s.head)
        s.norm = _gain(seed, 7, D)
        s.x, s.attn = torch.empty(T, D, device="cuda"), torch.empty(T, D, device="cuda")
        s.mlp = torch.zeros(T, D, device="cuda")
        s.logits = torch.empty(V, device="cuda")
        s.tok = torch.zeros(1, dtype=torch.int32, device="cuda")
        s.pos = torch.tensor([case["pos"]], dtype=torch.int32, device="cuda")
        s.scratch = torch.zeros(lib.cpg_head_scratch_bytes(V), dtype=torch.uint8, device="cuda")
        if T == 1:
            torch.cuda.synchronize()
            C.check(lib.cpg_capture_begin(), "capture")
            _model_pass(s)
            s.graph = _made(lib.cpg_capture_end())
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------- one pass

def _model_pass(s):
    """enqueue embedding, layers and head for the case's T tokens"""
    lib, T, pos = C.lib(), s.case["T"], s.case["pos"]
    x, attn = s.x.data_ptr(), s.attn.data_ptr()
    rc = lib.cpg_embed_rows(Q8, s.embed.data_ptr(), EMB_ROWS, D, s.ids.data_ptr(), T, x)
    for l in range(s.case["L"]):
        kc, vc = s.kc[l].data_ptr(), s.vc[l].data_ptr()
        if T == 1:
            rc = rc or lib.cpg_attn_forward_at(ctypes.byref(s.att[l]), x, 1, s.pos.data_ptr(), kc, vc,
                                               s.cap, attn, s.attn_ws)
        else:
            rc = rc or lib.cpg_attn_forward(ctypes.byref(s.att[l]), x, T, pos, kc, vc, s.cap, attn,
                                            s.attn_ws)
        rc = rc or lib.cpg_moe_forward_res(ctypes.byref(s.moe[l]), x, attn, T, s.topk[l].data_ptr(),
                                           s.mlp.data_ptr(), s.moe_ws)
    rc = rc or lib.cpg_head_next(Q8, s.head.data_ptr(), D, V, x + 4 * D * (T - 1), s.norm.data_ptr(),
                                 EPS, s.logits.data_ptr(), s.tok.data_ptr(), Q8, s.embed.data_ptr(),
                                 EMB_ROWS, s.scratch.data_ptr())
    C.check(rc, "model pass")


def run(s):
    lib, c = C.lib(), s.case
    T, L = c["T"], c["L"]
    if c["kind"] == "moe":
        # mlp is accumulated into, so each pass starts it at zero
        C.check(lib.cpg_memset(s.mlp.data_ptr(), 0, 4 * L * T * D), "memset")
        x, attn, mlp, topk, wt, ws = (s.x.data_ptr(), s.attn.data_ptr(), s.mlp.data_ptr(),
                                      s.topk.data_ptr(), s.wt.data_ptr(), s.moe_ws)
        for l in range(L):
            C.check(lib.cpg_moe_forward(ctypes.byref(s.moe[l]), x, attn, T, None, None,
                                        topk + 4 * l * T * K, wt + 4 * l * T * K,
                                        mlp + 4 * l * T * D, ws), "cpg_moe_forward")
        return {"mlp": s.mlp, "topk": s.topk, "wt": s.wt}
    pos, cap = c["pos"], s.cap
    rows = {"k": s.kc[:, pos:pos + T], "v": s.vc[:, pos:pos + T]}
    if c["kind"] == "attn":
        x, kc, vc, out = s.x.data_ptr(), s.kc.data_ptr(), s.vc.data_ptr(), s.out.data_ptr()
        row = 4 * cap * KV * HD
        for l in range(L):
            C.check(lib.cpg_attn_forward(ctypes.byref(s.att[l]), x, T, pos, kc + l * row,
                                         vc + l * row, cap, out + 4 * l * T * D, s.attn_ws),
                    "cpg_attn_forward")
        return dict(rows, attn=s.out)
    if s.graph:
        C.check(lib.cpg_graph_launch(s.graph), "cpg_graph_launch")
    else:
        _model_pass(s)
    return dict(rows, logits=s.logits, topk=s.topk)


# ---------------------------------------------------------------- what a pass cannot do without

def _distinct(T, skew):
    """experts that T tokens choose between them: a token takes each expert with the chance
    1 - exp(-m p), m so that it takes K"""
    p = ZIPF if skew else [1.0 / E] * E
    lo, hi = 0.0, 1e4
    for _ in range(60):
        m = (lo + hi) / 2
        lo, hi = (m, hi) if sum(1 - math.exp(-m * q) for q in p) < K else (lo, m)
    return sum(1 - math.exp(-m * q * T) for q in p)


def work(case):
    T, L, b = case["T"], case["L"], BITS[case["enc"]] / 8
    total, flops = 0.0, 0.0
    if case["kind"] != "attn":
        weights = _distinct(T, case.get("skew")) * 3 * F * D * b + 4 * E * D + 4 * D
        total += L * (weights + 4 * T * (3 * D + 2 * K))
        flops += L * 2.0 * T * (K * 3 * F * D + E * D)
    if case["kind"] != "moe":
        pos = case["pos"]
        total += L * ((NQKV * D + D * H * HD) * b + 4 * (D + 2 * HD) + 8 * KV * HD * (pos + T) +
                      8 * KV * HD * T + 4 * T * (2 * D + HD))
        flops += L * (2.0 * T * (NQKV * D + D * H * HD) + 4.0 * H * HD * sum(range(pos + 1, pos + T + 1)))
    if case["kind"] == "model":
        total += V * D * BITS[Q8] / 8 + T * D * BITS[Q8] / 8 + 4 * V + 4 * D
        flops += 2.0 * V * D
    return {"bytes": total, "flops": flops}


def tolerance(case):
    """Sums of 32-bit products in another order: measured up to 1.5e-6 from the 64-bit values.
    Expert ids change only where two router logits differ by less than a rounding; a model's
    layers see each other's roundings, so there a few may."""
    return {"rel": 6e-6, "differ": 0.01 if case["kind"] == "model" else 0.001}


# ---------------------------------------------------------------- the same in 64 bits

def _norm64(x, g):
    x = x.double()
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * g.double()


def _moe64(enc, w, hh):
    """(weighted sum of the experts' outputs, ids, weights) for the rows hh"""
    T = hh.shape[0]
    xn = _norm64(hh, w["ln2"])
    p, ids = (xn @ w["wgate"].double().T).softmax(-1).topk(K, -1)
    wt = p / p.sum(-1, keepdim=True)
    out = torch.zeros(T, D, dtype=torch.float64, device="cuda")
    m = {k: w[k].view(E, -1, w[k].shape[1]) for k in ("gate", "up", "down")}
    for e in ids.unique().tolist():
        t, j = (ids == e).nonzero(as_tuple=True)
        g = xn[t] @ _values(enc, m["gate"][e]).view(F, D).T
        u = xn[t] @ _values(enc, m["up"][e]).view(F, D).T
        y = (g * g.sigmoid() * u) @ _values(enc, m["down"][e]).view(D, F).T
        out.index_add_(0, t, y * wt[t, j, None])
    return out, wt


def _rotate64(x, pos):
    """x (T, heads, HD) at positions pos..: pairs (i, i + HD/2) turned by the position's angle,
    the angles being the 32-bit products that the model defines"""
    i = torch.arange(HD // 2, dtype=torch.float64)
    inv = (THETA ** (-2.0 * i / HD)).float()
    ang = (torch.arange(pos, pos + x.shape[0], dtype=torch.float32)[:, None] * inv).double().cuda()
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x[..., : HD // 2], x[..., HD // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attn64(enc, w, x, k0, v0):
    T, pos = x.shape[0], k0.shape[0]
    qkv = _norm64(x, w["ln1"]) @ _values(enc, w["wqkv"]).view(NQKV, D).T
    q, k, v = qkv.split([H * HD, KV * HD, KV * HD], -1)
    q = _rotate64(_norm64(q.view(T, H, HD), w["qn"]), pos)
    k = _rotate64(_norm64(k.view(T, KV, HD), w["kn"]), pos)
    kk = torch.cat([k0.double().view(pos, KV, HD), k])
    vv = torch.cat([v0.double().view(pos, KV, HD), v.view(T, KV, HD)])
    ahead = torch.arange(pos + T, device="cuda")[None] > torch.arange(pos, pos + T, device="cuda")[:, None]
    o = torch.empty(T, H, HD, dtype=torch.float64, device="cuda")
    for h in range(H):
        sc = q[:, h] @ kk[:, h // (H // KV)].T / math.sqrt(HD)
        o[:, h] = sc.masked_fill(ahead, -math.inf).softmax(-1) @ vv[:, h // (H // KV)]
    return (o.view(T, H * HD) @ _values(enc, w["wo"]).view(D, H * HD).T, k.reshape(T, -1), v)


def exact(case, seed):
    kind, T, L, enc = case["kind"], case["T"], case["L"], case["enc"]
    osig = _out_sigma(case)
    mw = lambda l: _moe_weights(enc, seed, l, case.get("skew"), osig)          # noqa: E731
    aw = lambda l: _attn_weights(enc, seed, l, osig)                          # noqa: E731
    if kind == "moe":
        x, attn = _tokens(case, seed)
        got = [_moe64(enc, mw(l), x.double() + attn.double()) for l in range(L)]
        return {"mlp": torch.stack([g[0] for g in got]), "topk": None,
                "wt": torch.stack([g[1] for g in got])}
    if kind == "attn":
        x = _normal(seed, 1, T, D)
        got = [_attn64(enc, aw(l), x, *_cache(seed, l, case["pos"])) for l in range(L)]
        o, k, v = (torch.stack(z) for z in zip(*got))
        return {"attn": o, "k": k, "v": v}
    table = _values(Q8, _matrix(Q8, seed, 5, EMB_ROWS, D, 1.0)).view(EMB_ROWS, D)
    x, ks, vs = table[_model_ids(case, seed).long()], [], []
    for l in range(L):
        a, k, v = _attn64(enc, aw(l), x, *_cache(seed, l, case["pos"]))
        x = x + a + _moe64(enc, mw(l), x + a)[0]
        ks.append(k)
        vs.append(v)
    xn = _norm64(x[-1:], _gain(seed, 7, D))
    head = _matrix(Q8, seed, 6, V, D, SIGMA)
    logits = torch.cat([(xn @ _values(Q8, b).view(-1, D).T)[0]
                        for b in head.view(16, -1, head.shape[1])])
    return {"k": torch.stack(ks), "v": torch.stack(vs), "logits": logits, "topk": None}
