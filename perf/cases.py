"""Performance cases of the INT8 training framework: what a user of `jatai_amd` has it do, through its public entry
points (`OpsHip`, `Modelo.passo`, `PassoGravado`), from a two-layer step of 256 tokens to the 24-layer step of 16,384.

Every output is an integer tensor (or the float64 loss computed from integers) that the format defines bit for bit,
so every tolerance is "exact". `exact` restates the format's rules for single layers and blocks in plain 64-bit torch.
"""
import math
import os
import tempfile

import torch

from jatai_amd import ops as O
from jatai_amd.modelo import Modelo, PassoGravado
from jatai_amd.registro import Registro

E_ZERO, GA = -127, 4
DEV = "cuda"


def listed():
    return [
        # the smallest whole step a user runs: two layers at the reference's own widths, op by op (no graph), as when
        # a model is brought up or a test steps it; host and launch cost
        dict(name="passo_2_camadas", tipo="passo", grafo=False, L=2, D=256, H=64, FF=1024, V=256, T=128, Bt=2, blk=128, r16=False),
        # the reference's published training run: 12 layers, 64 heads of 4, blocks of 128, 2048 tokens, captured graph
        dict(name="passo_referencia", tipo="passo", grafo=True, L=12, D=256, H=64, FF=1024, V=256, T=128, Bt=16, blk=128, r16=False),
        # the framework's headline training step: 12 layers, d_model 512, 8 heads of 64, 2048 tokens, captured graph
        dict(name="passo_12_camadas", tipo="passo", grafo=True, L=12, D=512, H=8, FF=2048, V=256, T=256, Bt=8, blk=32, r16=False),
        # the largest training step: 24 layers, 16,384 tokens, 16-bit residual stream, captured graph
        dict(name="passo_24_camadas", tipo="passo", grafo=True, L=24, D=512, H=8, FF=2048, V=256, T=256, Bt=64, blk=32, r16=True),
        # the forward pass alone, op by op, to the logits and the loss: evaluation of one batch
        dict(name="avalia", tipo="avalia", L=12, D=512, H=8, FF=2048, V=256, T=256, Bt=8, blk=32),
        # one small product on its own: 512 x 512 x 512, the smallest of the configurations
        dict(name="gemm_512", tipo="gemm", modo="bloco", M=512, N=512, K=512, blk=32),
        # the Q/K/V projection of a large batch
        dict(name="gemm_qkv", tipo="gemm", modo="bloco", M=16384, N=1536, K=512, blk=32),
        # the MLP block of a layer, forward and backward (the five products and the norm around them)
        dict(name="mlp", tipo="mlp", M=16384, D=512, FF=2048, blk=32),
        # the weight gradients of a layer: transposes and the grouped products over all tokens
        dict(name="grad_pesos", tipo="grad", M=16384, D=512, FF=2048, blk=32),
        # attention of a large batch, forward and backward: 8 heads of 64 over 256 tokens
        dict(name="atencao_64", tipo="atencao", Bt=64, T=256, H=8, hd=64, blk=32),
        # attention at another head width and a longer sequence, where the raw outputs are quantized separately
        dict(name="atencao_32", tipo="atencao", Bt=8, T=512, H=16, hd=32, blk=32),
        # the row operations around the layers: norm and its backward with the residual, softmax cross-entropy, loss
        dict(name="linhas", tipo="linhas", M=16384, D=512, V=256, blk=32),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _mult(x, m, lo, hi):
    """The multiple of m nearest to x within [lo, hi]."""
    return int(min(max(round(x / m), -(-lo // m)), hi // m)) * m


def _tokens(rng, blk, hi=16384):
    """A token count the transposes and the weight gradients take: a multiple of 128, past 4096 of 16 blocks."""
    m = _mult(_log(rng, 128, hi), 128, 128, hi)
    return m if m <= 4096 else _mult(m, 16 * blk, 4096, hi)


def _modelo(rng):
    blk = rng.choice([32, 32, 128])
    if rng.random() < 0.3:                      # the reference's head width, up to 64 heads
        H, T, hd = rng.choice([32, 64]), rng.choice([32, 64, 96, 128, 256]), 4
    else:
        hd, T = rng.choice([64, 64, 32, 16]), rng.choice([64, 128, 192, 256, 512])
        H = rng.choice([h for h in (2, 4, 6, 8, 12, 16, 32) if h * hd % 128 == 0 and h * hd <= 1024])
    D, passo = H * hd, 128 // math.gcd(T, 128)
    Bt = _mult(_log(rng, 1, 4096 / T), passo, passo, max(passo, 4096 // T))
    return dict(L=rng.randint(1, 8), D=D, H=H, FF=D * rng.choice([2, 3, 4]), V=rng.choice([256, 256, 128, 384]), T=T, Bt=Bt, blk=blk)


def draw(rng):
    tipo = rng.choice(["passo", "passo", "avalia", "gemm", "gemm", "mlp", "grad", "atencao", "linhas"])
    blk = rng.choice([32, 32, 32, 128])
    if tipo == "passo":
        return dict(tipo=tipo, grafo=rng.random() < 0.7, r16=rng.random() < 0.25, **_modelo(rng))
    if tipo == "avalia":
        return dict(tipo=tipo, **_modelo(rng))
    if tipo == "gemm":
        modo = rng.choice(["bloco", "cru", "soma", "relu2", "relu2_back"])
        return dict(tipo=tipo, modo=modo, M=_mult(_log(rng, 32, 16384), 32, 32, 16384), N=_mult(_log(rng, 128, 2048), 128, 128, 2048),
                    K=_mult(_log(rng, blk, 4096), blk, blk, 4096), blk=blk)
    if tipo in ("mlp", "grad"):
        return dict(tipo=tipo, M=_tokens(rng, blk), D=rng.choice([128, 256, 384, 512, 768, 1024]), FF=128 * rng.randint(2, 16), blk=blk)
    if tipo == "atencao":
        hd = rng.choice([64, 64, 32, 16, 4])
        T = rng.choice([32, 64, 96, 128, 256]) if hd == 4 else 64 * rng.randint(1, 8)
        H = rng.choice([32, 64]) if hd == 4 else rng.choice([h for h in (2, 4, 6, 8, 16) if h * hd % 128 == 0])
        return dict(tipo=tipo, Bt=_mult(_log(rng, 1, 16384 / T), 1, 1, 64), T=T, H=H, hd=hd, blk=blk)
    return dict(tipo=tipo, M=_mult(_log(rng, 32, 65536), 1, 32, 65536), D=128 * rng.randint(1, 8), V=128 * rng.randint(1, 8), blk=blk)


# ------------------------------------------------------------------------------------------------ inputs
def _quant(v, e, blk):
    """The INT8 block format's quantization of the integers v (|v| < 2^52) with exponents e: one exponent E per block
    of blk columns, E = max(e + bitlen(v)) - 7, one higher where a rounded mantissa passes 127, half to even; a zero
    block (or one below 2^-126) has mantissas 0 and E = -127."""
    R, C = v.shape
    v, e = v.view(R, C // blk, blk), e.expand(R, C).reshape(R, C // blk, blk)
    topo = torch.where(v != 0, e + _bitlen(v), -100000).amax(2, keepdim=True)
    E = topo - 7
    E = E + (_rnd(v, E - e).abs() > 127).any(2, keepdim=True)
    zero = (topo == -100000) | (E < -126)
    q = torch.where(zero, 0, _rnd(v, E - e))
    return q.view(R, C).to(torch.int8), torch.where(zero, E_ZERO, E).view(R, C // blk).to(torch.int8)


def _bitlen(v):
    return torch.frexp(v.abs().double())[1].long()


def _rnd(x, s):
    """x 2^-s for integers, half to even; s <= 0 is a left shift."""
    s = torch.as_tensor(s, device=x.device).clamp(-62, 62)
    d, esq = s.clamp(min=0), (-s).clamp(min=0)
    q = x >> d
    resto, meio = x - (q << d), (torch.ones_like(d) << d) >> 1
    q = q + ((resto > meio) | ((resto == meio) & (d > 0) & (q & 1 == 1))).long()
    return torch.where(s > 0, q, x << esq)


def _bloco(g, R, C, blk, sigma=1.0, por_linha=0.0):
    """N(0, sigma^2) values in the block format; por_linha > 0: rows scaled by a log-normal factor, as the gradients of
    different tokens are."""
    x = torch.randn(R, C, generator=g, device=DEV, dtype=torch.float64) * sigma
    if por_linha:
        x = x * torch.exp(por_linha * torch.randn(R, 1, generator=g, device=DEV, dtype=torch.float64))
    m, e = torch.frexp(x)
    return _quant((m * 2.0 ** 24).long(), (e - 24).long(), blk)


def _gerador(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _tok(g, c, n=None):
    return torch.randint(0, c["V"], (n,) if n else (c["Bt"], c["T"]), generator=g, device=DEV)


GRAD = 2.0 ** -12                               # gradients are a few thousandths of the activations


def _entradas(c, seed):
    """The tensors of a single layer or block, from the seed alone."""
    g, blk = _gerador(seed), c["blk"]
    if c["tipo"] == "gemm":
        t = dict(A=_bloco(g, c["M"], c["K"], blk), B=_bloco(g, c["N"], c["K"], blk, 0.02))
        if c["modo"] in ("soma", "relu2_back"):
            t["X"] = _bloco(g, c["M"], c["N"], blk)
        return t
    if c["tipo"] == "mlp":
        M, D, FF = c["M"], c["D"], c["FF"]
        return dict(x=_bloco(g, M, D, blk), Wup=_bloco(g, FF, D, blk, D ** -0.5), Wd=_bloco(g, D, FF, blk, FF ** -0.5),
                    gx=_bloco(g, M, D, blk, GRAD, 0.7))
    if c["tipo"] == "grad":
        M, D, FF = c["M"], c["D"], c["FF"]
        return dict(gx=_bloco(g, M, D, blk, GRAD, 0.7), a=_bloco(g, M, FF, blk), gh=_bloco(g, M, FF, blk, GRAD, 0.7), n2=_bloco(g, M, D, blk),
                    gq=_bloco(g, M, 3 * D, blk, GRAD, 0.7), n1=_bloco(g, M, D, blk))
    if c["tipo"] == "avalia":
        D, FF = c["D"], c["FF"]
        camadas = [dict(Wqkv=_bloco(g, 3 * D, D, blk, D ** -0.5), Wo=_bloco(g, D, D, blk, D ** -0.5), Wup=_bloco(g, FF, D, blk, D ** -0.5),
                        Wd=_bloco(g, D, FF, blk, FF ** -0.5)) for _ in range(c["L"])]
        return dict(emb=_bloco(g, c["V"], D, blk), camadas=camadas, out=_bloco(g, c["V"], D, blk, D ** -0.5),
                    tok=_tok(g, c, c["Bt"] * c["T"]).to(torch.int32), alvo=_tok(g, c, c["Bt"] * c["T"]).to(torch.int32))
    if c["tipo"] == "atencao":
        D = c["H"] * c["hd"]
        return dict(qkv=_bloco(g, c["Bt"] * c["T"], 3 * D, blk), go=_bloco(g, c["Bt"] * c["T"], D, blk, GRAD, 0.7))
    M, D, V = c["M"], c["D"], c["V"]
    logits = torch.randn(M, V, generator=g, device=DEV, dtype=torch.float64) * 2
    return dict(x=_bloco(g, M, D, blk), gn=_bloco(g, M, D, blk, GRAD, 0.7), gx=_bloco(g, M, D, blk, GRAD, 0.7),
                logits=((logits * 2.0 ** 16).to(torch.int32), torch.full((M, V), -16, dtype=torch.int16, device=DEV)),
                alvo=_tok(g, c, M).to(torch.int32))


_OPS = {}


def _ops(blk):
    """The program's operator object: one per process, at the program's block size."""
    if not _OPS:
        _OPS["reg"] = Registro(os.path.join(tempfile.gettempdir(), "jatai_perf"), "casos", eco=False)
        _OPS["ops"] = O.OpsHip(_OPS["reg"])
    O.BLK = blk
    return _OPS["ops"], _OPS["reg"]


def _contiguos(d):
    """Every block tensor of d moved into two flat buffers (mantissas, exponents), as a program that saves its state in
    one piece keeps them; returns the buffers."""
    flat = [torch.cat([t[i].reshape(-1) for t in d.values()]) for i in range(2)]
    ini = [0, 0]
    for n, t in d.items():
        d[n] = tuple(flat[i][ini[i]:ini[i] + t[i].numel()].view(t[i].shape) for i in range(2))
        ini = [ini[i] + t[i].numel() for i in range(2)]
    return flat


def prepare(case, seed):
    c = case
    ops, reg = _ops(c["blk"])
    reg.novo_passo(0)
    s = dict(case=c)
    if c["tipo"] != "passo":
        s.update(_entradas(c, seed))
        return s
    g = _gerador(seed)
    m = s["modelo"] = Modelo(c["V"], c["D"], c["H"], c["FF"], c["L"], seed, DEV, ops, reg, r16=c["r16"])
    s["estado"] = [t for d in (m.p, m.mom, m.res) for t in _contiguos(d)]
    s["tok"], s["alvo"] = _tok(g, c), _tok(g, c)
    if c["grafo"]:                            # one step op by op, then the capture, as a training program starts
        m.passo(_tok(g, c), _tok(g, c), k_lr=4)
        reg.fim_passo()
        s["grafo"] = PassoGravado(m, c["Bt"], c["T"], 4)
    return s


# ------------------------------------------------------------------------------------------------ one pass
def run(state):
    c = state["case"]
    ops, reg = _ops(c["blk"])
    reg.novo_passo(0)
    return globals()["_run_" + c["tipo"]](c, state, ops, reg)


def _run_passo(c, s, ops, reg):
    m = s["modelo"]
    perda = s["grafo"](s["tok"], s["alvo"]) if c["grafo"] else m.passo(s["tok"], s["alvo"], k_lr=4)
    reg.fim_passo()                             # a training loop reads the device's error record after each step
    return dict(perda=perda, estado=s["estado"])


def _run_avalia(c, s, ops, reg):
    Bt, T, H = c["Bt"], c["T"], c["H"]
    x = ops.embed(s["emb"], s["tok"])
    for W in s["camadas"]:
        om, _ = ops.atencao_q(ops.gemm(ops.rms(x)[0], W["Wqkv"]), Bt, T, H)
        x = ops.gemm_soma(om, W["Wo"], x)
        x = ops.gemm_soma(ops.gemm_relu2(ops.rms(x)[0], W["Wup"])[1], W["Wd"], x)
    logits = ops.gemm(ops.rms(x)[0], s["out"], cru=True)
    _, d, soma = ops.softmax_ce(logits, s["alvo"])
    return dict(x=x, logits=logits, d=d, soma=soma, perda=ops.perda(d, soma))


def _run_gemm(c, s, ops, reg):
    A, B = s["A"], s["B"]
    if c["modo"] == "bloco":
        return ops.gemm(A, B)
    if c["modo"] == "cru":
        return ops.gemm(A, B, cru=True)
    if c["modo"] == "soma":
        return ops.gemm_soma(A, B, s["X"])
    if c["modo"] == "relu2":
        return ops.gemm_relu2(A, B)
    return ops.gemm_relu2_back(A, B, s["X"])


def _run_mlp(c, s, ops, reg):
    n, cache = ops.rms(s["x"])
    h, a, ta = ops.gemm_relu2_t(n, s["Wup"])
    y = ops.gemm_soma(a, s["Wd"], s["x"])
    gh, tgh = ops.gemm_relu2_back_t(s["gx"], ops.transpoe(s["Wd"]), h)
    gn = ops.gemm(gh, ops.transpoe(s["Wup"]))
    return dict(n=n, h=h, a=a, ta=ta, y=y, gh=gh, tgh=tgh, gx=ops.rms_back_soma(gn, n, cache, s["gx"]))


def _run_grad(c, s, ops, reg):
    tgx, ta, tgh, tn2, tgq, tn1 = ops.transpoe_lote([s[k] for k in ("gx", "a", "gh", "n2", "gq", "n1")])
    return ops.gemm_cru_lote([(tgx, ta, None), (tgh, tn2, None), (tgx, tn2, None), (tgq, tn1, None)])


def _run_atencao(c, s, ops, reg):
    om, P = ops.atencao_q(s["qkv"], c["Bt"], c["T"], c["H"])
    return dict(om=om, P=P, gqkv=ops.atencao_back_q(s["go"], s["qkv"], P, c["Bt"], c["T"], c["H"]))


def _run_linhas(c, s, ops, reg):
    n, cache = ops.rms(s["x"])
    gx = ops.rms_back_soma(s["gn"], n, cache, s["gx"])
    g, d, soma = ops.softmax_ce(s["logits"], s["alvo"])
    return dict(n=n, cache=cache, gx=gx, g=g, d=d, soma=soma, perda=ops.perda(d, soma))


# ------------------------------------------------------------------------------------------------ work and tolerance
def work(case):
    c, b = case, 1 + 1 / case["blk"]
    if c["tipo"] in ("passo", "avalia"):
        M, D, FF, V, L = c["Bt"] * c["T"], c["D"], c["FF"], c["V"], c["L"]
        W = L * (4 * D * D + 2 * D * FF) + 2 * V * D
        # products over weights; attention's causal half of q.k and p.v (four products of that size in its backward)
        prod, at = 2 * M * (W - V * D), 2 * L * M * c["T"] * D
        if c["tipo"] == "avalia":
            return dict(bytes=W * b + 12 * M, flops=prod + at)
        return dict(bytes=6 * b * W + 8 * M, flops=3 * prod + 3.5 * at)
    if c["tipo"] == "gemm":
        M, N, K = c["M"], c["N"], c["K"]
        saida = {"bloco": b, "cru": 6, "soma": 2 * b, "relu2": 2 * b, "relu2_back": 2 * b}[c["modo"]]
        return dict(bytes=b * (M * K + N * K) + saida * M * N, flops=2 * M * N * K)
    if c["tipo"] == "mlp":
        M, D, FF = c["M"], c["D"], c["FF"]
        return dict(bytes=b * (2 * M * D + 2 * D * FF + 3 * M * D + 5 * M * FF), flops=8 * M * D * FF)
    if c["tipo"] == "grad":
        M, D, FF = c["M"], c["D"], c["FF"]
        P = 2 * D * FF + 4 * D * D
        return dict(bytes=b * M * (6 * D + 2 * FF) + 6 * P, flops=2 * M * P)
    if c["tipo"] == "atencao":
        M, D, T = c["Bt"] * c["T"], c["H"] * c["hd"], c["T"]
        return dict(bytes=b * 8 * M * D + M * T * c["H"], flops=7 * M * T * D)
    M, D, V = c["M"], c["D"], c["V"]
    return dict(bytes=M * (b * 5 * D + (6 + b) * V + 20), flops=M * (20 * D + 20 * V))


def tolerance(case):
    return "exact"


# ------------------------------------------------------------------------------------------------ plain 64-bit restatement
def _exp(E, blk):
    return E.long().repeat_interleave(blk, 1)


def _gemm(A, B, blk):
    """Raw product: per K-block the exact dot product, times 16, rounded at the row's and the column's exponents."""
    (a, ea), (b, eb) = A, B
    a, b, ea, eb = a.double(), b.double(), ea.long(), eb.long()
    RA, RB = ea.amax(1, keepdim=True), eb.amax(1, keepdim=True)
    acc = torch.zeros(a.shape[0], b.shape[0], dtype=torch.int64, device=a.device)
    for k in range(ea.shape[1]):
        p = (a[:, k * blk:(k + 1) * blk] @ b[:, k * blk:(k + 1) * blk].T).long()
        acc += _rnd(p << 4, (RA - ea[:, k:k + 1]) + (RB - eb[:, k:k + 1]).T)
    return acc, RA + RB.T - 4


def _soma(X, Y, blk):
    ex, ey = _exp(X[1], blk), _exp(Y[1], blk)
    ec = torch.maximum(ex, ey) - 21
    return _quant(_rnd(X[0].long(), ec - ex) + _rnd(Y[0].long(), ec - ey), ec, blk)


def _relu2(H, blk):
    return _quant(H[0].long().clamp(min=0) ** 2, 2 * _exp(H[1], blk), blk)


def _relu2_back(G, H, blk):
    return _quant(G[0].long() * H[0].long().clamp(min=0) * 2, _exp(G[1], blk) + _exp(H[1], blk), blk)


def _transpoe(X, blk):
    return _quant(X[0].long().T.contiguous(), _exp(X[1], blk).T.contiguous(), blk)


def _g_rms(D, blk):
    return 2 * ((8 - int(math.log2(D // blk))) // 2), 14 - int(math.log2(D))


def _isqrt(n):
    r = n.clamp(min=0).double().sqrt().long()
    r = r - (r * r > n).long()
    r = r + ((r + 1) * (r + 1) <= n).long()
    return r.clamp(min=1)


def _rms(X, blk):
    m, E = X[0].long(), X[1].long()
    M, D = m.shape
    G, _ = _g_rms(D, blk)
    emax = E.amax(1, keepdim=True)
    ss = _rnd((m * m).view(M, -1, blk).sum(2) << G, 2 * (emax - E)).sum(1, keepdim=True)
    r = _isqrt(ss >> int(math.log2(D)))
    k = _bitlen(r) + 10
    Y = _quant(m * ((torch.ones_like(k) << k) // r), _exp(E, blk) - k - emax + G // 2, blk)
    return Y, (r[:, 0].to(torch.int32), emax[:, 0].to(torch.int32))


def _rms_back(Gg, Y, cache, blk):
    g, y, eg, ey = Gg[0].long(), Y[0].long(), _exp(Gg[1], blk), _exp(Y[1], blk)
    D = g.shape[1]
    G, GB = _g_rms(D, blk)
    lg = int(math.log2(D))
    r, emax = cache[0].long()[:, None], cache[1].long()[:, None]
    smax = (eg + ey).amax(1, keepdim=True)
    S = _rnd((g * y) << GB, smax - (eg + ey)).sum(1, keepdim=True)
    sh = (_bitlen(S) - 15).clamp(min=0)
    S, eS = _rnd(S, sh), smax - GB - lg + sh
    k = _bitlen(r) + 10
    ec = torch.maximum(eg + 7, ey + eS + 22) - 28
    d = _rnd(g, ec - eg) - _rnd(y * S, ec - (ey + eS))
    sh2 = (_bitlen(d) - 18).clamp(min=0)
    return _quant(_rnd(d, sh2) * ((torch.ones_like(k) << k) // r), ec + sh2 - k - (emax - G // 2), blk)


def _exp_int(d):
    t = d.clamp(max=6000) * 23637
    n, f = t >> 22, (t & ((1 << 22) - 1)) >> 7
    p = torch.full_like(t, -1295)
    for c in (7556, -22645, 32765):
        p = ((p * f) >> 15) + c
    return torch.where(n > 30, 0, p >> n.clamp(max=30))


def _softmax_ce(L, alvo, blk):
    acc, e = L[0].long(), L[1].long()
    u = _rnd(acc, -(e + 8))
    umax = u.amax(1, keepdim=True)
    ex = _exp_int(umax - u) >> 3
    s = ex.sum(1, keepdim=True)
    v = (ex * ((1 << 28) // s) + (1 << 15)) >> 16
    t = alvo.long()[:, None]
    v = v.scatter_add(1, t, torch.full_like(t, -4096))
    d = (umax - u.gather(1, t))[:, 0]
    ev = torch.full((1, 1), -12 - int(math.log2(acc.shape[0])), dtype=torch.int64, device=acc.device)
    return _quant(v, ev, blk), d.to(torch.int32), s[:, 0].to(torch.int32)


def _perda(d, soma):
    return (d.double() / 256 + torch.log(soma.double() / 4096)).mean()


def _alinha(m, E, c, H, hd):
    """Values of every head aligned to the largest exponent the head holds over its sequence: [Bt H, T, hd] and that
    exponent less the guard bits, [Bt H, 1, 1]."""
    Bt, T = c["Bt"], c["T"]
    sep = lambda x: x.view(Bt, T, H, hd).transpose(1, 2).reshape(Bt * H, T, hd)
    x, e = sep(m.long()), sep(_exp(E, c["blk"]))
    emx = e.amax((1, 2), keepdim=True)
    return _rnd(x << GA, emx - e), emx - GA


def _mm(a, b):
    return torch.bmm(a.double().contiguous(), b.double().contiguous()).long()


def _atencao(qkv, go, c, H, hd):
    """The attention's outputs, quantized, and P; with go (the gradient of the first) the quantized gradient of qkv too."""
    Bt, T, blk = c["Bt"], c["T"], c["blk"]
    D, dev = H * hd, qkv[0].device
    parte = lambda i: (qkv[0][:, i * D:(i + 1) * D], qkv[1][:, i * D // blk:(i + 1) * D // blk])
    (q, eq), (k, ek), (v, ev) = [_alinha(*parte(i), c, H, hd) for i in range(3)]
    h = torch.arange(H, device=dev).repeat(Bt)[:, None, None]
    incl = 8 - h // 8 if hd == 4 else 8 - (8 * h) // H
    i, j = torch.arange(T, device=dev)[None, :, None], torch.arange(T, device=dev)[None, None, :]
    causal = j <= i
    alibi = torch.where(incl >= 0, ((i - j).clamp(min=0)) << incl.clamp(min=0), 0)
    u = _rnd(_mm(q, k.transpose(1, 2)), -(eq + ek - int(math.log2(hd)) // 2 + 8)) - alibi
    mx = torch.where(causal, u, -(1 << 62)).amax(2, keepdim=True)
    ex = torch.where(causal, _exp_int((mx - u).clamp(min=0)) >> 3, 0)
    P = ((ex * ((1 << 28) // ex.sum(2, keepdim=True)) + (1 << 19)) >> 20).clamp(max=255)
    junta = lambda x: x.view(Bt, H, T, hd).transpose(1, 2).reshape(Bt * T, D)
    espalha = lambda e: e.view(Bt, H, 1, 1).expand(Bt, H, T, hd).transpose(1, 2).reshape(Bt * T, D)
    om = _quant(junta(_mm(P, v)), espalha(ev - 8), blk)
    if go is None:
        return om, P, None
    go, ego = _alinha(*go, c, H, hd)
    gP = _mm(go, v.transpose(1, 2))
    sh = (_bitlen(torch.where(causal, gP, 0).abs().amax((1, 2), keepdim=True)) - 15).clamp(min=0)
    gP = _rnd(gP, sh)
    dS = P * (gP - _rnd((P * gP).sum(2, keepdim=True), 8))
    bits = 12 - max(0, int(math.log2(2 * T - 1)) - 7)
    sh2 = (_bitlen(dS.abs().amax((1, 2), keepdim=True)) - bits).clamp(min=0)
    dS, eds = _rnd(dS, sh2), ego + ev + sh - 9 + sh2
    partes = [(_mm(dS, k), eds + ek), (_mm(dS.transpose(1, 2), q), eds + eq), (_mm(P.transpose(1, 2), go), ego - 8)]
    gqkv = _quant(torch.cat([junta(x) for x, _ in partes], 1), torch.cat([espalha(e) for _, e in partes], 1), blk)
    return om, P.transpose(1, 2).to(torch.uint8).contiguous(), gqkv


def exact(case, seed):
    c, blk = case, case["blk"]
    if c["tipo"] == "passo":                    # whole training steps: their layers have cases of their own
        return None
    s = _entradas(c, seed)
    if c["tipo"] == "avalia":
        x = tuple(t[s["tok"].long()] for t in s["emb"])
        for W in s["camadas"]:
            qkv = _quant(*_gemm(_rms(x, blk)[0], W["Wqkv"], blk), blk)
            om = _atencao(qkv, None, c, c["H"], c["D"] // c["H"])[0]
            x = _soma(x, _quant(*_gemm(om, W["Wo"], blk), blk), blk)
            a = _relu2(_quant(*_gemm(_rms(x, blk)[0], W["Wup"], blk), blk), blk)
            x = _soma(x, _quant(*_gemm(a, W["Wd"], blk), blk), blk)
        acc, e = _gemm(_rms(x, blk)[0], s["out"], blk)
        _, d, soma = _softmax_ce((acc, e), s["alvo"], blk)
        return dict(x=x, logits=(acc.to(torch.int32), e.to(torch.int16)), d=d, soma=soma, perda=_perda(d, soma))
    if c["tipo"] == "gemm":
        acc, e = _gemm(s["A"], s["B"], blk)
        if c["modo"] == "cru":
            return acc.to(torch.int32), e.to(torch.int16)
        C = _quant(acc, e, blk)
        if c["modo"] == "soma":
            return _soma(s["X"], C, blk)
        if c["modo"] == "relu2":
            return C, _relu2(C, blk)
        return _relu2_back(C, s["X"], blk) if c["modo"] == "relu2_back" else C
    if c["tipo"] == "mlp":
        n, cache = _rms(s["x"], blk)
        h = _quant(*_gemm(n, s["Wup"], blk), blk)
        a = _relu2(h, blk)
        y = _soma(s["x"], _quant(*_gemm(a, s["Wd"], blk), blk), blk)
        gh = _relu2_back(_quant(*_gemm(s["gx"], _transpoe(s["Wd"], blk), blk), blk), h, blk)
        gn = _quant(*_gemm(gh, _transpoe(s["Wup"], blk), blk), blk)
        return dict(n=n, h=h, a=a, ta=_transpoe(a, blk), y=y, gh=gh, tgh=_transpoe(gh, blk), gx=_soma(s["gx"], _rms_back(gn, n, cache, blk), blk))
    if c["tipo"] == "grad":
        tgx, ta, tgh, tn2, tgq, tn1 = [_transpoe(s[k], blk) for k in ("gx", "a", "gh", "n2", "gq", "n1")]
        crus = [_gemm(A, B, blk) for A, B in ((tgx, ta), (tgh, tn2), (tgx, tn2), (tgq, tn1))]
        return [(acc.to(torch.int32), e.to(torch.int16)) for acc, e in crus]
    if c["tipo"] == "atencao":
        om, P, gqkv = _atencao(s["qkv"], s["go"], c, c["H"], c["hd"])
        return dict(om=om, P=P, gqkv=gqkv)
    n, cache = _rms(s["x"], blk)
    g, d, soma = _softmax_ce(s["logits"], s["alvo"], blk)
    return dict(n=n, cache=cache, gx=_soma(s["gx"], _rms_back(s["gn"], n, cache, blk), blk), g=g, d=d, soma=soma, perda=_perda(d, soma))
