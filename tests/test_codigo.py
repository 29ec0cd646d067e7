"""The code object inside the built library, read with the compiler's own tools (no GPU): no kernel keeps registers in scratch
memory, and no result of a matrix instruction is used too early on any path. Both depend on the compiler's choices, which
a change of a kernel or of the compiler can undo without changing a result on most runs."""
import os
import re
import shutil
import subprocess

import pytest

from jatai_amd.build import HIPCC
from jatai_amd.ops import LIB

LLVM = os.path.join(os.path.dirname(os.path.dirname(HIPCC)), "llvm", "bin")
ESTADOS = 8                                     # MFMAs of 4 passes (every one used here) before a use by another unit


@pytest.fixture(scope="module")
def objeto(tmp_path_factory):
    if not os.path.exists(os.path.join(LLVM, "llvm-readelf")):
        pytest.skip("no LLVM tools beside hipcc")
    d = tmp_path_factory.mktemp("codigo")
    subprocess.run([os.path.join(LLVM, "llvm-objdump"), "--offloading", shutil.copy(LIB, d)], check=True, capture_output=True, cwd=d)
    co, = d.glob("*gfx950*")
    return co


def _saida(*cmd):
    return subprocess.run([os.path.join(LLVM, cmd[0]), *map(str, cmd[1:])], check=True, capture_output=True, text=True).stdout


def test_kernels_sem_scratch(objeto):
    notas = _saida("llvm-readelf", "--notes", objeto)
    campos = lambda c: re.findall(rf"^\s*-?\s*\.{c}:\s+(\S+)", notas, re.M)
    nomes = [n for n in campos("symbol") if n.endswith(".kd")]
    scratch, derramados = campos("private_segment_fixed_size"), campos("vgpr_spill_count")
    assert len(nomes) == len(scratch) == len(derramados) > 100
    assert not [x for x in zip(nomes, scratch, derramados) if x[1:] != ("0", "0")]


def _regs(txt):
    r = set()
    for u, n, v, a, b in re.findall(r"\b([va])(\d+)\b|\b([va])\[(\d+):(\d+)\]", txt):
        r.update([(u, int(n))] if u else [(v, i) for i in range(int(a), int(b) + 1)])
    return r


def cedo_demais(listagem, minimo):
    """(function, address, states, instruction) of every MFMA whose result another instruction reads or overwrites within
    fewer than `minimo` wait states on some path; s_nop n counts n + 1, any other instruction 1. An MFMA that accumulates
    on the same registers takes them from the matrix unit itself."""
    funcoes, ins = {}, None
    for l in listagem.splitlines():
        if m := re.match(r"^[0-9a-f]+ <(.+)>:", l):
            ins = funcoes.setdefault(m.group(1), [])
        elif ins is not None and (m := re.match(r"^\s+(\S+)(?:\s+(.*?))?\s*//\s*([0-9A-F]+):", l)):
            ins.append((int(m.group(3), 16), m.group(1), (m.group(2) or "").split(" <")[0]))
    achados = []
    for f, ins in funcoes.items():
        onde = {e: i for i, (e, _, _) in enumerate(ins)}

        def segue(i):
            e, op, arg = ins[i]
            alvo = [onde[e + 4 + 4 * ((int(arg) ^ 0x8000) - 0x8000)]] if op.startswith(("s_cbranch", "s_branch")) else []
            return alvo + ([] if op in ("s_branch", "s_endpgm", "s_setpc_b64") or i + 1 == len(ins) else [i + 1])
        for i, (e, op, arg) in enumerate(ins):
            if not op.startswith("v_mfma"):
                continue
            destino, visto, fila = _regs(arg.split(",")[0]), {}, [(j, 0) for j in segue(i)]
            while fila:
                j, n = fila.pop()
                if n >= minimo or visto.get(j, minimo) <= n:
                    continue
                visto[j] = n
                _, o, a = ins[j]
                if _regs(a) & destino:
                    p = re.split(r",\s*(?![^\[]*\])", a)
                    if not (o.startswith("v_mfma") and _regs(p[3]) == destino and not (_regs(p[1]) | _regs(p[2])) & destino):
                        achados.append((f, hex(e), n, f"{o} {a}"))
                    continue
                fila += [(k, n + (int(a, 0) + 1 if o == "s_nop" else 1)) for k in segue(j)]
    return achados


def test_resultados_de_mfma_com_estados_de_espera(objeto):
    listagem = _saida("llvm-objdump", "-d", "--no-show-raw-insn", objeto)
    assert listagem.count("v_mfma") > 1000
    assert not cedo_demais(listagem, ESTADOS)


def test_cedo_demais_acha_o_caminho_curto():
    """The search itself, on a listing where a branch leaves 3 states before the use and the straight path 11."""
    linhas = ["v_mfma_f32_16x16x16_f16 v[0:3], v[4:5], v[6:7], 0", "v_mfma_f32_16x16x16_f16 v[0:3], v[4:5], v[6:7], v[0:3]", "s_mov_b32 s0, 0",
              "s_mov_b32 s1, 0", "s_cbranch_scc1 1", "s_nop 7", "v_add_f32_e32 v8, v2, v9", "s_endpgm"]
    tam, e, txt = [8, 8, 4, 4, 4, 4, 4, 4], 0, "0000000000000000 <f>:\n"
    for l, t in zip(linhas, tam):
        txt, e = txt + f"\t{l}    // {e:012X}:\n", e + t
    assert cedo_demais(txt, 8) == [("f", "0x8", 3, "v_add_f32_e32 v8, v2, v9")]
    assert not cedo_demais(txt, 3) and not cedo_demais(txt.replace("scc1 1", "scc1 0"), 8)
