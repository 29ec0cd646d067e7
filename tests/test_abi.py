"""The C-ABI library loads (without touching a GPU) and exports every symbol include/jatai.h declares."""
import ctypes
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declarados():
    txt = open(os.path.join(ROOT, "include", "jatai.h")).read()
    txt = re.sub(r"/\*.*?\*/", "", txt, flags=re.S)
    return sorted(set(re.findall(r"\b(jt_\w+)\s*\(", txt)))


def test_exporta_tudo_do_cabecalho():
    import torch  # noqa: F401  (the library binds to the HIP runtime torch loads)
    from jatai_amd import ops as O
    lib = O.carrega_lib()
    nomes = _declarados()
    assert len(nomes) >= 29
    faltam = [n for n in nomes if not hasattr(lib, n)]
    assert not faltam, f"missing exports: {faltam}"


def test_superficie_python_usa_so_simbolos_declarados():
    from jatai_amd import ops as O
    assert set(O.FUNCOES) | set(O.VOIDS) <= set(_declarados())


def test_guardas_de_host_sem_gpu():
    """Format guards fire on the host before any launch (the reference's guards: jatai_cuda/registro.py:161-189)."""
    import pytest
    import torch
    from jatai_amd import ops as O
    from jatai_amd.registro import ErroJatai, Registro
    reg = Registro("/tmp/jatai_testes", "abi", eco=False)
    with pytest.raises(ErroJatai, match="not on the GPU"):
        reg.confere_bloco("A", (torch.zeros(4, 128, dtype=torch.int8), torch.zeros(4, 1, dtype=torch.int8)))
    O.BLK = 32
    try:
        with pytest.raises(ErroJatai, match="exponent shape"):
            reg.confere_bloco("A", (torch.zeros(4, 128, dtype=torch.int8), torch.zeros(4, 1, dtype=torch.int8)))
    finally:
        O.BLK = 128
    with pytest.raises(ErroJatai, match="int16"):
        reg.confere_cru("C", (torch.zeros(4, 128, dtype=torch.int32), torch.zeros(4, 128, dtype=torch.int32)))


def test_registro_estatistica_e_mensagens(tmp_path, capsys):
    """Host registry without a GPU: the block-tensor statistics (zero blocks, exponent range and median, mantissa
    bits of block maxima, zero and saturated mantissas) on a hand-built tensor, the warnings they trigger, and the
    error text (step and scope first, then the message) with its log record."""
    import json
    import pytest
    import torch
    from jatai_amd import ops as O
    from jatai_amd.registro import ErroJatai, Registro
    old = O.BLK
    O.BLK = 32
    try:
        reg = Registro(str(tmp_path), "r", eco=False)
        reg.novo_passo(3)
        m = torch.zeros(2, 64, dtype=torch.int8)
        m[0, :32] = torch.arange(-16, 16, dtype=torch.int8)          # block maximum 16: 5 bits; one zero
        m[1, 32:] = 127                                              # saturated block
        E = torch.tensor([[-115, -127], [-127, 3]], dtype=torch.int8)  # two zero blocks
        rec = reg.estatistica("x", (m, E))
        assert rec["blocos"] == 4 and rec["blocos_zero"] == 0.5
        assert (rec["exp_min"], rec["exp_max"]) == (-115, 3) and rec["bits_usados"] == 6.0
        assert rec["zeros_em_vivos"] == round(1 / 64, 4) and rec["saturados"] == 0.5
        err = capsys.readouterr().err
        assert "within 16 of the INT8 exponent range" in err and "mantissa bits" not in err
        z = reg.estatistica("z", (torch.zeros(1, 32, dtype=torch.int8), torch.full((1, 1), -127, dtype=torch.int8)))
        assert z["blocos_zero"] == 1.0 and "every block is zero" in capsys.readouterr().err
        with reg.trecho("forward"), reg.trecho("mlp"):
            with pytest.raises(ErroJatai) as e:
                reg.exige(False, "bad shape")
        assert str(e.value) == "step 3, forward / mlp:\nbad shape"
        linhas = [json.loads(l) for l in open(tmp_path / "r.jsonl")]
        assert [l["tipo"] for l in linhas].count("estatistica") == 2 and linhas[-1]["tipo"] == "erro"
        assert linhas[-1]["trecho"] == "forward / mlp" and linhas[-1]["passo"] == 3
    finally:
        O.BLK = old


def test_formato_aceita_e_recusa_sem_gpu(tmp_path):
    """What the block-format guard accepts and refuses, over dtypes, layouts, shapes and sizes, on tensors that report
    a GPU; one on the CPU and an operand that is no tensor are refused too."""
    import pytest
    import torch
    from jatai_amd import ops as O
    from jatai_amd.registro import ErroJatai, Registro

    class NaGpu(torch.Tensor):
        is_cuda = property(lambda self: True)

    def z(*forma, tipo=torch.int8):
        return torch.zeros(*forma, dtype=tipo).as_subclass(NaGpu)

    reg, old = Registro(str(tmp_path), "f", eco=False), O.BLK
    try:
        for blk in (32, 128):
            O.BLK = blk
            for R, C in ((4, 2 * blk), (1, blk), (0, blk), (3, 0)):
                reg.confere_bloco("A", (z(R, C), z(R, C // blk)))
                reg.confere_r16("A", (z(R, C, tipo=torch.int16), z(R, C // blk)))
            m, E = z(4, 2 * blk), z(4, 2)
            for a, b, msg in ((z(4, 2 * blk, tipo=torch.int16), E, "mantissa torch.int16"), (m, z(4, 2, tipo=torch.int16), "exponent torch.int16"),
                              (z(2 * blk, 4).t(), E, "mantissa not contiguous"), (m, z(2, 4).t(), "exponent not contiguous"),
                              (z(4, 4 * blk)[:, ::2], E, "mantissa not contiguous"), (z(8 * blk), E, "1 dimensions"),
                              (z(1, 4, 2 * blk), E, "3 dimensions"), (z(4, 2 * blk - 1), E, "not a multiple"), (m, z(4, 3), "exponent shape"),
                              (m, z(2, 4), "exponent shape"), (m, z(8), "exponent shape"), (m, None, "not a tensor"), ([0], E, "not a tensor"),
                              (torch.zeros(4, 2 * blk, dtype=torch.int8), E, "mantissa not on the GPU"),
                              (m, torch.zeros(4, 2, dtype=torch.int8), "exponent not on the GPU")):
                with pytest.raises(ErroJatai, match=msg):
                    reg.confere_bloco("A", (a, b))
    finally:
        O.BLK = old


def test_argumentos_c():
    """An argument as the C call receives it: addresses (null for None and for empty tensors), ints within 32 bits,
    and longer ones; the library's int parameters read the low 32 bits that ctypes passes."""
    import torch
    from jatai_amd.ops import OpsHip
    t = torch.zeros(8, dtype=torch.int8)
    assert OpsHip._a(t).value == t.data_ptr() and OpsHip._a(t[3:]).value == t.data_ptr() + 3
    assert all(not OpsHip._a(x).value for x in (None, torch.empty(0), t[4:4]))
    eco = ctypes.CDLL(None).abs                     # int abs(int): what an int parameter receives
    for x in (0, 1, -1, 2**31 - 1, 1 - 2**31, True):
        assert eco(OpsHip._a(x)) == abs(x)
    for x in (2**31, -2**31, 2**40):
        assert isinstance(OpsHip._a(x), ctypes.c_longlong) and OpsHip._a(x).value == x


def test_linhas_do_tile_sem_gpu():
    """The GEMM's automatic tile on both sides of each line of its rule: tiles per CU, an uneven load, short K, raw
    outputs, the LDS of a long K, and an M that a taller tile does not divide; forced tiles ignore the rule."""
    from jatai_amd.ops import carrega_lib
    lib = carrega_lib()
    antes = lib.jt_bloco_atual()
    try:
        for blk, M, N, K, modo, linhas in (
                (32, 1984, 1024, 512, 0, 32), (32, 2048, 1024, 512, 0, 64),                                    # one 64-row tile per CU
                (32, 2048, 1536, 512, 0, 32), (32, 3584, 1024, 512, 0, 64), (32, 5120, 1024, 512, 0, 32),      # even and uneven loads
                (128, 2048, 1536, 256, 0, 32), (128, 3584, 1024, 256, 0, 64), (32, 9216, 1024, 512, 0, 64),
                (32, 2048, 2048, 32, 0, 32), (32, 2048, 2048, 64, 0, 64), (32, 2048, 2048, 480, 1, 32), (32, 2048, 2048, 512, 1, 64),
                (32, 16384, 2048, 480, 0, 32), (32, 16384, 2048, 512, 0, 64), (128, 2048, 1024, 128, 1, 32), (128, 4096, 1024, 128, 1, 64),
                (32, 2048, 2048, 3936, 4, 64), (32, 2048, 2048, 3968, 4, 128), (32, 2048, 2048, 4096, 0, 128), (32, 2048, 1024, 4096, 0, 32),
                (32, 8256, 1024, 4096, 0, 32), (32, 5120, 1024, 4096, 0, 32), (32, 7168, 1024, 4096, 3, 128), (32, 2048, 2048, 8192, 0, 64),
                (128, 2048, 2048, 256, 4, 128), (128, 2048, 2048, 896, 3, 64), (128, 2048, 2048, 1024, 3, 128),
                (128, 5120, 1024, 384, 0, 32), (128, 7168, 1024, 384, 0, 64), (128, 5120, 1024, 512, 0, 64), (32, 4128, 1024, 512, 0, 32)):
            lib.jt_bloco(blk)
            assert lib.jt_gemm_tile_k(M, N, K, modo) == linhas, (blk, M, N, K, modo)
            if K == 512:
                assert lib.jt_gemm_tile(M, N, modo) == linhas
            for bm in (32, 64, 128):
                lib.jt_gemm_bm(bm)
                assert lib.jt_gemm_tile_k(M, N, K, modo) == max(r for r in (32, 64, 128) if r <= bm and M % r == 0)
            lib.jt_gemm_bm(0)
    finally:
        lib.jt_gemm_bm(0)
        lib.jt_bloco(antes)
