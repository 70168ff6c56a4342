"""Which contraction kernel an apply launches (xtr_op_contract_kernel, what the benchmark reports), and each of them
against the generic per-wavenumber kernel and the oracle on either side of the lines where another one takes over.

Tolerances: a result sums 3 nz <= 258 products, so two orders of summation differ by at most about 258 eps of the sum
of magnitudes, a few times that of the result for random data: 1e-13 (complex128), and 1e-12 against the oracle, whose
transforms differ too; with the transforms in float32 as well 2e-6 (complex64)."""
import os
import re
import struct
import subprocess

import numpy as np
import pytest

from extreme_amd import cartesian_model as cm
from extreme_amd import xtreme as X
from tests.conftest import rel
from tests.test_gpu_folded import _mirror_symmetric_green

pytestmark = pytest.mark.gpu


def _op(oracle, shape, nrhs, precision, seed):
    """An operator with a random tensor, scaled (by the resistivity times the layer thickness) so that the convolution
    is of the size of its input and a wrong block shows as its share of the result."""
    m = cm.small_model(*shape, seed=seed)
    w = cm.omega_of(m.frequencies[0])
    G = {c: g * (1e4 / np.sqrt(3 * m.nz)) for c, g in _mirror_symmetric_green(oracle, m, seed).items()}
    op = X.ConvolutionOperator(m, w, precision=precision, max_rhs=nrhs)
    op.set_green_tensor(G)
    assert op.green_layout()[0] == "folded"
    op.prepare_operator("A")
    return m, w, G, op


def _x(m, nrhs, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal((nrhs, m.n)) + 1j * rng.standard_normal((nrhs, m.n))


# a wave per block from 6 blocks a CU (2 up to 5 layers) on; (24, 20), (20, 20): 525 and 441 blocks; (40, 40), (40, 32): 1681, 1353
@pytest.mark.parametrize("grid,nz,nrhs,direct", [((24, 20), 5, 2, True), ((20, 20), 5, 2, False), ((24, 20), 3, 8, True),
                                                 ((20, 20), 3, 8, False), ((40, 40), 8, 2, True), ((40, 32), 8, 2, False),
                                                 ((40, 40), 10, 5, True), ((40, 32), 10, 5, False), ((40, 40), 11, 2, False)])
@pytest.mark.parametrize("precision,tol_g,tol_o", [("fp64", 1e-13, 1e-12), ("fp32", 2e-6, 2e-6)])
def test_few_layers_on_either_side(oracle, torch_cuda, monkeypatch, grid, nz, nrhs, direct, precision, tol_g, tol_o):
    if torch_cuda.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the grids lie on either side of the line of a chip with 256 CUs")
    m, w, G, op = _op(oracle, (*grid, nz), nrhs, precision, nz + nrhs)
    assert op.contract_kernel(nrhs) is None
    xs = _x(m, nrhs, nz)
    y = op.apply(xs)
    kernel = op.contract_kernel(nrhs)
    assert kernel.startswith(f"contract_{'direct' if direct else 'block'}_kernel<{'double' if precision == 'fp64' else 'float'}, {nz}, ")
    monkeypatch.setenv("XTR_CONTRACT_KERNEL", "generic")
    g = op.apply(xs)
    assert op.contract_kernel(nrhs) == f"contract_kernel<{'double' if precision == 'fp64' else 'float'}>"
    oop = oracle.Operator(m, G)
    oop.prepare("A", m.zeta(w).reshape(-1), m.zeta0(w))
    eg = max(rel(y[r], g[r]) for r in range(nrhs))
    eo = max(rel(y[r], oop.apply(xs[r])) for r in {0, nrhs - 1})
    print(f"{grid} nz {nz} nrhs {nrhs} {kernel}: vs generic {eg:.1e}, vs oracle {eo:.1e}", flush=True)
    assert eg < tol_g and eo < tol_o


@pytest.mark.parametrize("nz,nrhs,precision,layout,kernel", [
    (32, 2, "fp64", None, "contract_block_kernel<double, 32, 2>"), (47, 1, "fp64", None, "contract_block_kernel<double, 47, 1>"),
    (24, 3, "fp64", None, "contract_block_kernel<double, 24, 2>"), (48, 2, "fp64", None, "contract_rows_kernel<double, 1>"),
    (48, 2, "fp32", None, "contract_block_kernel<float, 48, 2>"), (85, 3, "fp64", None, "contract_rows_kernel<double, 2>"),
    (86, 2, "fp64", None, "contract_kernel<double>"), (64, 2, "fp64", None, "contract_fold64_kernel<double>"),
    (64, 3, "fp32", None, "contract_fold64_kernel<float>"), (32, 2, "fp64", "full", "contract_stream_kernel<double>"),
    (64, 2, "fp64", "full", "contract_stream64_kernel<double, 2>"), (24, 2, "fp64", "full", "contract_kernel<double>")])
def test_kernel_by_depth_and_layout(oracle, torch_cuda, monkeypatch, nz, nrhs, precision, layout, kernel):
    if layout:
        monkeypatch.setenv("XTR_GREEN_LAYOUT", layout)
    m = cm.small_model(4, 5, nz, seed=nz)
    op = X.ConvolutionOperator(m, cm.omega_of(m.frequencies[0]), precision=precision, max_rhs=nrhs)
    op.calculate_green_tensor()
    op.prepare_operator("A")
    op.apply(_x(m, nrhs, nz))
    assert op.contract_kernel(nrhs) == kernel
    if nrhs > 1:
        assert op.contract_kernel(1) is None
    with pytest.raises(X.XtrError, match="nrhs"):
        op.contract_kernel(nrhs + 1)


def _spills(tmp_path):
    """{mangled kernel name: spilled vector registers} from the metadata of the library's device code."""
    data, magic, out = open(X.LIB_PATH, "rb").read(), b"__CLANG_OFFLOAD_BUNDLE__", {}
    for at in (m.start() for m in re.finditer(magic, data)):
        count, pos = struct.unpack_from("<Q", data, at + len(magic))[0], at + len(magic) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, pos)
            triple = data[pos + 24:pos + 24 + length]
            pos += 24 + length
            if not triple.endswith(b"gfx950"):
                continue
            (tmp_path / "code").write_bytes(data[at + offset:at + offset + size])
            notes = subprocess.run([os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-readelf"), "--notes",
                                    str(tmp_path / "code")], check=True, capture_output=True, text=True).stdout
            for kernel in re.split(r"\n\s*- \.agpr_count", notes)[1:]:
                name, spilled = re.search(r"\.name:\s*(\S+)", kernel), re.search(r"\.vgpr_spill_count:\s*(\d+)", kernel)
                out[name.group(1)] = int(spilled.group(1))
    return out


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_up_to_four_right_hand_sides_do_not_spill(torch_cuda, tmp_path, precision):
    """A kernel that spills runs its copies in step with its scratch accesses: the dispatch of up to four right-hand
    sides chooses none. From 26 layers on, where groups of four begin (below them no kernel comes near its registers)."""
    spills, seen = _spills(tmp_path), set()
    letter = {"double": "d", "float": "f"}
    for nz in range(26, 64):
        m = cm.small_model(4, 5, nz, seed=nz)
        op = X.ConvolutionOperator(m, cm.omega_of(m.frequencies[0]), precision=precision, max_rhs=4)
        op.calculate_green_tensor()
        op.prepare_operator("A")
        for nrhs in range(1, 5):
            op.apply(_x(m, nrhs, nz))
            name = op.contract_kernel(nrhs)
            t, *args = re.search(r"<(.*)>", name).group(1).split(", ")
            mangled = name.split("<")[0] + "I" + letter[t] + "".join(f"Li{a}E" for a in args) + "E"
            found = [v for k, v in spills.items() if mangled in k]
            assert found and max(found) == 0, (nz, nrhs, name, found)
            seen.add(name)
    assert len(seen) > 38


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-13), ("fp32", 2e-6)])
@pytest.mark.parametrize("nrhs", [1, 2, 3, 4, 8])
def test_every_depth_where_the_convolution_weighs(oracle, torch_cuda, monkeypatch, nrhs, precision, tol):
    worst = (0.0, None)
    for nz in range(1, 86):
        if 3 * nz * nrhs > 1024:
            continue
        m, _, _, op = _op(oracle, (4, 5, nz), nrhs, precision, nz + nrhs)
        xs = _x(m, nrhs, nz)
        y = op.apply(xs)
        kernel = op.contract_kernel(nrhs)
        monkeypatch.setenv("XTR_CONTRACT_KERNEL", "generic")
        g = op.apply(xs)
        monkeypatch.delenv("XTR_CONTRACT_KERNEL")
        e = max(rel(y[r], g[r]) for r in range(nrhs))
        worst = max(worst, (e, kernel))
        assert e < tol, (kernel, e)
    print(f"nrhs {nrhs} {precision}: worst {worst[0]:.1e}, {worst[1]}", flush=True)
