"""CPU checks of the drop-in boundary: the library loads and exports every
symbol include/acetn_hip.h declares (no compute calls without a GPU)."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    txt = open(os.path.join(ROOT, "include", "acetn_hip.h")).read()
    txt = re.sub(r"/\*.*?\*/", "", txt, flags=re.S)
    return sorted(set(re.findall(r"\b(acetn_hip_\w+)\s*\(", txt)))


def test_header_declares_entry_points():
    syms = declared_symbols()
    assert "acetn_hip_half_projectors" in syms and "acetn_hip_renormalize_boundary" in syms
    assert len(syms) >= 12


def test_library_exports_every_declared_symbol():
    from acetn import _hip
    assert os.path.exists(_hip.LIB_PATH), "build the library first (__graft_entry__.build())"
    lib = ctypes.CDLL(_hip.LIB_PATH)
    missing = [s for s in declared_symbols() if not hasattr(lib, s)]
    assert not missing, missing


def test_hip_backend_refuses_without_gpu():
    import torch
    from acetn import _hip
    if torch.cuda.is_available():
        pytest.skip("GPU present")
    with pytest.raises(RuntimeError):
        _hip.require_gpu()


def test_config_validation():
    import torch
    from acetn.ipeps.ipeps_config import IpepsConfig
    cfg = IpepsConfig(TN={'nx': 2, 'ny': 2, 'dims': {'phys': 2, 'bond': 2, 'chi': 8}},
                      evolution={'backend': 'cutensor'}, device="cpu")
    assert cfg.evolution.backend == "hip"
    assert cfg.device.type == "cuda"
    # the reference's default backend name runs on the engine too
    cfg = IpepsConfig(TN={'nx': 2, 'ny': 2}, evolution={'backend': 'torch'})
    assert cfg.evolution.backend == "hip"
    with pytest.raises(ValueError):
        IpepsConfig(TN={'nx': 2, 'ny': 2}, evolution={'backend': 'numpy'})
    with pytest.raises(TypeError):
        IpepsConfig(TN={'nx': 2, 'ny': 2}, ctmrg={'no_such_key': 1})
    assert IpepsConfig(TN={'nx': 2, 'ny': 2}, dtype="float32").dtype == torch.float64
    assert IpepsConfig(TN={'nx': 2, 'ny': 2}, dtype=torch.float32).dtype == torch.float64
    with pytest.raises(NotImplementedError, match="real"):
        IpepsConfig(TN={'nx': 2, 'ny': 2}, dtype="complex128")


def test_ctmrg_graph_config_raises_while_switched_off():
    """config.graph=True fails before any work while the capture is off
    (runs without a GPU: the check precedes every device call)."""
    from acetn.renormalization.ctmrg import ctmrg

    class C:
        graph = True
    with pytest.raises(NotImplementedError, match="switched off"):
        ctmrg(None, C())


def test_learned_start_network_save_load_roundtrip(tmp_path):
    """MLP.save writes plain tensors that load with weights_only=True; the
    layer sizes are checked (host-side, no kernels)."""
    import torch
    from acetn.evolution.learned_start import MLP
    m = MLP(40, 12, hidden=16, seed=3, device="cpu")
    p = tmp_path / "net.pt"
    m.save(str(p))
    st = torch.load(str(p), weights_only=True)
    assert st["fin"] == 40 and st["hidden"] == 16 and st["fout"] == 12
    m2 = MLP.load(str(p), device="cpu")
    assert torch.equal(m2.params, m.params)
    st["params"] = st["params"][:-1]
    torch.save(st, str(p))
    with pytest.raises(ValueError, match="parameter count"):
        MLP.load(str(p), device="cpu")


def test_boundary_refuses_host_and_non_float64_tensors():
    """The kernels read FP64 device memory: a float32 (or complex) site
    tensor is refused at the boundary instead of being read as FP64 bytes,
    and a host tensor instead of being handed to a kernel as a device
    address (both guards run before any device call)."""
    import torch
    from acetn import _hip
    A = torch.zeros(2, 2, 2, 2, 2, dtype=torch.float64)
    C = [torch.zeros(4, 4, dtype=torch.float64) for _ in range(4)]
    E = [torch.zeros(4, 4, 2, 2, dtype=torch.float64) for _ in range(4)]
    for bad in (torch.float32, torch.complex128):
        with pytest.raises(TypeError, match="float64"):
            _hip.make_site(A.to(bad), C, E)
        with pytest.raises(TypeError, match="float64"):
            _hip.make_site(A, C[:3] + [C[3].to(bad)], E)
    with pytest.raises(ValueError, match="GPU"):
        _hip.make_site(A, C, E)
    with pytest.raises(ValueError, match="GPU"):
        _hip.ptr(A)
    assert _hip.ptr(None).value is None


def _site(D, C_dim, E_dim):
    """An acetn_site whose tensors are never read (a call that fails before
    its first launch)."""
    from acetn import _hip
    s = _hip.AcetnSite()
    s.A, s.D, s.d = 4096, D, 2
    for k in range(4):
        s.C[k] = s.E[k] = 4096
        s.C_dim[k][0], s.C_dim[k][1] = C_dim[k]
        s.E_dim[k][0], s.E_dim[k][1] = E_dim[k]
    return s


@pytest.mark.parametrize("precision", [0, 1, 0x100, 0x101])
@pytest.mark.parametrize("D,dims,chi,p", [
    (3, (51, 3, 9, 1, 1, 6), 23, 9), (1, (1, 4, 41, 12, 2, 15), 36, 1),
    (2, (1, 25, 24, 1, 52, 5), 21, 9), (4, (4, 19, 4, 1, 3, 2), 39, 7),
    (2, (20, 20, 20, 20, 20, 20), 20, 2), (6, (144, 144, 144, 144, 144, 144), 144, 2)])
def test_pair_scratch_does_not_depend_on_trust(D, dims, chi, p, precision):
    """Both phases of a projector pair carve one workspace, the products'
    scratch first: begin and end plan the same scratch with and without
    RF_TRUST.  A workspace of 512 bytes fails at that first buffer, before
    anything is launched, and the message names its size."""
    from acetn import _hip
    lib = _hip.lib()
    ca, cb, n1, n2, x, n4 = dims
    s1 = _site(D, [(ca, cb)] * 4, [(cb, n1), (cb, n1), (cb, n1), (n2, ca)])
    s4 = _site(D, [(x, x)] * 4, [(x, x), (x, x), (n4, x), (x, n2)])
    arr = (ctypes.POINTER(_hip.AcetnSite) * 4)(*[ctypes.pointer(s) for s in (s1, s1, s1, s4)])
    buf = ctypes.create_string_buffer(1024)
    ws = ctypes.cast(buf, ctypes.c_void_p)

    def planned(rc):
        msg = lib.acetn_hip_last_error().decode()
        m = re.match(r"workspace too small: (\d+) bytes at 0 of", msg)
        assert rc != 0 and m, msg
        return int(m.group(1))

    sizes = set()
    for bits in (precision, precision | _hip.RF_TRUST):
        sizes.add(planned(lib.acetn_hip_projectors_begin(
            arr, 0, chi, p, 2, 0.0, 1, 1, 0, 0, bits, ws, None, ws, 512, None)))
        sizes.add(planned(lib.acetn_hip_projectors_end(
            arr, 0, chi, p, 2, 0, 0, bits, 1, ws, ws, ws, 512, None)))
    assert len(sizes) == 1 and sizes.pop() > 512


def test_trust_bit_is_refused_where_no_one_can_start_over():
    """RF_TRUST is a bit of projectors_begin[_mark] and projectors_end; every
    other entry point that takes a precision refuses it, before anything else
    could fail (null outputs and workspaces here)."""
    from acetn import _hip
    lib = _hip.lib()
    s = _site(2, [(4, 4)] * 4, [(4, 4)] * 4)
    one = ctypes.byref(s)
    arr = (ctypes.POINTER(_hip.AcetnSite) * 4)(*[ctypes.pointer(s)] * 4)
    calls = {
        "quarter_tensor": lambda b: lib.acetn_hip_quarter_tensor(one, 0, b, None, None, 0, None),
        "half_projectors": lambda b: lib.acetn_hip_half_projectors(
            one, one, 0, 4, 2, 2, 0.0, 1, 1, b, None, None, None, None, None, 0, None),
        "half_projectors_begin": lambda b: lib.acetn_hip_half_projectors_begin(
            one, one, 0, 4, 2, 2, 0.0, 1, 1, b, None, None, None, 0, None),
        "half_projectors_end": lambda b: lib.acetn_hip_half_projectors_end(
            one, one, 0, 4, 2, 2, b, 1, None, None, None, 0, None),
        "projectors_begin_graph": lambda b: lib.acetn_hip_projectors_begin_graph(
            arr, 0, 4, 2, 2, 0.0, 1, 1, None, 0, 0, b, None, None, None, 0, None),
        "projectors_end_padded": lambda b: lib.acetn_hip_projectors_end_padded(
            arr, 0, 4, 2, 2, 0, 0, b, 1, None, None, None, 0, None),
        "renormalize_boundary": lambda b: lib.acetn_hip_renormalize_boundary(
            one, 0, None, None, 4, None, None, 4, b, None, None, None, None, 0, None),
        "renormalize_boundary_part": lambda b: lib.acetn_hip_renormalize_boundary_part(
            one, 0, 1, 0, None, None, 4, None, None, 4, 4, b, None, None, None, None, 0, None),
    }
    for name, call in calls.items():
        for base in (0, 1, 0x100):
            assert call(base) != 0
            assert "precision" not in lib.acetn_hip_last_error().decode(), name
            assert call(base | _hip.RF_TRUST) != 0
            assert "precision" in lib.acetn_hip_last_error().decode(), name
    # the pair's own two calls take it (and fail on what else is missing)
    for call in (lambda: lib.acetn_hip_projectors_begin(
                     arr, 0, 4, 2, 2, 0.0, 1, 1, 0, 0, _hip.RF_TRUST, None, None, None, 0, None),
                 lambda: lib.acetn_hip_projectors_end(
                     arr, 0, 4, 2, 2, 0, 0, _hip.RF_TRUST, 1, None, None, None, 0, None)):
        assert call() != 0
        assert "null" in lib.acetn_hip_last_error().decode()
