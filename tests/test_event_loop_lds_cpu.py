"""The LDS of the event loop: whatever is accepted (by the layout of the earlier
event tree, up to 64 KiB) fits a CU's 160 KiB as the loop lays it out now."""
import ctypes as C
import itertools

from spatialpy_amd import _abi

NSM = "_ZN3ssa13nsm_lds_bytesEiiiiii"       # nsm_lds_bytes(nodes, S, R, T, n_code, n_consts)
SSA = "_ZN3ssa13ssa_lds_bytesEiiiiiiii"     # ssa_lds_bytes(tree_nodes, S, R, T, nnzN, nnzG, n_code, n_consts)


def test_what_is_accepted_fits():
    lib = _abi.load_library()
    nsm, ssa = lib[NSM], lib[SSA]
    nsm.restype, ssa.restype = C.c_size_t, C.c_size_t
    most = 0
    for nodes, S, R, T, code in itertools.product((1, 64, 1024, 4096), (1, 2, 8, 16), (0, 1, 6, 16), (1, 2, 63),
                                                  (0, 1, 3000, 11000, 15000)):
        consts = code // 16
        # the least tables of such a model: no stoichiometry, no dependencies
        if ssa(nodes, S, R, T, 0, 0, code, consts) > 65536:
            continue
        most = max(most, nsm(nodes, S, R, T, code, consts))
    assert 65536 < most <= 160 << 10
