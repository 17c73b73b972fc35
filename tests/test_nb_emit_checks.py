"""upf_nb_emit refuses statistics that no extraction gives before it launches anything (no GPU)."""
import ctypes

import pytest

from unnatural_planets_amd import spec as S


@pytest.mark.parametrize("blocks,vertices,triangles", [(0, 3, 1), (0, 0, 1), (4, -1, 0), (4, 0, -1), (4, -(2 ** 40), 2), (4, 4 * 2187 + 1, 1),
                                                       (4, 3, 4 * 2560 + 1)])
def test_impossible_counts(upf, blocks, vertices, triangles):
    L, g, s = upf.lib(), S.uniform_grid(-1.6, 1.6, 33), S.field_spec("sphere", (1.0,), [])
    room = (ctypes.c_float * 3)()
    st, mb = S.NbStats(), S.MeshBuffers()
    st.blocks, st.active_blocks, st.n_vertices, st.n_triangles = 64, blocks, vertices, triangles
    mb.positions = mb.normals = mb.indices = ctypes.addressof(room)  # never touched
    mb.cap_vertices = mb.cap_triangles = 1 << 40
    size = L.upf_nb_workspace_bytes(ctypes.byref(g), 64)
    assert L.upf_nb_emit(ctypes.byref(s), ctypes.byref(g), 0.0, ctypes.byref(mb), None, ctypes.addressof(room), size,
                         ctypes.byref(st), None) == S.ERR_INVALID_VALUE
    assert mb.n_vertices == mb.n_triangles == 0
