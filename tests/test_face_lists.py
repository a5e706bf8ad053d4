"""The flux kernel's face lists, walked on the CPU as the kernel walks them:
the entry that a cell's slot points at is that slot's face, in regular meshes
and in mesh arrays that list a face twice in a cell, in one of its cells only,
or between a cell and itself."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HARNESS = r"""
#include "layout.hpp"
#include "device.hpp"
using namespace mlr;
// Slots whose list entry is not their face, or -1 - k when a list of block k is malformed.
extern "C" long check_face_lists(uint32_t n_nodes, const double* xy, uint32_t n_cells, const uint32_t* off,
                                 const uint32_t* noc, const uint32_t* foc, uint32_t n_faces, const uint32_t* nof,
                                 const int32_t* cof, uint32_t n_zones, const char* const* names, const uint32_t* zoff,
                                 const uint32_t* zf) {
    const Mesh m = make_from_arrays(n_nodes, xy, n_cells, off, noc, foc, n_faces, nof, cof, n_zones, names, zoff, zf);
    std::vector<BoundarySpec> bcs;
    for (uint32_t z = 1; z < n_zones; ++z) {
        BoundarySpec b;
        b.zone = names[z];
        b.type = (BCType)0;
        bcs.push_back(b);
    }
    const Layout L = build_layout(m, Recon::FO, TenoSpec{}, bcs, 1, false);
    long bad = 0;
    for (uint32_t c = 0; c < L.N; ++c) {
        const uint32_t b = c / 64, first = L.face_off[b], n = L.face_off[b + 1] - first, sum = L.cell_sum[c];
        if (n > 256) return -1 - (long)b;
        const uint32_t count = (sum >> dev::kSumCountShift) & 7u;
        if (count != ((L.info[c] >> 16) & 7u)) return -1 - (long)b;
        for (uint32_t r = 0; r < count; ++r) {
            const uint32_t l = (sum >> (2 * r)) & 3u, i = (L.cell_faces[c] >> (8 * l)) & 0xFFu;
            const size_t o = (size_t)l * L.N + c, e = (size_t)first + i;
            const uint32_t inf = L.info[o], side = (inf >> 2) & 1u, nb = (uint32_t)L.nb[o], nbs = inf & 3u;
            const bool bnd = (inf & kSlotBoundary) != 0;
            bool ok = i < n && ((sum >> (dev::kSumSideShift + l)) & 1u) == side &&
                      (((sum >> (dev::kSumBoundaryShift + l)) & 1u) != 0) == bnd;
            if (ok) {
                const uint32_t meta = L.face_meta[e], s0 = meta & 3u, s1 = (meta >> dev::kFaceSlot1Shift) & 3u;
                ok = L.face_c0[e] == (side ? nb : c) && L.face_c1[e] == (side ? c : nb) &&
                     ((meta & dev::kFaceBoundary) != 0) == bnd &&
                     s0 == (side ? nbs : l) && (bnd || s1 == (side ? l : nbs)) &&
                     L.face_nx[e] == L.nx[o] && L.face_ny[e] == L.ny[o] && L.face_area[e] == L.area[o];
            }
            bad += ok ? 0 : 1;
        }
    }
    return bad;
}
"""


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    d = tmp_path_factory.mktemp("face_lists")
    (d / "h.cpp").write_text(HARNESS)
    lib = os.path.join(ROOT, "mallard_amd", "lib")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "mallard_amd", "csrc"), str(d / "h.cpp"), "-o", str(d / "h.so"),
                    "-L" + lib, "-lmallard_amd", "-Wl,-rpath," + lib], check=True)
    fn = C.CDLL(str(d / "h.so")).check_face_lists
    fn.restype = C.c_long

    def run(a):
        keep = [np.ascontiguousarray(a[k], t) for k, t in (
            ("node_coords", np.float64), ("offsets_nodes_of_cell", np.uint32), ("nodes_of_cell", np.uint32),
            ("faces_of_cell", np.uint32), ("nodes_of_face", np.uint32), ("cells_of_face", np.int32),
            ("zone_offsets", np.uint32), ("zone_faces", np.uint32))]
        names = (C.c_char_p * len(a["zone_names"]))(*[z.encode() for z in a["zone_names"]])
        p = [k.ctypes.data_as(C.c_void_p) for k in keep]
        return fn(C.c_uint32(keep[0].size // 2), p[0], C.c_uint32(keep[1].size - 1), p[1], p[2], p[3],
                  C.c_uint32(keep[4].size // 2), p[4], p[5], C.c_uint32(len(names)), names, p[6], p[7])

    return run


def arrays(oracle, kind, nx, ny):
    """Mesh arrays of a generated mesh in the form Solver(mesh=...) takes."""
    m = oracle.Mesh(kind, nx, ny)
    z = ["interior", "right", "top", "left", "bottom"]
    lists = [np.asarray(m.zones[k], np.uint32) for k in z]
    per = 4 if kind == "cartesian" else 3
    return dict(node_coords=m.node_coords.ravel().copy(), nodes_of_cell=m.nodes_of_cell.ravel().copy(),
                offsets_nodes_of_cell=np.arange(m.n_cells + 1, dtype=np.uint32) * per,
                faces_of_cell=m.faces_of_cell.ravel().copy().reshape(-1, per),
                nodes_of_face=m.nodes_of_face.ravel()[:2 * m.n_faces].copy(),
                cells_of_face=m.cells_of_face.ravel().copy().reshape(-1, 2), zone_names=z,
                zone_offsets=np.concatenate([[0], np.cumsum([len(v) for v in lists])]).astype(np.uint32),
                zone_faces=np.concatenate(lists))


def irregular(oracle, how, nx, ny):
    """self: quads one cell high whose top and bottom are one face of the cell
    with itself. twice: a cell lists one of its faces in two slots, so a
    neighbour's face is listed by the neighbour alone. wrap: the top row's
    neighbours above are the bottom row (two faces between the same cells
    where the mesh is two cells high)."""
    a = arrays(oracle, "cartesian", nx, ny)
    f, c = a["faces_of_cell"], a["cells_of_face"]  # slots: right, top, left, bottom
    moved = []
    if how == "twice":
        for k in range(1, nx * ny, 5):
            f[k, 0] = f[k, 2]
    else:
        for i in range(nx):
            lo, hi = i * ny, i * ny + ny - 1
            top = f[hi, 1]
            f[lo, 3] = top
            c[top] = (hi, lo)
            moved.append(top)
    o, z = a["zone_offsets"], a["zone_faces"]
    lists = [z[o[k]:o[k + 1]] for k in range(5)]
    lists = [np.sort(np.concatenate([lists[0], np.array(moved, np.uint32)])).astype(np.uint32)] + \
            [v[~np.isin(v, moved)] for v in lists[1:]]
    a["zone_offsets"] = np.concatenate([[0], np.cumsum([len(v) for v in lists])]).astype(np.uint32)
    a["zone_faces"] = np.concatenate(lists)
    return a


IRREGULAR = [("self", 1, 1), ("self", 70, 1), ("twice", 9, 9), ("twice", 13, 11), ("wrap", 40, 2), ("wrap", 9, 8)]


@pytest.mark.parametrize("kind,nx,ny", [("cartesian", 1, 1), ("cartesian", 8, 8), ("cartesian", 13, 5),
                                        ("cartesian_tri", 3, 43), ("cartesian_tri", 11, 9)])
def test_regular_meshes(oracle, check, kind, nx, ny):
    assert check(arrays(oracle, kind, nx, ny)) == 0


@pytest.mark.parametrize("how,nx,ny", IRREGULAR)
def test_irregular_arrays(oracle, check, how, nx, ny):
    assert check(irregular(oracle, how, nx, ny)) == 0
