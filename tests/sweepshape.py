"""sweep_shape of csrc/sweep.h (host code), compiled for the host and called
through ctypes: the tile, threads and x chunk of a sweep's launch."""
import ctypes
import os
import subprocess

from opesci import compilation

SOURCE = r"""
#include "sweep.h"
using namespace opesci;
template <int M>
static void fill(const Geom& g, const InteriorLaunch& cfg, int bytes, int elem, int per_cu, int row_items, int* out) {
    const SweepShape s = sweep_shape<M>(g, cfg, nullptr, bytes, elem, [&](int) { return per_cu; }, row_items);
    const int v[] = {s.tile.rows, s.tile.ntz, s.threads, s.nb, s.boxes.xc[0], s.boxes.tyn[0], SweepPlane<M>::SIZE,
                     sweep_second_halo<M>()};
    for (int i = 0; i < 8; ++i) out[i] = v[i];
}
extern "C" void shape(const int* dims, int m, int pitch, const int* cfg, int bytes, int elem, int per_cu, int row_items,
                      int* out) {
    Geom g = {};
    g.nx = dims[0], g.ny = dims[1], g.nz = dims[2];
    g.m = m;
    g.pitch = pitch;
    g.sy = pitch;
    g.sx = (int64_t)g.ny * pitch;
    const InteriorLaunch c{cfg[0], cfg[1], cfg[2]};
    m == 1   ? fill<1>(g, c, bytes, elem, per_cu, row_items, out)
    : m == 2 ? fill<2>(g, c, bytes, elem, per_cu, row_items, out)
    : m == 3 ? fill<3>(g, c, bytes, elem, per_cu, row_items, out)
             : fill<4>(g, c, bytes, elem, per_cu, row_items, out);
}
"""
NAMES = ('rows', 'ntz', 'threads', 'nb', 'xc', 'tyn', 'plane', 'second')


def build(folder):
    """shape(dims, m, cfg, elem, ...) -> dict, from the sources as they are"""
    src, lib = os.path.join(str(folder), 'shape.hip'), os.path.join(str(folder), 'shape.so')
    with open(src, 'w') as f:
        f.write(SOURCE)
    subprocess.run([compilation.HIPCC, '--offload-host-only', '-O1', '-std=c++17', '-fPIC', '-shared', '-I',
                    compilation.CSRC, '-I', compilation.INCLUDE, src, '-o', lib], check=True)
    fn = ctypes.CDLL(lib).shape

    def shape(dims, m, cfg=(0, 0, 0), elem=4, bytes_per_point=60, per_cu=3, row_items=0):
        align = 128 // elem
        pitch = (dims[2] + align - 1) // align * align
        out = (ctypes.c_int * 8)()
        fn((ctypes.c_int * 3)(*dims), m, pitch, (ctypes.c_int * 3)(*cfg), bytes_per_point, elem, per_cu, row_items, out)
        return dict(zip(NAMES, out), pitch=pitch)
    return shape
