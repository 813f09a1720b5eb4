// m2l_children.h -- neighbour parents of a tile of M2L targets.
#pragma once
#include "device_common.h"
#include "m2l64.h"

namespace lfmm {

// Uniform tables read by scalar loads: pointers into the constant address space.
template <typename V>
using m64_const = const V __attribute__((address_space(4)));
template <typename V>
__device__ __forceinline__ m64_const<V>* m64_scalar(const V* p)
{
    return (m64_const<V>*)(uintptr_t)p;
}
typedef int m64_i2 __attribute__((ext_vector_type(2)));
typedef int m64_i4 __attribute__((ext_vector_type(4)));

typedef double m64_v2 __attribute__((ext_vector_type(2)));

// kids[k][j]: the first child and the child classes present (bit per class)
// of the parent at offset k = 9 (dx + 1) + 3 (dy + 1) + dz + 1 from the parent
// of target j; targets are the children of the parents pbeg .. pend - 1 of the
// level or of its list.  An M2L step then finds its source by one LDS read
// instead of a key interleave, a bounds check and a table lookup per lane.
// Entries K0 .. K1 - 1 only (13: the parent itself).
template <int TILE, int NT, int K0 = 0, int K1 = 27>
__device__ __forceinline__ void m64_children(const M64Level& A, int pbeg, int pend, int2 (*kids)[TILE])
{
    const RtrLevel& L = A.L;
    const int pside = 1 << (L.level - 1);
    for (int e = K0 * TILE + threadIdx.x; e < K1 * TILE; e += NT) {
        const int k = e / TILE, j = e - k * TILE;
        int2 v = make_int2(0, 0);
        if (pbeg + j < pend) {
            const int Pj = L.plist ? L.plist[pbeg + j] : pbeg + j;
            int Pk = Pj;
            if (k != 13) {
                const uint64_t key = A.pkeys[Pj];
                const int px = (int)compact3(key >> 2) + k / 9 - 1, py = (int)compact3(key >> 1) + k / 3 % 3 - 1,
                          pz = (int)compact3(key) + k % 3 - 1;
                Pk = -1;
                if (px >= 0 && py >= 0 && pz >= 0 && px < pside && py < pside && pz < pside)
                    Pk = find_box(morton3(px, py, pz), A.plut, A.pkeys, A.psize);
            }
            if (Pk >= 0) {
                v.x = L.child_begin[Pk];
                const int ce = L.child_begin[Pk + 1];
                for (int i = v.x; i < ce; ++i) v.y |= 1 << (int)(L.child_keys[i] & 7u);
            }
        }
        kids[k][j] = v;
    }
}

// near[k][j]: the index of that neighbour parent at its level, -1 if absent.
template <int TILE, int NT>
__device__ __forceinline__ void m64_parents(const M64Level& A, int pbeg, int pend, int (*near)[TILE])
{
    const RtrLevel& L = A.L;
    const int pside = 1 << (L.level - 1);
    for (int e = threadIdx.x; e < 27 * TILE; e += NT) {
        const int k = e / TILE, j = e - k * TILE;
        int v = -1;
        if (pbeg + j < pend) {
            const int Pj = L.plist ? L.plist[pbeg + j] : pbeg + j;
            const uint64_t key = A.pkeys[Pj];
            const int px = (int)compact3(key >> 2) + k / 9 - 1, py = (int)compact3(key >> 1) + k / 3 % 3 - 1,
                      pz = (int)compact3(key) + k % 3 - 1;
            if (px >= 0 && py >= 0 && pz >= 0 && px < pside && py < pside && pz < pside)
                v = find_box(morton3(px, py, pz), A.plut, A.pkeys, A.psize);
        }
        near[k][j] = v;
    }
}

}  // namespace lfmm
