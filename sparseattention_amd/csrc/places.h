// Planes side by side: which plane and tile a workgroup of the backward takes (bwd_spread), as sparse_fwd_kernel<..., SD> has it.  Plain C++, so
// that the map can be looked at on the host.
#pragma once

#ifdef __HIPCC__
#define SA_PLACES_FN __host__ __device__ __forceinline__
#else
#define SA_PLACES_FN inline
#endif

namespace sa {

// Which of an XCD's `per` places its i-th workgroup takes: the second 32, which come to the compute units of the first 32, the other way round.
SA_PLACES_FN int side_turn(int i, int per) { return (i >> 5) == 1 && (i | 31) < per ? i ^ 31 : i; }

struct SidePlace {
    int plane, order;  // order 0: the tile that is heaviest under causal-like masks
};
// Place n (8 times the XCD's place, and the XCD) of `planes` planes of `tiles` tiles, `spread` planes together: a row of tiles of these planes
// after the other, from the heaviest one on.  Planes that are an odd number of fours are shared by two XCDs: orders 0, 3, 4, 7, 8 ... of a plane on
// one and 1, 2, 5, 6 ... on the other: as much work where it falls evenly, and neighbours, which share keys under a window, by twos.  Orders 0, 2, 4 ...
// on one of them gave it the longer list of every two, in every group of planes.  Backward with prepare, us, in turn | by twos: causal B19 H4
// S1024 142.4 | 137.1, B11 H4 S1536 136.9 | 131.5, window of 512 keys there 97.9 | 91.3; one group of planes and every key within 1.3 %.
SA_PLACES_FN SidePlace side_place(int n, int spread, int planes, int tiles) {
    int group = 0;
    if (spread != planes) {
        group = n / (spread * tiles);
        n -= group * (spread * tiles);
    }
    int order = n / spread;
    const int plane = group * spread + n - order * spread;
    if ((spread & 4) != 0 && (order | 1) < tiles) order ^= (order >> 1) & 1;
    return {plane, order};
}

}  // namespace sa
