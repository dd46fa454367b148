// Planes side by side: which plane and tile a workgroup of the backward takes (bwd_spread), as sparse_fwd_kernel<..., SD> has it.  Plain C++, so
// that the map can be looked at on the host.
#pragma once

#include <stdint.h>

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
// Place n (8 times the XCD's place, and the XCD) of `planes` planes of `tiles` tiles, `spread` planes together (the last ones: those left): a row of
// tiles of these planes after the other, from the heaviest one on.  Planes that are an odd number of fours are shared by two XCDs: orders 0, 3, 4, 7, 8 ... of a plane on
// one and 1, 2, 5, 6 ... on the other: as much work where it falls evenly, and neighbours, which share keys under a window, by twos.  Orders 0, 2, 4 ...
// on one of them gave it the longer list of every two, in every group of planes.  Backward with prepare, us, in turn | by twos: causal B19 H4
// S1024 142.4 | 137.1, B11 H4 S1536 136.9 | 131.5, window of 512 keys there 97.9 | 91.3; one group of planes and every key within 1.3 %.
SA_PLACES_FN SidePlace side_place(int n, int spread, int planes, int tiles) {
    int group = 0;
    if (spread != planes) {
        group = n / (spread * tiles);
        n -= group * (spread * tiles);
    }
    const int first = group * spread;
    if (planes - first < spread) spread = planes - first;
    int order = n / spread;
    const int plane = first + n - order * spread;
    if ((spread & 4) != 0 && (order | 1) < tiles) order ^= (order >> 1) & 1;
    return {plane, order};
}

// How many planes the passes of the backward with dS walk together: eights of them, or fours that two XCDs share, in groups of even size of which
// an XCD meets no more than 9 MiB (K and V, or q and dO, of the longer side).  Side by side the longest lists of all planes go to different compute
// units; with more than the caches near an XCD hold, its tiles fetch each other's rows again.  Backward with prepare, us, two by two | this
// (all planes of an XCD up to nine, if nine or fewer divide them, else one by one):
//   1/2 MiB a plane: B19 H4, B13 H8, B33 H4, B8 H32 S1024
//     causal        127 | 117 (142)   158 | 139 (161)   192 | 172 (193)   339 | 315 (313)
//     documents     124 | 118 (138)   155 | 133 (162)   190 | 172 (194)   330 | 318 (318)
//     blocks        133, 119 | 130, 111 (140, 127)   166, 149 | 157, 136 (167, 142)   193, 170 | 193, 175 (202, 181)   354, 310 | 348, 299 (346, 303)
//     window of 512 106 | 93 (119)   138 | 127 (136)   169 | 165 (166)   295 | 284 (286)
//     every key     173 | 169 (180)   220 | 219 (216)   281 | 278 (272)   479 | 478 (484)
//   1 MiB: B8 H16, B3 H24, B5 H8 S2048
//     causal        529 | 513 (513)   336 | 299 (290)   196 | 176 (173)
//     documents     321 | 293 (294)   195 | 170 (175)   127 | 111 (109)
//     blocks        566, 499 | 564, 496 (574, 497)   340, 299 | 328, 296 (335, 300)   213, 188 | 211, 177 (208, 172)
//     window of 512 316 | 318 (314)   200 | 184 (187)   126 | 111 (109)
//     every key     851 | 839 (850)   515 | 516 (515)   312 | 303 (314)
//   2 MiB: B8 H16, B7 H8, B1 H24, B3 H12, B19 H4 S4096
//     causal        1696 | 1636 (1634)   803 | 741 (725)   400 | 339 (338)   608 | 539 (485)   1060 | 1040 (1120)
//     documents     539 | 523 (530)   258 | 247 (245)   142 | 123 (124)   194 | 182 (173)   337 | 337 (359)
//     blocks        1774, 1656 | 1808, 1662 (1844, 1711)   810, 770 | 812, 762 (839, 785)   411, 374 | 402, 367 (414, 375)   565, 541 | 568, 523 (577, 537)   1077, 1009 | 1068, 1009 (1094, 1028)
//     window of 512 620 | 619 (608)   287 | 278 (288)   141 | 131 (134)   219 | 208 (200)   378 | 381 (397)
//     every key     2987 | 3034 (3012)   1344 | 1331 (1354)   635 | 635 (627)   934 | 924 (930)   1834 | 1823 (1817)
//   4 MiB: B2 H16, B1 H24 S8192
//     causal        1547 | 1538 (1511)   1292 | 1221 (1163)
//     documents     290 | 303 (284)   238 | 229 (225)
//     blocks        1683, 1621 | 1670, 1649 (1721, 1674)   1275, 1261 | 1283, 1235 (1307, 1277)
//     window of 512 326 | 321 (324)   261 | 251 (251)
//     every key     2917 | 2918 (2916)   2211 | 2189 (2200)
// The passes apart, keys + queries, two by two | with 4.5, 9 and 18 MiB held (two, four and eight planes of B8 H16 S4096):
//   B8 H16 S4096  causal 1187 + 488 | 1179 + 487   1203 + 432   1200 + 412   blocks 1243 + 502 | 1269 + 508   1262 + 510   1282 + 524   every key 2209 + 724 | 2213 + 733   2196 + 745   2205 + 757
//   B8 H16 S2048  causal  346 + 153 |  319 + 151    318 + 146    328 + 140   blocks  378 + 162 |  369 + 167    366 + 159    364 + 178   documents 200 + 88 | 202 + 91   178 + 83   185 + 77
//   B2 H16 S8192  causal 1098 + 408 | 1112 + 439   1115 + 402   1116 + 378   blocks 1201 + 451 | 1176 + 454   1183 + 452   1200 + 470   documents 191 + 79 | 184 + 75   178 + 73   173 + 70
// Runs of one side differ by up to 3 %.  Causal lists of few rounds of workgroups would gain by more planes than that, where blocks lose.
// The three passes in one launch and the two at D = 64 gain nothing by it (D = 64 causal B1 H16 S4096 144 | 138, B8 H16 S1024 92.8 | 94.4).
inline int bwd_spread(int planes, int64_t plane_bytes) {
    if (planes % 4 != 0) return 0;
    const int unit = planes % 8 != 0 ? 4 : 8, each = planes / unit;
    const int64_t held = ((int64_t)9 << 20) / plane_bytes, most = held < 1 ? 1 : (held < each ? held : each);
    const int groups = (int)((each + most - 1) / most);
    return unit * ((each + groups - 1) / groups);
}

}  // namespace sa
