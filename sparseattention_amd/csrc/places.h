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
// units; with more than the caches near an XCD hold, its tiles fetch each other's rows again.  Launches of up to four rounds of workgroups (512 run at once) end
// with their longest lists and take nine planes in any case: with 9 MiB there causal gained half as much (B3 H12 S4096 608 | 539, B1 H24 S8192 1292 | 1221).
// Backward with prepare, us, two by two | this (all planes of an XCD if they are nine or fewer, else as many up to nine as divide them):
//   1/2 MiB a plane: B19 H4, B13 H8, B33 H4, B8 H32 S1024
//     causal        126 | 114 (138)   165 | 135 (154)   191 | 171 (193)   332 | 318 (316)
//     documents     128 | 118 (139)   164 | 135 (162)   190 | 168 (191)   331 | 312 (319)
//     blocks        139, 117 | 126, 110 (144, 126)   168, 149 | 154, 140 (166, 144)   194, 173 | 194, 170 (198, 185)   350, 295 | 337, 301 (351, 294)
//     window of 512 106 | 92 (123)   142 | 119 (135)   165 | 160 (167)   293 | 283 (286)
//     every key     170 | 172 (171)   235 | 227 (209)   268 | 272 (280)   475 | 481 (482)
//   1 MiB: B8 H16, B3 H24, B5 H8 S2048
//     causal        543 | 511 (500)   321 | 290 (295)   196 | 170 (177)
//     documents     321 | 295 (296)   201 | 170 (171)   127 | 108 (112)
//     blocks        558, 492 | 565, 497 (562, 482)   343, 298 | 333, 295 (329, 297)   207, 182 | 209, 172 (209, 173)
//     window of 512 319 | 315 (316)   199 | 183 (187)   125 | 111 (109)
//     every key     841 | 839 (836)   513 | 509 (515)   303 | 304 (302)
//   2 MiB, up to 2048 tiles: B7 H8, B1 H24, B3 H12 S4096
//     causal        792 | 730 (719)   404 | 350 (349)   613 | 501 (506)
//     documents     259 | 239 (243)   151 | 122 (125)   199 | 176 (172)
//     blocks        796, 748 | 831, 759 (822, 769)   404, 388 | 402, 372 (402, 364)   565, 532 | 579, 532 (578, 551)
//     window of 512 295 | 280 (279)   149 | 134 (137)   216 | 204 (200)
//     every key     1330 | 1335 (1317)   632 | 618 (623)   917 | 920 (916)
//   2 MiB, more: B8 H16, B19 H4 S4096
//     causal        1695 | 1632 (1615)   1061 | 1024 (1107)
//     documents     529 | 523 (518)   345 | 330 (357)
//     blocks        1772, 1660 | 1758, 1635 (1814, 1699)   1072, 1019 | 1066, 984 (1075, 1018)
//     window of 512 619 | 616 (612)   377 | 378 (398)
//     every key     2952 | 2979 (2992)   1811 | 1798 (1797)
//   4 MiB: B2 H16, B1 H24 S8192
//     causal        1531 | 1496 (1511)   1283 | 1152 (1154)
//     documents     285 | 280 (285)   242 | 228 (223)
//     blocks        1634, 1603 | 1691, 1654 (1690, 1660)   1266, 1228 | 1279, 1260 (1284, 1250)
//     window of 512 329 | 325 (343)   267 | 249 (247)
//     every key     2885 | 2891 (2918)   2169 | 2194 (2207)
// The passes apart, keys + queries, two by two | with 4.5, 9 and 18 MiB held (two, four and eight planes of B8 H16 S4096):
//   B8 H16 S4096  causal 1187 + 488 | 1179 + 487   1203 + 432   1200 + 412   blocks 1243 + 502 | 1269 + 508   1262 + 510   1282 + 524   every key 2209 + 724 | 2213 + 733   2196 + 745   2205 + 757
//   B8 H16 S2048  causal  346 + 153 |  319 + 151    318 + 146    328 + 140   blocks  378 + 162 |  369 + 167    366 + 159    364 + 178   documents 200 + 88 | 202 + 91   178 + 83   185 + 77
//   B2 H16 S8192  causal 1098 + 408 | 1112 + 439   1115 + 402   1116 + 378   blocks 1201 + 451 | 1176 + 454   1183 + 452   1200 + 470   documents 191 + 79 | 184 + 75   178 + 73   173 + 70
// Runs of one side differ by up to 3 %.
// The three passes in one launch and the two at D = 64 gain nothing by it (D = 64 causal B1 H16 S4096 144 | 138, B8 H16 S1024 92.8 | 94.4).
inline int bwd_spread(int planes, int tiles) {
    if (planes % 4 != 0) return 0;
    const int unit = planes % 8 != 0 ? 4 : 8, each = planes / unit;
    const int held = (9 << 20) / 65536 / tiles, together = (int64_t)planes * tiles <= 4 * 512 && held < 9 ? 9 : held;  // (64 KiB a tile)
    const int most = together < 1 ? 1 : (together < each ? together : each), groups = (each + most - 1) / most;
    return unit * ((each + groups - 1) / groups);
}

}  // namespace sa
