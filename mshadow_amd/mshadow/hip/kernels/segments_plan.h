/*
 * Which sums over dense planes ReduceSegmentsKernel takes, and how it deals the planes out: plain C++, for the
 * library, the expression headers and host code alike.
 */
#ifndef MSHADOW_HIP_KERNELS_SEGMENTS_PLAN_H_
#define MSHADOW_HIP_KERNELS_SEGMENTS_PLAN_H_

#include <stdint.h>

namespace mshadow {
namespace hip {

const uint32_t kSegMostWaves = 16;  //!< waves of a workgroup

/*! \brief how (n, c) planes of `len` elements are dealt out */
struct SegmentsPlan {
  bool use;        //!< false: the kernels of reduce_dma.h and reduce.h are the sooner ones
  int lanes;       //!< planes of a wave
  uint32_t kept, waves;  //!< kept indices and waves of a workgroup
};
/*! \brief few kept indices (fewer than three quarters of the CUs): whether a workgroup that takes all planes of its
 *  index is done before the other kernels would be, which deal the planes of an index out.
 *  The split kernel takes, in us, 8 + 0.08 n or 6 + 0.085 n (its last workgroup's chains) and 8 TB/s of what it reads;
 *  binary16 10 + 0.09 n and 2 TB/s. A workgroup of this kernel takes 3 us and 32 GB/s, 47 where planes begin with their
 *  cache lines (binary16 30 and 39), and an element of a chain 5 ns (binary16 6) where the chains
 *  of a CU are few. As measured, split and this one: floats
 *  (256,16,1024) 29 and 24, (1024,8,1024) 91 and 84, (2048,32,784) 215 and 196, (2048,16,1024) 197 and 166, (200,100,400)
 *  38 and 16, (60,190,1500) 30 and 19; but (512,16,784) 49.4 and 50.7, (512,16,1500) 54 and 93, (1024,16,1500) 105 and
 *  176, (2048,1,784) 151 and 179, (2048,4,2048) 178 and 400, (160,40,2296) 27 and 45, (64,64,12544) 52 and 78. Binary16
 *  (512,16,784) 56 and 32, (826,31,1936) 131 and 95, (64,128,2048) 29 and 15, but (2048,4,2048) 184 and 315; odd planes, which
 *  the generic kernel has otherwise, (512,16,2025) 141 and 96. Short reductions: 32 planes of 196 6.2 and 4.9, 41 of 132
 *  5.6 and 4.7, 128 of 100 8.8 and 6.5, but 64 of 100 5.4 and 5.7, 35 of 56 4.3 and 5.1, binary16 40 of 255 7.7 and 8.4. */
inline bool SegmentsOfFewKept(uint64_t n_out, uint64_t planes, uint64_t len, uint32_t cus, int least_len) {
  const bool half = least_len == 8;
  if (n_out <= 4 && !half) return false;  // a chain lane a plane and nothing to deal out: (2,16,11445) 54 and 58
  if (n_out * len < 1u << 16) {  // the end of a plane costs more: half a slice of 128 halves takes longer
    return n_out > 64 || (len >= 128 && (!half || len >= 256 || len % 128 <= 64));
  }
  /* more planes than the split kernel has room for, which leaves a workgroup per index either way: (2048,48,196) 121 and
     77, (1618,41,100) 75 and 48, (1024,128,100) 49 and 32; binary16 86 and 69, 58 and 54, 39 and 34 */
  if (planes > 65536) return true;
  /* what the generic kernel has otherwise, whose large workgroups (from 2^18 values an index on) are the sooner ones where
     its 16 chain lanes are in use and this kernel has two waves: (10,46,40001) 176 and 199, (16,64,31251) 130 and 139, but
     (8,46,40001) 251 and 143, (16,46,10001) 68 and 52, (16,180,20001) 82 and 71 */
  if (half && len % 2 != 0) return n_out < 9 || n_out > 16 || n_out * len < 1u << 18 || planes >= 100 * n_out;
  const uint64_t bytes = n_out * len * (16u / least_len), all = planes / n_out * bytes;
  const bool lines = bytes / n_out % 128 == 0;
  if (half) {
    const uint64_t split = 10000 + 90 * n_out + all / 2000;  // ns, as below; rates are bytes a ns
    if (bytes > split * (lines ? 39 : 30) || len * 6 > split) return false;
    /* One round of workgroups of the split kernel, 16 planes of whole packs each or 32: it takes, in us, 5 + 0.085 n and 3.5 ns
       an element (5.3 + 0.056 n and 4.4). Of this kernel's chains an element takes 5.5 ns, where there are eight to a wave 6 to
       4, the fewer the more indices are kept and while every wave has a SIMD to itself: (64,46,5000) 28 and 33, (40,46,3000) 20 and 24, (64,64,8000) 38 and 45, (81,50,6384) 34.5 and
       39, but (64,46,1400) 15.4 and 12.9, (72,46,3000) 22 and 19.5, (32,100,2048) 15.2 and 13.5, and in two rounds (64,80,5000) 45
       and 30, (81,64,8000) 65 and 46 */
    const bool packs = len % 8 == 0;
    if (planes > (packs ? 16u : 32u) * cus) return true;
    const uint64_t kept = planes / n_out;
    const uint64_t ps = n_out > 64 ? 5500 : kept < 64 ? 6000 : kept < 96 ? 5000 : n_out > 32 ? 4600 : 4000;  // an element
    return 4500 + len * ps / 1000 <= (packs ? 5000 + 85 * n_out + len * 7 / 2 : 5300 + 56 * n_out + len * 22 / 5);
  }
  const uint64_t split = (n_out <= 400 ? 8000 + 80 * n_out : 6000 + 85 * n_out) + all / 8000;
  return 3000 + bytes / (lines ? 47 : 32) <= split && 3000 + len * 5 <= split;
}
/*! \brief short reductions of many kept indices (fewer than 65536 values of each) that are not this kernel's: mostly where the
 *  ends of their planes - what is left of the last slice of 64 floats or 128 halves: floats come from LDS by packs and are
 *  selected by the plane's length, halves by whole packs and then one by one - cost more than it wins. In us, the kernel of a
 *  workgroup per index and this one: floats (46,409,120) 6.3 and 7.0, (95,745,50) 9.7 and 10.7,
 *  (4,667,756) 8.0 and 10.0, but (65,208,117) 8.8 and 6.7, (4,1928,637) 14.2 and 12.3; binary16 (38,1675,55) 7.3 and 10.9,
 *  (20,346,231) 7.2 and 8.0, (2,1439,1005) 10.2 and 15.9, but (112,335,56) 8.7 and 7.0, (22,422,198) 7.3 and 6.7, (4,1800,840)
 *  level, and planes of two slices and more, (43,835,1275) 38.8 and 27.0. */
inline bool ShortSumsGoElsewhere(uint32_t n_out, uint32_t n_keep, uint64_t planes, uint64_t len, uint32_t cus, int least_len) {
  const bool one_round = n_out > 64 && n_keep <= 2 * cus;  // few workgroups of several rounds each with the other kernel
  if (least_len == 8) {
    if (n_out <= 4) return len % 128 > 72;
    if (n_out <= 16 && len < 256) return true;  // (15,1400,133) 5.1 and 7.1, (9,1400,161) 5.2 and 5.4
    return (len < 128 && !one_round) || (len >= 128 && len < 256 && len % 128 > 72);
  }
  if (n_out <= 4) return n_keep <= cus || (len > 600 && planes < 2800 && len % 64 >= 44);  // (3,220,1000) 6.8 and 7.8
  if (n_out <= 16) {
    /* short planes, (14,600,161) 3.8 and 4.2, (11,686,234) 4.3 and 4.6, and more than the memory-side cache has, (15,8000,2385) 195 and 226, (13,4000,4000)
       151 and 170, but (14,2947,1500) 47 and 37 */
    return (len < (n_out < 9 ? 200u : 256u) && n_keep <= 4 * cus) || (n_out >= 12 && planes * len > 80000000);
  }
  return len < 128 && len % 64 >= 44 && n_out >= 24 && !one_round;
}
/*! \brief kept indices of a workgroup where an index has five to sixteen planes: what two to eight waves hold. What counts are the
 *  waves of the CU that has the most: (14,906,881) two indices and four waves a workgroup, two of those a CU, 10.2 us, three
 *  indices and six waves 12.4; (9,1024,2385) four indices, five waves, one workgroup a CU 16.8, three indices, four waves, two 18.8.
 *  Within an eighth the fewer workgroups: (11,1079,2385) three indices, ten waves a CU 22.7, two, nine waves 24.1. */
inline uint32_t KeptOfMiddling(uint32_t n_out, uint32_t n_keep, uint32_t lanes, uint32_t cus) {
  const uint32_t kMost = 8;
  uint32_t kept[kMost + 1], load[kMost + 1], least = ~0u, best = 1;
  for (uint32_t waves = 2; waves <= kMost; ++waves) {
    kept[waves] = waves * lanes / n_out;
    if (kept[waves] > n_keep / cus) kept[waves] = n_keep / cus;
    if (kept[waves] < 1) kept[waves] = 1;
    const uint32_t groups = (n_keep + kept[waves] - 1) / kept[waves];
    load[waves] = (groups + cus - 1) / cus * ((kept[waves] * n_out + lanes - 1) / lanes);
    if (load[waves] < least) least = load[waves];
  }
  for (uint32_t waves = 2; waves <= kMost; ++waves) {
    if (static_cast<uint64_t>(load[waves]) * 8 <= static_cast<uint64_t>(least) * 9) best = kept[waves];
  }
  return best;
}
/*! \brief Measured on (n, c, len), us, the other kernels and this one; floats, binary16 gains as much.
 *  A workgroup per kept index that fills a CU: (248,552,280) 70 and 42, (30,600,2500) 74
 *  and 44, (19,304,5760) 93 and 35, (5,1144,8320) 115 and 49, (114,246,896) 22 and 18, (248,416,450) 54 and 42, where chain
 *  lanes (n up to the next 64, 16 or 4) and the last round of workgroups are idle for more than a tenth; (64,256,3136) 35.6
 *  and 40, (64,512,1600) 43 and 41, (16,249,5512) 27 and 29.
 *  Up to a kept index a CU there is one round of either, and up to 64 planes an index what counts are the lanes:
 *  (32,192,3136) 28 and 23, (48,192,3136) 29 and 26, but (48,255,3136) 29 and 31, (64,192,3136) 29.5 and 31; binary16
 *  (32,192,3136) 19.5 and 16.8, but (48,192,3136) 19.6 and 21, (64,192,1640) 14.3 and 16.2.
 *  A workgroup of four waves per kept index, for fewer than 65536 values of each: (17,896,260) 11.7 and 7.2,
 *  (39,957,384) 14.9 and 11.9, (5,1519,3920) 63 and 28, (12,1448,592) 15.7 and 9.5, (16,1400,140) 7.1 and 4.9, (2,1912,2048)
 *  25.6 and 13.3, (7,216,3392) 24 and 20, and with few kept indices (24,24,2208) 35 and 18, (28,184,1536) 25.5 and 11.4; small
 *  ones are level within 0.4 us, which is less than their launch. One plane per kept index, which is one lane there:
 *  (1,2048,3136) 46 and 20, (1,536,5184) 36 and 26, (1,512,32768) 144 and 142, (1,1100,50000) 347 and 229, (1,512,400000)
 *  2740 and 1735, but (1,59,3696) 16.5 and 20, (1,512,50000) 203 and 217, (1,1000,40000) 173 and 184, (1,1000,65500) 263 and
 *  298; binary16 (1,72,1392) 8.8 and 7.3, (1,64,200000) 773 and 691, (1,512,50176) 205 and 154. */
inline SegmentsPlan PlanSegments(uint32_t n_out, uint32_t n_keep, uint64_t len, uint32_t cus, int least_len) {
  SegmentsPlan p = {false, 16, 1, 1};
  const uint64_t planes = static_cast<uint64_t>(n_out) * n_keep;
  /* 32-bit numbers of planes, fewer than 2^32 threads */
  if (len < static_cast<uint64_t>(least_len) || n_out < 1 || n_out > 2048 || n_keep > 1u << 21 || len >= 1ull << 31 ||
      planes >= 1ull << 31) {
    return p;
  }
  const bool few_kept = static_cast<uint64_t>(n_keep) * 4 < 3ull * cus;
  const uint32_t side = n_out > 16 ? 64 : n_out > 4 ? 16 : n_out > 1 ? 4 : 1;
  const uint64_t lanes = (n_out + side - 1) / side * side, turns = (n_keep + cus - 1) / cus * cus;
  if (few_kept) {
    p.use = n_out == 1 ? least_len == 8 && n_keep >= 64 && len >= 512 : SegmentsOfFewKept(n_out, planes, len, cus, least_len);
  } else if (n_out == 1) {
    /* up to a workgroup of the other kernel for every SIMD, and long planes below its own limit */
    const bool other = least_len == 4 && n_keep <= 4 * cus && len > 36000 && len < 1u << 16;
    p.use = (n_keep >= 2 * cus && !other) || (least_len == 8 && len >= 512);
  } else if (n_out * len >= 1u << 16) {
    p.use = planes >= 2048 && lanes * turns * 100 > planes * 112;
    if (n_out > 40 && n_out <= 64 && n_keep <= cus) {
      p.use = p.use && least_len == 4 && n_out <= 48 && n_keep * 16ull < 15ull * cus;
    }
  } else {
    p.use = !ShortSumsGoElsewhere(n_out, n_keep, planes, len, cus, least_len);
  }
  if (!p.use) return p;
  /* more waves: (32,512,784) 12.4, with sixteen 13.3; up to two waves a SIMD of a workgroup's CU, which take turns
     beyond that */
  if (len >= 512 && planes / 16 < 4 * cus && n_out <= 64) p.lanes = 8;
  /* workgroups of four waves or so where planes are few per kept index, but one for every CU */
  if (n_out >= 5 && n_out <= 16) {
    p.kept = KeptOfMiddling(n_out, n_keep, p.lanes, cus);
  } else {
    while (p.kept * n_out < 4u * p.lanes && n_keep / (p.kept + 1) >= cus) ++p.kept;
  }
  const uint32_t all = (p.kept * n_out + p.lanes - 1) / p.lanes;
  /* a CU holds 20 waves of this kernel: where there are more of them, small workgroups that go round again fill it,
     but not where few kept indices are few workgroups ((1024,128,100): 62 of them that way, now 32) */
  const uint32_t most = !few_kept && planes / p.lanes >= 20ull * cus ? 4 : kSegMostWaves;
  const uint32_t rounds = (all + most - 1) / most;
  p.waves = (all + rounds - 1) / rounds;
  return p;
}

}  // namespace hip
}  // namespace mshadow
#endif  // MSHADOW_HIP_KERNELS_SEGMENTS_PLAN_H_
