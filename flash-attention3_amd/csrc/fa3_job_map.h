// XCD-aware job map of the main kernels' default plans and of the split
// plan's descriptors: which (group, position) each workgroup id runs (job_of
// in fa3_bwd_main_kernel.h reads the fields set here).  Host code.
#pragma once

#include <algorithm>

#include "fa3_bwd_main_kernel.h"
#include "fa3_bwd_reg_kernel.h"

namespace fa3 {

// An XCD runs its K virtual groups one after another, or position by
// position across them (longest jobs of all of them first).  Run one after
// another, the last group's longest job starts when about share / K of a
// CU's share of the work is left, and may set the kernel's end; one group at
// a time keeps the XCD's L2 on fewer heads.  The map interleaves with at
// most kInterleaveJobsPerCu jobs per CU, or when the longest job is at least
// kInterleaveTail x share / K (all in dKV steps) and the XCD's virtual
// groups belong to at most kInterleaveSpan groups.  Measured: B1 H9 S2048
// D128 causal -20.7 % (2.25 jobs per CU), B1 Hq28 Hkv7 S4096 -20.2 % (8.75,
// longest 256 against share / K 57), B1 H19 S4096 -4.3 % (9.5; 64 against
// 14; 3 groups per XCD); interleaving P4 (20 per CU; 256 against 455) left
// its time unchanged and raised its L2 misses 1.9x, B1 H36 S4096 (18; 64
// against 57) +6.9 %, B2 H24 S2048 D64 (12; 32 against 29) +1.3 %, P5 (32;
// 128 against 896) +6.5 %, B8 H16 S1024 D128 (16; 16 against 7.4, but 16
// groups per XCD) +20 %, B4 H32 S1024 +20 %.
inline constexpr int kInterleaveJobsPerCu = 8;
inline constexpr double kInterleaveTail = 2.0;
inline constexpr int kInterleaveSpan = 4;

// The smallest split of the groups into parts that deals whole parts to the
// XCDs: n_groups * parts % 8 == 0.
inline int xcd_split(int n_groups) {
    int gcd8 = 8;
    while (n_groups % gcd8 != 0) gcd8 >>= 1;
    return 8 / gcd8;
}

// XCD-aware job map of a.n_groups groups of a.jobs_per_group jobs, an XCD's
// groups one after another or interleaved (A: FusedArgs, or RegArgs of
// fa3_bwd_reg_kernel.h); by_parts false: without the XCDs' parts.
template <typename A, typename Choose>
inline void set_job_map_with(A& a, Choose&& interleave_of, bool by_parts = true) {
    const int parts = xcd_split(a.n_groups);
    const bool fits = by_parts && a.jobs_per_group % parts == 0;
    a.xcd_parts = fits ? parts : 0;
    a.xcd_vgroups = fits ? a.n_groups * parts / 8 : 0;
    // the groups an XCD's virtual groups belong to (one more where its
    // first part is not a group's first)
    const int span = fits ? (a.xcd_vgroups + parts - 1) / parts : a.n_groups;
    const bool interleave = interleave_of(span);
    a.xcd_interleave = interleave ? 1 : 0;
    a.xcd_mode = a.xcd_parts | a.xcd_interleave << 8;
    a.map_radix = !fits ? 0 : interleave ? a.xcd_vgroups : a.jobs_per_group / parts;
    a.div_parts = make_fastdiv(a.xcd_parts);
    a.div_radix = make_fastdiv(a.map_radix);
    a.div_jpg = make_fastdiv(a.jobs_per_group);
    a.div_groups = make_fastdiv(a.n_groups);
}

// The map of bwd_main_kernel's plans.  longest: the longest job, share: a
// CU's share of the work (both in dKV steps), cus: the CU count -- for the
// interleave choice above (the defaults: one group after another).
inline void set_job_map(FusedArgs& a, double longest = 0.0, double share = 1.0, int cus = 0) {
    set_job_map_with(a, [&](int span) {
        const long long jobs = (long long)a.n_groups * a.jobs_per_group;
        return jobs <= (long long)kInterleaveJobsPerCu * cus ||
               (span <= kInterleaveSpan && longest * a.xcd_vgroups >= kInterleaveTail * share);
    });
}

// The map of bwd_reg_kernel's launches (seqlen, group, chunks, heads and
// n_groups set).  Always position by position across an XCD's groups, longest
// jobs first: the hardware deals the jobs out in this order, and with small
// workgroups a late long job costs more than the L2 gains from one group at a
// time (bf16: B2 Hq32 Hkv8 S4096 D128 causal 914 -> 798 us, B4 H16 S1024 80.5
// -> 70.1, B4 H16 S2048 261.5 -> 230.7, B1 H16 S8192 771 -> 755; full attention,
// B2 H12 S1664 D64 68.3 -> 61.4, B2 H16 S8192 D64 1 521 -> 1 541, where five
// times the algorithmic bytes are fetched).
// Groups cut into parts of one job have no order inside an XCD: all roles and
// lengths come mixed, group after group.  With three heads per dKV job or more,
// which is then several times as long as a dQ job, the positions run across
// all groups instead (106 shapes of S 128 and 256, parts -> across against
// bwd_main_kernel: D 128 0.93, up to 1.10 -> 0.81, up to 0.85; D 64 0.82 -> 0.68);
// so they do at D 128 causal with one head and parts of one or two jobs, S >=
// 512 (67 shapes: 0.95, up to 1.05 -> 0.87, up to 0.91).  Elsewhere the parts' L2
// gain is worth as much or more (across 0.9 to 1.25 of their time).
inline void set_reg_job_map(RegArgs& r, const RegPlan& plan, int head_dim, bool causal) {
    r.jobs_per_group =
        r.seqlen / 128 * (std::max(plan.split_kv, 1) * r.chunks + plan.split_q * r.group) +
        plan.halved * r.chunks;
    const int parts = xcd_split(r.n_groups);
    const int most = r.heads > 2 ? 1
                     : r.heads == 1 && head_dim == 128 && causal && r.seqlen >= 512 ? 2
                                                                                     : 0;
    set_job_map_with(r, [](int) { return true; },
                     parts < 4 || r.jobs_per_group > most * parts);
}

}  // namespace fa3
