// Main FA3 backward kernel for gfx950: the fast instantiations and the host
// side (job map, split plan, workspace plan, launch).  The kernels and their
// device helpers are in fa3_bwd_main_kernel.h.
#include "fa3_bwd_main_kernel.h"
#include "fa3_bwd_reg_kernel.h"
#include "fa3_job_map.h"
#include "fa3_split_plan.h"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <memory>
#include <mutex>
#include <random>
#include <vector>

namespace fa3 {
namespace {

FusedArgs base_args(const BwdProblem& p, const BwdTensors& t) {
    FusedArgs a{};
    a.q = (const _Float16*)t.q;
    a.k = (const _Float16*)t.k;
    a.v = (const _Float16*)t.v;
    a.dout = (const _Float16*)t.dout;
    a.dq = t.dq;
    a.dk = t.dk;
    a.dv = t.dv;
    a.out_f32 = p.out_f32 ? 1 : 0;
    a.q_rs = p.bshd ? p.heads_q * p.head_dim : p.head_dim;
    a.q_hs = p.bshd ? p.head_dim : p.seqlen * p.head_dim;
    a.kv_rs = p.bshd ? p.heads_kv * p.head_dim : p.head_dim;
    a.kv_hs = p.bshd ? p.head_dim : p.seqlen * p.head_dim;
    a.seqlen = p.seqlen;
    a.heads_q = p.heads_q;
    a.heads_kv = p.heads_kv;
    a.group = p.heads_q / p.heads_kv;
    a.div_hq = make_fastdiv(p.heads_q);
    a.div_hkv = make_fastdiv(p.heads_kv);
    a.div_group = make_fastdiv(a.group);
    a.div_g1 = make_fastdiv(a.group + 1);
    a.n_groups = p.batch * p.heads_kv;
    a.scale_log2 = p.scale * kLog2e;
    a.scale = p.scale;
    a.spin_limit = 1;
    return a;
}

std::atomic<int> g_spin_limit{1 << 24};
std::atomic<bool> g_debug_kernels{false};

// Compute units of device `dev` (cached per device); 0 if unknown.
int cu_count(int dev) {
    static std::mutex mu;
    static int cache[64] = {};
    if (dev < 0 || dev >= 64) return 0;
    std::lock_guard<std::mutex> lock(mu);
    if (cache[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return 0;
        cache[dev] = n;
    }
    return cache[dev];
}

// Epochs: a process-wide counter started at a random 64-bit value, so a
// word left in a workspace by an earlier launch (of this or another
// process) practically never equals the current launch's epoch.  The
// launches of this process have used the epochs [g_epoch0, g_epoch) (0
// skipped), which lets the host tell an error word written by one of them
// from whatever an uninitialised workspace holds.
unsigned long long epoch_seed() {
    std::random_device rd;
    unsigned long long x = ((unsigned long long)rd() << 32) ^ rd();
    x ^= (unsigned long long)std::chrono::steady_clock::now().time_since_epoch().count();
    return x | 1;
}
const unsigned long long g_epoch0 = epoch_seed();
std::atomic<unsigned long long> g_epoch{g_epoch0};

unsigned long long next_epoch() {
    unsigned long long e;
    do e = g_epoch.fetch_add(1, std::memory_order_relaxed);
    while (e == 0);
    return e;
}

// size_t arithmetic that reports overflow instead of wrapping
struct Checked {
    size_t v = 0;
    bool ok = true;
    Checked add(size_t x) const {
        Checked r = *this;
        r.ok = ok && !__builtin_add_overflow(v, x, &r.v);
        return r;
    }
    Checked mul(size_t x) const {
        Checked r = *this;
        r.ok = ok && !__builtin_mul_overflow(v, x, &r.v);
        return r;
    }
    Checked align() const { return add(255).and_mask(); }
    Checked and_mask() const {
        Checked r = *this;
        r.v &= ~(size_t)255;
        return r;
    }
};

}  // namespace

void set_split_spin_limit(int polls) { g_spin_limit.store(polls < 0 ? 0 : polls); }

void set_debug_kernels(bool on) { g_debug_kernels.store(on); }

bool epoch_issued(unsigned long long word) {
    return word != 0 && word - g_epoch0 < g_epoch.load(std::memory_order_relaxed) - g_epoch0;
}

// Workspace of the no-allocation entry.  Each GPU holds its own copy of the
// array; in host code `scratch` is only a handle for the runtime, never a
// device address, so the kernels receive the address hipGetSymbolAddress
// reports for the launch's device.  Nothing in it needs clearing between
// calls: the split words are tagged with each launch's epoch, and everything
// else is written before it is read within a call.
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];
// Split waits that gave up on this GPU since the library was loaded (the
// kernels count them; shaobo_fa3_ext_split_error_count reads them).
static __device__ unsigned long long split_giveups[1];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_symbol_mu;
void* g_scratch_ptr[kMaxDevices] = {};
void* g_giveups_ptr[kMaxDevices] = {};

// Device address of a __device__ array on device dev, looked up once per
// device with that device current (the caller's launches run on it).
hipError_t symbol_address(int dev, const void* symbol, void* (&cache)[kMaxDevices], void** ptr) {
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_symbol_mu);
    if (cache[dev] == nullptr) {
        int cur = -1;
        hipError_t e = hipGetDevice(&cur);
        if (e != hipSuccess) return e;
        if (cur != dev) return hipErrorInvalidDevice;
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, symbol);
        if (e != hipSuccess) return e;
        if (p == nullptr) return hipErrorInvalidSymbol;
        cache[dev] = p;
    }
    *ptr = cache[dev];
    return hipSuccess;
}
}  // namespace

hipError_t noalloc_scratch(int dev, void** ptr) {
    return symbol_address(dev, HIP_SYMBOL(scratch), g_scratch_ptr, ptr);
}

hipError_t split_giveup_count(int dev, unsigned long long** ptr) {
    void* p = nullptr;
    const hipError_t e = symbol_address(dev, HIP_SYMBOL(split_giveups), g_giveups_ptr, &p);
    *ptr = static_cast<unsigned long long*>(p);
    return e;
}

// The split plan runs its workgroups in one round: past one job per CU the
// default plan (one job per workgroup, or the persistent queues from 512
// jobs on) measured faster for every shape tried -- 384 jobs: B1 H12 S1024
// D128 -18 %, B1 H6 S2048 D64 -24 %; 512 jobs: B1 H8 S2048 D128 -4.8 %,
// B1 H2 S8192 D64 -10.6 %, B1 H16 S1024 D64 +0.3 %.
constexpr long long kSplitMaxJobs = 256;
static_assert(kSplitMaxJobs <= kMaxSplitWgs, "one descriptor per split-plan workgroup");

// Head-split plan choice.  Work in dKV steps (a dQ step ~0.75 of one); a
// CU's share = all steps / kHeadSplitCus (an MI355X's CU count: the plan,
// and so the workspace size, depends on the shape only).  The merged plan
// takes max(share, G QT) -- its longest job, G heads' query tiles against
// key tile 0 -- and chunks of G / f heads take max(share, G QT / f), times
// 1 + kHeadSplitPerChunk f (the fp32 contributions' traffic and the extra
// prologues), plus kHeadSplitFixed for the reduction launch.  The plan picks
// the f with the least estimate, if it is below kHeadSplitGain x the merged
// plan's: near the boundary the estimate's error exceeds the gain (B2 Hq16
// Hkv4 S2048 D128 causal: estimated -3 %, measured +9 %).  Measured (D 128
// causal): 32 chunks at B1 Hq32 Hkv1 S4096 run each step of the share ~12 %
// slower than the merged plan runs a full machine's; 8 chunks there take
// the backward from 1 596 to 532 us, 2 chunks at B4 from 2 099 to 1 982.
constexpr int kHeadSplitCus = 256;
constexpr double kHeadSplitPerChunk = 0.004;
constexpr double kHeadSplitFixed = 8.0;
constexpr double kHeadSplitGain = 0.92;
constexpr int kHeadSplitMaxChunks = 64;

// The chunk count f (a divisor of G, >= 2) of the head-split plan for this
// shape, or 0 for the merged plan.  (G QT > share needs QT + 1 < 2 x 256 /
// (1.75 B Hkv) causal, QT < 256 / (1.75 B Hkv) full: the plan never meets a
// sequence long enough to strain the reduction's 32-bit indices.)
int head_split_chunks(const BwdProblem& p, int qt) {
    const int group = p.heads_kv > 0 ? p.heads_q / p.heads_kv : 0;
    if (group < 2 || qt <= 0 || p.out_f32 || p.no_head_split) return 0;
    const double steps = p.causal ? 0.5 * qt * (qt + 1.0) : (double)qt * qt;
    const double share = (double)p.batch * p.heads_q * steps * 1.75 / kHeadSplitCus;
    const double merged = std::max(share, (double)group * qt);
    int best = 0;
    double best_t = kHeadSplitGain * merged;
    // beyond 64 chunks the chunks' own cost (+26 %) outweighs any split
    for (int f = 2; f <= std::min(group, kHeadSplitMaxChunks); ++f) {
        if (group % f != 0) continue;
        const double t = std::max(share, (double)(group / f) * qt) * (1.0 + kHeadSplitPerChunk * f) +
                         kHeadSplitFixed;
        if (t < best_t) {
            best_t = t;
            best = f;
        }
    }
    return best;
}

WorkspacePlan plan_workspace(const BwdProblem& p) {
    WorkspacePlan w;
    if (p.batch <= 0 || p.heads_q <= 0 || p.seqlen <= 0 || p.head_dim <= 0) return w;
    const Checked rows = Checked{(size_t)p.batch}.mul((size_t)p.heads_q).mul((size_t)p.seqlen);
    Checked at{256};  // the error word's region
    w.err_off = kErrWordOffset;
    w.nlse2_off = at.v;
    at = at.add(rows.mul(sizeof(float)).v).align();
    w.ndelta_off = at.v;
    at = at.add(rows.mul(sizeof(float)).v).align();
    w.queue_off = at.v;
    at = at.add(kQueueBytes).align();
    if (!rows.ok) return w;
    // Split plan for causal shapes with one query head per KV head and few
    // jobs (at most one per CU of an MI355X): see bwd_main_kernel.
    const int qt = p.seqlen / kTileM;
    const long long jobs = 2LL * p.batch * p.heads_q * qt;
    if (p.causal && p.heads_q == p.heads_kv && qt >= 4 && qt % 2 == 0 && jobs <= kSplitMaxJobs) {
        w.bal_m = qt / 2;  // <= kMaxBalM since jobs <= kSplitMaxJobs
        w.n_split = p.batch * p.heads_q * w.bal_m;
        const size_t kv_piece = (size_t)4 * 2 * (p.head_dim / 64) * 4096;
        const size_t q_piece = (size_t)4 * (p.head_dim / 64) * 4096;
        w.sync_off = at.v;
        at = at.add((size_t)w.n_split * 4 * sizeof(unsigned long long)).align();
        w.pkv_off = at.v;
        at = at.add((size_t)w.n_split * kv_piece).align();
        w.pq_off = at.v;
        at = at.add((size_t)w.n_split * q_piece).align();
        // the kernel addresses the partial sums with 32-bit buffer offsets
        if (w.pq_off - w.pkv_off > 0xFFFFFFFFull || at.v - w.pq_off > 0xFFFFFFFFull) return w;
    }
    // Head-split default plan for GQA: when one dKV job (G heads' query
    // tiles against one key tile) is much longer than a CU's share of the
    // work, it alone sets the kernel's length (MQA at batch 1), so each dKV
    // job runs for a chunk of the heads and the chunks' fp32 contributions
    // are summed afterwards.
    if (w.bal_m == 0) {
        w.hs_chunks = head_split_chunks(p, qt);
        if (w.hs_chunks > 0) {
            w.hsd_off = at.v;
            const Checked parts = Checked{(size_t)p.batch}
                                      .mul((size_t)p.heads_kv)
                                      .mul((size_t)w.hs_chunks)
                                      .mul((size_t)p.seqlen)
                                      .mul((size_t)p.head_dim);
            at = at.add(parts.mul(sizeof(float) * 2).v).align();
            if (!parts.ok) return w;
        }
    }
    if (!at.ok || !rows.ok || rows.v > (size_t)INT32_MAX) return w;
    w.total = at.v;
    w.ok = true;
    return w;
}

// Which launches run the register-operand kernel, and how it cuts its jobs.
// Work in units of 128 keys x 64 query rows of a dKV job (a dQ unit ~0.75):
// share = a CU's part of it, longest = the longest dKV job of 128 keys
// (group / chunks heads' query rows).  x = longest / share decides between
// the kernels, because two (D 128) or three (D 64) workgroups share a CU and
// each then runs at a part of its speed, while bwd_main_kernel's one
// workgroup has the CU to itself.  Measured against bwd_main_kernel over 110
// random shapes (bf16, both head dims, causal and full, G 1..8):
//   x <= 0.75: -6 to -40 %;
//   0.75 < x <= 1.3: G > 1 -3 to -21 % (with its longest dKV jobs halved,
//     below), but with one head per dKV job (G = 1, or a chunk per head) a dQ
//     job is as long as a dKV job.  G = 1: both halved from 0.9 on, -4 to
//     -33 % at D 64, within 5 % at D 128, which stays with bwd_main_kernel.
//     D 64 causal: from 0.6 on for S >= 512 (109 shapes of 0.6 .. 0.9, whole ->
//     both halved against bwd_main_kernel: S >= 2048 0.97, up to 1.11 -> 0.85,
//     up to 0.91; S 1024 .. 2047 0.91 -> 0.79; S 512 .. 1023 0.77 -> 0.72;
//     below S 512 equal).
//     A chunk per head (x in 0.75 .. 1.3, 320 shapes, dKV halved alone -> the
//     rule, both against bwd_main_kernel): D 64 full from 1.12 on +2 to +25 %
//     -> -5 to -10 % with both halved, causal up to +28 % -> -12 to -20 %
//     (below S 512 dKV halved alone is 3 to 7 % faster up to 1.12);
//     D 128 full below 1.12 -7 to -12 %, above +2 to +15 %, and causal the
//     longer the sequence the worse (S 256, 512: -4 to -13 %; S 1024 .. 2047:
//     -1 to -5 % below 1.12, +2 to +6 % above; S >= 2048: +1 to +19 %; S 128:
//     +5 % above 1.12): those run bwd_main_kernel;
//     D 64 causal with more heads and S >= 3072 is up to 9 % slower than
//     bwd_main_kernel from 1.15 on (354 shapes, 4 % on average), but not than
//     its unscaled instantiation (below), and stays;
//   x > 1.3: bwd_main_kernel.  Whole jobs are 8 to 100 % slower there the fewer
//     they are; with every dKV job halved (both roles with one head) 1.3 .. 1.6
//     is 5 to 18 % faster on average, single shapes up to 14 % slower.
// Launches below 1.3 with G > 1 that bwd_main_kernel runs take its unscaled
// instantiation: S c in fp32 as in this kernel, not K c or Q c rounded (fp16
// error against 64 bits 3.0e-4, scaled 3.7e-4), at the same speed (1 859 shapes
// at D 128: 1.000 of the scaled one's time, up to 1.08).
// A dKV job longer than a workgroup slot's share sets the launch's end: such
// tiles run as two jobs of 64 keys, at ~10 % more per unit.  Causal, only the
// longest tiles (B2 Hq32 Hkv8 S2048 D128, of 16 tiles 0 / 4 / 8 / 12 / 16
// halved: 315 / 263 / 233 / 236 / 245 us, the rule 9; B1 Hq32 Hkv1 S4096, of
// 32 tiles 0 / 8 / 16 / 20 / 32: 622 / 510 / 449 / 431 / 451, the rule 18; B2
// Hq32 Hkv8 S4096 within 1 % from 0 to 12, the rule 4).  Against whole or all
// halved by x alone, with the longest jobs at raised priority: B4 Hq20 Hkv5
// S384 40.4 -> 36.5 us, B1 Hq32 Hkv16 S3328 296.2 -> 287.5, B2 Hq32 Hkv8 S2048
// 221.9 -> 219.8, S4096 827.9 -> 820.2, B4 Hq12 Hkv3 S2304 229.1 -> 230.5; the
// priority alone is worth at most 1.5 % either way and went.
// With one head per dKV job the dQ jobs are as long and stay whole at D 128,
// so halving dKV only adds work: none from 0.54 to 0.75 (103 shapes against
// bwd_main_kernel: the line above 0.93 on average and up to 1.08, none halved
// 0.84, up to 1.05; nearer 0.5 the line halves a tile or two, as fast).
// Full attention's jobs of a role are all alike, so all are halved or none:
// halved from 0.9 on, with these other lines (times against bwd_main_kernel):
//   D 64, more than one head, S >= 512: from 0.7 on (71 shapes of 0.7 .. 0.9,
//     whole -> halved: S >= 1024 1.00, up to 1.13 -> 0.84, up to 0.90; S 512 ..
//     1023 0.87 -> 0.74; shorter 0.75 -> 0.69, but some 18 % slower halved);
//     two heads from 0.76 on, where halved dKV and dQ jobs fit one round of
//     three workgroups per CU (0.76 .. 0.8: halved 0.85 of whole, 0.7 .. 0.76
//     1.04);
//   D 128, two heads: from 1.14 on, where the halved jobs are at most one per
//     CU (above it whole 1.07, halved 0.82); of 0.9 .. 1.14 whole below S 1024
//     (28 shapes, halved -> whole: 0.97, up to 1.11 -> 0.89, up to 1.02), and
//     bwd_main_kernel from there on (whole 1.01 to 1.12, halved 1.02 to 1.14);
//   D 128, four heads or more, S >= 1024: from 0.8 on (12 shapes of 0.8 .. 0.9,
//     whole -> halved: 0.99, up to 1.03 -> 0.90);
//   D 128: also with 1 to 4/3 rounds of two workgroups per CU, less than two
//     thirds of the slots of two rounds filled (B2 H12 S1792: 672 jobs, -6 %
//     whole, -11 % halved), but not with two heads and S >= 1024 (15 shapes,
//     halved -> whole: 0.96, up to 1.02 -> 0.90).
RegPlan reg_plan(const BwdProblem& p, const WorkspacePlan& w) {
    RegPlan r;
#ifdef FA3_TIMELINE
    return r;  // the stamps are bwd_main_kernel's
#endif
    if (w.bal_m > 0 || p.out_f32) return r;  // (its outputs are 16-bit)
    const int group = p.heads_q / p.heads_kv, chunks = std::max(w.hs_chunks, 1);
    const int heads = group / chunks, qt = p.seqlen / 64;  // (qt even)
    const double units = p.causal ? 0.25 * qt * (qt + 2.0) : 0.5 * qt * qt;
    const double share = (double)p.batch * p.heads_q * units * 1.75 / kHeadSplitCus;
    const double x = (double)heads * qt / share;
    if (x > 1.3) return r;
    const bool d64 = p.head_dim == 64;
    if (heads == 1) {
        double most;
        if (d64 && p.seqlen >= 512) most = p.causal ? 0.6 : 0.9;
        else if (d64) most = group == 1 ? 0.9 : 1.12;
        else if (group == 1) most = 0.75;
        else if (!p.causal) most = 1.12;
        else most = p.seqlen >= 2048 ? 0.75 : p.seqlen >= 1024 || p.seqlen < 256 ? 1.12 : 1.3;
        if (x > most) {
            r.on = d64;
            r.unscaled = group > 1;
            r.split_kv = r.split_q = 2;
            return r;
        }
    }
    r.on = true;
    const double slot = share / (p.head_dim == 64 ? 3 : 2);
    if (p.causal) {
        // tile k's job: heads x (qt - 2 k) units
        const double k = 0.5 * (qt - slot / heads);
        r.split_kv = 0;
        r.halved = heads == 1 && !d64 && x > 0.54 && x <= 0.75
                       ? 0
                       : std::min(std::max((int)std::ceil(k), 0), qt / 2);
    } else {
        const double rounds = (double)p.batch * p.heads_kv * (chunks + group) * (qt / 2) /
                              (2 * kHeadSplitCus);
        double most = 0.9;
        if (d64 && heads > 1 && p.seqlen >= 512) most = heads == 2 ? 0.76 : 0.7;
        if (!d64 && heads == 2) {
            most = 1.14;
            if (x > 0.9 && x <= most && p.seqlen >= 1024) {
                r.on = false;
                r.unscaled = true;
            }
        }
        if (!d64 && heads > 3 && p.seqlen >= 1024) most = 0.8;
        if (x > most ||
            (!d64 && !(heads == 2 && p.seqlen >= 1024) && rounds > 1.0 &&
             std::ceil(rounds) / rounds > 1.5))
            r.split_kv = 2;
    }
    return r;
}

// The register-operand kernel's arguments, from a default-plan launch's.
RegArgs reg_args(const FusedArgs& a, RegPlan plan, int head_dim, bool causal) {
    RegArgs r{};
    r.q = a.q;
    r.k = a.k;
    r.v = a.v;
    r.dout = a.dout;
    r.nlse2 = a.nlse2;
    r.ndelta = a.ndelta;
    r.dq = a.dq;
    r.dq_f32 = 0;
    r.q_rs = a.q_rs;
    r.q_hs = a.q_hs;
    r.kv_rs = a.kv_rs;
    r.kv_hs = a.kv_hs;
    r.seqlen = a.seqlen;
    r.heads_q = a.heads_q;
    r.heads_kv = a.heads_kv;
    r.group = a.group;
    if (a.part_dk != nullptr) {  // head split: fp32 contributions [B][Hkv chunks][S][D]
        r.chunks = a.hs_chunks;
        r.heads = a.hs_heads;
        r.dk = a.part_dk;
        r.dv = a.part_dv;
        r.dkv_f32 = 1;
        r.o_rs = head_dim;
        r.o_hs = a.seqlen * head_dim;
        r.o_heads = a.heads_kv * a.hs_chunks;
    } else {
        r.chunks = 1;
        r.heads = a.group;
        r.dk = a.dk;
        r.dv = a.dv;
        r.dkv_f32 = 0;
        r.o_rs = a.kv_rs;
        r.o_hs = a.kv_hs;
        r.o_heads = a.heads_kv;
    }
    r.scale_log2 = a.scale_log2;
    r.scale = a.scale;
    r.n_groups = a.n_groups;
    r.halved = plan.halved;
    set_reg_job_map(r, plan, head_dim, causal);
    r.div_hkv = a.div_hkv;
    r.div_group = a.div_group;
    r.div_chunks = make_fastdiv(r.chunks);
    return r;
}

void describe_launch(const BwdProblem& p, const WorkspacePlan& w, ShaoboFa3ExtPlan* out) {
    const int group = p.heads_q / p.heads_kv, chunks = std::max(w.hs_chunks, 1);
    const RegPlan reg = reg_plan(p, w);
    ShaoboFa3ExtPlan o{};
    o.struct_size = out->struct_size;
    o.kernel = reg.on ? SHAOBO_FA3_EXT_KERNEL_REG : SHAOBO_FA3_EXT_KERNEL_MAIN;
    o.split_plan = w.bal_m > 0 ? 1 : 0;
    o.chunks = chunks;
    o.unscaled = reg.on || w.bal_m > 0 || !main_scaled(p.scale * kLog2e, reg.unscaled) ? 1 : 0;
    if (reg.on) {
        RegArgs r{};
        r.seqlen = p.seqlen;
        r.group = group;
        r.chunks = chunks;
        r.heads = group / chunks;
        r.n_groups = p.batch * p.heads_kv;
        set_reg_job_map(r, reg, p.head_dim, p.causal);
        o.jobs = r.n_groups * r.jobs_per_group;
        o.split_kv = reg.split_kv;
        o.halved = reg.halved;
        o.split_q = reg.split_q;
        o.xcd_parts = r.xcd_parts;
    } else {
        o.jobs = p.batch * p.heads_kv * (p.seqlen / kTileN) * (chunks + group);
    }
    *out = o;
}

hipError_t launch_component(const BwdProblem& p, const BwdTensors& t, int role) {
    FusedArgs a = base_args(p, t);
    a.packed = t.packed_in;
    a.smax = t.aux0;
    a.ssum = t.aux1;
    a.delta = t.delta_in;
    a.jobs_per_group = p.seqlen / kTileN;
    set_job_map(a);
    const dim3 grid(a.n_groups * a.jobs_per_group);
    if (p.head_dim == 128) {
        if (role == 1) hipLaunchKernelGGL((bwd_component_kernel<128, 1>), grid, dim3(kThreads), 0, t.stream, a);
        else hipLaunchKernelGGL((bwd_component_kernel<128, 2>), grid, dim3(kThreads), 0, t.stream, a);
    } else {
        if (role == 1) hipLaunchKernelGGL((bwd_component_kernel<64, 1>), grid, dim3(kThreads), 0, t.stream, a);
        else hipLaunchKernelGGL((bwd_component_kernel<64, 2>), grid, dim3(kThreads), 0, t.stream, a);
    }
    return hipGetLastError();
}

#ifdef FA3_TIMELINE
namespace {
unsigned long long* g_timeline = nullptr;
}
// Timeline build only (no product entry point): the device buffer that the
// main-kernel launches that follow fill with per-workgroup timestamps (null:
// none).  At least 2^21 + 32 x workgroups 64-bit words, zeroed by the caller.
extern "C" __attribute__((visibility("default"))) void fa3_timeline_set(void* buffer) {
    g_timeline = static_cast<unsigned long long*>(buffer);
}
#endif

hipError_t launch_backward(const BwdProblem& p, const BwdTensors& t, void* workspace,
                           unsigned long long* epoch) {
    const WorkspacePlan plan = plan_workspace(p);
    if (!plan.ok) return hipErrorInvalidValue;
    char* ws = static_cast<char*>(workspace);
    FusedArgs a = base_args(p, t);
    float* nlse2 = reinterpret_cast<float*>(ws + plan.nlse2_off);
    float* ndelta = reinterpret_cast<float*>(ws + plan.ndelta_off);
    auto mark = [&](int i) {
        return t.events[i] != nullptr ? hipEventRecord(t.events[i], t.stream) : hipSuccess;
    };
    hipError_t err = mark(0);
    if (err != hipSuccess) return err;
    unsigned int* queue = reinterpret_cast<unsigned int*>(ws + plan.queue_off);
    if (t.stages & 1) {
        err = t.packed_in != nullptr ? launch_rowstats(p, t, nlse2, ndelta, queue)
                                     : launch_preprocess(p, t, nlse2, ndelta, queue);
    }
    if (err == hipSuccess) err = mark(1);
    if (err != hipSuccess) return err;
    if (!(t.stages & 2)) return mark(2);
    a.nlse2 = nlse2;
    a.ndelta = ndelta;
    const int group = p.heads_q / p.heads_kv;
    // per key tile / query tile: one dKV job (head split: one per chunk of
    // G / chunks query heads) and G dQ jobs
    a.jobs_per_group = (p.seqlen / kTileN) * ((plan.hs_chunks > 0 ? plan.hs_chunks : 1) + group);
    if (plan.hs_chunks > 0) {
        a.part_dk = reinterpret_cast<float*>(ws + plan.hsd_off);
        a.part_dv = a.part_dk + (size_t)p.batch * p.heads_kv * plan.hs_chunks * p.seqlen * p.head_dim;
        a.hs_chunks = plan.hs_chunks;
        a.hs_heads = group / plan.hs_chunks;
        a.div_chunks = make_fastdiv(plan.hs_chunks);
    }
    const int cus = cu_count(t.device) & ~7;
    {
        // the longest job (a dKV job: its G, or G / chunks, heads' query
        // tiles) against a CU's share, in dKV steps (a dQ step ~0.75)
        const int qt = p.seqlen / kTileN;
        const double steps = p.causal ? 0.5 * qt * (qt + 1.0) : (double)qt * qt;
        const double share = (double)p.batch * p.heads_q * steps * 1.75 / std::max(cus, 8);
        const int heads = plan.hs_chunks > 0 ? group / plan.hs_chunks : group;
        set_job_map(a, (double)heads * qt, share, std::max(cus, 8));
    }
    a.n_jobs = a.n_groups * a.jobs_per_group;
    a.queue = queue;
    // persistent default plan once there are more than two jobs per CU: one
    // workgroup per CU (a multiple of 8, the XCD count) pulls jobs from the
    // queues, so no CU waits for the in-order dispatch of new workgroups.
    // At exactly two per CU the hardware's dispatch of one job per
    // workgroup measured faster (512 jobs: B1 H16 S1024 D128 -9.8 %, B1 H8
    // S2048 D64 -11.2 %, B1 H16 S1024 D64 full -19.3 %, B1 H4 S4096 D128
    // -1.1 %); from 576 jobs on the queues win (B1 H9 S2048 D128: +7.6 %
    // without them), and below 512 too (384 jobs: +6 to +16 % with them).
    a.persist = plan.bal_m == 0 && cus >= 8 && a.n_jobs > 2 * cus ? cus : 0;
    a.epoch = next_epoch();
    if (epoch != nullptr) *epoch = a.epoch;
    a.err = reinterpret_cast<unsigned long long*>(ws + plan.err_off);
    err = split_giveup_count(t.device, &a.giveups);
    if (err != hipSuccess) return err;
    a.spin_limit = g_spin_limit.load();
#ifdef FA3_TIMELINE
    a.tl = g_timeline;
#endif
    a.bal_m = plan.bal_m;
    if (plan.bal_m > 0) {
        a.n_split = plan.n_split;
        a.sync = reinterpret_cast<unsigned long long*>(ws + plan.sync_off);
        a.part_kv = reinterpret_cast<float*>(ws + plan.pkv_off);
        a.part_q = reinterpret_cast<float*>(ws + plan.pq_off);
        a.part_kv_bytes = (uint32_t)(plan.pq_off - plan.pkv_off);
        a.part_q_bytes = (uint32_t)(plan.total - plan.pq_off);
        // each workgroup's descriptor: its job id's kind x = pos mod M (pos
        // as the job map deals it), group, head-piece length and short job
        const int M = plan.bal_m;
        if (a.n_jobs > kMaxSplitWgs || a.n_groups > 64) return hipErrorInvalidValue;
        const SplitPlan& sp = split_plan(M);
        for (int id = 0; id < a.n_jobs; ++id) {
            int g = 0, pos = 0;
            job_of(a, id, g, pos);
            const int kind = pos / M, x = pos % M;
            const int len = kind == 1 || kind == 2 ? sp.head_kv[x] : sp.head_q[x];
            const int s = sp.shrt[kind][x];
            const int sfield = s < 0 ? kNoShort : sp.after[kind][x] ? kShortAfter + s : s;
            a.split_desc[id] = split_desc(kind, x, g, len, sfield);
        }
    }
    const RegPlan reg = reg_plan(p, plan);
    if (reg.on) {
        const RegArgs r = reg_args(a, reg, p.head_dim, p.causal);
        if (g_debug_kernels.load())
            launch_reg_race_check(r, reg, p.head_dim, p.causal, p.bf16, t.stream);
        else launch_reg_kernel<false>(r, reg, p.head_dim, p.causal, p.bf16, t.stream);
    }
    else if (g_debug_kernels.load())
        launch_race_check(a, p.head_dim, p.causal, p.bf16, reg.unscaled, t.stream);
    else if (p.head_dim == 128)
        launch_dd<128, false>(a, p.causal, p.bf16, reg.unscaled, t.stream);
    else launch_dd<64, false>(a, p.causal, p.bf16, reg.unscaled, t.stream);
    err = hipGetLastError();
    if (err == hipSuccess && plan.hs_chunks > 0) {
        const dim3 rg((unsigned)((p.seqlen * (p.head_dim / 4) + 255) / 256),
                      (unsigned)(p.batch * p.heads_kv));
        _Float16* dk = static_cast<_Float16*>(t.dk);
        _Float16* dv = static_cast<_Float16*>(t.dv);
        auto reduce = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, rg, dim3(256), 0, t.stream, a.part_dk, a.part_dv, dk, dv,
                               p.heads_kv, plan.hs_chunks, p.seqlen, a.kv_rs, a.kv_hs);
        };
        if (p.head_dim == 128)
            reduce(p.bf16 ? gqa_reduce_kernel<128, true> : gqa_reduce_kernel<128, false>);
        else
            reduce(p.bf16 ? gqa_reduce_kernel<64, true> : gqa_reduce_kernel<64, false>);
        err = hipGetLastError();
    }
    return err == hipSuccess ? mark(2) : err;
}

}  // namespace fa3
