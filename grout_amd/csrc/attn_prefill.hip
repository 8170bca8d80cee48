// Causal GQA flash-attention prefill on CDNA4 MFMA.
//
// Replaces fmha_prefill_causal (src/kernels.rs:1146-1295, grout's default
// prefill), fmha_prefill_gqa (:1322-1495), fmha_prefill_gqa_lpt (:1513-1862)
// and flash_attn_causal_seq_f16 (:1037-1127).  Semantics: query row m at
// position query_start+m attends keys n < min(kv_len, query_start+m+1) of the
// cache head q_head/G; base-2 online softmax with c = qk_scale/ln2:
//   m' = max(m, c*rowmax(s)); p = 2^(c*s - m'); alpha = 2^(m - m');
//   l = l*alpha + sum(p); acc = acc*alpha + f16(p) V; out = f16(acc/max(l,1e-8)).
//
// Shape of the kernel (MI355X-first):
//  * Workgroup = 8 wavefronts, two per SIMD.  A wavefront owns 32 query rows
//    of one query head; the 8 wavefront tasks of a workgroup belong to the
//    same KV head (GQA packing: a K/V tile is fetched once from HBM for all
//    of them), e.g. G=4: 4 heads x the same 64 positions.
//  * Ping-pong: waves 0-3 and 4-7 run the same per-tile program one phase
//    apart.  A tile is a GEMM phase (PV of the previous tile + S of this
//    tile, 32 MFMAs) and a softmax phase (VALU, v_exp_f32); each tile starts
//    with the two groups in opposite phases, so one wave of a SIMD feeds the
//    matrix core (at raised issue priority) while the other does its softmax.
//    One workgroup barrier per tile guards the stage ring.
//  * K/V tiles of 64 keys go straight from HBM into LDS (direct-to-LDS DMA,
//    no register staging) through a 4-stage ring; tile t+2 is issued in
//    tile step t, at the start of each wavefront's softmax phase.
//  * S^T = K Q^T on v_mfma_f32_32x32x16_f16 (K rows = A operand, 16-byte LDS
//    reads; Q^T = B operand held in registers for the whole loop), so each
//    lane owns one query row and the row softmax needs a single cross-lane
//    step (v_permlane32_swap).
//  * O^T += V^T P^T: P^T comes straight from the S^T accumulators (the
//    reduction slots are ordered to match), V^T from ds_read_b64_tr_b16.
//    LDS operands are read a few MFMAs ahead into a register ring.
//  * The running max is raised only when P would leave f16 range, so most
//    tiles need no row max and no rescale.
//  * Causal tile skipping per wavefront; masking only on diagonal tiles.
//  * Heavy (late-position) workgroups launch first (longest-processing-time
//    order) and all workgroups of one KV head go to one XCD so its K/V stay
//    in that XCD's L2.
//  * Small launches (row blocks of at most 8 key tiles, one workgroup per
//    query head and row block within the CU count) take a short form: the 8
//    wavefronts of a workgroup take one key tile each and merge in LDS.
#include <math.h>

#include <type_traits>

#include "abi_util.h"
#include "common.h"

namespace grout {

constexpr int kPfBN = 64;     // keys per tile
// LDS tile layout: key row n of a tile sits in 1 KB block n%16 at row n/16
// (256 B rows inside a block); blocks are 1040 B (K) / 1088 B (V) apart.
// One direct-to-LDS copy fills one block (rows b, b+16, b+32, b+48), the
// MFMA operand reads (8 or 16 consecutive keys, or 4 keys x 32 B for the
// transposing V reads) hit distinct banks, and every read address is a
// per-lane base plus an immediate offset.
constexpr int kPfKBlock = 1040;
constexpr int kPfVBlock = 1088;
constexpr int kPfKBytes = 16 * kPfKBlock;
constexpr int kPfVBytes = 16 * kPfVBlock;
constexpr int kPfStageBytes = kPfKBytes + kPfVBytes;
constexpr int kPfStages = 4;
constexpr int kPfOutBytes = 32 * 256;  // one wavefront's f16 output tile
static_assert(4 * kPfOutBytes <= kPfStageBytes, "a stage holds the output tiles of 4 wavefronts");
constexpr float kPfNegBig = -1.0e30f;
// Lazy rescale: the running max used for p = 2^(c*s - m) is only raised when
// some p of a tile would reach this bound (f16 holds up to 65504), so O is
// rescaled on few tiles and no per-tile row max is needed otherwise.
constexpr float kPfPsumLimit = 32768.0f;
// LDS operand read-ahead of the GEMM phase, in MFMAs.
constexpr int kPfAhead = 4;

struct PrefillArgs {
    const uint16_t* q;
    const uint16_t* k_cache;
    const uint16_t* v_cache;
    uint16_t* out;
    float scale_log2;
    int num_q_heads;
    int group;
    int q_len;
    int kv_len;
    int query_start;
    int max_seq_len;
    int n_pos_tiles;       // ceil(q_len / rows per wavefront) (split: padded to whole q blocks)
    int tasks_per_head;    // n_pos_tiles * group wavefront tasks per KV head
    int blocks_per_head;   // ceil(tasks_per_head / waves per workgroup)
    // Split-K form only (fmha_prefill_gqa_lpt_split's generics and scratch).
    uint16_t* att_partial;  // [tiles, num_splits*block_m*split_group, 128]
    float* lse_partial;     // [tiles, num_splits*block_m*split_group]
    int block_m;            // BM: query rows per q block (a multiple of 32)
    int block_n;            // BN: keys per split-range tile
    int split_group;        // GROUP: q heads per logical tile
    int num_splits;
    // Dynamic schedule only (kDyn): claim counters (kPfQueues XCD queues, the
    // shared pool, the exit counter; kPfSchedStride u32 apart, zero on entry
    // and exit), the number of persistent workgroups, the KV-head count and
    // the first block (per head) that goes to the shared pool.
    uint32_t* sched;
    int n_wg;
    int num_kv_heads;
    int pool_block0;
};

// Dynamic schedule.  A task is a workgroup-sized unit (one block of the static
// grid).  The KV heads h = q (mod kPfQueues) belong to XCD q: their blocks
// [0, pool_block0) form its heavy queue and the lighter blocks
// [pool_block0, blocks_per_head) its light queue, each heaviest first with the
// heads interleaved.  A persistent workgroup claims from the heavy queue of
// the XCD it runs on (a head's K/V stay in that XCD's L2), then from the
// fullest other heavy queue, then from its own light queue while that holds
// at least half as many tasks as the fullest light queue, else from the
// fullest: XCDs that run faster take over the slower ones' heavy blocks, the
// last tasks anywhere are light ones, and most light tasks still run where
// their head's K/V are cached.
constexpr int kPfQueues = 8;
constexpr int kPfLight = kPfQueues;             // counter index of light queue q: kPfLight + q
constexpr int kPfExit = 2 * kPfQueues;          // counter index of the exit counter
constexpr int kPfSchedCounters = 2 * kPfQueues + 1;
constexpr int kPfSchedStride = 64;  // u32: one 256-byte line per counter
constexpr int kPfClaimAttempts = 64;

// Asynchronous 16-byte HBM -> LDS copy (global_load_lds_dwordx4, scalar base
// + 32-bit per-lane byte offset): lane l's 16 bytes land at LDS byte
// lds_base + 16*l (lds_base wave-uniform).  Issued through inline asm so the
// compiler does not serialise consecutive copies behind vmcnt(0) waits; the
// kernel waits for them itself with s_waitcnt vmcnt before its workgroup
// barrier.  M0 carries the LDS base (this kernel keeps nothing else in M0);
// one wait state separates the M0 write from the copy.
__device__ __forceinline__ void lds_dma16(const void* gbase, uint32_t voff, uint32_t lds_base) {
    asm volatile(
        "s_mov_b32 m0, %2\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %0, %1"
        :
        : "v"(voff), "s"(gbase), "s"(lds_base)
        : "memory");
}

// A wave-uniform pointer held in SGPRs, where the compiler does not see that it
// is uniform.
__device__ __forceinline__ const uint16_t* uniform_ptr(const uint16_t* p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
    return reinterpret_cast<const uint16_t*>(static_cast<uint64_t>(hi) << 32 | lo);
}

// f16(f32(o / l)) for f32 o and l > 0, with rl = 1/l rounded to f64: the f64
// product o*rl is within 2^-52 (relative) of o/l, while a quotient of two f32
// values in the f32 normal range is never an f32 rounding midpoint and lies
// more than 2^-49 (relative) from every one; so the product rounds to the same
// f32 as the correctly rounded division.  Quotients below 2^-126 give +-0 in
// f16 either way.  About 4 instructions against the ~10 of an f32 division.
__device__ __forceinline__ half_t div_to_half(float o, double rl) {
    float f = static_cast<float>(static_cast<double>(o) * rl);
    // Keeps the two roundings: the code generator otherwise folds
    // f64 -> f32 -> f16 into a single f64 -> f16 rounding, another function.
    asm("" : "+v"(f));
    return static_cast<half_t>(f);
}

// s_waitcnt immediate for "at most n vector-memory ops outstanding" (gfx9
// encoding: vmcnt bits [3:0]+[15:14]; expcnt [6:4] and lgkmcnt [11:8] at their
// maximum, i.e. not waited on).
constexpr int waitcnt_vm(int n) { return (n & 15) | ((n >> 4) << 14) | 0x0F70; }

// Workgroup barrier that also orders LDS: this wavefront's LDS reads have
// completed (a stage may be refilled right after the barrier) and the
// compiler moves no memory access across it.
__device__ __forceinline__ void pf_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// GEMM phase of one tile: O^T += V^T P^T of the previous tile (MFMA slots 0-15:
// key step i/4, dim block i%4; `vb`: this lane's base in its V stage), then
// S^T = K Q^T of this tile (slots 16-31: dim step (i-16)/2, key block i%2;
// `kb`: this lane's base in its K stage).  One software pipeline over the 32
// slots: each slot's LDS operand is read kPfAhead slots before its MFMA into a
// ring of registers, so LDS latency hides behind ~kPfAhead MFMAs; a
// scheduling fence per slot keeps that order.
__device__ __forceinline__ void pf_gemm(const unsigned char* kb, const unsigned char* vb, const half8_t (&qop)[8],
                                        const half8_t (&pop)[4], float16_t (&o)[4], float16_t (&s)[2]) {
    constexpr int kRing = kPfAhead + 1;
    auto read_op = [&](int i) {
        if (i < 16) {
            // V^T[32 dims of block i%4, 16 keys of step i/4].
            const unsigned char* p0 = vb + 256 * (i >> 2) + 64 * (i & 3);
            return cat(lds_read_tr16(reinterpret_cast<const half_t*>(p0)),
                       lds_read_tr16(reinterpret_cast<const half_t*>(p0 + 8 * kPfVBlock)));
        }
        // K[32 keys of block i%2, 16 dims of step (i-16)/2].
        return *reinterpret_cast<const half8_t*>(kb + 512 * (i & 1) + 32 * ((i - 16) >> 1));
    };
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int r = 0; r < 16; ++r) s[mb][r] = 0.0f;
    half8_t ring[kRing];
    // Issue priority above the softmax-phase wave on the same SIMD while
    // feeding the matrix core (measured: ~1% faster; raising the softmax
    // phase instead does nothing).
    __builtin_amdgcn_s_setprio(2);
#pragma unroll
    for (int i = 0; i < kPfAhead; ++i) ring[i % kRing] = read_op(i);
#pragma unroll
    for (int i = 0; i < 32; ++i) {
        if (i + kPfAhead < 32) ring[(i + kPfAhead) % kRing] = read_op(i + kPfAhead);
        if (i < 16) {
            o[i & 3] = mfma32x32x16(ring[i % kRing], pop[i >> 2], o[i & 3]);
        } else {
            s[i & 1] = mfma32x32x16(ring[i % kRing], qop[(i - 16) >> 1], s[i & 1]);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_setprio(0);
}

// The GEMM phase of half a tile (32 keys: V rows of key steps 0-1 at `vb`, K
// rows of one key block at `kb`): 8 PV and 8 S MFMAs, alternating, because the
// 8 S MFMAs of one key block are one accumulation chain.
__device__ __forceinline__ void pf_gemm_half(const unsigned char* kb, const unsigned char* vb,
                                             const half8_t (&qop)[8], const half8_t (&pop)[2],
                                             float16_t (&o)[4], float16_t (&s)[1]) {
    constexpr int kRing = kPfAhead + 1;
    auto read_op = [&](int i) {
        const int n = i >> 1;
        if ((i & 1) == 0) {
            const unsigned char* p0 = vb + 256 * (n >> 2) + 64 * (n & 3);
            return cat(lds_read_tr16(reinterpret_cast<const half_t*>(p0)),
                       lds_read_tr16(reinterpret_cast<const half_t*>(p0 + 8 * kPfVBlock)));
        }
        return *reinterpret_cast<const half8_t*>(kb + 32 * n);
    };
#pragma unroll
    for (int r = 0; r < 16; ++r) s[0][r] = 0.0f;
    half8_t ring[kRing];
    __builtin_amdgcn_s_setprio(2);
#pragma unroll
    for (int i = 0; i < kPfAhead; ++i) ring[i % kRing] = read_op(i);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        if (i + kPfAhead < 16) ring[(i + kPfAhead) % kRing] = read_op(i + kPfAhead);
        const int n = i >> 1;
        if ((i & 1) == 0) {
            o[n & 3] = mfma32x32x16(ring[i % kRing], pop[n >> 2], o[n & 3]);
        } else {
            s[0] = mfma32x32x16(ring[i % kRing], qop[n], s[0]);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_setprio(0);
}

// Softmax of one (already masked) tile: P = 2^(c*s - m) into `pop`, its row
// sum into l, with the running max m raised only when it has to be.
// kBlocks: 32-key blocks of the tile (2: the grid's 64 keys, 1: half a tile).
// fill(i), i < 8 kBlocks, runs before the i-th pair of exponentials.
struct NoFill {
    __device__ __forceinline__ void operator()(int) const {}
};
template <int kBlocks, typename Fill = NoFill>
__device__ __forceinline__ void pf_softmax(const float16_t (&s)[kBlocks], half8_t (&pop)[2 * kBlocks],
                                           float16_t (&o)[4], float& m_run, float& l_run, float c, Fill fill = Fill{}) {
    // The row sum runs in four independent f32 chains.
    auto exp_tile = [&](float m_use, auto filler) {
        // Each chain starts from its first pair rather than from 0.0f: the
        // compiler keeps a float 0 + x (it is not x for x = -0), and those
        // four adds measured ~1% of the kernel's time.  p >= 0, so the
        // sums are the same values.
        float ps[4];
#pragma unroll
        for (int mb = 0; mb < kBlocks; ++mb)
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                filler(8 * mb + (r >> 1));
                const float p0 = __builtin_amdgcn_exp2f(fmaf(s[mb][r], c, -m_use));
                const float p1 = __builtin_amdgcn_exp2f(fmaf(s[mb][r + 1], c, -m_use));
                const int k = (r >> 1) & 3;
                ps[k] = (mb == 0 && r < 8) ? (p0 + p1) : ps[k] + (p0 + p1);
                pop[2 * mb + (r >> 3)][r & 7] = static_cast<half_t>(p0);
                pop[2 * mb + (r >> 3)][(r & 7) + 1] = static_cast<half_t>(p1);
            }
        return (ps[0] + ps[1]) + (ps[2] + ps[3]);
    };
    float psum = exp_tile(m_run, fill);
    // The max is only raised when P would leave f16 range: a lane's partial
    // row sum below 2^15 bounds each of its p below 2^15 (the test also
    // catches inf).  Then the tile's row max becomes the running max, O and
    // l are rescaled and P is recomputed.  Until then p <= 2^15 keeps full
    // f16 relative precision, so the normalised result is the same function.
    if (__any(!(psum < kPfPsumLimit))) {
        float mx = kPfNegBig;
#pragma unroll
        for (int mb = 0; mb < kBlocks; ++mb)
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[mb][r]);
        mx = fmaxf(mx, swap_halves(mx));
        const float m_new = fmaxf(m_run, mx * c);
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
        l_run *= alpha;
#pragma unroll
        for (int db = 0; db < 4; ++db) o[db] *= alpha;
        m_run = m_new;
        psum = exp_tile(m_run, NoFill{});
    }
    l_run += psum;
}

// S^T = K Q^T of one tile alone (`kb`: this lane's base in its K stage).
__device__ __forceinline__ void pf_scores(const unsigned char* kb, const half8_t (&qop)[8], float16_t (&s)[2]) {
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int r = 0; r < 16; ++r) s[mb][r] = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i)
        s[i & 1] = mfma32x32x16(*reinterpret_cast<const half8_t*>(kb + 512 * (i & 1) + 32 * (i >> 1)), qop[i >> 1], s[i & 1]);
}

// O^T += V^T P^T of one tile alone (`vb`: this lane's base in its V stage).
__device__ __forceinline__ void pf_values(const unsigned char* vb, const half8_t (&pop)[4], float16_t (&o)[4]) {
    constexpr int kRing = kPfAhead + 1;
    auto read_op = [&](int i) {
        const unsigned char* p0 = vb + 256 * (i >> 2) + 64 * (i & 3);
        return cat(lds_read_tr16(reinterpret_cast<const half_t*>(p0)),
                   lds_read_tr16(reinterpret_cast<const half_t*>(p0 + 8 * kPfVBlock)));
    };
    half8_t ring[kRing];
#pragma unroll
    for (int i = 0; i < kPfAhead; ++i) ring[i % kRing] = read_op(i);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        if (i + kPfAhead < 16) ring[(i + kPfAhead) % kRing] = read_op(i + kPfAhead);
        o[i & 3] = mfma32x32x16(ring[i % kRing], pop[i >> 2], o[i & 3]);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Workgroup: 8 wavefronts x 32 query rows, all on query heads of one KV head.
// Waves 0-3 (group A, one per SIMD) and 4-7 (group B) run the same per-tile
// program one phase apart ("ping-pong"): a tile is two phases, GEMM (PV of the
// previous tile + S of this tile, 32 MFMAs) and softmax (VALU + v_exp_f32).
// After each tile's barrier group A starts with its GEMM phase and group B
// with its softmax, so each SIMD has one wavefront feeding the matrix core
// while the other does its softmax.  Between the phases there is no barrier:
// a second one per tile, to hold the groups in step, measured 0.5% slower.
constexpr int kPfWaves = 8;
constexpr int kPfRows = 32;

// kSplit: the split-K form (fmha_prefill_gqa_lpt_split, src/kernels.rs:1872-2142).
// Workgroup (task, blockIdx.y = split); every wavefront restricts its keys to
// its split's range, computed from the reference's q block of its rows
// (block_m is a multiple of 32, so a wavefront's rows lie in one block), and
// stores a normalised partial and its log2 LSE instead of the output.
// kDyn: persistent workgroups that claim tasks from the per-XCD queues above
// instead of taking one task from blockIdx; each task runs exactly as in the
// static grid, so the output is bit-identical.
// kWaves = 4: group A alone (one computing wavefront per SIMD, no ping-pong
// partner) on 4 row tiles, and four wavefronts that only copy, for grids too
// small to fill the GPU: twice the workgroups, and a tile step takes one GEMM
// phase and one softmax phase.  A 1 KB copy holds up the wavefront that issues
// it for ~100 cycles; left to the computing wavefronts, their eight copies a
// step were ~800 of ~2850 cycles, with the copy wavefronts a step took ~2300
// (Qwen3-4B, 1000 tokens 24.3 -> 21.3 us; 509 tokens behind 6003 117 -> 95 us).
// Without a partner to alternate with, a step computes S of the next tile
// between the exponentials of this one, then this one's PV: ~2090 cycles (Qwen3-0.6B,
// 927 tokens 19.0 -> 17.8 us; 32/8 heads, 768 behind 4096 73.3 -> 71.7).  Of
// these 1390 are the softmax with its 16 S MFMAs and 620 PV: one wavefront's
// MFMAs and VALU hardly overlap, and spreading the softmax over PV's MFMAs of
// the tile before as well measured the same.
// Every wavefront computes exactly what it computes in the 8-wavefront
// workgroup, so the output is bit-identical.
template <bool kSplit, bool kDyn, int kWaves = kPfWaves>
__global__ __launch_bounds__(kPfWaves * kWave, 1) void attn_prefill_kernel(PrefillArgs a) {
    static_assert(!(kSplit && kDyn), "the split-K form keeps the static grid");
    static_assert(kWaves == kPfWaves || (kWaves == 4 && !kSplit && !kDyn),
                  "the 4-wavefront form is the plain static grid only");
    constexpr int kDmaPerWave = 16 / kWaves;  // K blocks (and V blocks) per wavefront
    __shared__ __attribute__((aligned(1024))) unsigned char pf_lds[kPfStages * kPfStageBytes];

    const int tid = threadIdx.x;
    const int wave_id = __builtin_amdgcn_readfirstlane(tid / kWave);
    const bool copies_only = kWaves == 4 && wave_id >= 4;
    const int wave = kWaves == 4 ? wave_id & 3 : wave_id;  // copy wavefront w fills blocks as wave w
    const int grp = wave >> 2;  // 0: group A, 1: group B (one phase behind)
    const int lane = tid % kWave;
    const int l32 = lane & 31;
    const int hl = lane >> 5;  // which half of the wavefront

    // XCD-aware, longest-first task order: consecutive workgroup ids go to
    // different XCDs, so T groups all workgroups of a KV head on one XCD, and
    // within a head the latest (heaviest) position tiles come first.  With
    // fewer than 8 KV heads a head spans hx = 8/Hkv XCDs, which take its blocks
    // in turn (block i*hx + j on the head's j-th XCD): each XCD then gets the
    // same mix of heavy and light blocks, not a contiguous (heavy or light) run.
    const int nb = gridDim.x;
    const int b = blockIdx.x;
    int T = b;
    if (nb % 8 == 0) {
        const int hkv = nb / a.blocks_per_head;
        const int x = b % 8, i = b / 8;
        if (hkv < 8 && 8 % hkv == 0) {
            const int hx = 8 / hkv;
            T = (x / hx) * a.blocks_per_head + i * hx + x % hx;
        } else {
            T = x * (nb / 8) + i;
        }
    }

    // Dynamic schedule state (wave 0 claims; the task goes to all waves
    // through LDS).  The claim on the own queue is issued one task ahead, after
    // the previous task's loop, so its round trip overlaps that epilogue.
    __shared__ int s_task;
    int my_q = 0, nhq_own = 0, nq_own = 0;
    bool own_live = false;
    uint32_t pre_j = 0xffffffffu;  // prefetched own-queue ticket (wave 0, lane 0)
    int pre_ticket = -1;           // the same, read back (wave 0, uniform); -1: none
    if constexpr (kDyn) {
        uint32_t xcc;
        asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
        my_q = static_cast<int>(xcc % kPfQueues);
        nhq_own = a.num_kv_heads > my_q ? (a.num_kv_heads - my_q + kPfQueues - 1) / kPfQueues : 0;
        nq_own = nhq_own * a.pool_block0;
        own_live = nq_own > 0;
        if (wave == 0 && lane == 0 && own_live)
            pre_j = __hip_atomic_fetch_add(a.sched + my_q * kPfSchedStride, 1u, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
        if (wave == 0 && own_live) pre_ticket = static_cast<int>(__shfl(pre_j, 0));
    }
    // Task j of heavy queue q: KV head q + kPfQueues*(j % nhq), block j / nhq;
    // of light queue q: the same head, block pool_block0 + j / nhq.
    auto queue_task = [&](int q, int nhq, int j) {
        return (q + kPfQueues * (j % nhq)) * a.blocks_per_head + j / nhq;
    };
    const int light_blocks = a.blocks_per_head - a.pool_block0;

    for (;;) {
    if constexpr (kDyn) {
        if (wave == 0) {
            int task = -1;
            const int j0 = pre_ticket;
            if (own_live && j0 >= 0 && j0 < nq_own) {
                // nhq_own passes through an empty asm so that the division's
                // constants are derived here, not held across the task loop.
                int nhq = nhq_own;
                asm volatile("" : "+s"(nhq));
                task = queue_task(my_q, nhq, j0);
            } else {
                own_live = false;
            }
            // Own heavy queue empty: claim from the fullest other heavy queue,
            // else from the own light queue if it holds at least half as many
            // tasks as the fullest light queue, else from the fullest; leave
            // once all are empty.  Lane i < 2*kPfQueues reads counter i.
            for (int attempt = 0; attempt < kPfClaimAttempts && task < 0; ++attempt) {
                int rem = 0;
                if (lane < 2 * kPfQueues) {
                    const int q = lane % kPfQueues;
                    const int nhq = a.num_kv_heads > q ? (a.num_kv_heads - q + kPfQueues - 1) / kPfQueues : 0;
                    const uint32_t nq = static_cast<uint32_t>(nhq * (lane < kPfQueues ? a.pool_block0 : light_blocks));
                    const uint32_t c = __hip_atomic_load(a.sched + lane * kPfSchedStride, __ATOMIC_RELAXED,
                                                         __HIP_MEMORY_SCOPE_AGENT);
                    rem = static_cast<int>(nq - min(c, nq));
                }
                int best = -1, best_rem = 0;
#pragma unroll
                for (int q = 0; q < kPfQueues; ++q) {
                    const int r = __shfl(rem, q);
                    if (r > best_rem) {
                        best_rem = r;
                        best = q;
                    }
                }
                if (best < 0) {
#pragma unroll
                    for (int q = 0; q < kPfQueues; ++q) {
                        const int r = __shfl(rem, kPfLight + q);
                        if (r > best_rem) {
                            best_rem = r;
                            best = kPfLight + q;
                        }
                    }
                    const int own_rem = __shfl(rem, kPfLight + my_q);
                    if (own_rem > 0 && (own_rem << 1) >= best_rem) best = kPfLight + my_q;
                }
                if (best < 0) break;
                uint32_t j = 0;
                if (lane == 0)
                    j = __hip_atomic_fetch_add(a.sched + best * kPfSchedStride, 1u, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
                j = __shfl(j, 0);
                const int q = best % kPfQueues;
                const int nhq = (a.num_kv_heads - q + kPfQueues - 1) / kPfQueues;
                if (best < kPfQueues) {
                    if (j < static_cast<uint32_t>(nhq * a.pool_block0)) task = queue_task(q, nhq, static_cast<int>(j));
                } else if (j < static_cast<uint32_t>(nhq * light_blocks)) {
                    task = queue_task(q, nhq, static_cast<int>(j)) + a.pool_block0;
                }
            }
            if (lane == 0) s_task = task;
        }
        pf_barrier();  // also: every wavefront is past the previous task's LDS reads
        T = s_task;
        if (T < 0) break;
    }
    const int kvh = T / a.blocks_per_head;
    const int rblk = T % a.blocks_per_head;
    const int u = rblk * kWaves + wave;
    const bool task_ok = u < a.tasks_per_head;
    const int pt = a.n_pos_tiles - 1 - u / a.group;
    const int g = u % a.group;
    const int qh = kvh * a.group + g;
    const int row0 = pt * kPfRows;
    const int pos0 = a.query_start + row0;

    const int pt_max = a.n_pos_tiles - 1 - (rblk * kWaves) / a.group;
    const int blk_kv_end = min(a.kv_len, a.query_start + pt_max * kPfRows + kPfRows);
    int wave_kv_end = task_ok ? min(a.kv_len, pos0 + kPfRows) : 0;
    // Key range [lo, hi) of this wavefront (all keys unless split) and the
    // workgroup's range of 64-key tiles [tile0, tile0 + ntiles).
    int key_lo = 0, key_hi = a.kv_len, tile0 = 0, blk_end = blk_kv_end;
    if constexpr (kSplit) {
        // src/kernels.rs:2036-2043 for q block bq: tc = ceil(min(m_end, kv_len)/BN),
        // tps = ceil(tc/NKS), split s covers tiles [s*tps, min(s*tps+tps, tc)).
        auto split_range = [&](int bq, int& lo, int& hi) {
            const int m_end = a.query_start + (bq + 1) * a.block_m;
            const int tc = (min(m_end, a.kv_len) + a.block_n - 1) / a.block_n;
            const int tps = (tc + a.num_splits - 1) / a.num_splits;
            const int st = static_cast<int>(blockIdx.y) * tps;
            const int et = min(st + tps, tc);
            lo = st * a.block_n;
            hi = max(lo, min(et * a.block_n, a.kv_len));
        };
        split_range(row0 / a.block_m, key_lo, key_hi);
        wave_kv_end = min(wave_kv_end, key_hi);
        if (wave_kv_end <= key_lo) wave_kv_end = 0;  // empty range: no tile
        // The ranges grow with the q block, so the workgroup's union runs from
        // its lowest block's start to its highest block's end.
        const int pt_min = max(0, a.n_pos_tiles - 1 - (rblk * kWaves + kWaves - 1) / a.group);
        int lo_min, hi_min, lo_max, hi_max;
        split_range(pt_min * kPfRows / a.block_m, lo_min, hi_min);
        split_range(pt_max * kPfRows / a.block_m, lo_max, hi_max);
        blk_end = min(blk_kv_end, hi_max);
        tile0 = lo_min / kPfBN;
        if (blk_end <= lo_min) blk_end = tile0 * kPfBN;  // no key in any range
    }
    const int ntiles = max(0, (blk_end + kPfBN - 1) / kPfBN - tile0);
    // This wavefront's active tiles [wave_t0, wave_tiles), relative to tile0.
    const int wave_t0 = (wave_kv_end > 0) ? key_lo / kPfBN - tile0 : 0;
    const int wave_tiles = (wave_kv_end > 0) ? (wave_kv_end + kPfBN - 1) / kPfBN - tile0 : 0;

    const uint16_t* kh = a.k_cache + static_cast<int64_t>(kvh) * a.max_seq_len * kHeadDim;
    const uint16_t* vh = a.v_cache + static_cast<int64_t>(kvh) * a.max_seq_len * kHeadDim;

    // HBM -> LDS copy of tile `tile` into stage `st`: this wavefront fills K
    // and V blocks wave*kDmaPerWave + r; lane l moves row b + 16*(l/16), 16-byte
    // column l%16.  On the block's last tile rows at or past blk_kv_end are
    // clamped to the last valid row (they are masked in the softmax).
    const uint32_t lds0 = static_cast<uint32_t>(
        (uintptr_t)((__attribute__((address_space(3))) unsigned char*)(pf_lds)));
    // kFresh: the lane terms are derived again from the lane id at this call,
    // so the compiler cannot hoist them out of the persistent task loop and
    // keep (or spill) them across it; used for the prologue's two tiles.
    auto issue_tile = [&](int tile, int st, auto fresh) {
        int ln = lane;
        if constexpr (decltype(fresh)::value) asm volatile("" : "+v"(ln));
        const uint32_t lane_off = 4096u * static_cast<uint32_t>(ln >> 4) + 16u * (ln & 15);
        const uint32_t kb = lds0 + st * kPfStageBytes;
        const uint32_t vb = kb + kPfKBytes;
        const int n0 = (tile0 + tile) * kPfBN;
        const bool clamp = n0 + kPfBN > blk_kv_end;
#pragma unroll
        for (int r = 0; r < kDmaPerWave; ++r) {
            const int blk = wave * kDmaPerWave + r;
            int64_t row_base = static_cast<int64_t>(n0 + blk) * kHeadDim;
            uint32_t off = lane_off;
            if (clamp) {
                // Address from the tile start: n0 <= blk_kv_end - 1, so every
                // clamped row is >= n0 and the unsigned offset stays in range.
                const int row = min(n0 + blk + 16 * (ln >> 4), blk_kv_end - 1);
                row_base = static_cast<int64_t>(n0) * kHeadDim;
                off = static_cast<uint32_t>(row - n0) * 256u + 16u * (ln & 15);
            }
            lds_dma16(uniform_ptr(kh + row_base), off, __builtin_amdgcn_readfirstlane(kb + kPfKBlock * blk));
            lds_dma16(uniform_ptr(vh + row_base), off, __builtin_amdgcn_readfirstlane(vb + kPfVBlock * blk));
        }
    };

    // Tiles 0 and 1 are copied ahead; tile t+2 is issued in tile step t
    // (after the barrier that opens it), into the stage of tile t-2, whose
    // last reader (group B's PV of tile t-2, in its GEMM(t-1)) ended before
    // that barrier.
    if (kWaves != 4 || copies_only) {
        if (ntiles > 0) issue_tile(0, 0, std::integral_constant<bool, kDyn>{});
        if (ntiles > 1) issue_tile(1, 1, std::integral_constant<bool, kDyn>{});
    }
    // Tile t is in LDS once at most the copies of tile t+1 are outstanding
    // (vector-memory loads retire in order).
    static_assert(kPfStages == 4, "the wait below assumes one tile in flight behind tile t");
    auto wait_tile = [&](int t) {
        if (t >= ntiles) return;
        if (t + 1 < ntiles) {
            __builtin_amdgcn_s_waitcnt(waitcnt_vm(2 * kDmaPerWave));
        } else {
            __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
        }
    };
    if constexpr (kWaves == 4) {
        if (copies_only) {
            for (int t = 0; t <= ntiles; ++t) {
                wait_tile(t);
                pf_barrier();
                if (t + 2 < ntiles) issue_tile(t + 2, (t + 2) % kPfStages, std::false_type{});
            }
            return;
        }
    }

    // Q^T (B operand): qop[kk] = Q[row0 + l32][16kk + 8hl + 0..7].
    half8_t qop[8];
    {
        const int row = row0 + l32;
        const bool ok = task_ok && row < a.q_len;
        const uint16_t* qr = a.q + (static_cast<int64_t>(ok ? row : 0) * a.num_q_heads + qh) * kHeadDim;
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) qop[kk] = load_half8(qr + 16 * kk + 8 * hl);
        if (!ok) {
#pragma unroll
            for (int kk = 0; kk < 8; ++kk) qop[kk] = half8_t{};
        }
    }
    // Settle the Q loads here.  The compiler's wait insertion does not see the
    // asm DMAs, so a Q load still pending at the loop would make it wait
    // for Q inside the loop with a vmcnt that, counted by the hardware, also
    // covers the next tile's copies: one stall per tile.  The asm "use" makes
    // it wait once, before the loop.
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) asm volatile("" : "+v"(qop[kk]));

    float16_t o[4];
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] = 0.0f;
    float m_run = kPfNegBig, l_run = 0.0f;
    const float c = a.scale_log2;
    float16_t s[2];  // S^T of the tile in flight
    half8_t pop[4];  // P^T of the last softmaxed tile
#pragma unroll
    for (int k = 0; k < 4; ++k) pop[k] = half8_t{};
    // The V half of the last stage is what GEMM(0) of the 8-wavefront forms
    // multiplies with P = 0: zero it (finite), before the first barrier.  Tile 3
    // refills it only after both groups are past GEMM(0).
    if constexpr (kWaves != 4) {
        uint4_t* vz = reinterpret_cast<uint4_t*>(pf_lds + (kPfStages - 1) * kPfStageBytes + kPfKBytes);
        for (int i = tid; i < kPfVBytes / 16; i += kWaves * kWave) vz[i] = uint4_t{0u, 0u, 0u, 0u};
    }

    // Per-lane LDS read offsets.  K (A operand of S^T = K Q^T): key 32mb + l32,
    // dims 16kk + 8hl.  V^T (A operand of O^T += V^T P^T) via the transposing
    // read: 16-lane group gi = lane/16 covers dims 32db + 16(gi&1) + [0,16) and
    // keys 16ks + 4(gi>>1) + [0,4) (+8 for reduction slots 4..7).
    const int gi = lane >> 4, ii = lane & 15;
    const uint32_t k_lane = (l32 & 15) * kPfKBlock + (l32 >> 4) * 256 + 16 * hl;
    const uint32_t v_lane = (4 * (gi >> 1) + (ii >> 2)) * kPfVBlock + 32 * (gi & 1) + 8 * (ii & 3);

    // GEMM phase of tile j (8-wavefront forms): PV of tile j-1, then S of tile j.
    //
    // Every GEMM phase runs all 32 slots (one code path keeps register
    // allocation tight): at j = 0 the PV half multiplies P = 0 with the V
    // stage zeroed above (adds exactly +0 to O); at j = wave_tiles the S half
    // reads a stage inside LDS and its result is never used.
    // A split wavefront whose range starts after the workgroup's first tile
    // runs the GEMM phases before it too: its P is still zero there (PV adds
    // exactly +0; the V tile is finite cache data) and those S tiles are
    // never softmaxed.  One skip condition keeps the accumulators in place.
    auto gemm_phase = [&](int j) {
        if (j > wave_tiles) return;
        pf_gemm(pf_lds + (j % kPfStages) * kPfStageBytes + k_lane,
                pf_lds + ((j + kPfStages - 1) % kPfStages) * kPfStageBytes + kPfKBytes + v_lane, qop, pop, o, s);
    };

    // Softmax phase of tile j: mask, running max (lazy), P = 2^(c*s - m), row sum.
    // Masked scores: -1e30 as the reference adds (src/kernels.rs:1242-1257).
    // The split form may have rows with every key of a range masked (the
    // range starts past the row's position); -inf gives them p = 0 and so
    // O = 0, LSE = -1e30, weight 0 in the merge (the reference's -1e30 gives
    // such rows p = 1 and an LSE near -1.3e29: also weight 0).
    constexpr float kMasked = kSplit ? -__builtin_inff() : kPfNegBig;
    auto mask_tile = [&](int j, float16_t (&sc)[2]) {
        const int n0 = (tile0 + j) * kPfBN;
        bool need_mask = (n0 + kPfBN - 1 > pos0) || (n0 + kPfBN > a.kv_len);
        if constexpr (kSplit) need_mask = need_mask || n0 < key_lo || n0 + kPfBN > key_hi;
        if (need_mask) {
            // Keys n in [key_lo, n_end) stay, n_end = min(position + 1, key_hi,
            // kv_len) clamped to >= key_lo: one unsigned compare per score.
            const int n_end = max(key_lo, min(min(pos0 + l32 + 1, key_hi), a.kv_len));
            const uint32_t span = static_cast<uint32_t>(n_end - key_lo);
            const int rel0 = n0 - key_lo + 4 * hl;
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int rel = rel0 + 32 * mb + 8 * (r >> 2) + (r & 3);
                    if (static_cast<uint32_t>(rel) >= span) sc[mb][r] = kMasked;
                }
        }
    };
    auto softmax_phase = [&](int j) {
        if (j < wave_t0 || j >= wave_tiles) return;
        mask_tile(j, s);
        pf_softmax<2>(s, pop, o, m_run, l_run, c);
    };

    // 8-wavefront forms, tile step t: group A runs GEMM(t) then softmax(t), group
    // B softmax(t-1) then GEMM(t).  GEMM(ntiles) is the last PV; softmax of a tile
    // outside the wavefront's range is a no-op.  Each group has its own
    // straight-line loop (B's is A's rotated by one phase); both pass the same
    // ntiles+1 barriers, one at the start of each step.  Tile t+2 is issued after
    // the barrier of step t into the stage of tile t-2, whose last reader (group
    // B's GEMM(t-1), the PV of tile t-2) ended before that barrier.
    auto open_tile_step = [&](int t) {
        wait_tile(t);
        pf_barrier();
    };
    // The copies of tile t+2 go out at the start of each wavefront's softmax
    // phase of step t: group A's after its GEMM phase, group B's at the
    // start of the step.  Issued by all eight wavefronts right after the
    // barrier, the copies queue behind each other and hold up the GEMM phase
    // of group A (measured ~1% slower, bit-identical output).
    if constexpr (kWaves == 4) {
        // One wavefront per SIMD: S of tile t+1 runs under the softmax of tile
        // t (an S MFMA before every pair of exponentials), then PV of tile t.
        // The barrier before step t opens tile t+1; tile t+3 goes into the
        // stage of tile t-1, whose PV ended before it.  Two score buffers
        // alternate.
        auto k_base = [&](int j) { return pf_lds + (j % kPfStages) * kPfStageBytes + k_lane; };
        auto step = [&](int t, float16_t (&cur)[2], float16_t (&nxt)[2]) {
            pf_barrier();
            if (t >= wave_tiles) return;
            mask_tile(t, cur);
            if (t + 1 < wave_tiles) {
                const unsigned char* kb = k_base(t + 1);
                constexpr int kRing = kPfAhead + 1;
                half8_t ring[kRing];
                auto read_op = [&](int i) {
                    return *reinterpret_cast<const half8_t*>(kb + 512 * (i & 1) + 32 * (i >> 1));
                };
#pragma unroll
                for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                    for (int r = 0; r < 16; ++r) nxt[mb][r] = 0.0f;
#pragma unroll
                for (int i = 0; i < kPfAhead; ++i) ring[i % kRing] = read_op(i);
                pf_softmax<2>(cur, pop, o, m_run, l_run, c, [&](int i) {
                    if (i + kPfAhead < 16) ring[(i + kPfAhead) % kRing] = read_op(i + kPfAhead);
                    nxt[i & 1] = mfma32x32x16(ring[i % kRing], qop[i >> 1], nxt[i & 1]);
                    __builtin_amdgcn_sched_barrier(0);
                });
            } else {
                pf_softmax<2>(cur, pop, o, m_run, l_run, c);
            }
            pf_values(pf_lds + (t % kPfStages) * kPfStageBytes + kPfKBytes + v_lane, pop, o);
        };
        float16_t s2[2];
        pf_barrier();
        if (wave_tiles > 0) pf_scores(k_base(0), qop, s);
        for (int t = 0; t < ntiles; t += 2) {
            step(t, s, s2);
            if (t + 1 < ntiles) step(t + 1, s2, s);
        }
    } else if (grp == 0) {
        for (int t = 0; t <= ntiles; ++t) {
            open_tile_step(t);
            gemm_phase(t);
            if (t + 2 < ntiles) issue_tile(t + 2, (t + 2) % kPfStages, std::false_type{});
            softmax_phase(t);
        }
    } else {
        for (int t = 0; t <= ntiles; ++t) {
            open_tile_step(t);
            if (t + 2 < ntiles) issue_tile(t + 2, (t + 2) % kPfStages, std::false_type{});
            softmax_phase(t - 1);
            gemm_phase(t);
        }
    }

    if constexpr (kDyn) {
        if (wave == 0 && lane == 0 && own_live)
            pre_j = __hip_atomic_fetch_add(a.sched + my_q * kPfSchedStride, 1u, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
    }
    if (task_ok) {
    // Row row0 + l32 of O^T holds dims d = 32db + 8(r/4) + 4hl + r%4.
    const float lt = l_run + swap_halves(l_run);
    const float l_safe = fmaxf(lt, 1.0e-8f);
    // O / l_safe is the reference's true division (src/kernels.rs:1289-1291),
    // rounded to f32 and then to f16: div_to_half gives that same f16 from one
    // f64 reciprocal per row.  (An f32 reciprocal and multiplies is not the
    // same operation: up to 1 f16 ulp away.)
    const double rl = 1.0 / static_cast<double>(l_safe);
    if constexpr (kSplit) {
        // Logical tile (q block, head group) = bq * (Hq/GROUP) + qh/GROUP; its
        // row r = (row % BM) * GROUP + qh % GROUP in split-major scratch
        // (src/kernels.rs:2105-2141).  Rows past q_len (zero Q) are written
        // too, as the reference's padded tile rows are.
        const int row = row0 + l32;
        const int m_eff = a.block_m * a.split_group;
        const int64_t tile = static_cast<int64_t>(row / a.block_m) * (a.num_q_heads / a.split_group) +
                             qh / a.split_group;
        const int64_t prow = (tile * a.num_splits + blockIdx.y) * m_eff +
                             (row % a.block_m) * a.split_group + qh % a.split_group;
        uint16_t* prow_p = a.att_partial + prow * kHeadDim;
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                half4_t h;
#pragma unroll
                for (int e = 0; e < 4; ++e) h[e] = div_to_half(o[db][4 * i + e], rl);
                *reinterpret_cast<half4_t*>(prow_p + 32 * db + 8 * i + 4 * hl) = h;
            }
        if (hl == 0) a.lse_partial[prow] = m_run + log2f(l_safe);
    } else {
        half4_t hv[16];
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) hv[4 * db + i][e] = div_to_half(o[db][4 * i + e], rl);
        if constexpr (kDyn) {
            // The ticket claimed after the loop is read back before the
            // stores go out: vmcnt also counts stores, so reading it after
            // them would wait for the stores as well.
            if (wave == 0) pre_ticket = own_live ? static_cast<int>(__shfl(pre_j, 0)) : -1;
            asm volatile("" ::: "memory");
        }
        // The 32 x 128 tile goes out in whole rows: written to LDS in the
        // accumulator layout, read back 16 bytes a lane, so one store covers 4
        // rows x 256 bytes.  (Stored from the accumulator layout, every store
        // touches 32 rows, 16 bytes each: 8x the write requests, ~2 us a task.)
        // Group A uses stage (ntiles+1) % 4, group B stage (ntiles+2) % 4: no
        // tile is copied into either after tile ntiles-1 and their last
        // readers ended before the last barrier.  16-byte chunk c of row r
        // sits at chunk c ^ (r % 16), so the row reads are free of bank
        // conflicts.
        // Lane terms derived here from the lane id (the empty asm stops the
        // compiler from hoisting them out of the persistent task loop and
        // spilling them across it).
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const int lr = ln & 31, lb = ln >> 4, cc = ln & 15;
        const int sw_w = 16 * (lr & 15);
        const int sw_r = 16 * (cc ^ lb);  // read row r = lb + 4k: r % 16 = lb | 4(k % 4)
        unsigned char* ot = pf_lds + ((ntiles + 1 + grp) % kPfStages) * kPfStageBytes + (wave & 3) * kPfOutBytes;
        unsigned char* wrow = ot + lr * 256 + 8 * (ln >> 5);
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<half4_t*>(wrow + ((16 * (4 * db + i)) ^ sw_w)) = hv[4 * db + i];
        // A wavefront's LDS accesses complete in order; the fence keeps the
        // compiler from moving the reads above the writes.
        asm volatile("" ::: "memory");
        const unsigned char* rrow = ot + lb * 256;
        uint16_t* orow = a.out + (static_cast<int64_t>(row0 + lb) * a.num_q_heads + qh) * kHeadDim + 8 * cc;
        const int64_t ostep = static_cast<int64_t>(4) * a.num_q_heads * kHeadDim;  // 4 rows
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const uint4_t v = *reinterpret_cast<const uint4_t*>(rrow + 1024 * k + (sw_r ^ (64 * (k & 3))));
            if (row0 + lb + 4 * k < a.q_len) *reinterpret_cast<uint4_t*>(orow + ostep * k) = v;
        }
    }
    } else if constexpr (kDyn) {
        if (wave == 0) pre_ticket = own_live ? static_cast<int>(__shfl(pre_j, 0)) : -1;
    }  // task_ok
    if constexpr (!kDyn) break;
    }  // task loop

    if constexpr (kDyn) {
        // The last workgroup to leave clears the counters for the next launch:
        // every other one has stopped claiming before its exit increment.
        if (tid == 0) {
            const uint32_t done = __hip_atomic_fetch_add(a.sched + kPfExit * kPfSchedStride, 1u,
                                                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (done + 1 == static_cast<uint32_t>(a.n_wg)) {
                for (int q = 0; q < kPfSchedCounters; ++q)
                    __hip_atomic_store(a.sched + q * kPfSchedStride, 0u, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
}

// Short prefill: for a launch whose row blocks need at most kSpWaves key tiles
// and whose (query head, 32-row block) pairs fit one workgroup per CU.  The
// grid above would walk up to 8 tiles in sequence in its heaviest workgroup;
// here one workgroup takes one (query head, row block), its 8 wavefronts take
// one 64-key tile each, and the 8 online-softmax partials (m, l, O) meet in
// LDS: the critical path is one tile and a merge.  Each wavefront computes
// S^T = K Q^T with K straight from global memory (an A operand is 16
// contiguous bytes of one key row) and O^T += V^T P^T with V copied into its
// own LDS region (the transposing reads need it there), in the LDS layout and
// lane mapping of the main kernel.  The merge follows the split-K reduction:
// M = max_w m_w, out = f16(sum_w 2^(m_w-M) O_w / max(sum_w 2^(m_w-M) l_w, 1e-8)).
// Keys outside a row's causal range are -inf (a wavefront whose tile holds no
// key of a row keeps m = -1e30, l = 0, O = 0 for it: weight 0); tile 0 holds
// key 0, which every row sees, so M is always a real score.
constexpr int kSpWaves = 8;
constexpr int kSpORow = 132;  // f32 per LDS row of a merge partial (16-lane groups hit distinct banks)
constexpr int kSpOBytes = 32 * kSpORow * 4;
static_assert(kSpOBytes + 256 <= kPfVBytes, "a wavefront's merge partial fits its V region");

__global__ __launch_bounds__(kSpWaves * kWave, 1) void attn_prefill_short_kernel(PrefillArgs a) {
    __shared__ __attribute__((aligned(1024))) unsigned char sp_lds[kSpWaves * kPfVBytes];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int lane = tid % kWave;
    const int l32 = lane & 31;
    const int hl = lane >> 5;

    // Heaviest row blocks first; the query heads of a row block are consecutive.
    const int qh = static_cast<int>(blockIdx.x % a.num_q_heads);
    const int pt = a.n_pos_tiles - 1 - static_cast<int>(blockIdx.x / a.num_q_heads);
    const int kvh = qh / a.group;
    const int row0 = pt * kPfRows;
    const int pos0 = a.query_start + row0;
    const int blk_kv_end = min(a.kv_len, pos0 + kPfRows);
    const int ntiles = (blk_kv_end + kPfBN - 1) / kPfBN;  // <= kSpWaves (host check)

    unsigned char* vw = sp_lds + wave * kPfVBytes;
    float16_t o[4];
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] = 0.0f;
    float m_w = kPfNegBig, l_w = 0.0f;

    if (wave < ntiles) {
        const int n0 = wave * kPfBN;
        const uint16_t* kh = a.k_cache + static_cast<int64_t>(kvh) * a.max_seq_len * kHeadDim;
        const uint16_t* vh = a.v_cache + static_cast<int64_t>(kvh) * a.max_seq_len * kHeadDim;
        // K operands: kop[mb][kk] = K[n0 + 32mb + l32][16kk + 8hl .. +8]; rows
        // at or past blk_kv_end read the last valid row (masked below).
        half8_t kop[2][8];
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) {
            const int key = min(n0 + 32 * mb + l32, blk_kv_end - 1);
#pragma unroll
            for (int kk = 0; kk < 8; ++kk)
                kop[mb][kk] = load_half8(kh + static_cast<int64_t>(key) * kHeadDim + 16 * kk + 8 * hl);
        }
        // V tile into this wavefront's region: copy r fills block r with rows
        // n0 + r + 16j, j = lane/16, clamped like the K rows.  K, V and Q are
        // in flight together (vector-memory ops retire in order, so the first
        // MFMA's wait covers all three): one memory round trip for the tile.
        const uint32_t vw0 = static_cast<uint32_t>(
            (uintptr_t)((__attribute__((address_space(3))) unsigned char*)(vw)));
        const bool clamp = n0 + kPfBN > blk_kv_end;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            int64_t row_base = static_cast<int64_t>(n0 + r) * kHeadDim;
            uint32_t off = 4096u * static_cast<uint32_t>(lane >> 4) + 16u * (lane & 15);
            if (clamp) {
                const int row = min(n0 + r + 16 * (lane >> 4), blk_kv_end - 1);
                row_base = static_cast<int64_t>(n0) * kHeadDim;
                off = static_cast<uint32_t>(row - n0) * 256u + 16u * (lane & 15);
            }
            lds_dma16(vh + row_base, off, vw0 + kPfVBlock * r);
        }
        half8_t qop[8];
        {
            const int row = row0 + l32;
            const bool ok = row < a.q_len;
            const uint16_t* qr = a.q + (static_cast<int64_t>(ok ? row : 0) * a.num_q_heads + qh) * kHeadDim;
#pragma unroll
            for (int kk = 0; kk < 8; ++kk) qop[kk] = ok ? load_half8(qr + 16 * kk + 8 * hl) : half8_t{};
        }
        float16_t s[2];
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int r = 0; r < 16; ++r) s[mb][r] = 0.0f;
#pragma unroll
        for (int kk = 0; kk < 8; ++kk)
#pragma unroll
            for (int mb = 0; mb < 2; ++mb) s[mb] = mfma32x32x16(kop[mb][kk], qop[kk], s[mb]);
        if (n0 + kPfBN - 1 > pos0 || n0 + kPfBN > a.kv_len) {
            const int n_end = min(pos0 + l32 + 1, a.kv_len);
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int key = n0 + 32 * mb + 8 * (r >> 2) + 4 * hl + (r & 3);
                    if (key >= n_end) s[mb][r] = -__builtin_inff();
                }
        }
        const float c = a.scale_log2;
        float mx = fmaxf(s[0][0], s[0][1]);
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int r = (mb == 0 ? 2 : 0); r < 16; r += 2) mx = fmaxf(mx, fmaxf(s[mb][r], s[mb][r + 1]));
        mx = fmaxf(mx, swap_halves(mx));
        m_w = fmaxf(kPfNegBig, mx * c);
        half8_t pop[4];
        float ps[4];
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const float p0 = __builtin_amdgcn_exp2f(fmaf(s[mb][r], c, -m_w));
                const float p1 = __builtin_amdgcn_exp2f(fmaf(s[mb][r + 1], c, -m_w));
                const int k = (r >> 1) & 3;
                ps[k] = (mb == 0 && r < 8) ? (p0 + p1) : ps[k] + (p0 + p1);
                pop[2 * mb + (r >> 3)][r & 7] = static_cast<half_t>(p0);
                pop[2 * mb + (r >> 3)][(r & 7) + 1] = static_cast<half_t>(p1);
            }
        l_w = (ps[0] + ps[1]) + (ps[2] + ps[3]);
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));  // this wavefront's V copies landed
        asm volatile("" ::: "memory");
        const int gi = lane >> 4, ii = lane & 15;
        const unsigned char* vb = vw + (4 * (gi >> 1) + (ii >> 2)) * kPfVBlock + 32 * (gi & 1) + 8 * (ii & 3);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const unsigned char* p0 = vb + 256 * (i >> 2) + 64 * (i & 3);
            const half8_t va = cat(lds_read_tr16(reinterpret_cast<const half_t*>(p0)),
                                   lds_read_tr16(reinterpret_cast<const half_t*>(p0 + 8 * kPfVBlock)));
            o[i & 3] = mfma32x32x16(va, pop[i >> 2], o[i & 3]);
        }
    }

    // Every wavefront's partial into its own region (its V reads are done
    // after the barrier), rows of kSpORow f32, then m and the row sum l.
    pf_barrier();
    {
        float* orow = reinterpret_cast<float*>(vw) + l32 * kSpORow;
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float4_t v = {o[db][4 * j], o[db][4 * j + 1], o[db][4 * j + 2], o[db][4 * j + 3]};
                *reinterpret_cast<float4_t*>(orow + 32 * db + 8 * j + 4 * hl) = v;
            }
        const float lt = l_w + swap_halves(l_w);
        float* ml = reinterpret_cast<float*>(vw + kSpOBytes);
        if (hl == 0) {
            ml[l32] = m_w;
            ml[32 + l32] = lt;
        }
    }
    pf_barrier();
    // Thread (row, 8 dims): the 8 partials of its row.
    const int row = tid >> 4, d8 = tid & 15;
    float mw[kSpWaves];
    float M = kPfNegBig;
#pragma unroll
    for (int w = 0; w < kSpWaves; ++w) {
        mw[w] = reinterpret_cast<const float*>(sp_lds + w * kPfVBytes + kSpOBytes)[row];
        M = fmaxf(M, mw[w]);
    }
    float L = 0.0f;
    float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < kSpWaves; ++w) {
        const float wt = __builtin_amdgcn_exp2f(mw[w] - M);
        const float* base = reinterpret_cast<const float*>(sp_lds + w * kPfVBytes);
        L += wt * base[kSpOBytes / 4 + 32 + row];
        const float4_t x0 = *reinterpret_cast<const float4_t*>(base + row * kSpORow + 8 * d8);
        const float4_t x1 = *reinterpret_cast<const float4_t*>(base + row * kSpORow + 8 * d8 + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            acc[e] += wt * x0[e];
            acc[4 + e] += wt * x1[e];
        }
    }
    const double rl = 1.0 / static_cast<double>(fmaxf(L, 1.0e-8f));
    half8_t h;
#pragma unroll
    for (int e = 0; e < 8; ++e) h[e] = div_to_half(acc[e], rl);
    if (row0 + row < a.q_len)
        store_half8(a.out + (static_cast<int64_t>(row0 + row) * a.num_q_heads + qh) * kHeadDim + 8 * d8, h);
}

// Key-split prefill, for a few query rows behind many keys (a chunk of a prompt,
// drafted tokens checked against a long context), where the grids above leave
// most CUs idle and walk the keys in sequence.  gridDim.y workgroups share a
// row block's keys and leave f32 partials (O, m, l) in a workspace, which
// attn_prefill_split32_merge_kernel combines.
//  * Rows are packed position-major over the query heads of the KV head: tile
//    row i is position i / G, head i % G.  A few positions then fill a tile
//    (7 rows of 4 heads are one tile, not four).
//  * Workgroup = 4 row tiles; two wavefronts share a tile and take the first and
//    the second 32 keys of every 64-key tile.  Group A (waves 0-3) and group B
//    (waves 4-7) ping-pong as in the grid above, half a tile per phase; waves
//    8-11 only copy.  (12 wavefronts leave 168 VGPRs each; half a tile needs
//    154.)  At the end each wavefront takes over half of its partner's O
//    through LDS, so a row tile leaves one partial per split.
//  * LDS: four K and four V slots.  The copy wavefronts issue V(t+2) and K(t+3)
//    after the barrier of step t, into the slots that GEMM(t-1) read last, three
//    steps before GEMM(t+2) and GEMM(t+3) need them.
// Bound by the copies with one or two row tiles per KV head (a CU takes ~40
// bytes a cycle into LDS, HBM gives each ~28 GB/s, 12 bytes a cycle), by the
// phases' fixed latencies (~2000 cycles a 64-key step) with more.  Measured,
// the 4-tile grid above -> split kernel and merge: 32/8 heads, 7 rows behind
// 12001 keys 156 -> 18.7 us (2.6 TB/s of K/V), 509 behind 6003 90 -> 67; 64/8
// heads, 10 behind 28683 366 -> 30.8 (3.8 TB/s); 16/8 heads, 5 behind 3000 42.5
// -> 10.5.
constexpr int kPrWaves = 8;      // computing wavefronts
constexpr int kPrCopyWaves = 4;  // and copying ones
constexpr int kPrThreads = (kPrWaves + kPrCopyWaves) * kWave;
constexpr int kPrTiles = 4;  // row tiles per workgroup
constexpr int kPrSlots = 4;
constexpr int kPrLdsBytes = kPrSlots * (kPfKBytes + kPfVBytes);
constexpr int kPrExchBytes = 8 * kWave * 16;       // half of O of one wavefront
constexpr int kPrMlOff = kPrWaves * kPrExchBytes;  // then m[32], l[32] per wavefront
constexpr int kPrPartFloats = 32 * kHeadDim;       // O of one (tile, split)
constexpr int kPrMaxSplits = 64;
static_assert(kPrMlOff + kPrWaves * 256 <= kPrLdsBytes, "the exchange reuses the slots");

struct Split32Args {
    const uint16_t* q;
    const uint16_t* k_cache;
    const uint16_t* v_cache;
    uint16_t* out;
    float scale_log2;
    int num_q_heads;
    int group;
    int rows;             // q_len * group packed rows per KV head
    int kv_len;
    int query_start;
    int max_seq_len;
    int n_tiles;          // ceil(rows / 32)
    int blocks_per_head;  // ceil(n_tiles / kPrTiles)
    int num_splits;       // gridDim.y
    float* part_o;        // [Hkv, n_tiles, num_splits][32 * 128], accumulator order
    float* part_ml;       // [Hkv, n_tiles, num_splits][m 32, l 32]
};

__global__ __launch_bounds__(kPrThreads, 1) void attn_prefill_split32_kernel(Split32Args a) {
    __shared__ __attribute__((aligned(1024))) unsigned char pr_lds[kPrLdsBytes];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int grp = wave >> 2;  // 0: A, 1: B (2: copies)
    const int w4 = wave & 3;
    const int lane = tid % kWave;
    const int l32 = lane & 31;
    const int hl = lane >> 5;

    // The order of the grids above: a head's blocks on one XCD, heaviest first.
    const int nb = gridDim.x;
    int T = blockIdx.x;
    if (nb % 8 == 0) {
        const int hkv = nb / a.blocks_per_head;
        const int x = T % 8, i = T / 8;
        if (hkv < 8 && 8 % hkv == 0) {
            const int hx = 8 / hkv;
            T = (x / hx) * a.blocks_per_head + i * hx + x % hx;
        } else {
            T = x * (nb / 8) + i;
        }
    }
    const int kvh = T / a.blocks_per_head;
    const int u0 = (T % a.blocks_per_head) * kPrTiles;
    const bool task_ok = u0 + w4 < a.n_tiles;
    const int pt = a.n_tiles - 1 - (u0 + w4);  // row tile, heaviest first
    // Keys of row tile p end at the limit of its last position.
    auto tile_end = [&](int p) {
        return min(a.kv_len, a.query_start + min(32 * p + 31, a.rows - 1) / a.group + 1);
    };
    const int blk_kv_end = tile_end(a.n_tiles - 1 - u0);
    // Split y's tiles: an even share of the workgroup's.
    const int64_t n_kt = (blk_kv_end + kPfBN - 1) / kPfBN;
    const int tile0 = static_cast<int>(n_kt * blockIdx.y / a.num_splits);
    const int tile1 = static_cast<int>(n_kt * (blockIdx.y + 1) / a.num_splits);
    const int steps = tile1 - tile0;

    if (wave >= kPrWaves) {
        // Copy wavefront: blocks 4 w4 + r of every tile.
        const uint16_t* kh = a.k_cache + static_cast<int64_t>(kvh) * a.max_seq_len * kHeadDim;
        const uint16_t* vh = a.v_cache + static_cast<int64_t>(kvh) * a.max_seq_len * kHeadDim;
        const uint32_t lds0 = static_cast<uint32_t>(
            (uintptr_t)((__attribute__((address_space(3))) unsigned char*)(pr_lds)));
        auto issue = [&](int j, const uint16_t* src, uint32_t slot, int block_bytes) {
            if (j >= steps) return;
            const int n0 = (tile0 + j) * kPfBN;
            const bool clamp = n0 + kPfBN > blk_kv_end;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int blk = 4 * w4 + r;
                int64_t row_base = static_cast<int64_t>(n0 + blk) * kHeadDim;
                uint32_t off = 4096u * static_cast<uint32_t>(lane >> 4) + 16u * (lane & 15);
                if (clamp) {
                    // Rows at or past blk_kv_end repeat the last valid one.
                    const int row = min(n0 + blk + 16 * (lane >> 4), blk_kv_end - 1);
                    row_base = static_cast<int64_t>(n0) * kHeadDim;
                    off = static_cast<uint32_t>(row - n0) * 256u + 16u * (lane & 15);
                }
                lds_dma16(uniform_ptr(src + row_base), off,
                          __builtin_amdgcn_readfirstlane(slot + static_cast<uint32_t>(block_bytes * blk)));
            }
        };
        auto issue_k = [&](int j) { issue(j, kh, lds0 + (j % kPrSlots) * kPfKBytes, kPfKBlock); };
        auto issue_v = [&](int j) {
            issue(j, vh, lds0 + kPrSlots * kPfKBytes + (j % kPrSlots) * kPfVBytes, kPfVBlock);
        };
        issue_k(0);
        issue_v(0);
        issue_k(1);
        issue_v(1);
        issue_k(2);
        for (int t = 0; t <= steps; ++t) {
            // GEMM(t) needs K(t) and V(t-1); V(t), K(t+1), V(t+1) and K(t+2),
            // four copies each as far as they are in range, are younger.
            if (t + 2 < steps) {
                __builtin_amdgcn_s_waitcnt(waitcnt_vm(16));
            } else if (t + 1 < steps) {
                __builtin_amdgcn_s_waitcnt(waitcnt_vm(12));
            } else if (t < steps) {
                __builtin_amdgcn_s_waitcnt(waitcnt_vm(4));
            } else {
                __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
            }
            pf_barrier();
            issue_v(t + 2);
            issue_k(t + 3);
        }
        // The two barriers of the merge below.
        pf_barrier();
        pf_barrier();
        return;
    }

    // This wavefront's tiles: tile0 + j, j < cnt.
    int cnt = 0;
    if (task_ok) cnt = max(0, min(tile1, (tile_end(pt) + kPfBN - 1) / kPfBN) - tile0);

    // Q^T (B operand) of packed row 32 pt + l32, and that row's key limit.
    const int ridx = min(max(32 * pt + l32, 0), a.rows - 1);
    const int rpos = ridx / a.group;
    const int n_end = min(a.query_start + rpos + 1, a.kv_len);
    const bool row_ok = task_ok && 32 * pt + l32 < a.rows;
    half8_t qop[8];
    {
        const uint16_t* qr = a.q + (static_cast<int64_t>(rpos) * a.num_q_heads + kvh * a.group +
                                    (ridx - rpos * a.group)) * kHeadDim;
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) qop[kk] = load_half8(qr + 16 * kk + 8 * hl);
        if (!row_ok) {
#pragma unroll
            for (int kk = 0; kk < 8; ++kk) qop[kk] = half8_t{};
        }
    }
    // Settled before the loop, as in the grid above.
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) asm volatile("" : "+v"(qop[kk]));

    float16_t o[4];
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] = 0.0f;
    float m_run = kPfNegBig, l_run = 0.0f;
    const float c = a.scale_log2;
    float16_t s[1];
    half8_t pop[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) pop[i] = half8_t{};
    // GEMM(0) multiplies P = 0 with V slot 3: zero it (finite); V(3) is copied
    // there after the barrier of step 1.
    {
        uint4_t* vz = reinterpret_cast<uint4_t*>(pr_lds + kPrSlots * kPfKBytes + (kPrSlots - 1) * kPfVBytes);
        for (int i = tid; i < kPfVBytes / 16; i += kPrWaves * kWave) vz[i] = uint4_t{0u, 0u, 0u, 0u};
    }
    // This wavefront's half of a tile: key block grp (K), key steps 2 grp and
    // 2 grp + 1 (V).
    const int gi = lane >> 4, ii = lane & 15;
    const uint32_t k_lane = (l32 & 15) * kPfKBlock + (l32 >> 4) * 256 + 16 * hl + 512 * grp;
    const uint32_t v_lane = kPrSlots * kPfKBytes + (4 * (gi >> 1) + (ii >> 2)) * kPfVBlock + 32 * (gi & 1) +
                            8 * (ii & 3) + 512 * grp;
    // First key limit in the row tile: keys below it need no mask.
    const int n_min = min(a.query_start + max(32 * pt, 0) / a.group + 1, a.kv_len);

    auto gemm_phase = [&](int j) {
        if (j > cnt) return;
        pf_gemm_half(pr_lds + (j % kPrSlots) * kPfKBytes + k_lane,
                     pr_lds + ((j + kPrSlots - 1) % kPrSlots) * kPfVBytes + v_lane, qop, pop, o, s);
    };
    // A row may have no key in a wavefront's halves: masked scores are -inf,
    // which leaves m = -1e30 (or the -1.3e29 of a scaled -1e30), l = 0, O = 0
    // and so weight 0 in the merge.
    auto softmax_phase = [&](int j) {
        if (j < 0 || j >= cnt) return;
        const int n0 = (tile0 + j) * kPfBN + 32 * grp;
        if (n0 + 32 > n_min) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int key = n0 + 4 * hl + 8 * (r >> 2) + (r & 3);
                if (key >= n_end) s[0][r] = -__builtin_inff();
            }
        }
        pf_softmax<1>(s, pop, o, m_run, l_run, c);
    };
    if (grp == 0) {
        for (int t = 0; t <= steps; ++t) {
            pf_barrier();
            gemm_phase(t);
            softmax_phase(t);
        }
    } else {
        for (int t = 0; t <= steps; ++t) {
            pf_barrier();
            softmax_phase(t - 1);
            gemm_phase(t);
        }
    }

    // Merge of the pair: each wavefront hands over the 64 dims the other one
    // finishes (A keeps dim blocks 0-1, B 2-3).  No copy is outstanding: the
    // last ones were waited for at the barrier of the last step.
    pf_barrier();
    const float lt = l_run + swap_halves(l_run);
    unsigned char* exch = pr_lds + wave * kPrExchBytes;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int i = k & 3;
        float4_t v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float lo = o[k >> 2][4 * i + e], hi = o[2 + (k >> 2)][4 * i + e];
            v[e] = grp ? lo : hi;
        }
        *reinterpret_cast<float4_t*>(exch + (k * kWave + lane) * 16) = v;
    }
    float* ml = reinterpret_cast<float*>(pr_lds + kPrMlOff);
    if (hl == 0) {
        ml[wave * 64 + l32] = m_run;
        ml[wave * 64 + 32 + l32] = lt;
    }
    pf_barrier();
    if (!task_ok) return;
    const int other = wave ^ 4;
    const float m_o = ml[other * 64 + l32], l_o = ml[other * 64 + 32 + l32];
    const float M = fmaxf(m_run, m_o);
    const float f_own = __builtin_amdgcn_exp2f(m_run - M), f_o = __builtin_amdgcn_exp2f(m_o - M);
    const float L = lt * f_own + l_o * f_o;
    const unsigned char* oexch = pr_lds + other * kPrExchBytes;
    float4_t x[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int i = k & 3;
        const float4_t y = *reinterpret_cast<const float4_t*>(oexch + (k * kWave + lane) * 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float own = grp ? o[2 + (k >> 2)][4 * i + e] : o[k >> 2][4 * i + e];
            x[k][e] = own * f_own + y[e] * f_o;
        }
    }
    const int64_t part = (static_cast<int64_t>(kvh) * a.n_tiles + pt) * a.num_splits + blockIdx.y;
    float* po = a.part_o + part * kPrPartFloats + grp * (kPrPartFloats / 2);
#pragma unroll
    for (int k = 0; k < 8; ++k) *reinterpret_cast<float4_t*>(po + (k * kWave + lane) * 4) = x[k];
    if (grp == 0 && hl == 0) {
        a.part_ml[part * 64 + l32] = M;
        a.part_ml[part * 64 + 32 + l32] = L;
    }
}

// Merge of the key splits.  Workgroup (row tile, dim block of
// 32): the split weights w_s = 2^(m_s - M) of the 32 rows go to LDS, then
// thread t sums float4 t of the block over the splits (coalesced, 16 bytes a
// thread) and the block leaves through LDS in 64-byte row pieces.
__global__ __launch_bounds__(256) void attn_prefill_split32_merge_kernel(Split32Args a) {
    __shared__ float s_w[kPrMaxSplits * 32];
    __shared__ float s_red[8 * 32];
    __shared__ float s_sum[8 * 32];
    __shared__ __attribute__((aligned(16))) half_t s_out[32 * 40];
    const int tid = threadIdx.x;
    const int kvh = static_cast<int>(blockIdx.x) / a.n_tiles;
    const int pt = static_cast<int>(blockIdx.x) % a.n_tiles;
    const int db = blockIdx.y;
    const int NS = a.num_splits;
    const int64_t part = static_cast<int64_t>(blockIdx.x) * NS;
    const float* ml = a.part_ml + part * 64;
    const int row = tid & 31, sg = tid >> 5;
    float mx = kPfNegBig;
    for (int s = sg; s < NS; s += 8) mx = fmaxf(mx, ml[s * 64 + row]);
    s_red[sg * 32 + row] = mx;
    __syncthreads();
#pragma unroll
    for (int g = 0; g < 8; ++g) mx = fmaxf(mx, s_red[g * 32 + row]);
    float sum = 0.0f;
    for (int s = sg; s < NS; s += 8) {
        const float w = __builtin_amdgcn_exp2f(ml[s * 64 + row] - mx);
        s_w[s * 32 + row] = w;
        sum += w * ml[s * 64 + 32 + row];
    }
    s_sum[sg * 32 + row] = sum;
    __syncthreads();
    // tid = i * 64 + lane: dims 32 db + 8 i + 4 hl + [0, 4) of row lane % 32.
    const int i = tid >> 6, hl = (tid >> 5) & 1;
    const float* po = a.part_o + part * kPrPartFloats + (db * 256 + tid) * 4;
    float4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 8
    for (int s = 0; s < NS; ++s) {
        const float4_t v = *reinterpret_cast<const float4_t*>(po + static_cast<int64_t>(s) * kPrPartFloats);
        const float w = s_w[s * 32 + row];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] += w * v[e];
    }
    float L = 0.0f;
#pragma unroll
    for (int g = 0; g < 8; ++g) L += s_sum[g * 32 + row];
    const double rl = 1.0 / static_cast<double>(fmaxf(L, 1.0e-8f));
    half4_t h;
#pragma unroll
    for (int e = 0; e < 4; ++e) h[e] = div_to_half(acc[e], rl);
    *reinterpret_cast<half4_t*>(s_out + row * 40 + 8 * i + 4 * hl) = h;
    __syncthreads();
    if (tid < 128) {
        const int r = tid >> 2, j = tid & 3;
        const int idx = 32 * pt + r;
        if (idx < a.rows) {
            const int pos = idx / a.group;
            uint16_t* dst = a.out + (static_cast<int64_t>(pos) * a.num_q_heads + kvh * a.group + (idx - pos * a.group)) * kHeadDim;
            store_half8(dst + 32 * db + 8 * j, *reinterpret_cast<const half8_t*>(s_out + r * 40 + 8 * j));
        }
    }
}

// The short form applies when every row block needs at most kSpWaves key
// tiles and the (query head, row block) pairs number at most one per CU.
// (The last row block's key range ends at min(kv_len, query_start + 32 *
// row blocks), as the kernel computes it.)
static bool prefill_short_fits(const PrefillArgs& a, int cus) {
    const int64_t n_blocks = (static_cast<int64_t>(a.q_len) + kPfRows - 1) / kPfRows;
    const int64_t last_end = min(static_cast<int64_t>(a.kv_len),
                                 static_cast<int64_t>(a.query_start) + kPfRows * n_blocks);
    return last_end <= static_cast<int64_t>(kSpWaves) * kPfBN && n_blocks * a.num_q_heads <= cus;
}

// Time of a grid of `blocks` workgroups (one per CU) that walk from `most` down
// to `least` key tiles, longest first, in tile steps: one round takes the
// longest; in a second round the k-th workgroup past the CUs follows the k-th
// shortest of the first, and with evenly spaced lengths all those pairs have the
// same sum.  Launch, first loads and output stores count as `fixed` steps, 3
// more for a second workgroup on a CU.
static int64_t prefill_rounds(int64_t blocks, int64_t cus, int64_t most, int64_t least, int64_t fixed) {
    int64_t t = most + fixed;
    if (blocks > cus) t = max(t, 2 * most - (most - least) * (2 * cus - 1) / (blocks - 1) + fixed + 3);
    return t;
}

// Whether 4-tile workgroups (blocks4) beat 8-tile ones (blocks8).  In steps of
// prefill_rounds the launches below took 0.92-1.15 us a step with the former,
// 1.22-1.50 with the latter, 0.67 to 0.82 of it at one shape.  The rule counts
// 4/5: the former lose once the grid needs that many more rounds.  Measured, 4
// against 8 tiles: 32/8 heads 1500 tokens 30.4 / 37.4 us, 2048 46.9 / 50.5, 3000
// 91.2 / 81.1; 64/8 heads 1024 tokens 26.9 / 29.9, 1500 52.3 / 45.8, 2048 82.9 /
// 72.5; 16/8 heads 3000 tokens 49.2 / 61.5, 4096 77.2 / 89.2; 32/8 heads, 1024
// tokens behind 8192, 149 / 168, 1100 behind 1000 44.5 / 45.2, 1500 behind 8192
// 259 / 214.  1500 behind 1000, 56.4 / 57.6, goes to 8 tiles.
static bool prefill_narrow_wins(const PrefillArgs& a, int64_t blocks8, int64_t blocks4, int64_t cus) {
    if (blocks4 <= cus) return true;
    if (blocks4 > 2 * cus) return false;
    const int64_t most = (min(static_cast<int64_t>(a.kv_len),
                              static_cast<int64_t>(a.query_start) + kPfRows * static_cast<int64_t>(a.n_pos_tiles)) +
                          kPfBN - 1) / kPfBN;
    const int64_t least = (min(static_cast<int64_t>(a.kv_len), static_cast<int64_t>(a.query_start) + kPfRows) +
                           kPfBN - 1) / kPfBN;
    return 4 * prefill_rounds(blocks4, cus, most, least, 5) <= 5 * prefill_rounds(blocks8, cus, most, least, 4);
}

static int32_t launch_prefill(PrefillArgs a, int num_kv_heads, hipStream_t stream) {
    a.n_pos_tiles = (a.q_len + kPfRows - 1) / kPfRows;
    a.tasks_per_head = a.n_pos_tiles * a.group;
    a.blocks_per_head = (a.tasks_per_head + kPfWaves - 1) / kPfWaves;
    const int64_t blocks = static_cast<int64_t>(a.blocks_per_head) * num_kv_heads;
    if (blocks > 0x7fffffff) return GROUT_ERR_KV_LEN;
    int dev = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return static_cast<int32_t>(e);
    if (prefill_short_fits(a, cus)) {
        const int64_t sblocks = static_cast<int64_t>(a.n_pos_tiles) * a.num_q_heads;
        hipLaunchKernelGGL(attn_prefill_short_kernel, dim3(static_cast<unsigned>(sblocks)),
                           dim3(kSpWaves * kWave), 0, stream, a);
        return launch_status();
    }
    const int64_t bph4 = (static_cast<int64_t>(a.tasks_per_head) + 3) / 4;
    if (prefill_narrow_wins(a, blocks, bph4 * num_kv_heads, cus)) {
        a.blocks_per_head = static_cast<int>(bph4);
        hipLaunchKernelGGL((attn_prefill_kernel<false, false, 4>), dim3(static_cast<unsigned>(bph4 * num_kv_heads)),
                           dim3(kPfWaves * kWave), 0, stream, a);
        return launch_status();
    }
    hipLaunchKernelGGL((attn_prefill_kernel<false, false>), dim3(static_cast<unsigned>(blocks)),
                       dim3(kPfWaves * kWave), 0, stream, a);
    return launch_status();
}

// Dynamic schedule: one persistent workgroup per CU (the kernel's LDS allows
// one) when the static grid would run more than two rounds of workgroups;
// smaller grids keep the static launch, which then leaves the counters alone.
static int32_t launch_prefill_sched(PrefillArgs a, int num_kv_heads, uint32_t* sched,
                                    hipStream_t stream) {
    a.n_pos_tiles = (a.q_len + kPfRows - 1) / kPfRows;
    a.tasks_per_head = a.n_pos_tiles * a.group;
    a.blocks_per_head = (a.tasks_per_head + kPfWaves - 1) / kPfWaves;
    const int64_t blocks = static_cast<int64_t>(a.blocks_per_head) * num_kv_heads;
    if (blocks > 0x7fffffff) return GROUT_ERR_KV_LEN;
    int dev = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return static_cast<int32_t>(e);
    if (cus <= 0 || blocks <= 2 * static_cast<int64_t>(cus)) return launch_prefill(a, num_kv_heads, stream);
    a.sched = sched;
    a.n_wg = cus;
    a.num_kv_heads = num_kv_heads;
    // The lightest quarter of each head's blocks goes to the XCD light queues.
    a.pool_block0 = a.blocks_per_head - a.blocks_per_head / 4;
    hipLaunchKernelGGL((attn_prefill_kernel<false, true>), dim3(static_cast<unsigned>(cus)),
                       dim3(kPfWaves * kWave), 0, stream, a);
    return launch_status();
}

// How a launch is split over its keys; num_splits 0: it is not.
struct Split32Plan {
    int n_tiles, blocks_per_head, num_splits;
};

// Splits only where the 4-tile workgroups leave at least half the CUs idle and
// the short form does not apply, and only when the estimate says it pays.
// Estimates in ns, fitted to the measurements at the kernel and here: unsplit
// 828 per key tile + 4500; split 870 per key tile of a split + 8000 (second
// launch, more stores) + the partials' way out and back at 3.5 TB/s.  Measured
// at the fewest key tiles that split, unsplit / split: 32/8 heads, 5 rows and 9
// tiles 11.9 / 8.8 us, 33 and 9 12.6 / 12.9, 130 and 15 18.0 / 16.8, 512 and 36
// 35.1 / 35.4; 64/8 heads, 33 and 12 15.2 / 14.4; 16/8 heads, 64 and 9 12.6 /
// 13.1, 512 and 21 22.6 / 21.9; 8/1 heads, 130 and 9 12.7 / 13.1; at five more
// tiles the split takes 0.59-0.97 of the unsplit time in each.  Split counts:
// 8/1 heads, 300 rows behind 1000 keys: 1 / 2 / 4 / 8 splits 23.7 / 18.3 / 15.9 /
// 16.7 us; 32/8 heads, 7 behind 12001: 16 / 24 / 32 splits 18.3 / 17.0 / 18.1.
static Split32Plan split32_plan(const PrefillArgs& a, int num_kv_heads, int cus) {
    Split32Plan p = {};
    const int64_t rows = static_cast<int64_t>(a.q_len) * a.group;
    const int64_t n_tiles = (rows + 31) / 32;
    const int64_t bph = (n_tiles + kPrTiles - 1) / kPrTiles;
    const int64_t blocks = bph * num_kv_heads;
    if (2 * blocks > cus || prefill_short_fits(a, cus)) return p;
    const int64_t end = min(static_cast<int64_t>(a.kv_len), static_cast<int64_t>(a.query_start) + a.q_len);
    const int64_t key_tiles = (end + kPfBN - 1) / kPfBN;
    // The fixed cost alone exceeds what a short walk can save; callers skip the
    // question for kv_len <= 512.
    if (key_tiles <= 8) return p;
    const int64_t part_bytes = n_tiles * num_kv_heads * (kPrPartFloats + 64) * 4;
    int64_t best = 828 * key_tiles + 4500;
    const int64_t most = min(min(static_cast<int64_t>(kPrMaxSplits), cus / blocks), key_tiles);
    for (int64_t ns = 2; ns <= most; ++ns) {
        const int64_t t = 870 * ((key_tiles + ns - 1) / ns) + 8000 + 2 * part_bytes * ns / 3500;
        if (t < best) {
            best = t;
            p.num_splits = static_cast<int>(ns);
        }
    }
    p.n_tiles = static_cast<int>(n_tiles);
    p.blocks_per_head = static_cast<int>(bph);
    return p;
}

static int64_t split32_workspace_bytes(const Split32Plan& p, int num_kv_heads) {
    return static_cast<int64_t>(num_kv_heads) * p.n_tiles * p.num_splits * (kPrPartFloats + 64) * 4;
}

static int32_t launch_prefill_split32(const PrefillArgs& a, const Split32Plan& p, int num_kv_heads, void* workspace,
                                      hipStream_t stream) {
    Split32Args b = {};
    b.q = a.q;
    b.k_cache = a.k_cache;
    b.v_cache = a.v_cache;
    b.out = a.out;
    b.scale_log2 = a.scale_log2;
    b.num_q_heads = a.num_q_heads;
    b.group = a.group;
    b.rows = a.q_len * a.group;
    b.kv_len = a.kv_len;
    // A start at or past kv_len sees every key, as kv_len itself does.
    b.query_start = min(a.query_start, a.kv_len);
    b.max_seq_len = a.max_seq_len;
    b.n_tiles = p.n_tiles;
    b.blocks_per_head = p.blocks_per_head;
    b.num_splits = p.num_splits;
    const int64_t parts = static_cast<int64_t>(num_kv_heads) * p.n_tiles * p.num_splits;
    b.part_o = static_cast<float*>(workspace);
    b.part_ml = b.part_o + parts * kPrPartFloats;
    hipLaunchKernelGGL(attn_prefill_split32_kernel,
                       dim3(static_cast<unsigned>(p.blocks_per_head * num_kv_heads), static_cast<unsigned>(p.num_splits)),
                       dim3(kPrThreads), 0, stream, b);
    const int32_t st = launch_status();
    if (st != GROUT_OK) return st;
    hipLaunchKernelGGL(attn_prefill_split32_merge_kernel, dim3(static_cast<unsigned>(num_kv_heads * p.n_tiles), 4),
                       dim3(256), 0, stream, b);
    return launch_status();
}

// Merge of the split-K partials (prefill_splitk_reduce_merge,
// src/kernels.rs:2151-2323): thread = (row < q_len, q head, 8 dims); weights
// w_s = 2^(lse_s - max) / max(sum, 1e-8), out = f16(sum_s w_s * att_s).
__global__ __launch_bounds__(256) void attn_prefill_split_merge_kernel(
    const uint16_t* __restrict__ att, const float* __restrict__ lse, uint16_t* __restrict__ out,
    int num_q_heads, int q_len, int block_m, int group, int num_splits) {
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const int64_t total = static_cast<int64_t>(q_len) * num_q_heads * (kHeadDim / 8);
    if (idx >= total) return;
    const int d0 = static_cast<int>(idx % (kHeadDim / 8)) * 8;
    const int64_t rh = idx / (kHeadDim / 8);
    const int head = static_cast<int>(rh % num_q_heads);
    const int row = static_cast<int>(rh / num_q_heads);
    const int m_eff = block_m * group;
    const int64_t tile = static_cast<int64_t>(row / block_m) * (num_q_heads / group) + head / group;
    const int r = (row % block_m) * group + head % group;
    const float* l = lse + tile * num_splits * m_eff + r;
    float mx = l[0];
    for (int s = 1; s < num_splits; ++s) mx = fmaxf(mx, l[static_cast<int64_t>(s) * m_eff]);
    float sum = 0.0f;
    for (int s = 0; s < num_splits; ++s) sum += __builtin_amdgcn_exp2f(l[static_cast<int64_t>(s) * m_eff] - mx);
    const float inv = 1.0f / fmaxf(sum, 1.0e-8f);
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    const uint16_t* p = att + (tile * num_splits * m_eff + r) * kHeadDim + d0;
    for (int s = 0; s < num_splits; ++s) {
        const float w = __builtin_amdgcn_exp2f(l[static_cast<int64_t>(s) * m_eff] - mx) * inv;
        const half8_t x = load_half8(p + static_cast<int64_t>(s) * m_eff * kHeadDim);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += static_cast<float>(x[e]) * w;
    }
    half8_t o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = static_cast<half_t>(acc[e]);
    store_half8(out + (static_cast<int64_t>(row) * num_q_heads + head) * kHeadDim + d0, o);
}

static int32_t launch_prefill_split(PrefillArgs a, int num_kv_heads, hipStream_t stream) {
    const int64_t q_blocks = (static_cast<int64_t>(a.q_len) + a.block_m - 1) / a.block_m;
    const int64_t pos_tiles = q_blocks * (a.block_m / kPfRows);
    const int64_t tasks = pos_tiles * a.group;
    const int64_t bph = (tasks + kPfWaves - 1) / kPfWaves;
    const int64_t blocks = bph * num_kv_heads;
    if (pos_tiles > 0x3fffffff || blocks > 0x7fffffff) return GROUT_ERR_KV_LEN;
    a.n_pos_tiles = static_cast<int>(pos_tiles);
    a.tasks_per_head = static_cast<int>(tasks);
    a.blocks_per_head = static_cast<int>(bph);
    hipLaunchKernelGGL((attn_prefill_kernel<true, false>), dim3(static_cast<unsigned>(blocks), a.num_splits),
                       dim3(kPfWaves * kWave), 0, stream, a);
    return launch_status();
}

// Scratch geometry of the split-K form: tiles = ceil(q_len/BM) * (Hq/GROUP),
// rows per tile num_splits * BM * GROUP (src/kernels.rs:1922-1944).
static int64_t prefill_split_rows(int32_t num_q_heads, int32_t q_len, int32_t block_m,
                                  int32_t group, int32_t num_splits) {
    if (num_q_heads <= 0 || q_len < 0 || block_m <= 0 || group <= 0 || num_splits <= 0 ||
        num_q_heads % group != 0)
        return GROUT_ERR_ARG;
    const int64_t tiles = (static_cast<int64_t>(q_len) + block_m - 1) / block_m * (num_q_heads / group);
    return tiles * num_splits * block_m * group;
}

}  // namespace grout

using namespace grout;

// Size checks shared by the prefill entry points: the ensure!s of
// attend_seq_arc_into_ctx_with_position (src/model.rs:5564-5637).
static int32_t check_prefill_sizes(int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim, int32_t q_len,
                                   int32_t kv_len, int32_t query_start, int32_t max_seq_len) {
    GROUT_REQUIRE(head_dim == kHeadDim, GROUT_ERR_HEAD_DIM);
    GROUT_REQUIRE(num_q_heads > 0 && num_kv_heads > 0 && num_q_heads % num_kv_heads == 0,
                  GROUT_ERR_HEADS);
    GROUT_REQUIRE(max_seq_len > 0, GROUT_ERR_SEQ_RANGE);
    GROUT_REQUIRE(q_len >= 0 && query_start >= 0, GROUT_ERR_KV_LEN);
    GROUT_REQUIRE(kv_len >= 1 && kv_len <= max_seq_len, GROUT_ERR_KV_LEN);
    return GROUT_OK;
}

// The key-split plan of a call on the current device.
static int32_t plan_on_device(const PrefillArgs& a, int num_kv_heads, Split32Plan* p) {
    int dev = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return static_cast<int32_t>(e);
    *p = split32_plan(a, num_kv_heads, cus);
    return GROUT_OK;
}

// Shared by the prefill entry points: the key split where a workspace is given
// and it pays, else the dynamic schedule (sched != nullptr) or the static grid.
static int32_t prefill_entry(const uint16_t* q, const uint16_t* k_cache, const uint16_t* v_cache,
                             uint16_t* out, float qk_scale, int32_t num_q_heads,
                             int32_t num_kv_heads, int32_t head_dim, int32_t q_len, int32_t kv_len,
                             int32_t query_start, int32_t max_seq_len, uint32_t* sched,
                             void* workspace, int64_t workspace_bytes, grout_stream_t stream) {
    GROUT_REQUIRE_PTR(q);
    GROUT_REQUIRE_PTR(k_cache);
    GROUT_REQUIRE_PTR(v_cache);
    GROUT_REQUIRE_PTR(out);
    const int32_t sizes = check_prefill_sizes(num_q_heads, num_kv_heads, head_dim, q_len, kv_len, query_start,
                                              max_seq_len);
    if (sizes != GROUT_OK) return sizes;
    GROUT_REQUIRE(qk_scale > 0.0f && qk_scale < 1.0e30f, GROUT_ERR_ARG);
    if (q_len == 0) return GROUT_OK;

    PrefillArgs a = {};
    a.q = q;
    a.k_cache = k_cache;
    a.v_cache = v_cache;
    a.out = out;
    // src/kernels.rs:1170-1174: qk_scale / ln(2) in f32.
    a.scale_log2 = qk_scale / logf(2.0f);
    a.num_q_heads = num_q_heads;
    a.group = num_q_heads / num_kv_heads;
    a.q_len = q_len;
    a.kv_len = kv_len;
    a.query_start = query_start;
    a.max_seq_len = max_seq_len;
    if (workspace != nullptr) {
        Split32Plan p;
        const int32_t st = plan_on_device(a, num_kv_heads, &p);
        if (st != GROUT_OK) return st;
        if (p.num_splits >= 2 && workspace_bytes >= split32_workspace_bytes(p, num_kv_heads))
            return launch_prefill_split32(a, p, num_kv_heads, workspace, to_hip(stream));
    }
    if (sched == nullptr) return launch_prefill(a, num_kv_heads, to_hip(stream));
    return launch_prefill_sched(a, num_kv_heads, sched, to_hip(stream));
}

extern "C" int32_t grout_attn_prefill(const uint16_t* q, const uint16_t* k_cache,
                                      const uint16_t* v_cache, uint16_t* out, float qk_scale,
                                      int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                      int32_t q_len, int32_t kv_len, int32_t query_start,
                                      int32_t max_seq_len, grout_stream_t stream) {
    return prefill_entry(q, k_cache, v_cache, out, qk_scale, num_q_heads, num_kv_heads, head_dim,
                         q_len, kv_len, query_start, max_seq_len, nullptr, nullptr, 0, stream);
}

extern "C" int32_t grout_attn_prefill_sched(const uint16_t* q, const uint16_t* k_cache,
                                            const uint16_t* v_cache, uint16_t* out,
                                            float qk_scale, int32_t num_q_heads,
                                            int32_t num_kv_heads, int32_t head_dim, int32_t q_len,
                                            int32_t kv_len, int32_t query_start,
                                            int32_t max_seq_len, uint32_t* sched_counters,
                                            grout_stream_t stream) {
    GROUT_REQUIRE(sched_counters != nullptr, GROUT_ERR_NULL_POINTER);
    GROUT_REQUIRE((reinterpret_cast<uintptr_t>(sched_counters) & 3u) == 0, GROUT_ERR_ALIGNMENT);
    return prefill_entry(q, k_cache, v_cache, out, qk_scale, num_q_heads, num_kv_heads, head_dim,
                         q_len, kv_len, query_start, max_seq_len, sched_counters, nullptr, 0, stream);
}

extern "C" int32_t grout_attn_prefill_ws(const uint16_t* q, const uint16_t* k_cache,
                                         const uint16_t* v_cache, uint16_t* out, float qk_scale,
                                         int32_t num_q_heads, int32_t num_kv_heads,
                                         int32_t head_dim, int32_t q_len, int32_t kv_len,
                                         int32_t query_start, int32_t max_seq_len,
                                         uint32_t* sched_counters, void* workspace,
                                         int64_t workspace_bytes, grout_stream_t stream) {
    GROUT_REQUIRE((reinterpret_cast<uintptr_t>(sched_counters) & 3u) == 0, GROUT_ERR_ALIGNMENT);
    GROUT_REQUIRE(aligned16(workspace), GROUT_ERR_ALIGNMENT);
    return prefill_entry(q, k_cache, v_cache, out, qk_scale, num_q_heads, num_kv_heads, head_dim,
                         q_len, kv_len, query_start, max_seq_len, sched_counters, workspace, workspace_bytes,
                         stream);
}

extern "C" int64_t grout_attn_prefill_workspace_bytes(int32_t num_q_heads, int32_t num_kv_heads,
                                                      int32_t head_dim, int32_t q_len,
                                                      int32_t kv_len, int32_t query_start,
                                                      int32_t max_seq_len) {
    const int32_t sizes = check_prefill_sizes(num_q_heads, num_kv_heads, head_dim, q_len, kv_len, query_start,
                                              max_seq_len);
    if (sizes != GROUT_OK) return sizes;
    if (q_len == 0) return 0;
    PrefillArgs a = {};
    a.num_q_heads = num_q_heads;
    a.group = num_q_heads / num_kv_heads;
    a.q_len = q_len;
    a.kv_len = kv_len;
    a.query_start = query_start;
    a.max_seq_len = max_seq_len;
    Split32Plan p;
    const int32_t st = plan_on_device(a, num_kv_heads, &p);
    // Without a device there is nothing to plan for: 0, as for a call that does not split.
    if (st != GROUT_OK) return 0;
    return split32_workspace_bytes(p, num_kv_heads);
}

extern "C" int64_t grout_attn_prefill_sched_counter_bytes(void) {
    return static_cast<int64_t>(kPfSchedCounters) * kPfSchedStride * 4;
}

extern "C" int32_t grout_attn_prefill_split(const uint16_t* q, const uint16_t* k_cache,
                                            const uint16_t* v_cache, uint16_t* att_partial,
                                            float* lse_partial, float qk_scale, int32_t num_q_heads,
                                            int32_t num_kv_heads, int32_t head_dim, int32_t q_len,
                                            int32_t kv_len, int32_t query_start,
                                            int32_t max_seq_len, int32_t block_m, int32_t block_n,
                                            int32_t group, int32_t num_splits,
                                            grout_stream_t stream) {
    // The prefill checks, plus the microbench's group check
    // (benchmarks/src/bin/attention_microbench.rs:411-421) and this
    // kernel's tile limits.
    GROUT_REQUIRE_PTR(q);
    GROUT_REQUIRE_PTR(k_cache);
    GROUT_REQUIRE_PTR(v_cache);
    GROUT_REQUIRE_PTR(att_partial);
    GROUT_REQUIRE_PTR(lse_partial);
    GROUT_REQUIRE(head_dim == kHeadDim, GROUT_ERR_HEAD_DIM);
    GROUT_REQUIRE(num_q_heads > 0 && num_kv_heads > 0 && num_q_heads % num_kv_heads == 0,
                  GROUT_ERR_HEADS);
    GROUT_REQUIRE(max_seq_len > 0, GROUT_ERR_SEQ_RANGE);
    GROUT_REQUIRE(q_len >= 0 && query_start >= 0, GROUT_ERR_KV_LEN);
    GROUT_REQUIRE(kv_len >= 1 && kv_len <= max_seq_len, GROUT_ERR_KV_LEN);
    GROUT_REQUIRE(qk_scale > 0.0f && qk_scale < 1.0e30f, GROUT_ERR_ARG);
    GROUT_REQUIRE(group >= 1 && (num_q_heads / num_kv_heads) % group == 0, GROUT_ERR_GROUP);
    GROUT_REQUIRE(block_m >= kPfRows && block_m % kPfRows == 0 && block_m <= 65536, GROUT_ERR_ARG);
    GROUT_REQUIRE(block_n >= 1 && block_n <= 65536, GROUT_ERR_SPLITS);
    GROUT_REQUIRE(num_splits >= 1 && num_splits <= GROUT_MAX_PREFILL_SPLITS, GROUT_ERR_SPLITS);
    if (q_len == 0) return GROUT_OK;

    PrefillArgs a = {};
    a.q = q;
    a.k_cache = k_cache;
    a.v_cache = v_cache;
    a.out = nullptr;
    a.scale_log2 = qk_scale / logf(2.0f);
    a.num_q_heads = num_q_heads;
    a.group = num_q_heads / num_kv_heads;
    a.q_len = q_len;
    a.kv_len = kv_len;
    a.query_start = query_start;
    a.max_seq_len = max_seq_len;
    a.att_partial = att_partial;
    a.lse_partial = lse_partial;
    a.block_m = block_m;
    a.block_n = block_n;
    a.split_group = group;
    a.num_splits = num_splits;
    return launch_prefill_split(a, num_kv_heads, to_hip(stream));
}

extern "C" int32_t grout_attn_prefill_split_merge(const uint16_t* att_partial,
                                                  const float* lse_partial, uint16_t* out,
                                                  int32_t num_q_heads, int32_t head_dim,
                                                  int32_t q_len, int32_t block_m, int32_t group,
                                                  int32_t num_splits, grout_stream_t stream) {
    GROUT_REQUIRE_PTR(att_partial);
    GROUT_REQUIRE_PTR(lse_partial);
    GROUT_REQUIRE_PTR(out);
    GROUT_REQUIRE(head_dim == kHeadDim, GROUT_ERR_HEAD_DIM);
    GROUT_REQUIRE(num_q_heads > 0, GROUT_ERR_HEADS);
    GROUT_REQUIRE(q_len >= 0, GROUT_ERR_KV_LEN);
    GROUT_REQUIRE(group >= 1 && num_q_heads % group == 0, GROUT_ERR_GROUP);
    GROUT_REQUIRE(block_m >= 1 && block_m <= 65536, GROUT_ERR_ARG);
    GROUT_REQUIRE(num_splits >= 1 && num_splits <= GROUT_MAX_PREFILL_SPLITS, GROUT_ERR_SPLITS);
    if (q_len == 0) return GROUT_OK;
    const int64_t threads = static_cast<int64_t>(q_len) * num_q_heads * (kHeadDim / 8);
    const int64_t blocks = (threads + 255) / 256;
    if (blocks > 0x7fffffff) return GROUT_ERR_KV_LEN;
    hipLaunchKernelGGL(attn_prefill_split_merge_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0,
                       to_hip(stream), att_partial, lse_partial, out, num_q_heads, q_len, block_m,
                       group, num_splits);
    return launch_status();
}

extern "C" int64_t grout_attn_prefill_split_partial_bytes(int32_t num_q_heads, int32_t head_dim,
                                                          int32_t q_len, int32_t block_m,
                                                          int32_t group, int32_t num_splits) {
    if (head_dim <= 0) return GROUT_ERR_ARG;
    const int64_t rows = prefill_split_rows(num_q_heads, q_len, block_m, group, num_splits);
    return rows < 0 ? rows : rows * head_dim * 2;
}

extern "C" int64_t grout_attn_prefill_split_lse_bytes(int32_t num_q_heads, int32_t q_len,
                                                      int32_t block_m, int32_t group,
                                                      int32_t num_splits) {
    const int64_t rows = prefill_split_rows(num_q_heads, q_len, block_m, group, num_splits);
    return rows < 0 ? rows : rows * 4;
}
