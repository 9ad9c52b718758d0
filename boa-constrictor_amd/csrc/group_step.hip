// Decode steps for few lanes: G workgroups (CUs) share each group of 16 lanes, where the fused kernels (fused_step.hip,
// fused_step512.hip) give one CU a whole group.
//
// What bounds the fused kernels at few lanes is one CU's share of the work, whatever the others do: every step streams
// all weights of the model through one CU (31.6 MB at d_model 256 x 8 layers, fp32) and multiplies them there.
//
// Here member m of a group owns d_inner / G channels (in_proj's x and z columns, conv, scan state, in whole 64-channel
// x_proj K blocks) and 1 / G of the output columns of every other GEMM, so each weight block is read by one member.
// What the next phase needs from the others goes through device memory, five times per layer: x_proj partials, y, the
// mixer output, the hidden layer, the residual stream.  Values travel in 8-byte packets (value, sequence number): a
// reader polls the packets themselves until each carries the sequence number it expects, so there is no separate flag,
// no fence and no ordering between packets to rely on, and an exchange costs one store-to-load latency.  The members of a
// group are placed on one XCD, which they verify (HW_REG_XCC_ID): the packets then stay in its L2.
//
// Loads return in order within a wave, so what a phase needs is requested one phase ahead of the wait in front of it: the
// weights of the next GEMM (held in registers), conv history, SSM state and parameters; and with few rows per thread the
// state is stored only after the next exchange has arrived.
//
// us per boa_model_step, fused kernel -> this one (G) and the fused launch behind it that leaves at once:
//   d 256 x 8, fp32:    1 lane 597 -> 190 (8), 64: 668 -> 227 (8), 512: 684 -> 249 (8), 1000: 703 -> 332 (4), 2048: 731 -> 528 (2)
//   d 256 x 8, bf16x3:  1: 429 -> 137 (8), 64: 493 -> 176 (8), 512: 497 -> 202 (8), 1000: 501 -> 276 (4), 2048: 526 -> 456 (2)
//   d 512 x 16, bf16w:  1: 2924 -> 353 (16), 256: 3713 -> 526 (16), 1000: 3813 -> 990 (4), 2048: 4074 -> 1838 (2)
//   d 512 x 16, bf16x3: 1: 3860 -> 411 (16), 256: 4633 -> 627 (16), 1000: 4590 -> 1548 (4), 2048: 5118 -> 3496 (2)
// What remains at 64 lanes (fp32, 8 launches of 125 steps, hardware counters): the matrix cores of the 32 CUs are busy 50
// of a step's 225 us, in chains of dependent MFMAs (256 per FF2 output), and the waves wait 48% of their cycles: for
// packets, at barriers, for their own loads.
// Registers: every form spills 70 to 113 scalar registers to vector lanes.  At d_model 512 with G = 2, where a member
// holds most, vector registers go to scratch memory too: bf16w 67, bf16x3 188.
//
// A packet is rewritten only by the same exchange of the next layer (or step), and its writer gets there only after
// every member has sent its packets of a later exchange of this layer, which it does after reading this one (a barrier
// between): no packet is overwritten before all have read it.  Sequence numbers grow from launch to launch, so what
// earlier launches left never matches; a packet holds their low 32 bits, and before those wrap the host zeroes all packets
// (launch_fused; 0 is never expected).
//
// All workgroups have to be resident at once (at most one per CU).  They meet at a gate first, before anything is read or
// written: the last to arrive opens it; the first to find its time up (another kernel holds the CUs) closes it for this
// launch, all of them leave, and the fused launch that follows does the work (left_out).  Beyond the gate every wait ends
// because its partners run.  (A cooperative launch gives the same guarantee but took 80 us longer per launch, of a step's
// 187.)  The waits are bounded all the same (wait_ticks): if one expires (the process was taken off the GPU for seconds),
// the workgroup stops waiting for good, goes through the rest of the launch on whatever it holds, and notes it in
// CTL_EXPIRED and, with the launch, for the host.  What the others make of its packets is as void as its own results: the
// launch that follows sees the note and sets all logits to NaN, as do all steps until the state is reset, and the host
// refuses the next call.  With more groups than CUs / 2 the fused kernels, one workgroup per group, fill the GPU and have
// no exchange.
//
// Arithmetic: every GEMM output accumulates its K steps in ascending order through mfma_split_step_t, x_proj is the left
// fold of 64-channel partials, and every elementwise step is the shared function of model_dev.h, as in the fused and
// compress kernels: same logits bit for bit.  The members fold, normalise and decode redundantly, from the same packets.
// Measured and not kept: one kernel-wide ring per GEMM under a wave-uniform branch (spills), packets of one XCD through
// group-scope loads (they may hit the L1 and then never see the packet), the packets received by the waves without
// fragments alone (the loads of a wave are issued at a fixed rate: 4% slower at 64 lanes).
#include "model_dev.h"
#include "model_internal.h"

#include <algorithm>
#include <type_traits>

namespace boa {

namespace {

constexpr int ROWS = 16, NTHR = 512, NWAVE = 8, NS = 16, VV = 256;
// Wait at the gate, in 10 ns, of a launch behind one that was shut out.  With room, the last of a launch's workgroups is
// there about 3 us after the first (up to 256 workgroups, 1200 launches: 5 us passed in 45, 10 us in none).  With the whole
// wait (0.5 ms and more) every step of a context beside other work paid it.
constexpr uint32_t SHUT_TICKS = 2000;
typedef uint64_t Packet;

typedef __attribute__((address_space(4))) const FusedArgs KArgs;
// kernel arguments through an opaque pointer (kept out of SGPRs across the step loop and the waits)
__device__ __forceinline__ KArgs& kargs() {
    auto kp = (__attribute__((address_space(4))) const char*)__builtin_amdgcn_kernarg_segment_ptr();
    __asm__ volatile("" : "+s"(kp));
    return *reinterpret_cast<KArgs*>(kp);
}

// exchange regions of one group, in packets
template <int D>
struct Xch {
    static constexpr int DI = 2 * D, HID = 4 * D, FW = D / 16 + 2 * NS, QB = DI / XPROJ_KB;
    static constexpr int P = 0;                     // x_proj partials [QB][ROWS][FW]
    static constexpr int Y = P + QB * ROWS * FW;    // y [ROWS][DI]
    static constexpr int M = Y + ROWS * DI;         // mixer output [ROWS][D]
    static constexpr int H = M + ROWS * D;          // hidden layer [ROWS][HID]
    static constexpr int X = H + ROWS * HID;        // residual stream [ROWS][D]
    static constexpr int T = X + ROWS * D;          // head's hidden layer [ROWS][D]
    static constexpr int LG = T + ROWS * D;         // logits [ROWS][VV]
    static constexpr int W = LG + ROWS * VV;        // where each member runs [16]
    static constexpr int SIZE = W + 16;
};

// Packets through a buffer descriptor over the group's regions, two adjacent ones per access where they are: each 8-byte
// packet is whole by itself.  near: every member runs on the same XCD, whose CUs share the L2: stores go through the L1 to
// it anyway, and a reader drops its L1 before each poll.  Otherwise both use the agent scope (SC1: past the L2 too).
constexpr int CPOL_GROUP = 1, CPOL_AGENT = 16;
typedef uint32_t bufv2 __attribute__((vector_size(8)));
struct Link {
    __amdgpu_buffer_rsrc_t x;
    bool near;
    volatile uint32_t* limit;  // of a wait, in ticks of the 100 MHz wall clock; 0: the workgroup waits no more
};
__device__ __forceinline__ void send(const Link& k, uint32_t at, uint32_t seq, uint32_t v) {
    if (k.near) __builtin_amdgcn_raw_buffer_store_b64(bufv2{v, seq}, k.x, at * 8, 0, CPOL_GROUP);
    else __builtin_amdgcn_raw_buffer_store_b64(bufv2{v, seq}, k.x, at * 8, 0, CPOL_AGENT);
}
__device__ __forceinline__ void send4(const Link& k, uint32_t at, uint32_t seq, uint32_t v0, uint32_t v1, uint32_t v2, uint32_t v3) {
    const bufv4 a = {v0, seq, v1, seq}, b = {v2, seq, v3, seq};
    if (k.near) {
        __builtin_amdgcn_raw_buffer_store_b128(a, k.x, at * 8, 0, CPOL_GROUP);
        __builtin_amdgcn_raw_buffer_store_b128(b, k.x, at * 8 + 16, 0, CPOL_GROUP);
    } else {
        __builtin_amdgcn_raw_buffer_store_b128(a, k.x, at * 8, 0, CPOL_AGENT);
        __builtin_amdgcn_raw_buffer_store_b128(b, k.x, at * 8 + 16, 0, CPOL_AGENT);
    }
}

// Waits for the N pairs of packets at (at[i], at[i] + 1), at even; v receives their values.
template <int N>
__device__ __forceinline__ void receive(const Link& k, const uint32_t (&at)[N], uint32_t seq, uint32_t (&v)[2 * N]) {
    uint64_t t0 = 0;
    for (;;) {
        u32x4 w[N];
#pragma unroll
        for (int i = 0; i < N; ++i) w[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(k.x, at[i] * 8, 0, CPOL_AGENT));
        pin_loads();  // read again on every pass
        uint32_t off = 0;  // no branch per packet
#pragma unroll
        for (int i = 0; i < N; ++i) {
            off |= (w[i].y ^ seq) | (w[i].w ^ seq);
            v[2 * i] = w[i].x;
            v[2 * i + 1] = w[i].z;
        }
        if (off == 0u) return;
        const uint32_t limit = *k.limit;
        if (limit == 0u) return;
        const uint64_t now = wall_clock64();
        if (t0 == 0) t0 = now;
        if (now - t0 >= limit) {
            KArgs& a = kargs();
            *k.limit = 0u;
            __hip_atomic_store(a.ctl + CTL_EXPIRED, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(a.host_expired, 2ull * a.seq0 + 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            return;
        }
    }
}

// GEMM operand in LDS, K columns: fp32 rows (NT 1) or split bf16 rows (the lo array behind the hi array)
template <int NT, int K> constexpr int op_bytes() { return NT == 1 ? ROWS * (K + 4) * 4 : 2 * ROWS * (K + 8) * 2; }
template <int NT, int K>
__device__ __forceinline__ void op_store4(unsigned char* op, int r, int k, float4 y) {
    if constexpr (NT == 1) {
        *reinterpret_cast<float4*>(reinterpret_cast<float*>(op) + r * (K + 4) + k) = y;
    } else {
        uint16_t* h = reinterpret_cast<uint16_t*>(op);
        uint2 hp, lp;
        split4(y.x, y.y, y.z, y.w, hp, lp);
        *reinterpret_cast<uint2*>(h + r * (K + 8) + k) = hp;
        *reinterpret_cast<uint2*>(h + ROWS * (K + 8) + r * (K + 8) + k) = lp;
    }
}
template <int NT, int K>
__device__ __forceinline__ void op_store1(unsigned char* op, int r, int k, float y) {
    if constexpr (NT == 1) {
        reinterpret_cast<float*>(op)[r * (K + 4) + k] = y;
    } else {
        uint16_t* h = reinterpret_cast<uint16_t*>(op);
        uint32_t hi, lo;
        split2(y, hi, lo);
        h[r * (K + 8) + k] = (uint16_t)hi;
        h[ROWS * (K + 8) + r * (K + 8) + k] = (uint16_t)lo;
    }
}
// an operand value as it travels: fp32 bits, or its split parts
template <int NT>
__device__ __forceinline__ uint32_t pack_value(float y) {
    if constexpr (NT == 1) return __float_as_uint(y);
    uint32_t hi, lo;
    split2(y, hi, lo);
    return hi | (lo << 16);
}
template <int NT, int K>
__device__ __forceinline__ void op_store_pair(unsigned char* op, int r, int k, uint32_t v0, uint32_t v1) {
    if constexpr (NT == 1) {
        *reinterpret_cast<uint2*>(reinterpret_cast<float*>(op) + r * (K + 4) + k) = make_uint2(v0, v1);
    } else {
        uint16_t* h = reinterpret_cast<uint16_t*>(op);
        *reinterpret_cast<uint32_t*>(h + r * (K + 8) + k) = (v0 & 0xFFFFu) | (v1 << 16);
        *reinterpret_cast<uint32_t*>(h + ROWS * (K + 8) + r * (K + 8) + k) = (v0 >> 16) | (v1 & 0xFFFF0000u);
    }
}
template <int NT, int K>
__device__ __forceinline__ void op_frag(const unsigned char* op, int row, int kg, int s, bf16x8& ah, bf16x8& al) {
    if constexpr (NT == 1) {
        const float* p = reinterpret_cast<const float*>(op) + row * (K + 4) + 32 * s + 4 * kg;
        ah = __builtin_bit_cast(bf16x8, *reinterpret_cast<const float4*>(p));
        al = __builtin_bit_cast(bf16x8, *reinterpret_cast<const float4*>(p + 16));
    } else {
        const uint16_t* p = reinterpret_cast<const uint16_t*>(op) + row * (K + 8) + 32 * s + 8 * kg;
        ah = *reinterpret_cast<const bf16x8*>(p);
        al = *reinterpret_cast<const bf16x8*>(p + ROWS * (K + 8));
    }
}
// N packets per row, all rows below nb, into the operand: pairs of columns, BP of them per thread in flight
template <int NT, int N>
__device__ __forceinline__ void receive_operand(const Link& k, uint32_t region, uint32_t seq, int nb,
                                                unsigned char* op, int tid) {
    constexpr int BP = 8;
    const int total = nb * (N / 2);
    for (int i0 = 0; i0 < total; i0 += NTHR * BP) {
        uint32_t at[BP], v[2 * BP];
#pragma unroll
        for (int u = 0; u < BP; ++u) {
            const int i = i0 + u * NTHR + tid;
            at[u] = region + 2 * (i < total ? i : total - 1);  // past the end: the last pair again
        }
        receive(k, at, seq, v);
#pragma unroll
        for (int u = 0; u < BP; ++u) {
            const int e = (int)(at[u] - region);
            op_store_pair<NT, N>(op, e / N, e % N, v[2 * u], v[2 * u + 1]);
        }
    }
}

// How the NF output fragments of one GEMM are shared among the waves: FPW fragments each, or, with fewer fragments than
// waves, one fragment for KS waves in turn, each with the next K / KS of its K steps.  (Such a fragment's products are one
// chain in any case; the waves' parts of its weights load at the same time.)
template <int NF> struct Share {
    static constexpr int KS = NF < NWAVE ? NWAVE / NF : 1, FPW = NF < NWAVE ? 1 : NF / NWAVE;
};
// A wave's part of one GEMM, its weight blocks in a ring of RD K steps (REGS registers' worth; the whole part where it
// fits): start() requests the first of them, long before the operand is there, run() multiplies.  Block (f, s) is 2 KB (hi
// and lo parts, or two fp32 groups) or 1 KB.
template <int NT, int K, int NF, int REGS>
struct Gemm {
    static constexpr int KS = Share<NF>::KS, FPW = Share<NF>::FPW, S = K / 32, SL = S / KS, BLKB = NT == 2 ? 1024 : 2048;
    static constexpr int FIT = REGS / (FPW * (NT == 2 ? 4 : 8)), RD = FIT >= SL ? SL : (FIT < 2 ? 2 : FIT);
    static constexpr int PRE = RD == SL ? SL : RD - 1;
    static_assert(SL * KS == S, "whole parts");
    u32x4 h[RD][FPW], l[RD][FPW];
    __amdgpu_buffer_rsrc_t w;
    uint32_t fo[FPW];
    __device__ __forceinline__ void issue(int s, int lane16) {
#pragma unroll
        for (int j = 0; j < FPW; ++j) {
            const uint32_t o = fo[j] + (uint32_t)s * BLKB;
            h[s % RD][j] = wbuf_ld16(w, lane16, o);
            l[s % RD][j] = h[s % RD][j];
            if constexpr (NT != 2) l[s % RD][j] = wbuf_ld16(w, lane16, o + 1024);
        }
    }
    // local fragment j of this wave (of the member's NF)
    static __device__ __forceinline__ int local(int wave, int j) { return KS > 1 ? wave % NF : wave + NWAVE * j; }
    static __device__ __forceinline__ int part(int wave) { return KS > 1 ? wave / NF : 0; }
    // frag(i): the matrix's fragment of the member's i-th
    template <class F> __device__ __forceinline__ void start(const uint16_t* Wp, int lane16, int wave, F&& frag) {
        w = wbuf(Wp);
#pragma unroll
        for (int j = 0; j < FPW; ++j)
            fo[j] = (uint32_t)__builtin_amdgcn_readfirstlane((frag(local(wave, j)) * S + part(wave) * SL) * BLKB);
#pragma unroll
        for (int i = 0; i < PRE; ++i) issue(i, lane16);
        pin_loads();
    }
    // acc[j]: columns 16 frag(j) + 4 (lane / 16) .. + 3 of row lane % 16
    __device__ __forceinline__ void multiply(const unsigned char* op, int wave, int lane, floatx4 (&acc)[FPW]) {
        const int row = lane & 15, kg = lane >> 4, lane16 = lane * 16;
        op += part(wave) * SL * 32 * (NT == 1 ? 4 : 2);
        bf16x8 ah, al;
        op_frag<NT, K>(op, row, kg, 0, ah, al);
        // unrolled over the whole part: at the end of a loop pass the compiler would wait for most of the ring
#pragma unroll
        for (int s = 0; s < SL; ++s) {
            if (RD < SL && s + RD - 1 < SL) issue(s + RD - 1, lane16);
            bf16x8 nh = ah, nl = al;
            if (s + 1 < SL) op_frag<NT, K>(op, row, kg, s + 1, nh, nl);
            // the reads stay a K step ahead of their MFMAs (one dependent chain per fragment: a read in front of its use
            // would stop it)
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < FPW; ++j)
                acc[j] = mfma_split_step_t<NT>(acc[j], ah, al, __builtin_bit_cast(bf16x8, h[s % RD][j]),
                                               __builtin_bit_cast(bf16x8, l[s % RD][j]));
            ah = nh;
            al = nl;
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // All waves call it.  Returns whether this wave holds the outputs (with KS > 1, the waves of the last part).  sAcc
    // [NF][64]: the sums on their way from wave to wave.
    __device__ __forceinline__ bool run(const unsigned char* op, int wave, int lane, floatx4 (&acc)[FPW], floatx4* sAcc) {
#pragma unroll
        for (int j = 0; j < FPW; ++j) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
        if constexpr (KS == 1) {
            multiply(op, wave, lane, acc);
            return true;
        } else {
#pragma unroll 1
            for (int p = 0; p < KS; ++p) {
                if (part(wave) == p) {
                    if (p > 0) acc[0] = sAcc[local(wave, 0) * 64 + lane];
                    multiply(op, wave, lane, acc);
                    if (p + 1 < KS) sAcc[local(wave, 0) * 64 + lane] = acc[0];
                }
                if (p + 1 < KS) __syncthreads();
            }
            return part(wave) == KS - 1;
        }
    }
};

// Lane-derived values from an opaque copy of the thread index, formed again in every phase: derived once, dozens of
// per-lane addresses of all phases would be held (and spilled) across the step and layer loops.
struct Ids {
    int tid, lane, lane16, row, cq;  // row, cq: this lane's row and first column of an output fragment
};
__device__ __forceinline__ Ids ids() {
    int t = (int)threadIdx.x;
    __asm__ volatile("" : "+v"(t));
    const int lane = t & 63;
    return {t, lane, lane * 16, lane & 15, 4 * (lane >> 4)};
}
#define IDS                                                                                             \
    const Ids id_ = ids();                                                                              \
    const int tid = id_.tid, lane = id_.lane, lane16 = id_.lane16, row = id_.row, cq = id_.cq;          \
    const bool live = row < nb;                                                                         \
    (void)tid; (void)lane; (void)lane16; (void)row; (void)cq; (void)live;
// the layer's parameter table entry from opaque copies of its index (its pointers are loaded again where they are used)
#define LAYER                                 \
    int l_ = l;                               \
    __asm__ volatile("" : "+s"(l_));          \
    CFusedLayer& w = layer_at(a.layers, l_);

template <int NT, int D, int G>
__global__ void __launch_bounds__(NTHR, 1) k_group_step(FusedArgs a0) {
    using XC = Xch<D>;
    constexpr int DI = XC::DI, HID = XC::HID, R = D / 16, FW = XC::FW, QB = XC::QB, LNV = D / 256;
    constexpr int CPG = DI / G, QPG = CPG / XPROJ_KB, XF = FW / 16;  // channels and x_proj K blocks per member
    constexpr int NFI = 2 * CPG / 16, FPI = NFI / NWAVE;              // in_proj fragments per member, per wave
    constexpr int NFO = D / 16 / G, FPO = Share<NFO>::FPW;  // out_proj, FF2, head1
    constexpr int NFF = HID / 16 / G, FPF = NFF / NWAVE;              // FF1
    constexpr int NFV = VV / 16 / G, FPV = Share<NFV>::FPW; // head2
    constexpr int XT = (QPG * XF + NWAVE - 1) / NWAVE;                // x_proj (block, fragment) pairs per wave
    constexpr int RSTEP = NTHR / CPG, RPT = ROWS / RSTEP;             // conv and scan: rows tid / CPG + RSTEP i
    static_assert(CPG % XPROJ_KB == 0 && FPI * NWAVE == NFI && FPF * NWAVE == NFF && RPT * RSTEP == ROWS, "shares");
    constexpr int LXZ = 2 * CPG + 4;
    // few rows per thread: the conv history and the SSM state are stored after the next exchange has arrived (a load that
    // follows a store in the queue is not seen before the store has been acknowledged)
    constexpr bool HOLD = RPT <= 4;
    // one LDS region: the operand of the GEMM at hand; during in_proj .. scan also xz and the conv output's operand
    constexpr int OFF_XZ = (op_bytes<NT, D>() + 15) / 16 * 16, OFF_CV = OFF_XZ + ROWS * LXZ * 4;
    constexpr int SZ1 = OFF_CV + op_bytes<NT, CPG>(), SZ2 = op_bytes<NT, HID>();
    constexpr int SZ = SZ1 > SZ2 ? SZ1 : SZ2;
    static_assert(SZ + ROWS * FW * 4 + NWAVE * 64 * 8 + 256 <= 160 * 1024 && op_bytes<NT, DI>() <= SZ, "LDS budget");
    __shared__ __attribute__((aligned(16))) unsigned char op[SZ];
    __shared__ __attribute__((aligned(16))) float sDbc[ROWS * FW];
    __shared__ floatx4 sAcc[NWAVE * 64 / 2];
    __shared__ int sTok[ROWS];
    __shared__ int sMaxLen, sGo;
    __shared__ uint32_t sLimit;
    float* sXZ = reinterpret_cast<float*>(op + OFF_XZ);
    unsigned char* sCv = op + OFF_CV;

    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    // the members of a group on one XCD (workgroup i runs on XCD i mod 8)
    const int bi = (int)blockIdx.x >> 3, member = bi % G, group = bi / G * 8 + ((int)blockIdx.x & 7);
    const int64_t b0 = (int64_t)group * ROWS;
    if (b0 >= a0.B) return;
    const int nb = (int)((a0.B - b0) < ROWS ? (a0.B - b0) : ROWS);
    volatile uint32_t* limit = &sLimit;
    // ---- the gate
    if (threadIdx.x == 0) {
        const uint64_t open = 2ull * a0.seq0, shut = open + 1ull;
        const uint64_t total = (uint64_t)((a0.B + ROWS - 1) / ROWS) * G;
        uint64_t* const gate = a0.ctl + CTL_GATE;
        auto state = [&]() { return __hip_atomic_load(gate, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
        // the first to decide for this launch: `was` holds an earlier launch's decision
        auto decide = [&](uint64_t was, uint64_t how) {
            if (was != open && was != shut)
                return __hip_atomic_compare_exchange_strong(gate, &was, how, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return false;
        };
        const uint64_t n = __hip_atomic_fetch_add(a0.ctl + CTL_ARRIVED, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        uint64_t st = state();
        if (n - a0.arrived == total - 1) decide(st, open);
        // if the launch before found no room, other work most likely still has the CUs: a short wait (SHUT_TICKS)
        const uint32_t ticks = (st & 1ull) != 0 && st != shut && a0.gate_ticks > SHUT_TICKS ? SHUT_TICKS : a0.gate_ticks;
        const uint64_t t0 = wall_clock64();
        while (st != open && st != shut) {
            st = state();
            if (wall_clock64() - t0 > ticks && decide(st, shut))
                __hip_atomic_fetch_add(a0.ctl + CTL_SHUT_OUT, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        sGo = st == open ? 1 : 0;
    }
    __syncthreads();
    if (!sGo) return;
    {
        const int tid = (int)threadIdx.x;
        if (tid < ROWS) sTok[tid] = tid < nb ? a0.tokens_in[b0 + tid] : 0;
        if (tid == 0) {
            int ml = 0;
            if (a0.decode)
                for (int r = 0; r < nb; ++r) ml = a0.lens[b0 + r] > ml ? a0.lens[b0 + r] : ml;
            sMaxLen = ml;
            sLimit = a0.wait_ticks;
        }
    }
    // coder state of this wave's rows 2 wave, 2 wave + 1 (every member keeps its own copy)
    DecState st[2];
    if (a0.decode) {
#pragma unroll
        for (int q = 0; q < 2; ++q)
            if (2 * wave + q < nb) st[q] = a0.dec[b0 + 2 * wave + q];
    }
    __syncthreads();
    // whether every member found itself on the same XCD (HW_REG_XCC_ID)
    bool near;
    {
        const Link far = {buf_rsrc(reinterpret_cast<Packet*>(a0.xch) + (int64_t)group * XC::SIZE, XC::SIZE * 8), false, limit};
        const uint32_t xcc = __builtin_amdgcn_s_getreg(20 | (3 << 11));
        if (threadIdx.x == 0) send(far, XC::W + member, a0.seq_first, xcc);
        uint32_t at[G / 2], v[G], differ = 0;
#pragma unroll
        for (int i = 0; i < G / 2; ++i) at[i] = XC::W + 2 * i;
        receive(far, at, (uint32_t)a0.seq0, v);
#pragma unroll
        for (int i = 0; i < G; ++i) differ |= v[i] ^ xcc;
        near = __builtin_amdgcn_readfirstlane(differ) == 0u;
    }
    // the matrix fragments of this member's: out_proj, FF2 and head1; in_proj (x, then z); FF1; head2
    auto o_frag = [&](int i) { return member * NFO + i; };
    auto in_frag = [&](int i) { return i < NFI / 2 ? member * (NFI / 2) + i : DI / 16 + member * (NFI / 2) + i - NFI / 2; };
    auto f_frag = [&](int i) { return member * NFF + i; };
    auto v_frag = [&](int i) { return member * NFV + i; };
    using GIn = Gemm<NT, D, NFI, 64>;
    using GOut = Gemm<NT, DI, NFO, 64>;
    using GF1 = Gemm<NT, D, NFF, 64>;
    using GF2 = Gemm<NT, HID, NFO, 64>;
    using GH1 = Gemm<NT, D, NFO, 64>;
    using GH2 = Gemm<NT, D, NFV, 64>;
    static_assert(GIn::FPW == FPI && GOut::FPW == FPO && GF1::FPW == FPF && GH2::FPW == FPV, "fragments per wave");
    auto own = [&](int j) { return o_frag(GOut::local(wave, j)); };

    int p0m3 = a0.p0m3;
#pragma unroll 1
    for (int step = 0; step < a0.nsteps; ++step) {
        KArgs& a = kargs();
        const int t = a.t + step;
        if (a.decode && t >= sMaxLen) break;  // every lane of the group is complete (the same for every member)
        const Link xc = {buf_rsrc(reinterpret_cast<Packet*>(a.xch) + (int64_t)group * XC::SIZE, XC::SIZE * 8), near, limit};
        const uint32_t seq0 = (uint32_t)a.seq0 + 1u + (uint32_t)step * (uint32_t)(a.L + 1);
        const int s1 = p0m3 == 2 ? 0 : p0m3 + 1, s2 = p0m3 == 0 ? 2 : p0m3 - 1;
        const int V = a.V;
        auto tok_of = [&](int r) {
            const int tk = sTok[r];
            return tk < 0 ? 0 : (tk >= V ? V - 1 : tk);
        };
        floatx4 xo[FPO];  // residual stream of this wave's FF2 outputs
        {
            IDS
#pragma unroll
            for (int j = 0; j < FPO; ++j) {
                const float4 e = ldg_f4(boa::G(a.emb) + (int64_t)tok_of(row) * D + 16 * own(j) + cq);
                xo[j] = floatx4{e.x, e.y, e.z, e.w};
            }
        }
        struct Ln {
            float4 w[LNV], b[LNV];
        };
        auto ln_load = [&](const float* lw, const float* lb, int lane) {
            Ln p;
#pragma unroll
            for (int i = 0; i < LNV; ++i) {
                p.w[i] = ldg_f4(boa::G(lw) + 256 * i + 4 * lane);
                p.b[i] = ldg_f4(boa::G(lb) + 256 * i + 4 * lane);
            }
            return p;
        };
        auto ln_store = [&](int r, const float (&v)[4 * LNV], const Ln& p, int lane) {
            float mu, rs;
            ln_stats_row<LNV>(v, mu, rs);
#pragma unroll
            for (int i = 0; i < LNV; ++i)
                op_store4<NT, D>(op, r, 256 * i + 4 * lane,
                                 make_float4(ln_apply(v[4 * i], mu, rs, p.w[i].x, p.b[i].x), ln_apply(v[4 * i + 1], mu, rs, p.w[i].y, p.b[i].y),
                                             ln_apply(v[4 * i + 2], mu, rs, p.w[i].z, p.b[i].z), ln_apply(v[4 * i + 3], mu, rs, p.w[i].w, p.b[i].w)));
        };
        // rows 2 wave, 2 wave + 1 (clamped to the last) of an exchanged fp32 [ROWS][W] array, in LayerNorm's lane layout
        auto receive_rows = [&](uint32_t region, auto width, uint32_t seq, float (&v)[2][4 * (decltype(width)::value / 256)], int lane) {
            constexpr int W = decltype(width)::value, NV = W / 256;
            uint32_t at[4 * NV], u[8 * NV];
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int i = 0; i < 2 * NV; ++i) {
                    const int r = 2 * wave + q < nb ? 2 * wave + q : nb - 1;
                    at[2 * NV * q + i] = region + r * W + 256 * (i / 2) + 4 * lane + 2 * (i & 1);
                }
            receive(xc, at, seq, u);
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int i = 0; i < 4 * NV; ++i) v[q][i] = __uint_as_float(u[4 * NV * q + i]);
        };
        using WD = std::integral_constant<int, D>;
        using WV = std::integral_constant<int, VV>;
        const bool rows_here = 2 * wave < nb;  // whether this wave has rows (uniform)

        GIn gin;  // requested a phase ahead, as every GEMM's weights: during the FF2 of the layer before
        {
            IDS
            gin.start(layer_at(a.layers, 0).in_p, lane16, wave, in_frag);
        }
#pragma unroll 1
        for (int l = 0; l < a.L; ++l) {
            const uint32_t seq = seq0 + (uint32_t)l;
            float4 bin[FPI], cw;
            float cb, h0[RPT], h1[RPT], h2[RPT];
            u32x4 xh[XT][2], xl[XT][2];
            {
                // ---- requests of this half of the layer, ahead of the wait for the residual stream
                IDS
                LAYER
                const Ln lnp = ln_load(w.ln1_w, w.ln1_b, lane);
#pragma unroll
                for (int j = 0; j < FPI; ++j) bin[j] = ldg_f4(boa::G(w.in_b) + 16 * in_frag(wave + NWAVE * j) + cq);
                const __amdgpu_buffer_rsrc_t xp = wbuf(w.x_p);
                constexpr int XS = DI / 32, BLKB = NT == 2 ? 1024 : 2048;
#pragma unroll
                for (int j = 0; j < XT; ++j) {
                    int i = wave + NWAVE * j;
                    i = i < QPG * XF ? i : QPG * XF - 1;
                    const int f = i % XF, q = member * QPG + i / XF;
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        const uint32_t o = (uint32_t)__builtin_amdgcn_readfirstlane((f * XS + 2 * q + s) * BLKB);
                        xh[j][s] = wbuf_ld16(xp, lane16, o);
                        xl[j][s] = xh[j][s];
                        if constexpr (NT != 2) xl[j][s] = wbuf_ld16(xp, lane16, o + 1024);
                    }
                }
                const int c = member * CPG + tid % CPG, r0 = tid / CPG;
                cw = ldg_f4(boa::G(w.conv_w) + 4 * c);
                cb = boa::G(w.conv_b)[c];
                const __amdgpu_buffer_rsrc_t hr3 = buf_rsrc(a.hist + ((int64_t)l * a.max_lanes + b0) * 3 * DI, (uint32_t)nb * 3 * DI * 4);
#pragma unroll
                for (int i = 0; i < RPT; ++i) {
                    const uint32_t o = (uint32_t)((r0 + RSTEP * i) * 3 * DI + c) * 4;
                    h0[i] = buf_ld1(hr3, o + p0m3 * DI * 4);
                    h1[i] = buf_ld1(hr3, o + s1 * DI * 4);
                    h2[i] = buf_ld1(hr3, o + s2 * DI * 4);
                }
                pin_loads();
                // ---- LN1 of the residual stream (layer 0: of the embedding rows)
                if (rows_here) {
                    float v[2][4 * LNV];
                    if (l == 0) {
#pragma unroll
                        for (int q = 0; q < 2; ++q)
#pragma unroll
                            for (int i = 0; i < LNV; ++i) {
                                const float4 e = ldg_f4(boa::G(a.emb) + (int64_t)tok_of(2 * wave + q) * D + 256 * i + 4 * lane);
                                v[q][4 * i] = e.x; v[q][4 * i + 1] = e.y; v[q][4 * i + 2] = e.z; v[q][4 * i + 3] = e.w;
                            }
                    } else {
                        receive_rows(XC::X, WD{}, seq - 1u, v, lane);
                    }
                    ln_store(2 * wave, v[0], lnp, lane);
                    ln_store(2 * wave + 1, v[1], lnp, lane);
                }
            }
            __syncthreads();
            // ---- in_proj of this member's channels
            {
                IDS
                floatx4 acc[FPI];
                gin.run(op, wave, lane, acc, sAcc);
#pragma unroll
                for (int j = 0; j < FPI; ++j)
                    *reinterpret_cast<float4*>(sXZ + row * LXZ + 16 * (wave + NWAVE * j) + cq) =
                        make_float4(epi_value<EPI_BIAS>(acc[j][0], bin[j].x), epi_value<EPI_BIAS>(acc[j][1], bin[j].y),
                                    epi_value<EPI_BIAS>(acc[j][2], bin[j].z), epi_value<EPI_BIAS>(acc[j][3], bin[j].w));
            }
            __syncthreads();
            // ---- conv + SiLU of this thread's (channel, row) pairs
            {
                IDS
                const int ch = tid % CPG, r0 = tid / CPG, c = member * CPG + ch;
                [[maybe_unused]] const __amdgpu_buffer_rsrc_t hr3 = buf_rsrc(a.hist + ((int64_t)l * a.max_lanes + b0) * 3 * DI, (uint32_t)nb * 3 * DI * 4);
#pragma unroll
                for (int i = 0; i < RPT; ++i) {
                    const int r = r0 + RSTEP * i;
                    const float x = sXZ[r * LXZ + ch];
                    const float y = conv_point(cw, cb, h0[i], h1[i], h2[i], x);
                    sXZ[r * LXZ + ch] = y;
                    op_store1<NT, CPG>(sCv, r, ch, y);
                    if constexpr (HOLD) h0[i] = x;
                    else buf_st1(hr3, (uint32_t)(r * 3 * DI + p0m3 * DI + c) * 4, x);
                }
            }
            __syncthreads();
            // ---- x_proj partials of this member's K blocks
            {
                IDS
#pragma unroll
                for (int j = 0; j < XT; ++j) {
                    const int i = wave + NWAVE * j;
                    if (i < QPG * XF) {
                        const int f = i % XF, ql = i / XF;
                        floatx4 part = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int s = 0; s < 2; ++s) {
                            bf16x8 ah, al;
                            op_frag<NT, CPG>(sCv, row, lane >> 4, 2 * ql + s, ah, al);
                            part = mfma_split_step_t<NT>(part, ah, al, __builtin_bit_cast(bf16x8, xh[j][s]),
                                                         __builtin_bit_cast(bf16x8, xl[j][s]));
                        }
                        if (live) {
                            const uint32_t at = XC::P + ((member * QPG + ql) * ROWS + row) * FW + 16 * f + cq;
                            send4(xc, at, seq, __float_as_uint(part[0]), __float_as_uint(part[1]),
                              __float_as_uint(part[2]), __float_as_uint(part[3]));
                        }
                    }
                }
            }
            constexpr int PF = RPT < 4 ? RPT : 4;  // rows of state in flight per thread
            f32x4 hs[PF][NS / 4];
            GOut gout;
            // ---- dt_proj + softplus + selective scan + D + gate; y to the others.  Requested ahead of the wait for the
            //      partials: the state of the first PF rows and the channel's parameters
            {
                IDS
                LAYER
                const int ch = tid % CPG, r0 = tid / CPG, c = member * CPG + ch;
                const __amdgpu_buffer_rsrc_t sr = buf_rsrc(a.ssm + ((int64_t)l * a.max_lanes + b0) * DI * NS, (uint32_t)nb * DI * NS * 4);
                auto h_off = [&](int r, int n) { return (uint32_t)((r * (NS / 4) + n) * DI + c) * 16; };
                float av[NS], wr[R];
#pragma unroll
                for (int n = 0; n < NS; n += 4) {
                    const float4 p = ldg_f4(boa::G(w.Aneg) + ((int64_t)(n / 4) * DI + c) * 4);
                    av[n] = p.x; av[n + 1] = p.y; av[n + 2] = p.z; av[n + 3] = p.w;
                }
#pragma unroll
                for (int r = 0; r < R; r += 4) {
                    const float4 q = ldg_f4(boa::G(w.dt_w) + (int64_t)c * R + r);
                    wr[r] = q.x; wr[r + 1] = q.y; wr[r + 2] = q.z; wr[r + 3] = q.w;
                }
                const float bdt = boa::G(w.dt_b)[c], Dc = boa::G(w.D)[c];
#pragma unroll
                for (int i = 0; i < PF; ++i)
#pragma unroll
                    for (int n = 0; n < NS / 4; ++n) hs[i][n] = buf_ld4(sr, h_off(r0 + RSTEP * i, n));
                pin_loads();
                // dbc = P_0 + P_1 + ..., two columns per thread
                static_assert(ROWS * FW / 2 <= NTHR, "one pair of columns per thread");
                {
                    const int total = nb * FW / 2, i = tid < total ? tid : total - 1;
                    uint32_t at[QB], v[2 * QB];
#pragma unroll
                    for (int q = 0; q < QB; ++q) at[q] = XC::P + q * ROWS * FW + 2 * i;
                    receive(xc, at, seq, v);
                    float d0 = __uint_as_float(v[0]), d1 = __uint_as_float(v[1]);
#pragma unroll
                    for (int q = 1; q < QB; ++q) {
                        d0 = d0 + __uint_as_float(v[2 * q]);
                        d1 = d1 + __uint_as_float(v[2 * q + 1]);
                    }
                    *reinterpret_cast<float2*>(&sDbc[2 * i]) = make_float2(d0, d1);
                }
                gout.start(w.out_p, lane16, wave, o_frag);
                __syncthreads();
#pragma unroll
                for (int i = 0; i < RPT; ++i) {
                    const int r = r0 + RSTEP * i;
                    float h[NS];
#pragma unroll
                    for (int n = 0; n < NS / 4; ++n) {
                        const f32x4 q = hs[i % PF][n];
                        h[4 * n] = q.x; h[4 * n + 1] = q.y; h[4 * n + 2] = q.z; h[4 * n + 3] = q.w;
                        if (i + PF < RPT) hs[i % PF][n] = buf_ld4(sr, h_off(r + RSTEP * PF, n));
                    }
                    const float y = scan_position<NS, R>(sDbc + r * FW, wr, bdt, av, Dc, sXZ[r * LXZ + ch], sXZ[r * LXZ + CPG + ch], h);
                    if (r < nb) send(xc, XC::Y + r * DI + c, seq, pack_value<NT>(y));
#pragma unroll
                    for (int n = 0; n < NS / 4; ++n) {
                        const f32x4 q = {h[4 * n], h[4 * n + 1], h[4 * n + 2], h[4 * n + 3]};
                        if constexpr (HOLD) hs[i][n] = q;
                        else buf_st4(sr, h_off(r, n), q);
                    }
                }
            }
            // the held stores of this layer
            auto store_held = [&]() {
                if constexpr (HOLD) {
                    IDS
                    const int r0 = tid / CPG, c = member * CPG + tid % CPG;
                    const __amdgpu_buffer_rsrc_t hr3 = buf_rsrc(a.hist + ((int64_t)l * a.max_lanes + b0) * 3 * DI, (uint32_t)nb * 3 * DI * 4);
                    const __amdgpu_buffer_rsrc_t sr = buf_rsrc(a.ssm + ((int64_t)l * a.max_lanes + b0) * DI * NS, (uint32_t)nb * DI * NS * 4);
#pragma unroll
                    for (int i = 0; i < RPT; ++i) {
                        const int r = r0 + RSTEP * i;
                        buf_st1(hr3, (uint32_t)(r * 3 * DI + p0m3 * DI + c) * 4, h0[i]);
#pragma unroll
                        for (int n = 0; n < NS / 4; ++n) buf_st4(sr, (uint32_t)((r * (NS / 4) + n) * DI + c) * 16, hs[i][n]);
                    }
                }
            };
            // ---- out_proj
            GF1 gff1;
            {
                IDS
                LAYER
                float4 bo[FPO];
#pragma unroll
                for (int j = 0; j < FPO; ++j) bo[j] = ldg_f4(boa::G(w.out_b) + 16 * own(j) + cq);
                __syncthreads();  // xz is read; the operand region is free
                receive_operand<NT, DI>(xc, XC::Y, seq, nb, op, tid);
                store_held();
                gff1.start(w.ff1_p, lane16, wave, f_frag);
                __syncthreads();
                floatx4 acc[FPO];
                if (gout.run(op, wave, lane, acc, sAcc) && live) {
#pragma unroll
                    for (int j = 0; j < FPO; ++j)
                        send4(xc, XC::M + row * D + 16 * own(j) + cq, seq, __float_as_uint(epi_value<EPI_BIAS>(acc[j][0], bo[j].x)),
                              __float_as_uint(epi_value<EPI_BIAS>(acc[j][1], bo[j].y)), __float_as_uint(epi_value<EPI_BIAS>(acc[j][2], bo[j].z)),
                              __float_as_uint(epi_value<EPI_BIAS>(acc[j][3], bo[j].w)));
                }
            }
            // ---- LN2, FF1 + GELU; hidden units to the others
            GF2 gff2;
            {
                IDS
                LAYER
                const Ln lnp = ln_load(w.ln2_w, w.ln2_b, lane);
                float4 bf[FPF];
#pragma unroll
                for (int j = 0; j < FPF; ++j) bf[j] = ldg_f4(boa::G(w.ff1_b) + 16 * f_frag(wave + NWAVE * j) + cq);
                pin_loads();
                __syncthreads();  // y is read
                float v[2][4 * LNV] = {};
                if (rows_here) receive_rows(XC::M, WD{}, seq, v, lane);
                gff2.start(w.ff2_p, lane16, wave, o_frag);
                if (rows_here) {
                    ln_store(2 * wave, v[0], lnp, lane);
                    ln_store(2 * wave + 1, v[1], lnp, lane);
                }
                __syncthreads();
                floatx4 acc[FPF];
                gff1.run(op, wave, lane, acc, sAcc);
                if (live) {
#pragma unroll
                    for (int j = 0; j < FPF; ++j)
                        send4(xc, XC::H + row * HID + 16 * f_frag(wave + NWAVE * j) + cq, seq,
                              pack_value<NT>(epi_value<EPI_GELU>(acc[j][0], bf[j].x)), pack_value<NT>(epi_value<EPI_GELU>(acc[j][1], bf[j].y)),
                              pack_value<NT>(epi_value<EPI_GELU>(acc[j][2], bf[j].z)), pack_value<NT>(epi_value<EPI_GELU>(acc[j][3], bf[j].w)));
                }
            }
            // ---- FF2 + block residual
            {
                IDS
                LAYER
                float4 bo[FPO];
#pragma unroll
                for (int j = 0; j < FPO; ++j) bo[j] = ldg_f4(boa::G(w.ff2_b) + 16 * own(j) + cq);
                __syncthreads();  // the LN2 operand is read
                receive_operand<NT, HID>(xc, XC::H, seq, nb, op, tid);
                gin.start(layer_at(a.layers, l + 1 < a.L ? l + 1 : l).in_p, lane16, wave, in_frag);  // (the last: unused)
                __syncthreads();
                floatx4 acc[FPO];
                if (gff2.run(op, wave, lane, acc, sAcc)) {
#pragma unroll
                    for (int j = 0; j < FPO; ++j) {
                        const float bv[4] = {bo[j].x, bo[j].y, bo[j].z, bo[j].w};
#pragma unroll
                        for (int e = 0; e < 4; ++e) xo[j][e] = xo[j][e] + epi_value<EPI_RESID>(acc[j][e], bv[e]);
                        if (live)
                            send4(xc, XC::X + row * D + 16 * own(j) + cq, seq, __float_as_uint(xo[j][0]), __float_as_uint(xo[j][1]),
                                  __float_as_uint(xo[j][2]), __float_as_uint(xo[j][3]));
                    }
                }
            }
            __syncthreads();  // the hidden layer is read: the next LN1 rewrites the operand
        }

        // ---- head: Linear -> ReLU -> Linear
        const uint32_t seqh = seq0 + (uint32_t)a.L;
        GH2 g2;
        {
            IDS
            GH1 g1;
            g1.start(a.h1_p, lane16, wave, o_frag);
            float4 bo[FPO];
#pragma unroll
            for (int j = 0; j < FPO; ++j) bo[j] = ldg_f4(boa::G(a.h1_b) + 16 * own(j) + cq);
            float v[2][4 * LNV] = {};
            if (rows_here) receive_rows(XC::X, WD{}, seqh - 1u, v, lane);
            g2.start(a.h2_p, lane16, wave, v_frag);
            if (rows_here) {
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int i = 0; i < LNV; ++i)
                        op_store4<NT, D>(op, 2 * wave + q, 256 * i + 4 * lane, make_float4(v[q][4 * i], v[q][4 * i + 1], v[q][4 * i + 2], v[q][4 * i + 3]));
            }
            __syncthreads();
            floatx4 acc[FPO];
            if (g1.run(op, wave, lane, acc, sAcc) && live) {
#pragma unroll
                for (int j = 0; j < FPO; ++j)
                    send4(xc, XC::T + row * D + 16 * own(j) + cq, seqh, pack_value<NT>(epi_value<EPI_RELU>(acc[j][0], bo[j].x)),
                          pack_value<NT>(epi_value<EPI_RELU>(acc[j][1], bo[j].y)), pack_value<NT>(epi_value<EPI_RELU>(acc[j][2], bo[j].z)),
                          pack_value<NT>(epi_value<EPI_RELU>(acc[j][3], bo[j].w)));
            }
        }
        {
            IDS
            float4 bo[FPV];
#pragma unroll
            for (int j = 0; j < FPV; ++j) bo[j] = ldg_f4(boa::G(a.h2_b) + 16 * v_frag(GH2::local(wave, j)) + cq);
            __syncthreads();
            receive_operand<NT, D>(xc, XC::T, seqh, nb, op, tid);
            __syncthreads();
            floatx4 acc[FPV];
            if (g2.run(op, wave, lane, acc, sAcc) && live) {
#pragma unroll
                for (int j = 0; j < FPV; ++j)
                    send4(xc, XC::LG + row * VV + 16 * v_frag(GH2::local(wave, j)) + cq, seqh,
                          __float_as_uint(epi_value<EPI_BIAS>(acc[j][0], bo[j].x)), __float_as_uint(epi_value<EPI_BIAS>(acc[j][1], bo[j].y)),
                          __float_as_uint(epi_value<EPI_BIAS>(acc[j][2], bo[j].z)), __float_as_uint(epi_value<EPI_BIAS>(acc[j][3], bo[j].w)));
            }
        }
        // ---- logits of rows 2 wave, 2 wave + 1 (4 consecutive per lane); decode
        if (rows_here) {
            IDS
            float v[2][4];
            receive_rows(XC::LG, WV{}, seqh, v, lane);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int r = 2 * wave + q;
                if (r >= nb) continue;
                const float4 l4 = make_float4(v[q][0], v[q][1], v[q][2], v[q][3]);
                if (a.logits && member == r % G) stg_f4(boa::GM(a.logits) + (b0 + r) * VV + 4 * lane, l4);
                if (a.decode && t < a.lens[b0 + r]) {
                    const LaneWords words = lane_words(a.payload, a.payload_words, a.off, a.nwords, b0 + r);
                    const int s = decode_l4(l4, VV, lane, st[q], words.p, words.n);
                    if (lane == 0) {
                        sTok[r] = s;
                        if (member == 0) a.out[(b0 + r) * a.out_stride + t] = (uint8_t)s;
                    }
                }
            }
        }
        __syncthreads();
        p0m3 = p0m3 == 2 ? 0 : p0m3 + 1;
    }
    if (a0.decode && member == 0) {
        const int tid = (int)threadIdx.x;
        if (tid < nb) a0.tokens_out[b0 + tid] = sTok[tid];
#pragma unroll
        for (int q = 0; q < 2; ++q)
            if (2 * wave + q < nb && (tid & 63) == 0) a0.dec[b0 + 2 * wave + q] = st[q];
    }
}

template <int NT, int D, int G>
hipError_t launch(const FusedArgs& a, hipStream_t s) {
    hipLaunchKernelGGL((k_group_step<NT, D, G>), dim3((unsigned)((a.B + 8 * ROWS - 1) / (8 * ROWS) * 8 * G)), dim3(NTHR), 0, s, a);
    return hipGetLastError();
}
template <int NT, int D>
hipError_t launch_g(const FusedArgs& a, int g, hipStream_t s) {
    if constexpr (D == 512) {
        if (g == 16) return launch<NT, D, 16>(a, s);
    }
    if (g == 8) return launch<NT, D, 8>(a, s);
    if (g == 4) return launch<NT, D, 4>(a, s);
    return launch<NT, D, 2>(a, s);
}

}  // namespace

int64_t group_step_bytes(int d_model, int64_t max_lanes) {
    const int64_t groups = std::min<int64_t>((max_lanes + ROWS - 1) / ROWS, GROUP_MAX);
    return groups * 8 * (d_model == 512 ? Xch<512>::SIZE : Xch<256>::SIZE);
}

int group_step_width(int d_model, int lanes, int cus) {
    const int groups = (lanes + ROWS - 1) / ROWS;
    if (groups > GROUP_MAX) return 1;
    for (int g = d_model == 512 ? 16 : 8; g > 1; g /= 2)
        if ((groups + 7) / 8 * 8 * g <= cus) return g;
    return 1;
}

int64_t group_step_blocks(int lanes, int g) { return (int64_t)((lanes + ROWS - 1) / ROWS) * g; }

hipError_t launch_group_step(const FusedArgs& a, int d_model, int nt, int g, hipStream_t s) {
    if (d_model == 512) return nt == 3 ? launch_g<3, 512>(a, g, s) : launch_g<2, 512>(a, g, s);
    if (nt == 3) return launch_g<3, 256>(a, g, s);
    if (nt == 2) return launch_g<2, 256>(a, g, s);
    return launch_g<1, 256>(a, g, s);
}

}  // namespace boa
