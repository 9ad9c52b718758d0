// Host/device interface between the model context (model.hip) and the fused decompress-step kernels
// (fused_step.hip for d_model 256, fused_step512.hip for d_model 512).  Internal to libboa_hip.so.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "boa_common.h"

namespace boa {

// Fragment-packed bfloat16 GEMM weights for MFMA 16x16x32 B operands: matrix W [N][K] (N % 16 == 0,
// K % 32 == 0) as blocks (f, s) for f < N/16, s < K/32, in order f-major; a block is 64 lanes x 8 values,
// lane l holding W[16f + (l % 16)][32s + 8(l / 16) + j], j < 8: the hi part, then (bf16x3) the lo part.
// One wavefront reads a block with one fully coalesced 16-byte load per lane.
struct FusedLayer {
    const float *ln1_w, *ln1_b, *in_b, *conv_w, *conv_b, *dt_w, *dt_b, *Aneg, *D, *out_b, *ln2_w, *ln2_b, *ff1_b,
        *ff2_b;
    const uint16_t *in_p, *x_p, *out_p, *ff1_p, *ff2_p;
};

// The layer table as the d_model 256 fused kernel reads it: constant memory (the table does not change while the
// kernel runs), so its pointers come through scalar loads, which wait on the scalar counter alone.  Read as global
// memory, each pointer is a vector load, and the wait for it is also a wait for every vector load and store
// issued before it (the counter is in order): at a phase boundary, the previous phase's state stores.  (The
// d_model 512 kernel, short of scalar registers, measured 4.5% slower with it and reads the table as global
// memory.)
typedef __attribute__((address_space(4))) const FusedLayer CFusedLayer;
__device__ __forceinline__ CFusedLayer& layer_at(const FusedLayer* table, int l) {
    return ((CFusedLayer*)table)[l];
}

struct FusedArgs {
    const FusedLayer* layers;  // device array [L]
    int L;
    int V;
    int B;                     // lanes in this launch
    int p0m3;                  // absolute position of this step, mod 3 (conv history ring slot)
    int64_t max_lanes;         // lane capacity of the state arrays
    const float *emb, *h1_b, *h2_b;
    const uint16_t *h1_p, *h2_p;
    float* ssm;                // [L][max_lanes][NS/4][di][4]
    float* hist;               // [L][max_lanes][3][di]
    const int32_t* tokens_in;  // [B] model input bytes
    float* logits;             // [B][V] output, or null
    // decode steps (decode != 0): positions t .. t + nsteps - 1, each step's symbol fed back as the next
    // step's input; the last one is left in tokens_out.  Without decode, nsteps must be 1.
    int decode;
    int t;
    int nsteps;
    int stagger_us;            // start offset between workgroup classes (multi-step launches), microseconds
    int stagger_classes;       // number of classes (1, 2, 4 or 8 sets of XCDs)
    const int32_t* lens;
    DecState* dec;
    const uint32_t* payload;
    int64_t payload_words;     // the payload's length: every lane's stream is clamped to it
    const int64_t* off;
    const int32_t* nwords;
    int32_t* tokens_out;
    uint8_t* out;
    int64_t out_stride;
    // d_model 512 kernel only: per-lane scratch in device memory (the context's workspace rows, row = lane): the
    // mixer's z | conv output [lanes][2 d_inner]
    float* scr;
    // group_step.hip: the exchange packets, the first sequence number of this launch (a packet carries its low 32 bits,
    // which a launch does not let wrap), its control words (below; arrivals before this launch: `arrived`, or GATE_NEVER),
    // how long its workgroups wait at the gate and for a packet, in 10 ns, and where an expired wait is reported to the
    // host
    uint64_t* xch;
    uint64_t seq0;
    uint32_t seq_first;        // what the first exchange's packets carry: seq0 (another number: that wait expires)
    uint64_t* ctl;
    uint64_t arrived;
    uint32_t gate_ticks;
    uint32_t wait_ticks;
    uint64_t* host_expired;
    // fused kernels: run only if the group launch with this decision word (2 seq0 + 1) did not start (0: always run)
    uint64_t only_if;
};
// Control words of a context's group launches: the last decision at the gate (2 seq0: open, 2 seq0 + 1: not all here),
// whether a wait expired since the state was reset (0: none did), arrivals at the gate, launches that were shut out.
enum { CTL_GATE, CTL_EXPIRED, CTL_ARRIVED, CTL_SHUT_OUT, CTL_WORDS };
constexpr uint64_t GATE_NEVER = 1ull << 63;  // `arrived` of a launch whose gate no count of arrivals opens

// Logits of a step that cannot be formed: NaN for every lane (all threads of the grid).
__device__ __forceinline__ void void_logits(float* logits, int64_t n) {
    const float nan = __builtin_nanf("");
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) logits[i] = nan;
}
// Whether a fused launch is left out: it follows a group launch that did run, or a wait between workgroups expired in it
// or in an earlier launch since the state was reset (ctl is null in contexts without group launches).
__device__ __forceinline__ bool left_out(const FusedArgs& a) {
    if (a.ctl == nullptr) return false;
    typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));
    const u64x2 ctl = *reinterpret_cast<const u64x2*>(a.ctl);  // both words in one access
    if (ctl[CTL_EXPIRED] != 0) {
        if (a.logits) void_logits(a.logits, (int64_t)a.B * a.V);
        return true;
    }
    return a.only_if != 0 && ctl[CTL_GATE] != a.only_if;
}

// Launches over several tiles at once (a tile: all lanes of a group at Tc consecutive positions, at one layer).
constexpr int PIPE_MAX = 16;  // tiles per launch at most

// out_proj + LN2 + feed-forward + residual of one tile's M rows.
struct FfnTile {
    const float *out_b, *ln_w, *ln_b, *ff1_b, *ff2_b;
    const uint16_t *out_p, *ff1_p, *ff2_p;
    float* x;
    const float* mm;          // out_proj's output where it ran on its own (k_ffn and k_ffn512 without OUTP)
    const uint16_t *yh, *yl;  // the scan's output: split parts, or fp32 at yh (fp32 mode)
    float* hid;               // [M][4 d], for k_ffn16 in two launches
    int64_t M;
};
struct FfnTiles {
    FfnTile t[PIPE_MAX];
};
__device__ __forceinline__ const FfnTile& ffn_tile(const FfnTile& a) { return a; }
__device__ __forceinline__ const FfnTile& ffn_tile(const FfnTiles& a) { return a.t[blockIdx.y]; }
// d_model 256, 16 rows per workgroup (fused_step.hip): for launches whose tiles are too few for k_ffn's 64-row workgroups
// split: workgroups per 16 rows (1, 4, in the fp32 mode also 2).
hipError_t launch_ffn16(const FfnTiles& a, int tiles, int64_t max_rows, int split, int nt, hipStream_t s);

// Head (Linear -> ReLU -> Linear) of M rows of x, 16 per workgroup (d_model 256): row m is position t0 + m % Tc of lane
// m / Tc.  Either the coder interval of the byte the position predicts (lf[m]), or the logits (logits[(lane * len + t0 +
// m % Tc) * V]).
struct HeadRows {
    const float *x, *h1_b, *h2_b;
    const uint16_t *h1_p, *h2_p;
    int64_t M;
    int V, t0, Tc;
    const uint8_t* bytes;
    int64_t stride;
    const int32_t* lens;
    uint2* lf;
    float* logits;
    int64_t len;
};
hipError_t launch_head16(const HeadRows& a, int nt, hipStream_t s);

// Supported shape of the fused kernel: d_model 256, d_state 16, dt_rank 16, d_conv 4, vocab % 16 == 0.
bool fused_step_supported(int d_model, int d_state, int dt_rank, int d_conv, int vocab);

// nt = 3 (bf16x3 weights, hi + lo) or 2 (bf16 weights); 512 threads per workgroup of 16 lanes
hipError_t launch_fused_step(const FusedArgs& a, int nt, hipStream_t s);

// The d_model 512 form (d_inner 1024, d_state 16, dt_rank 32, d_conv 4, vocab 256): 512 threads (8 waves) per
// workgroup of 32 lanes, one workgroup per CU (256 VGPRs per thread, 145 KB of LDS with the residual stream).
bool fused_step512_supported(int d_model, int d_state, int dt_rank, int d_conv, int vocab);
hipError_t launch_fused_step512(const FusedArgs& a, int nt, hipStream_t s);

// Decode steps with several workgroups per 16 lanes (group_step.hip): vocab 256, otherwise the fused kernels' shapes.
constexpr int GROUP_MAX = 128;  // groups of 16 lanes at most
int64_t group_step_bytes(int d_model, int64_t max_lanes);     // exchange packets, in bytes
int group_step_width(int d_model, int lanes, int cus);         // workgroups per group on a GPU of that many CUs; 1: none
// takes group_step_seqs sequence numbers from a.seq0 on; adds group_step_blocks to the gate's arrivals.  Does nothing
// (and says so at the gate) if its workgroups do not all get onto the GPU in time: a fused launch with only_if follows.
int64_t group_step_blocks(int lanes, int g);
inline uint32_t group_step_seqs(int nsteps, int L) { return 1u + (uint32_t)nsteps * (uint32_t)(L + 1); }
hipError_t launch_group_step(const FusedArgs& a, int d_model, int nt, int g, hipStream_t s);

}  // namespace boa
