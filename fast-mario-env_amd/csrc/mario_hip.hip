// mario_hip: batched Super Mario Bros env stepping on gfx950 — kernels and the C-ABI (include/mario_hip.h).
//
// One agent step of N envs is three kernels on the caller's stream:
//   k_step          a wave per env: sticky draw, K frames of 6502 + catch-up PPU, reward/done/info, hack
//                   frames, gray rendering of the max-pool pair into two frame buffers; then the 2-frame max +
//                   INTER_AREA of its last frames (obs_tail)
//   k_reset         one lane per env: finished envs take a cached (level, no-op count) start state
//   k_stack         frame-stack shift, final_obs, reset observation
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <tuple>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/mario_hip.h"
#include "lane_kernels.hpp"
#include "replay.hpp"

using namespace mh;

namespace {

// Stage PRG and the CHR banks (32 KB + 8 KB each) and the gray LUT in LDS; every thread of
// the block must call this.
__device__ __forceinline__ void stage_rom(const RomArgs& R, uint8_t* s_rom, uint8_t* s_lut) {
    const uint4* src = (const uint4*)R.rom;
    uint4* dst = (uint4*)s_rom;
    const int words = (0x8000 + R.n_chr * 0x2000) / 16;
    for (int i = threadIdx.x; i < words; i += blockDim.x) dst[i] = src[i];
    for (int i = threadIdx.x; i < 256; i += blockDim.x) s_lut[i] = R.lut[i];
    __syncthreads();
}

// Block-shared LDS of the emulator kernels: the cartridge, the gray LUT and each console's share.
#define ROM_LDS                                                     \
    __shared__ __attribute__((aligned(16))) uint8_t s_rom[0x8000 + MAX_CHR_BANKS * 0x2000]; \
    __shared__ uint8_t s_lut[256];                                  \
    __shared__ __attribute__((aligned(16))) uint32_t s_env[LDS_ENV_WORDS * LDS_LANES];
static_assert(0x8000 + MAX_CHR_BANKS * 0x2000 + 256 + 4 * LDS_ENV_WORDS * LDS_LANES <= 160 * 1024, "a CU's LDS");
static_assert(LDS_ENV_WORDS % 4 == 0, "a console's memory stays 16-byte aligned");

// Console slot of this wave in its block: wave-uniform, in a scalar register
__device__ __forceinline__ uint32_t wave_slot() { return uni(threadIdx.x >> 6); }
__device__ __forceinline__ LaneCtx lane_ctx(const RomArgs& R, const uint8_t* s_rom, const uint8_t* s_lut, uint32_t* s_env) {
    MH_LDS uint32_t* const own = (MH_LDS uint32_t*)s_env + wave_slot() * LDS_ENV_WORDS;
    return LaneCtx{make_cart(R, (const MH_LDS uint8_t*)s_rom, kDecode.w), (const MH_LDS uint8_t*)s_lut, own,
                   own + LDS_SP_WORDS, (uint8_t)(threadIdx.x & 63u)};
}

constexpr int EMU_THREADS = 64 * WAVES_PER_BLOCK;
#define EMU_BOUNDS __launch_bounds__(EMU_THREADS, EMU_WAVES_PER_SIMD)
// Launch shape of an emulator kernel over `count` consoles, a wave each, on a GPU with `cus` compute units: blocks of up
// to WAVES_PER_BLOCK waves (one block per CU: its LDS). When count is too small to give every CU a full block, the
// blocks shrink (down to one wave) so that the waves spread over all CUs instead of sharing a few CUs' SIMDs.
struct EmuLaunch { dim3 grid, block; };
static inline EmuLaunch emu_launch(int count, int cus) {
    if (cus < 1) cus = 1;
    int wpb = (count + cus - 1) / cus;
    wpb = wpb < 1 ? 1 : wpb > WAVES_PER_BLOCK ? WAVES_PER_BLOCK : wpb;
    return EmuLaunch{dim3((unsigned)((count + wpb - 1) / wpb)), dim3((unsigned)(64 * wpb))};
}
// this wave's console (the block's waves in order)
__device__ __forceinline__ uint32_t wave_console(uint32_t block) { return block * (blockDim.x >> 6) + wave_slot(); }

// The new observation of the wave's env into fresh[e * OBS_PIX + o]: the boot observation right after a reset, else
// INTER_AREA of the last frame, max-pooled with its partner frame (fastmario.cpp:377-386); `bits` as step_lane
// returns them. k_step runs it once the wave's frame loop is over, on the frames the wave has just drawn. 48 lanes
// take the 4 column periods of the tables (AreaPeriod: output columns 21 g .. 21 g + 20) times the 12 row periods (7
// output rows from 20 source rows each), so every lane runs the same code with constant taps and weights. A lane's 64
// pixels of a source row are 64 contiguous bytes: four 16-byte loads per frame. The float operations and their order
// are area_pixel's. Not inlined, so that its registers stay out of the frame loop's allocation.
typedef __attribute__((address_space(1))) uint8_t gbyte;       // global memory, addressed as such
__device__ __attribute__((noinline)) void obs_tail(const uint8_t* gray_, uint32_t np_, uint8_t* fresh_,
                                                   const uint8_t* boot_obs, uint32_t e, uint32_t lane, uint32_t bits_) {
    // The frames were stored by the lanes of this wave (streaming stores): wait for the stores, and drop the L1's
    // lines, before reading them.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    // the arguments a call passes in vector registers: the same in every lane but `lane`
    const gbyte* gray = (const gbyte*)uni64((uint64_t)gray_);
    gbyte* fresh = (gbyte*)uni64((uint64_t)fresh_) + (size_t)uni(e) * OBS_PIX;
    const uint32_t np = uni(np_), bits = uni(bits_);
    if (bits & 4) {
        const uint32_t* b = (const uint32_t*)(boot_obs + (size_t)(bits >> 8) * OBS_PIX);
        for (uint32_t i = lane; i < OBS_PIX / 4; i += 64) ((__attribute__((address_space(1))) uint32_t*)fresh)[i] = b[i];
        return;
    }
    if (lane >= 48) return;
    const uint32_t g = lane & 3u, p = lane >> 2;
    gbyte* out = fresh + 21 * g + 7 * 84 * p;                                  // row 0 of the lane's period
    const gbyte* f0 = gray + (size_t)uni(e) * GRAY_PIX;
    const gbyte* f1 = f0 + (size_t)GRAY_PIX * np;
    if (!(bits & 1)) { f0 = (bits & 2) ? f1 : f0; f1 = f0; }                   // one frame: its maximum with itself
    const uint32_t at = 20 * 256 * p + 64 * g;                                 // the lane's pixels of its first row
    float acc[21];
#pragma unroll
    for (int q = 0; q < 21; q++) acc[q] = 0.f;                                 // +0 at the period's start
#pragma nounroll
    for (int r = 0; r < 20; r++) {
        uint32_t ev[16], od[16];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // streaming loads: the frames are read once
            const mh_u32x4 a = __builtin_nontemporal_load((const __attribute__((address_space(1))) mh_u32x4*)(f0 + at + 256 * r) + i);
            const mh_u32x4 b = __builtin_nontemporal_load((const __attribute__((address_space(1))) mh_u32x4*)(f1 + at + 256 * r) + i);
#pragma unroll
            for (int k = 0; k < 4; k++) { ev[4 * i + k] = max_even_bytes(a[k], b[k]); od[4 * i + k] = max_odd_bytes(a[k], b[k]); }
        }
        float rs[21];
        obs_period_sums(ev, od, rs);
        obs_period_take(r, rs, acc, [&](int dy, const float (&v)[21]) {
            gbyte* o = out + dy * 84;
#pragma unroll
            for (int q = 0; q < 21; q++) o[q] = round_sat(v[q]);
        });
    }
}

__global__ void EMU_BOUNDS k_boot(BootArgs A) {
    ROM_LDS
    stage_rom(A.R, s_rom, s_lut);
    const int l = (int)wave_console(blockIdx.x);
    if (l < A.nl) boot_lane(A, lane_ctx(A.R, s_rom, s_lut, s_env), l);
}

__global__ void EMU_BOUNDS k_cache(CacheArgs A) {
    ROM_LDS
    stage_rom(A.R, s_rom, s_lut);
    const int ci = (int)wave_console(blockIdx.x);
    if (ci < A.nc) cache_lane(A, lane_ctx(A.R, s_rom, s_lut, s_env), ci);
}

// k_step's order when it has more envs than the GPU holds waves at once (past 4,096 on 256 CUs). The grid is then one
// block per CU, and a wave that is done with an env takes the next one from a counter, so that no wave waits for the
// slowest env of its block and the cartridge is staged once per CU. What is left is the end, when the last waves run
// alone: the envs start in order of the last step's executed 6502 instructions, most first, in half-octave buckets
// (longest-first list scheduling; a busy run, an area transition or a death, lasts several steps). k_step appends each
// env to the next step's buckets itself, and k_reset, which follows it on the stream, turns the two lists over: no
// launch and no pass of its own. The order within a bucket is that of the appends; no result depends on it.
// Measured at 32,768 / 65,536 envs when it came: k_step 9.0 / 18.8 ms, against 10.6 (unsorted) / 22.9 ms with blocks of 16 envs in
// the order of each block's slowest env (8.4 / 16.1 ms of it are the waves' mean busy time).
struct StepQueue {
    uint32_t side;                          // the lists this step reads; it appends to the others
    uint32_t next;                          // position of the next env to take, past the grid's first ones
    uint32_t count[2][WORK_BUCKETS];
};
// the envs of bucket b, side s: list[(s * WORK_BUCKETS + b) * np ..]

// What bounds it: scalar issue. A SIMD issues one scalar instruction per 4 cycles whichever of its waves it is from; the
// headline step (32,768 envs of 1-1) is 99,000 scalar, 67,000 vector and 15,000 branch instructions per env, of which
// the 5,150 6502 instructions are about 45,000 scalar ones (scalar issue 71% busy, vector 48%). Why one console per wave, against
// 16 per wave in lockstep (4 lanes each, every opcode's work as selects, 15 to 12 of 16 consoles active): a lockstep
// iteration issues ~470 instructions for ~12 6502 instructions but each env waits for all of them; here a 6502
// instruction is ~17 instructions and nothing waits for another console. Measured when it came (k_step, the same
// envs): 256 envs 11.6 -> 1.03 ms, 4,096 envs 19.9 -> 2.99 ms, 32,768 envs 14.57 -> 10.64 ms, 65,536 envs of 32 levels
// 40.9 -> 22.9 ms (9.0 and 18.8 with the queue; 7.4 and 14.6 now, by what run_frame, calls_to_hit and cpu_gfx950.hpp name).
// q null: every env has its wave.
__global__ void EMU_BOUNDS k_step(StepArgs A, StepQueue* q, uint32_t* list) {
    ROM_LDS
    stage_rom(A.R, s_rom, s_lut);
    const uint32_t lane = threadIdx.x & 63u, n = (uint32_t)A.n;
    uint32_t i = q ? wave_slot() * gridDim.x + blockIdx.x : wave_console(blockIdx.x);   // the heaviest, one per CU
    uint32_t side = 0, count = 0, upto = 0;   // lane k: bucket WORK_BUCKETS - 1 - k, and the envs up to its end
    if (q) {
        side = uni(q->side);
        if (lane < WORK_BUCKETS) count = q->count[side][WORK_BUCKETS - 1 - lane];
        upto = count;
        for (int d = 1; d < WORK_BUCKETS; d <<= 1) {
            const uint32_t o = (uint32_t)__shfl_up((int)upto, d);
            if ((int)lane >= d) upto += o;
        }
    }
    while (i < n) {
        uint32_t e = i;
        if (q) {
            const uint32_t k = (uint32_t)__builtin_popcountll(__ballot(lane < WORK_BUCKETS - 1 && upto <= i));
            const uint32_t first = uni((uint32_t)__shfl((int)(upto - count), (int)k));
            e = uni(list[(size_t)(side * WORK_BUCKETS + WORK_BUCKETS - 1 - k) * A.np + (i - first)]);
        }
        const uint32_t bits = step_lane(A, lane_ctx(A.R, s_rom, s_lut, s_env), e);
        __builtin_amdgcn_s_setprio(0);   // the frame loops of the other waves issue first
        obs_tail(A.gray, A.np, A.fresh, A.boot_obs, e, lane, bits);
        if (!q) return;
        if (lane == 0) {
            const uint32_t b = bits >> 4 & (WORK_BUCKETS - 1), o = side ^ 1u;
            list[(size_t)(o * WORK_BUCKETS + b) * A.np + atomicAdd(&q->count[o][b], 1u)] = e;
            i = atomicAdd(&q->next, 1u);   // grows past n by one per wave at most: every wave ends
        }
        i = uni(i);
    }
}

__global__ void EMU_BOUNDS k_raw(RawArgs A) {
    ROM_LDS
    stage_rom(A.R, s_rom, s_lut);
    const uint32_t e = wave_console(blockIdx.x);
    if (e < (uint32_t)A.n) raw_lane(A, lane_ctx(A.R, s_rom, s_lut, s_env), e);
}

// One wave of 64 envs per block: each lane draws its env's reset, then the wave copies the chosen cache
// consoles one env at a time with all 64 lanes.
__global__ void __launch_bounds__(64) k_reset(ResetArgs A, StepQueue* q, uint32_t first) {
    if (q && blockIdx.x == 0) {   // after a step: its lists are done, the next step reads the others
        const uint32_t s = q->side;
        if (threadIdx.x < WORK_BUCKETS) q->count[s][threadIdx.x] = 0;
        if (threadIdx.x == 0) { q->side = s ^ 1u; q->next = first; }
    }
    const uint32_t e = blockIdx.x * 64 + threadIdx.x;
    const int ci = e < (uint32_t)A.n ? reset_lane(A, e) : -1;
    uint64_t m = __ballot(ci >= 0);
    while (m) {
        const int l = __builtin_ctzll(m);
        m &= m - 1;
        const uint32_t el = (uint32_t)__shfl((int)e, l);
        const int cl = __shfl(ci, l);
        copy_console_wave(Region{A.mem, A.sc, A.np, el}, Region{(uint8_t*)A.cmem, (uint32_t*)A.csc, A.ncp, (uint32_t)cl},
                          threadIdx.x, 64);
    }
}

// Observation of a reset-cache entry or a boot state: the boot observation, or the resized last frame.
struct SmallObsArgs {
    const uint8_t* gray;                      // whole frames, entry i the i-th
    const uint8_t* use_boot;                  // per entry (nullable): take boot_obs[level(i)]
    const uint8_t* boot_obs; int nk;          // boot observations [level * OBS_PIX]
    uint8_t* out; int count;                  // [i * OBS_PIX + o]
    const AreaTables* T;
};
__global__ void k_small_obs(SmallObsArgs A) {
    const int i = blockIdx.y;
    const int o = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= A.count || o >= OBS_PIX) return;
    uint8_t v;
    if (A.use_boot && A.use_boot[i]) v = A.boot_obs[(size_t)(i / A.nk) * OBS_PIX + o];
    else v = area_pixel(Image{A.gray + (size_t)i * GRAY_PIX, 0, 0}, Image{}, false, o, A.T);
    A.out[(size_t)i * OBS_PIX + o] = v;
}

struct StackArgs {
    int n; uint32_t np; int K;
    uint8_t* obs; uint8_t* fin;   // [env][K][OBS_PIX]
    const int32_t* slot_env;      // env of each console slot
    const uint8_t* fresh;         // new observation of slot e at [e * OBS_PIX + o]
    const uint32_t* ev;
    const uint8_t* cobs;          // [ci * OBS_PIX + o]
    int mode;                     // 0 step, 1 reset
};
// Frame stack, final_obs, reset observation (fastmario.cpp:477-504). Block: 64 envs x 64 words of one
// frame; consecutive threads take consecutive words of one env.
__global__ void __launch_bounds__(256) k_stack(StackArgs A) {
    const uint32_t e0 = blockIdx.x * 64;   // env groups vary fastest: neighbouring workgroups read adjacent envs
    const int w0 = blockIdx.y * 64;        // word index within a frame (OBS_PIX / 4 = 1764 words)
    const int nw = OBS_PIX / 4;
    const size_t fw = (size_t)nw * A.K;   // words per env stack
    for (int idx = threadIdx.x; idx < 64 * 64; idx += 256) {
        const int j = idx >> 6, wl = idx & 63;
        const uint32_t e = e0 + j;
        const int w = w0 + wl;
        if (w >= nw || e >= (uint32_t)A.n) continue;
        const size_t env = (size_t)A.slot_env[e];
        uint32_t* st = (uint32_t*)A.obs + env * fw;
        const uint32_t ri = A.ev[(size_t)E_RESET_IDX * A.np + e];
        if (A.mode == 1) {
            for (int s = 0; s < A.K - 1; s++) st[(size_t)s * nw + w] = 0;
            st[(size_t)(A.K - 1) * nw + w] = ((const uint32_t*)A.cobs)[(size_t)ri * nw + w];
            continue;
        }
        const uint32_t fresh = ((const uint32_t*)A.fresh)[(size_t)e * nw + w];
        if (ri != 0xffffffffu) {
            uint32_t* fo = (uint32_t*)A.fin + env * fw;
            for (int s = 0; s < A.K - 1; s++) { fo[(size_t)s * nw + w] = st[(size_t)(s + 1) * nw + w]; st[(size_t)s * nw + w] = 0; }
            fo[(size_t)(A.K - 1) * nw + w] = fresh;
            st[(size_t)(A.K - 1) * nw + w] = ((const uint32_t*)A.cobs)[(size_t)ri * nw + w];
        } else {
            for (int s = 0; s < A.K - 1; s++) st[(size_t)s * nw + w] = st[(size_t)(s + 1) * nw + w];
            st[(size_t)(A.K - 1) * nw + w] = fresh;
        }
    }
}

// k_stack with 16-byte accesses, for obs / fin buffers (and the reset cache) 16-byte aligned: the same block
// (64 envs x 64 words of a frame), but a thread moves 4 consecutive words of one env per access (16 threads per
// env, 16 envs per pass, 4 passes), and reads the env's slot and reset index once per pass.
__global__ void __launch_bounds__(256) k_stack4(StackArgs A) {
    const uint32_t e0 = blockIdx.x * 64;
    const int w0 = blockIdx.y * 64;
    const int nw = OBS_PIX / 4;
    const size_t fw = (size_t)nw * A.K;   // words per env stack
    const int g = threadIdx.x & 15, w = w0 + 4 * g;   // this thread's 4 words: w .. w + 3 (nw is a multiple of 4)
    for (int pass = 0; pass < 4; pass++) {
        const int j = 16 * pass + (threadIdx.x >> 4);
        const uint32_t e = e0 + j;
        if (w >= nw || e >= (uint32_t)A.n) continue;
        const size_t env = (size_t)A.slot_env[e];
        uint4* st = (uint4*)((uint32_t*)A.obs + env * fw + w);          // frame s of the stack at st + s * nw / 4
        const uint32_t ri = A.ev[(size_t)E_RESET_IDX * A.np + e];
        const size_t fq = (size_t)nw / 4;
        if (A.mode == 1) {
            for (int s = 0; s < A.K - 1; s++) st[s * fq] = make_uint4(0, 0, 0, 0);
            st[(A.K - 1) * fq] = *(const uint4*)((const uint32_t*)A.cobs + (size_t)ri * nw + w);
            continue;
        }
        const uint4 fresh = *(const uint4*)((const uint32_t*)A.fresh + (size_t)e * nw + w);
        if (ri != 0xffffffffu) {
            uint4* fo = (uint4*)((uint32_t*)A.fin + env * fw + w);
            for (int s = 0; s < A.K - 1; s++) { fo[s * fq] = st[(s + 1) * fq]; st[s * fq] = make_uint4(0, 0, 0, 0); }
            fo[(A.K - 1) * fq] = fresh;
            st[(A.K - 1) * fq] = *(const uint4*)((const uint32_t*)A.cobs + (size_t)ri * nw + w);
        } else {
            // streaming stores: the stacks are read next by the caller, not by a kernel of this step
            // (0.453 -> 0.422 ms at 32,768 envs)
            typedef uint32_t v4u __attribute__((ext_vector_type(4)));
            v4u* sv = (v4u*)st;
            for (int s = 0; s < A.K - 1; s++) __builtin_nontemporal_store(sv[(s + 1) * fq], &sv[s * fq]);
            __builtin_nontemporal_store(*(const v4u*)&fresh, &sv[(A.K - 1) * fq]);
        }
    }
}

// The kernels that hand consoles out. A console's memory and its frame are contiguous, so that consecutive lanes take
// consecutive words of one console. slot_env (nullable: the identity): the output row of each console slot.

// A wave per console.
__global__ void __launch_bounds__(64) k_canon(const uint8_t* mem, const uint32_t* sc, uint32_t np, const int32_t* slot_env, uint8_t* out) {
    const uint32_t e = blockIdx.x;
    canon_lane(mem, sc, np, e, out + (size_t)(slot_env ? slot_env[e] : (int32_t)e) * MH_CANON_BYTES, threadIdx.x, 64);
}

// RAM of every console -> (n x 2048), W bytes at a time: 16, or 1 into an output that is not 16-byte aligned.
// 4,096 / 32,768 consoles: 46 / 355 us with lanes across the consoles, 8 (the launch) / 20 here.
template <class W>
__global__ void __launch_bounds__(256) k_ram_out(const uint8_t* mem, uint32_t np, int n, const int32_t* slot_env, uint8_t* out) {
    constexpr uint32_t PER = 2048 / sizeof(W);
    const uint32_t i = blockIdx.x * 256 + threadIdx.x, e = i / PER, w = i % PER;   // below 2^31 (MAX_ENVS)
    if (e >= (uint32_t)n) return;
    W* const to = (W*)(out + (size_t)(slot_env ? slot_env[e] : (int32_t)e) * 2048);
    to[w] = ((const W*)(mem + mem_offset(np, e, ROW_RAM)))[w];
}
static_assert(ROW_RAM % 16 == 0 && MEM_ROWS % 16 == 0 && (uint64_t)MAX_ENVS * 2048 < 1ull << 31, "16-byte words, 32-bit indexes");

// Frames of palette values -> (n x 240 x 256) RGB24 through a 64-entry RGB table (a palette value is taken & 63, as nes-py's
// screen). A thread's 4 pixels are three 32-bit words (`words`: out is 4-byte aligned), so that a wave writes 768 bytes
// in a row. Block: 1,024 of a console's 4-pixel words. Bound by memory: 4,096 frames (1.0 GB) 226 us, 495 with lanes
// across the consoles.
constexpr int RGB_WORDS = 1024;
static_assert(GRAY_PIX / 4 % RGB_WORDS == 0, "whole blocks");
__global__ void __launch_bounds__(256) k_frames_rgb(const uint8_t* src, const uint8_t* rgb64, uint8_t* out, int words) {
    __shared__ uint32_t tab[64];
    if (threadIdx.x < 64) {
        const uint8_t* t = rgb64 + 3 * threadIdx.x;
        tab[threadIdx.x] = t[0] | (uint32_t)t[1] << 8 | (uint32_t)t[2] << 16;
    }
    __syncthreads();
    const size_t w0 = (size_t)blockIdx.x * (GRAY_PIX / 4) + blockIdx.y * RGB_WORDS + threadIdx.x;
#pragma unroll
    for (int k = 0; k < RGB_WORDS / 256; k++) {
        const size_t w = w0 + 256 * k;
        const uint32_t v = ((const uint32_t*)src)[w];
        const uint32_t c0 = tab[v & 63u], c1 = tab[v >> 8 & 63u], c2 = tab[v >> 16 & 63u], c3 = tab[v >> 24 & 63u];
        const uint32_t o[3] = {c0 | c1 << 24, c1 >> 8 | c2 << 16, c2 >> 16 | c3 << 8};
        uint8_t* const to = out + 12 * w;
        if (words)
            for (int i = 0; i < 3; i++) ((uint32_t*)to)[i] = o[i];
        else
            for (int i = 0; i < 12; i++) to[i] = (uint8_t)(o[i >> 2] >> (8 * (i & 3)));
    }
}

// 240x256 gray images (env-major) -> 84x84.
__global__ void k_resize_images(const uint8_t* src, uint8_t* dst, int n, const AreaTables* T) {
    const int i = blockIdx.y;
    const int o = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || o >= OBS_PIX) return;
    dst[(size_t)i * OBS_PIX + o] = area_pixel(Image{src + (size_t)i * GRAY_PIX, 0, 0}, Image{}, false, o, T);
}

// ------------------------------------------------------------------ host side
thread_local std::string g_err;

static bool ok(hipError_t e, const char* what) {
    if (e == hipSuccess) return true;
    g_err = std::string(what) + ": " + hipGetErrorString(e);
    return false;
}
#define CK(expr) do { if (!ok((expr), #expr)) return -1; } while (0)
#define CKN(expr) do { if (!ok((expr), #expr)) { return nullptr; } } while (0)

static uint32_t pad64(int n) { return (uint32_t)((n + 63) / 64 * 64); }

struct DevBufs {
    std::vector<void*> ptrs;
    template <class T> T* alloc(size_t count, bool& good) {
        void* p = nullptr;
        if (hipMalloc(&p, count * sizeof(T) + 16) != hipSuccess) { good = false; g_err = "hipMalloc failed"; return nullptr; }
        if (hipMemset(p, 0, count * sizeof(T) + 16) != hipSuccess) { good = false; g_err = "hipMemset failed"; }
        ptrs.push_back(p);
        return (T*)p;
    }
    ~DevBufs() { for (void* p : ptrs) (void)hipFree(p); }
};

// iNES NROM image -> 0x8000 PRG (16 KB mirrored) + 0x2000 CHR and name-table offsets (nes_core.hpp:66-87).
static bool load_cart(const uint8_t* d, int64_t n, std::vector<uint8_t>& img, uint16_t nt[4]) {
    if (!d || n < 16 || d[0] != 'N' || d[1] != 'E' || d[2] != 'S' || d[3] != 0x1a) { g_err = "not an iNES image"; return false; }
    int mapper = ((d[6] >> 4) & 0xf) | (d[7] & 0xf0);
    if (mapper != 0 || (d[6] & 0x6)) { g_err = "unsupported ROM (mapper / PRG-RAM / trainer)"; return false; }
    int banks = d[4];
    if (banks < 1 || banks > 2 || d[5] != 1) { g_err = "unsupported ROM (PRG/CHR size)"; return false; }
    if (n < 16 + 0x4000LL * banks + 0x2000) { g_err = "truncated ROM"; return false; }
    img.assign(0xa000, 0);
    for (int i = 0; i < 0x8000; i++) img[i] = d[16 + (i % (0x4000 * banks))];
    memcpy(img.data() + 0x8000, d + 16 + 0x4000 * banks, 0x2000);
    switch (d[6] & 0xB) {
        case 0: nt[0] = 0; nt[1] = 0; nt[2] = 0x400; nt[3] = 0x400; break;
        case 1: nt[0] = 0; nt[1] = 0x400; nt[2] = 0; nt[3] = 0x400; break;
        default: nt[0] = nt[1] = nt[2] = nt[3] = 0; break;
    }
    return true;
}

// The program (the image's first 32 KB) as scalar_run's records.
static bool upload_records(uint32_t* d_recs, const std::vector<uint8_t>& img) {
    static constexpr dec::Table words{};
    std::vector<uint32_t> recs(REC_COUNT);
    decode_prg(img.data(), words.w, recs.data());
    return ok(hipMemcpy(d_recs, recs.data(), recs.size() * 4, hipMemcpyHostToDevice), "upload program records");
}

// ---- the PPO policy's input (the rollout harness's observation -> bf16 channels-last scaling)
// Observation stacks (n, k, 84, 84) u8 -> the bf16 (n, k, 84, 84) tensor in channels-last memory, i.e. element
// (b, c, h, w) at ((b * 84 + h) * 84 + w) * k + c, of value bf16(float(v) * float(1 / 255)) rounded to nearest
// even: what torch's float32 scaling followed by the bf16 cast gives. Thread: 4 consecutive pixels of one row of
// one image, all k channels (k u32 loads of 4 pixels, then 4 k bf16 values stored as 32-bit pairs).
__device__ __forceinline__ uint32_t bf16_rne(float f) {   // f finite and >= 0
    const uint32_t u = __float_as_uint(f);
    return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}
template <int K>
__global__ void __launch_bounds__(256) k_policy_input(const uint8_t* obs, uint32_t* out, int64_t groups) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= groups) return;
    const int64_t b = t / (OBS_PIX / 4);
    const int r = (int)(t - b * (OBS_PIX / 4));          // pixel group in the image: pixels 4 r .. 4 r + 3
    const float s = (float)(1.0 / 255.0);
    uint32_t v[K];
#pragma unroll
    for (int c = 0; c < K; c++) v[c] = ((const uint32_t*)obs)[(b * K + c) * (OBS_PIX / 4) + r];
    // pixel q of the group: its K channels at out halves (4 r + q) * K .. + K - 1 of image b
    uint32_t* o = out + (b * OBS_PIX + 4 * r) * K / 2;
#pragma unroll
    for (int q = 0; q < 4; q++) {
#pragma unroll
        for (int c = 0; c < K; c += 2) {
            const uint32_t lo = bf16_rne((float)((v[c] >> (8 * q)) & 0xffu) * s);
            const uint32_t hi = c + 1 < K ? bf16_rne((float)((v[c + 1] >> (8 * q)) & 0xffu) * s) : 0u;
            o[(q * K + c) / 2] = lo | hi << 16;
        }
    }
}

__global__ void __launch_bounds__(256) k_policy_input_k1(const uint8_t* obs, uint32_t* out, int64_t groups) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= groups) return;
    const float s = (float)(1.0 / 255.0);
    const uint32_t v = ((const uint32_t*)obs)[t];
    out[2 * t] = bf16_rne((float)(v & 0xffu) * s) | bf16_rne((float)((v >> 8) & 0xffu) * s) << 16;
    out[2 * t + 1] = bf16_rne((float)((v >> 16) & 0xffu) * s) | bf16_rne((float)(v >> 24) * s) << 16;
}

// ---- the PPO policy's convolutions on the matrix cores (Nature CNN: 4 -> 32 channels 8x8 stride 4, 84x84 -> 20x20;
// 32 -> 64 4x4 stride 2, 20x20 -> 9x9; 64 -> 64 3x3 stride 1, 9x9 -> 7x7), each an implicit GEMM with float32
// accumulation, its bias and its ReLU; activations bf16 in channels-last memory (pixel m's channels at m * C ..).
// A block stages whole images in LDS and a wave's tiles of 32 output pixels read their patches from there: a patch
// read from global memory touches a cache line per pixel (64 lines for the 1 KB of one MFMA step), and every input
// pixel is in 4 (9 in the third layer) patches of two waves, which is what bounded the kernels without staging. The
// weights stay in registers (lane l: output channel l % 32, K = 16 s + 8 (l / 32) .. + 7 of step s of
// v_mfma_f32_32x32x16_bf16); they are the first operand, so that a lane ends up with its pixel's channels
// 8 q + 4 (l / 32) .. + 3, q = 0 .. 3, and stores them 8 bytes at a time. The next images' loads are in flight while
// these compute. 32,768 images, before -> now (reading and writing the activations alone at a copy's 4.9 TB/s): first layer
// 600 -> 412 us (360), second 600 -> 257 (240), third 430 -> 150 (110).
typedef __bf16 mh_bf16x8 __attribute__((ext_vector_type(8)));
typedef float mh_f32x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ mh_bf16x8 as_bf16x8(mh_u32x4 q) { return __builtin_bit_cast(mh_bf16x8, q); }
typedef __bf16 mh_bf16x2 __attribute__((ext_vector_type(2)));
typedef float mh_f32x2 __attribute__((ext_vector_type(2)));
// lo | hi << 16 as bf16, rounded to nearest even: one instruction for the two, which an element at a time takes four
__device__ __forceinline__ uint32_t bf16_pair(float lo, float hi) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(mh_f32x2{lo, hi}, mh_bf16x2));
}
// four pixels, a byte each, as bf16(float(v) * sc)
__device__ __forceinline__ uint2 scaled_pixels(uint32_t v, float sc) {
    return make_uint2(bf16_pair((float)(v & 0xffu) * sc, (float)(v >> 8 & 0xffu) * sc),
                      bf16_pair((float)(v >> 16 & 0xffu) * sc, (float)(v >> 24) * sc));
}
// a lane's 16 sums (its pixel's channels) + bias, ReLU, bf16, to out (the pixel's first channel of these 32, + 4 kg);
// wide: out is 8-byte aligned
__device__ __forceinline__ void conv_out(const mh_f32x16& acc, const float (&bias)[16], uint16_t* out, bool wide) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
        float r[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            r[i] = acc[4 * q + i] + bias[4 * q + i];
            r[i] = r[i] > 0.f ? r[i] : 0.f;
        }
        const uint2 h = make_uint2(bf16_pair(r[0], r[1]), bf16_pair(r[2], r[3]));
        if (wide) *(uint2*)(out + 8 * q) = h;
        else
            for (int i = 0; i < 4; i++) out[8 * q + i] = (uint16_t)((i < 2 ? h.x : h.y) >> (16 * (i & 1)));
    }
}

// The products of a tile's STEPS steps, operand(s) of step s read from LDS a group of 4 ahead of the products that use it.
// (Left to itself the compiler reads one step ahead, and a read takes as long as 4 products: k_policy_conv12 606 us of
// 32,768 images against 535. The layers' own kernels have no registers left for it.)
template <int STEPS, class F>
__device__ __forceinline__ mh_f32x16 tile_products(const mh_bf16x8 (&w)[STEPS], F&& operand) {
    static_assert(STEPS % 4 == 0, "groups of 4 steps");
    mh_f32x16 acc = {};
    mh_u32x4 a[4], ahead[4];
#pragma unroll
    for (int i = 0; i < 4; i++) ahead[i] = operand(i);
#pragma unroll
    for (int s = 0; s < STEPS; s += 4) {
#pragma unroll
        for (int i = 0; i < 4; i++) a[i] = ahead[i];
        if (s + 4 < STEPS) {
#pragma unroll
            for (int i = 0; i < 4; i++) ahead[i] = operand(s + 4 + i);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; i++) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[s + i], as_bf16x8(a[i]), acc, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    }
    return acc;
}
// The weights have arrived. Before a loop that keeps loads in flight: else the compiler waits in it for the weights, and
// so for all that is in flight, ahead of every first product.
__device__ __forceinline__ void weights_arrived() { __builtin_amdgcn_s_waitcnt(0); }

// The first layer, with the input scaled as mh_policy_input scales it: K = 4 x 8 x 8 in the weight's own (ci, kh, kw)
// order. An image is 56,448 bytes of bf16 in LDS, scaled once (2.5 vector instructions a pixel; scaled per patch, 7 a
// patch element, it bounded the layer). A wave has all 32 channels and every fourth tile.
constexpr int CONV1_OUT = 20 * 20;   // output pixels per image
__global__ void __launch_bounds__(256, 2) k_policy_conv1(const uint8_t* obs, const uint16_t* w, const uint16_t* bias,
                                                         uint16_t* out, int64_t n, int wide) {
    constexpr int WORDS = 4 * OBS_PIX / 4, PER = (WORDS + 255) / 256;   // 4-pixel words an image, a thread
    __shared__ __attribute__((aligned(16))) uint16_t s_x[4 * OBS_PIX];
    const int tid = threadIdx.x, l = tid & 63, wv = tid >> 6, j = l & 31, kg = l >> 5;
    mh_bf16x8 wb[16];
#pragma unroll
    for (int s = 0; s < 16; s++) wb[s] = as_bf16x8(*(const mh_u32x4*)(w + (size_t)j * 256 + 16 * s + 8 * kg));
    float bj[16];
#pragma unroll
    for (int v = 0; v < 16; v++) bj[v] = __uint_as_float((uint32_t)bias[8 * (v >> 2) + 4 * kg + (v & 3)] << 16);
    const float sc = (float)(1.0 / 255.0);
    uint32_t raw[PER];
    auto load = [&](int64_t b) {
        const uint32_t* src = (const uint32_t*)(obs + (size_t)b * 4 * OBS_PIX);
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int c = tid + 256 * i;
            raw[i] = src[c < WORDS ? c : 0];
        }
    };
    weights_arrived();
    int64_t b = blockIdx.x;
    if (b < n) load(b);
    for (; b < n; b += gridDim.x) {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int c = tid + 256 * i;
            if (c < WORDS) *(uint2*)(s_x + 4 * c) = scaled_pixels(raw[i], sc);
        }
        __syncthreads();
        if (b + gridDim.x < n) load(b + gridDim.x);
        for (int t = wv; t * 32 < CONV1_OUT; t += 4) {
            const int m = t * 32 + j, p = m < CONV1_OUT ? m : CONV1_OUT - 1, oy = p / 20, ox = p - oy * 20;
            const uint16_t* at = s_x + (4 * oy + kg) * 84 + 4 * ox;
            mh_f32x16 acc = {};
#pragma unroll
            for (int s = 0; s < 16; s++) {   // K = 16 s + 8 kg ..: channel s / 4, rows 2 (s % 4) + kg
                const uint2* r = (const uint2*)(at + (s >> 2) * OBS_PIX + 2 * (s & 3) * 84);
                const uint2 a = r[0], c = r[1];
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wb[s], as_bf16x8(mh_u32x4{a.x, a.y, c.x, c.y}), acc, 0, 0, 0);
            }
            if (m < CONV1_OUT) conv_out(acc, bj, out + ((size_t)b * CONV1_OUT + m) * 32 + 4 * kg, wide);
        }
        __syncthreads();
    }
}

// The second and third layers: the weight is (64, KS, KS, CI), so K = (kh, kw, ci) and a step is 16 channels of one
// input pixel. IMGS images at a time: their output pixels in one row of tiles, the even and odd waves the two halves of
// the output channels, the block's two pairs of waves every second tile. A pixel takes 16 bytes more than its
// channels in LDS, so that the lanes of a 16-byte read are in different banks along an output row; across its end they
// still meet (bank conflicts on over a quarter of the third layer's cycles).
template <int CI, int KS, int ST, int HI, int HO, int IMGS>
__global__ void __launch_bounds__(256, 2) k_policy_conv(const uint16_t* x, const uint16_t* w, const uint16_t* bias,
                                                        uint16_t* y, int64_t n, int wide) {
    constexpr int CO = 64, K = KS * KS * CI, STEPS = K / 16, PIX = HO * HO, INP = HI * HI, PXW = CI + 8;
    constexpr int PARTS = CI / 8, CHUNKS = IMGS * INP * PARTS, PER = (CHUNKS + 255) / 256;   // 16-byte pieces
    static_assert(CI % 16 == 0, "whole MFMA steps");
    __shared__ __attribute__((aligned(16))) uint16_t s_x[IMGS * INP * PXW];
    const int tid = threadIdx.x, l = tid & 63, wv = tid >> 6, j = l & 31, kg = l >> 5, half = wv & 1;
    mh_bf16x8 wb[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; s++) wb[s] = as_bf16x8(*(const mh_u32x4*)(w + (size_t)(32 * half + j) * K + 16 * s + 8 * kg));
    float bj[16];
#pragma unroll
    for (int v = 0; v < 16; v++) bj[v] = __uint_as_float((uint32_t)bias[32 * half + 8 * (v >> 2) + 4 * kg + (v & 3)] << 16);
    const int64_t groups = (n + IMGS - 1) / IMGS;
    auto images = [&](int64_t g) { return n - g * IMGS < IMGS ? (int)(n - g * IMGS) : IMGS; };
    mh_u32x4 raw[PER];
    auto load = [&](int64_t g) {
        const mh_u32x4* src = (const mh_u32x4*)(x + (size_t)g * IMGS * INP * CI);
        const int last = images(g) * INP * PARTS - 1;
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int c = tid + 256 * i;
            raw[i] = src[c < last ? c : last];
        }
    };
    weights_arrived();
    int64_t g = blockIdx.x;
    if (g < groups) load(g);
    for (; g < groups; g += gridDim.x) {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int c = tid + 256 * i;
            if (c < CHUNKS) *(mh_u32x4*)(s_x + (c / PARTS) * PXW + 8 * (c % PARTS)) = raw[i];
        }
        __syncthreads();
        const int pixels = images(g) * PIX;
        if (g + gridDim.x < groups) load(g + gridDim.x);
        for (int t = wv >> 1; t * 32 < pixels; t += 2) {
            const int m = t * 32 + j, q = m < pixels ? m : pixels - 1;
            const int b = q / PIX, p = q - b * PIX, oy = p / HO, ox = p - oy * HO;
            const uint16_t* at = s_x + (b * INP + ST * oy * HI + ST * ox) * PXW + 8 * kg;
            mh_f32x16 acc = {};
#pragma unroll
            for (int s = 0; s < STEPS; s++) {
                const int k0 = 16 * s, kh = k0 / (KS * CI), kw = (k0 / CI) % KS, ci = k0 % CI;
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    wb[s], as_bf16x8(*(const mh_u32x4*)(at + (kh * HI + kw) * PXW + ci)), acc, 0, 0, 0);
            }
            if (m < pixels) conv_out(acc, bj, y + ((size_t)g * IMGS * PIX + m) * CO + 32 * half + 4 * kg, wide);
        }
        __syncthreads();
    }
}
// images a block takes at a time in the second and third layers once that leaves every CU a block: 162 pixels are 6
// tiles, 245 are 8 (one image is 81 and 49: 3 and 2)
constexpr int CONV2_IMGS = 2, CONV3_IMGS = 5;

// The first two layers in one pass, the first one's output in LDS alone (32,768 images: 1.7 GB less of memory traffic).
// A block of 8 waves a CU, in phases of half an image (10 of the first layer's 20 output rows): waves 0 .. 3 are the first
// layer's, of image i, while waves 4 .. 7 do the second layer of image i - 1 from the other of two LDS buffers; both
// stage the next half image, the first ones after their products and the second ones before, so that a SIMD, which has
// a wave of each, scales with one while it multiplies with the other. A row of s_y is padded so that pixel p of the second
// layer's 81 reads at p times a pixel's words, modulo the banks, across its rows too. Operands, sums and their order are
// those of the two kernels above, and so are the results. 300 / 32,768 images: 22 / 669 us as two kernels, 16.5 /
// 535 here (whole images at a time, all waves staging before the products: 16 / 578; operands read one step ahead: 606).
// No unit is full: matrix cores 38% busy, LDS accesses about half of the cycles (a quarter of it bank conflicts), vector
// issue 33%; a wave waits 40% of its time, with two a SIMD.
__global__ void __launch_bounds__(512, 2) k_policy_conv12(const uint8_t* obs, const uint16_t* w1, const uint16_t* bias1,
                                                          const uint16_t* w2, const uint16_t* bias2, uint16_t* y, int64_t n) {
    constexpr int ROWS = 44, CH = ROWS * 84 / 4, WORDS = 4 * CH, PER = (WORDS + 511) / 512;   // 4-pixel words of a half
    constexpr int PXW = 40, ROWW = 20 * PXW + 8, HALF_PIX = CONV1_OUT / 2, HO = 9, PIX = HO * HO;   // s_y's, in halfs
    __shared__ __attribute__((aligned(16))) uint16_t s_x[2][4 * WORDS];
    __shared__ __attribute__((aligned(16))) uint16_t s_y[2][20 * ROWW];
    const int tid = threadIdx.x, l = tid & 63, wv = (int)uni((uint32_t)tid >> 6), j = l & 31, kg = l >> 5;
    const float sc = (float)(1.0 / 255.0);
    const int64_t step = gridDim.x, phases = 2 * ((n - blockIdx.x + step - 1) / step);   // blockIdx.x < n
    uint32_t raw[PER];
    auto load = [&](int64_t q) {   // the half image of phase q
        if (q >= phases) return;
        const uint32_t* src = (const uint32_t*)(obs + (size_t)(blockIdx.x + (q >> 1) * step) * 4 * OBS_PIX) + (q & 1) * (40 * 21);
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int c = tid + 512 * i, d = c < WORDS ? c : 0;
            raw[i] = src[d / CH * (OBS_PIX / 4) + d % CH];
        }
    };
    auto stage = [&](int64_t q) {
        if (q >= phases) return;
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int c = tid + 512 * i;
            if (c < WORDS) *(uint2*)(s_x[q & 1] + 4 * c) = scaled_pixels(raw[i], sc);
        }
    };
    auto biases = [&](const uint16_t* bias, float (&bj)[16]) {
#pragma unroll
        for (int v = 0; v < 16; v++) bj[v] = __uint_as_float((uint32_t)bias[8 * (v >> 2) + 4 * kg + (v & 3)] << 16);
    };
    // both roles pass the same barriers: one before the first phase and one after each. Phase q reads s_x[q & 1], which
    // was staged in phase q - 1, and stages the other; an image's s_y is written in its two phases and read in the two after.
    load(0);
    stage(0);
    load(1);
    if (wv < 4) {
        mh_bf16x8 wb[16];
#pragma unroll
        for (int s = 0; s < 16; s++) wb[s] = as_bf16x8(*(const mh_u32x4*)(w1 + (size_t)j * 256 + 16 * s + 8 * kg));
        float bj[16];
        biases(bias1, bj);
        weights_arrived();
        __syncthreads();
        for (int64_t q = 0; q < phases; q++) {
            const int part = (int)(q & 1), turn = (int)(q >> 1 & 1);
            // of the half's 7 tiles two, two, two and one; one, one, three and two beside the second layer's third tile
            for (int t = wv, by = part ? (wv < 2 ? 8 : 2) : 4; t * 32 < HALF_PIX; t += by) {
                const int m = t * 32 + j, p = m < HALF_PIX ? m : HALF_PIX - 1, oy = p / 20, ox = p - oy * 20;
                const uint16_t* at = s_x[part] + (4 * oy + kg) * 84 + 4 * ox;
                const mh_f32x16 acc = tile_products<16>(wb, [&](int s) {
                    const uint2* r = (const uint2*)(at + (s >> 2) * (4 * CH) + 2 * (s & 3) * 84);
                    return mh_u32x4{r[0].x, r[0].y, r[1].x, r[1].y};
                });
                if (m < HALF_PIX) conv_out(acc, bj, s_y[turn] + (10 * part + oy) * ROWW + ox * PXW + 4 * kg, true);
            }
            stage(q + 1);
            load(q + 2);
            __syncthreads();
        }
    } else {
        const int half = wv & 1, first = (wv - 4) >> 1;
        mh_bf16x8 wb[32];
#pragma unroll
        for (int s = 0; s < 32; s++) wb[s] = as_bf16x8(*(const mh_u32x4*)(w2 + (size_t)(32 * half + j) * 512 + 16 * s + 8 * kg));
        float bj[16];
        biases(bias2 + 32 * half, bj);
        auto tile = [&](int64_t i, int t) {   // of the block's i-th image
            const int m = t * 32 + j, p = m < PIX ? m : PIX - 1, oy = p / HO, ox = p - oy * HO;
            const uint16_t* at = s_y[i & 1] + 2 * oy * ROWW + 2 * ox * PXW + 8 * kg;
            // K = 16 s + 8 kg ..: row s / 8, column s / 2 % 4, half a pixel's channels
            const mh_f32x16 acc = tile_products<32>(wb, [&](int s) {
                return *(const mh_u32x4*)(at + (s >> 3) * ROWW + ((s >> 1) & 3) * PXW + 16 * (s & 1));
            });
            if (m < PIX) conv_out(acc, bj, y + ((size_t)(blockIdx.x + i * step) * PIX + m) * 64 + 32 * half + 4 * kg, true);
        };
        weights_arrived();
        __syncthreads();
        // tiles 0 and 1 in an image's first phase, 2 in its second; in the end the last image's
        for (int64_t q = 0; q < phases + 2; q++) {
            if (q < phases) {
                stage(q + 1);
                load(q + 2);
            }
            if (q >= 2 && !(q & 1)) tile((q >> 1) - 1, first);
            else if (q >= 2 && first == 0) tile((q >> 1) - 1, 2);
            if (q < phases) __syncthreads();
        }
    }
}

// ---- the network's float32 parameters as the bf16 operands of a forward pass, in one launch: the first layer's weight
// as (co, ci, kh, kw), the others' as (co, kh, kw, ci), the fully connected one's columns from (c, h, w) to (h, w, c)
// order, and the biases. Bound by memory (6.7 MB in, 3.4 out); what it saves is launches: a small batch's pass spends
// its time on them, and these were 12 of 21 (casts and permutes): with it and k_policy_heads a pass is 6, and a pass over
// 300 observations takes 101 us instead of 197 (of it 8 for this). A row of the fully connected weight goes through LDS,
// so that it is read and written whole.
struct PackArgs {
    const float* w[3]; int64_t st[3][4];   // convolution weights and their strides (co, ci, kh, kw)
    const float* b[4];                     // biases
    const float* fc;                       // (512, 3136) contiguous
    uint16_t* out;
};
constexpr int PACK_W[4] = {0, 8192, 40960, 77824};          // the convolutions' weights in out; then the biases,
constexpr int PACK_B[5] = {77824, 77856, 77920, 77984, 78496}, PACK_FC = 78496, FC_IN = 64 * 49, FC_OUT = 512;
static_assert(PACK_FC + FC_OUT * FC_IN == MH_POLICY_PACKED, "the header's size");
constexpr int PACK_SMALL = (PACK_FC + 255) / 256;           // blocks of the small ones, after a block per row of fc
__global__ void __launch_bounds__(256) k_policy_pack(PackArgs A) {
    __shared__ float row[FC_IN];
    const int tid = threadIdx.x;
    auto half = [](float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); };   // to nearest even
    if (blockIdx.x < FC_OUT) {
        const float* src = A.fc + (size_t)blockIdx.x * FC_IN;
        for (int i = tid; i < FC_IN; i += 256) row[i] = src[i];
        __syncthreads();
        uint32_t* dst = (uint32_t*)(A.out + PACK_FC + (size_t)blockIdx.x * FC_IN);
        for (int i = tid; i < FC_IN / 2; i += 256) {   // channels c, c + 1 of pixel p
            const int p = i >> 5, c = 2 * (i & 31);
            dst[i] = half(row[c * 49 + p]) | (uint32_t)half(row[(c + 1) * 49 + p]) << 16;
        }
        return;
    }
    const int i = (int)(blockIdx.x - FC_OUT) * 256 + tid;
    if (i >= PACK_FC) return;
    float f;
    if (i >= PACK_B[0]) {
        int k = 0;
        while (i >= PACK_B[k + 1]) k++;
        f = A.b[k][i - PACK_B[k]];
    } else {
        const int k = i < PACK_W[1] ? 0 : i < PACK_W[2] ? 1 : 2, e = i - PACK_W[k];
        int co, ci, kh, kw;
        if (k == 0) { co = e >> 8; ci = e >> 6 & 3; kh = e >> 3 & 7; kw = e & 7; }
        else if (k == 1) { co = e >> 9; kh = e >> 7 & 3; kw = e >> 5 & 3; ci = e & 31; }
        else { co = e / 576; const int r = e - co * 576; kh = r / 192; kw = r / 64 - 3 * kh; ci = r & 63; }
        f = A.w[k][co * A.st[k][0] + ci * A.st[k][1] + kh * A.st[k][2] + kw * A.st[k][3]];
    }
    A.out[i] = half(f);
}

// ---- the two heads: logits and value of relu(h), h the bf16 (n, 512) output of the fully connected layer, in float32
// (products fused into the sums). A wave per row: a lane has 8 of the row's 512 features and of each of 8 outputs' weights
// (blockIdx.y: which 8 of the A + 1), then the lanes' 8 sums are added by halves (4 + 2 + 1 exchanges, then 3). Bound by
// launches for a small batch, by reading h for a large one. 300 / 32,768 rows: 4 / 23 us; as a ReLU, a conversion and two
// matrix products 30 / 70.
constexpr int HEAD_IN = 512;
__global__ void __launch_bounds__(256) k_policy_heads(const uint16_t* h, const float* w_pi, const float* b_pi, const float* w_vf,
                                                      const float* b_vf, float* logits, float* value, int64_t n, int A) {
    const int l = threadIdx.x & 63, first = 8 * (int)blockIdx.y;
    float w[8][8];
#pragma unroll
    for (int o = 0; o < 8; o++) {
        const int k = first + o;
        const float* src = k < A ? w_pi + (size_t)k * HEAD_IN : w_vf;
#pragma unroll
        for (int i = 0; i < 8; i++) w[o][i] = src[8 * l + i];
    }
    // this lane's output after the reduction: bits 5, 4, 3 of the lane choose the halves
    const int mine = first + (l >> 3 & 4) + (l >> 3 & 2) + (l >> 3 & 1);
    const float bias = mine < A ? b_pi[mine] : b_vf[0];
    const int64_t wave = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6), waves = (int64_t)gridDim.x * 4;
    for (int64_t r = wave; r < n; r += waves) {
        const mh_u32x4 q = *(const mh_u32x4*)(h + r * HEAD_IN + 8 * l);
        float s[8] = {};
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float f = __uint_as_float(i & 1 ? q[i >> 1] & 0xffff0000u : q[i >> 1] << 16), x = f < 0.f ? 0.f : f;
#pragma unroll
            for (int o = 0; o < 8; o++) s[o] = __builtin_fmaf(x, w[o][i], s[o]);
        }
#pragma unroll
        for (int half = 4, bit = 32; half >= 1; half >>= 1, bit >>= 1) {
            const bool upper = l & bit;
#pragma unroll
            for (int o = 0; o < half; o++) {
                const float give = upper ? s[o] : s[o + half], keep = upper ? s[o + half] : s[o];
                s[o] = keep + __shfl_xor(give, bit);
            }
        }
#pragma unroll
        for (int bit = 4; bit >= 1; bit >>= 1) s[0] += __shfl_xor(s[0], bit);
        if ((l & 7) == 0) {
            if (mine < A) logits[r * A + mine] = s[0] + bias;
            else if (mine == A) value[r] = s[0] + bias;
        }
    }
}

// ---- generalized advantage estimation (fast_mario_env_amd.rollout.gae): a lane per env, backwards over the T steps.
// Bound by memory: 17 bytes in and 8 out an env-step, every row read and written once, whole rows of 256 bytes a wave.
// Few waves run (an env is a serial chain: 512 waves for 32,768 envs), so each keeps GAE_AHEAD steps of loads in flight
// behind the chain. The float operations and their order are those of the row-by-row form
//   keep = 1 - s[t+1];  delta = (r[t] + (gamma v[t+1]) keep) - v[t];  a = delta + ((gamma lam) keep) a
// T 128, 32,768 envs: 20 us (3.6 TB/s of the 4.9 that a large copy reaches); the row-by-row form, 8 launches a row, took 5,700.
constexpr int GAE_AHEAD = 16;
__global__ void __launch_bounds__(64) k_gae(const float* __restrict__ rew, const float* __restrict__ val,
                                            const uint8_t* __restrict__ start, const float* __restrict__ next_val,
                                            const uint8_t* __restrict__ next_start, int64_t T, int64_t n, float gamma,
                                            float gamma_lam, float* __restrict__ adv, float* __restrict__ ret) {
    const int64_t e = (int64_t)blockIdx.x * 64 + threadIdx.x;
    if (e >= n) return;
    float nv = next_val[e], ns = next_start[e] ? 1.f : 0.f, last = 0.f;
    float r[2][GAE_AHEAD], v[2][GAE_AHEAD];
    uint8_t s[2][GAE_AHEAD];
    auto load = [&](int64_t t, int b) {         // steps t, t - 1, .. (past the start: step 0, not used)
#pragma unroll
        for (int i = 0; i < GAE_AHEAD; i++) {
            const int64_t at = (t > i ? t - i : 0) * n + e;
            r[b][i] = rew[at]; v[b][i] = val[at]; s[b][i] = start[at];
        }
    };
    auto run = [&](int64_t t, int b) {
#pragma unroll
        for (int i = 0; i < GAE_AHEAD; i++) {
            if (t < i) return;
            const float keep = 1.f - ns;
            const float delta = r[b][i] + gamma * nv * keep - v[b][i];
            last = delta + gamma_lam * keep * last;
            adv[(t - i) * n + e] = last;
            ret[(t - i) * n + e] = last + v[b][i];
            nv = v[b][i];
            ns = s[b][i] ? 1.f : 0.f;
        }
    };
    int64_t t = T - 1;
    load(t, 0);
    while (t >= 0) {
        load(t - GAE_AHEAD, 1);
        run(t, 0);
        t -= GAE_AHEAD;
        if (t < 0) break;
        load(t - GAE_AHEAD, 0);
        run(t, 1);
        t -= GAE_AHEAD;
    }
}

}  // namespace

// compute units of a device (the emulator kernels' launch shape depends on it)
static int device_cus(int device) {
    hipDeviceProp_t prop;
    return hipGetDeviceProperties(&prop, device) == hipSuccess ? prop.multiProcessorCount : 0;
}

struct MhEnv {
    int n = 0, K = 4, nl = 0, nk = 1, nc = 0, device = 0, cus = 0;
    uint32_t np = 0, nlp = 0, ncp = 0;
    Cfg cfg{};
    DevBufs B;
    RomArgs R{};
    AreaTables* T = nullptr;
    uint8_t *mem = nullptr, *gray = nullptr, *fresh = nullptr;
    EmuLaunch ls{};                    // k_step's launch shape
    StepQueue* queue = nullptr;        // k_step's order, when it has more envs than the GPU holds waves: null otherwise
    uint32_t* queue_list = nullptr;
    uint32_t queue_first = 0;          // waves of k_step's grid
    uint32_t *sc = nullptr, *ev = nullptr;
    uint8_t* snap_mem = nullptr;     // 2 snapshot slots of the live consoles (early-termination re-emulation)
    uint32_t* snap_sc = nullptr;
    uint8_t *boot_mem = nullptr, *boot_gray = nullptr, *boot_obs = nullptr;
    uint32_t* boot_sc = nullptr;
    int64_t *x0 = nullptr, *t0 = nullptr;
    uint8_t *cmem = nullptr, *cgray = nullptr, *cobs = nullptr, *cboot = nullptr;
    uint8_t* key_bank = nullptr;     // CHR bank of each (level, ROM) key
    int32_t* slot_env = nullptr;     // env of each console slot (slots grouped by (level, ROM) key)
    uint32_t *csc = nullptr;
    uint8_t* csnap_mem = nullptr;    // 2 snapshot slots of the cache consoles
    uint32_t* csnap_sc = nullptr;
    int64_t *cx = nullptr, *ct = nullptr;
    int32_t *clives = nullptr, *cdraws = nullptr;
    uint64_t *cframes = nullptr, *cinstr = nullptr, *cff = nullptr;
    uint32_t* cbad = nullptr;
    uint8_t *obs = nullptr, *fin = nullptr, *term = nullptr, *trunc = nullptr;
    float* rew = nullptr;
    int32_t *info = nullptr, *ep_len = nullptr;
    double* ep_ret = nullptr;
    // per-stage HIP event timing of mh_step_async (mh_timing / mh_timing_read)
    bool timing = false;
    std::vector<hipEvent_t> events;    // MH_STAGES + 1 events per timed step
    size_t timed_steps = 0;
    ~MhEnv() { for (hipEvent_t e : events) (void)hipEventDestroy(e); }

    ResetArgs reset_args(int all) const {
        return ResetArgs{n, np, cfg, nk, ncp, mem, sc, ev, cmem, csc, cx, ct, clives, cdraws, cboot,
                         cframes, cinstr, cff, cbad, all};
    }
    StackArgs stack_args(int mode) const { return StackArgs{n, np, K, obs, fin, slot_env, fresh, ev, cobs, mode}; }
};

// k_stack4 when the stacks (and the reset cache) allow 16-byte accesses, else k_stack
static void launch_stack(const MhEnv* h, hipStream_t s, int mode) {
    const dim3 grid(h->np / 64, (OBS_PIX / 4 + 63) / 64);
    const bool al = ((((uintptr_t)h->obs) | ((uintptr_t)h->fin) | ((uintptr_t)h->cobs)) & 15) == 0;
    if (al) hipLaunchKernelGGL(k_stack4, grid, dim3(256), 0, s, h->stack_args(mode));
    else hipLaunchKernelGGL(k_stack, grid, dim3(256), 0, s, h->stack_args(mode));
}

static int launch_ram(const uint8_t* mem, uint32_t np, int n, const int32_t* slot_env, uint8_t* out, hipStream_t s) {
    const bool wide = (((uintptr_t)out) & 15) == 0;
    const dim3 grid((unsigned)(((size_t)n * 2048 / (wide ? 16 : 1) + 255) / 256));
    if (wide) hipLaunchKernelGGL(k_ram_out<uint4>, grid, dim3(256), 0, s, mem, np, n, slot_env, out);
    else hipLaunchKernelGGL(k_ram_out<uint8_t>, grid, dim3(256), 0, s, mem, np, n, slot_env, out);
    CK(hipGetLastError());
    return 0;
}

struct MhRaw {
    int n = 0, device = 0, cus = 0;
    EmuLaunch lr{};                // k_raw's launch shape
    uint32_t np = 0;
    DevBufs B;
    RomArgs R{};
    uint8_t *mem = nullptr, *screen = nullptr, *bk_mem = nullptr;
    uint32_t *sc = nullptr, *bk_sc = nullptr, *bad = nullptr, *instr = nullptr, *ff = nullptr;
};

extern "C" {

const char* mh_last_error(void) { return g_err.c_str(); }

MhEnv* mh_create(const uint8_t* rom, int64_t rom_len, int n, const int* levels, const uint8_t* lut,
                 int skip, int max_steps, double sticky, int noop_max, int maxpool, int frame_stack,
                 const uint64_t* rng, int device) {
    return mh_create_roms(rom, &rom_len, 1, nullptr, n, levels, lut, skip, max_steps, sticky, noop_max, maxpool,
                          frame_stack, rng, device);
}

MhEnv* mh_create_roms(const uint8_t* roms, const int64_t* rom_lens, int n_roms, const int32_t* env_rom, int n,
                      const int* levels, const uint8_t* lut, int skip, int max_steps, double sticky, int noop_max,
                      int maxpool, int frame_stack, const uint64_t* rng, int device) {
    g_err.clear();
    if (n < 1 || skip < 1 || skip > MAX_SKIP || frame_stack < 1 || frame_stack > 16 || noop_max < 0 ||
        max_steps < 1 || !(sticky >= 0.0 && sticky <= 1.0) || !levels || !lut || !rng || !roms || !rom_lens ||
        n_roms < 1 || n_roms > MAX_CHR_BANKS || (n_roms > 1 && !env_rom)) {
        g_err = "invalid arguments";
        return nullptr;
    }
    if ((uint32_t)n > MAX_ENVS) { g_err = "too many envs (at most 979,648)"; return nullptr; }
    // the cartridge image: ROM 0's PRG, then the CHR of every ROM; the ROMs must agree on PRG and mirroring
    std::vector<uint8_t> img;
    uint16_t nt[4];
    int64_t off = 0;
    for (int r = 0; r < n_roms; r++) {
        std::vector<uint8_t> one;
        uint16_t ntr[4];
        if (!load_cart(roms + off, rom_lens[r], one, ntr)) return nullptr;
        off += rom_lens[r];
        if (r == 0) {
            img.assign(one.begin(), one.begin() + 0x8000);
            memcpy(nt, ntr, sizeof(nt));
        } else if (memcmp(img.data(), one.data(), 0x8000) != 0 || memcmp(nt, ntr, sizeof(nt)) != 0) {
            g_err = "per-env ROMs must share PRG and mirroring (rom_mode variants differ in CHR only)";
            return nullptr;
        }
        img.insert(img.end(), one.begin() + 0x8000, one.begin() + 0xa000);
    }
    for (int i = 0; i < n && env_rom; i++)
        if (env_rom[i] < 0 || env_rom[i] >= n_roms) { g_err = "env ROM index out of range"; return nullptr; }
    CKN(hipSetDevice(device));
    MhEnv* h = new MhEnv();
    auto fail = [&]() -> MhEnv* { delete h; return nullptr; };
    bool good = true;
    h->n = n; h->K = frame_stack; h->device = device; h->np = pad64(n); h->cus = device_cus(device);
    h->cfg = Cfg{skip, max_steps, noop_max, maxpool ? 1 : 0, sticky};
    // distinct (level, ROM) keys in order of first appearance (levels: fastmario.cpp:584-593); a key has its
    // own boot state and reset-cache entries
    std::vector<int> lv, env_level(n);
    std::vector<uint8_t> key_bank;
    for (int i = 0; i < n; i++) {
        const int ri = env_rom ? env_rom[i] : 0;
        int li = -1;
        for (size_t k = 0; k < key_bank.size(); k++)
            if (lv[3 * k] == levels[3 * i] && lv[3 * k + 1] == levels[3 * i + 1] && lv[3 * k + 2] == levels[3 * i + 2] &&
                key_bank[k] == ri) li = (int)k;
        if (li < 0) {
            li = (int)key_bank.size();
            lv.insert(lv.end(), levels + 3 * i, levels + 3 * i + 3);
            key_bank.push_back((uint8_t)ri);
        }
        env_level[i] = li;
    }
    h->nl = (int)lv.size() / 3; h->nlp = pad64(h->nl);
    // Console slots grouped by key, ordered by (world, stage, area, ROM), envs of a key in index order, so that envs
    // of one level, which do about the same, run beside one another. State lives in slot order; actions, outputs, RAM and state dumps stay in env order (slot_env).
    std::vector<int32_t> slot_env(h->np, 0), env_slot(n);
    {
        std::vector<int> order(n);
        for (int i = 0; i < n; i++) order[i] = i;
        auto key_of = [&](int i) {
            const int k = env_level[i];
            return std::make_tuple(lv[3 * k], lv[3 * k + 1], lv[3 * k + 2], (int)key_bank[k], i);
        };
        std::sort(order.begin(), order.end(), [&](int a, int b) { return key_of(a) < key_of(b); });
        for (int s = 0; s < n; s++) { slot_env[s] = order[s]; env_slot[order[s]] = s; }
        for (uint32_t s = (uint32_t)n; s < h->np; s++) slot_env[s] = (int32_t)s;   // padding slots: never used
    }
    h->nk = noop_max + 1; h->nc = h->nl * h->nk; h->ncp = pad64(h->nc);
    auto& B = h->B;
    uint8_t* d_rom = B.alloc<uint8_t>(img.size(), good);
    uint8_t* d_lut = B.alloc<uint8_t>(256, good);
    uint32_t* d_recs = B.alloc<uint32_t>(REC_COUNT, good);
    h->T = B.alloc<AreaTables>(1, good);
    int* d_levels = B.alloc<int>(lv.size(), good);
    h->key_bank = B.alloc<uint8_t>(key_bank.size(), good);
    h->slot_env = B.alloc<int32_t>(h->np, good);
    h->mem = B.alloc<uint8_t>((size_t)MEM_ROWS * h->np, good);
    h->sc = B.alloc<uint32_t>((size_t)S_COUNT * h->np, good);
    h->ev = B.alloc<uint32_t>((size_t)E_COUNT * h->np, good);
    h->gray = B.alloc<uint8_t>((size_t)2 * GRAY_PIX * h->np, good);
    h->snap_mem = B.alloc<uint8_t>((size_t)2 * MEM_ROWS * h->np, good);
    h->snap_sc = B.alloc<uint32_t>((size_t)2 * S_COUNT * h->np, good);
    h->fresh = B.alloc<uint8_t>((size_t)OBS_PIX * h->np, good);
    h->ls = emu_launch(h->n, h->cus);
    if ((int)h->ls.grid.x > h->cus && h->cus > 0) {
        h->ls.grid = dim3((unsigned)h->cus);
        h->queue_first = (uint32_t)h->cus * WAVES_PER_BLOCK;
        h->queue = B.alloc<StepQueue>(1, good);
        h->queue_list = B.alloc<uint32_t>((size_t)2 * WORK_BUCKETS * h->np, good);
    }
    h->boot_mem = B.alloc<uint8_t>((size_t)MEM_ROWS * h->nlp, good);
    h->boot_sc = B.alloc<uint32_t>((size_t)S_COUNT * h->nlp, good);
    h->boot_gray = B.alloc<uint8_t>((size_t)GRAY_PIX * h->nlp, good);
    h->boot_obs = B.alloc<uint8_t>((size_t)OBS_PIX * h->nl, good);
    h->x0 = B.alloc<int64_t>(h->nl, good); h->t0 = B.alloc<int64_t>(h->nl, good);
    h->cmem = B.alloc<uint8_t>((size_t)MEM_ROWS * h->ncp, good);
    h->csc = B.alloc<uint32_t>((size_t)S_COUNT * h->ncp, good);
    h->cgray = B.alloc<uint8_t>((size_t)2 * GRAY_PIX * h->ncp, good);
    h->csnap_mem = B.alloc<uint8_t>((size_t)2 * MEM_ROWS * h->ncp, good);
    h->csnap_sc = B.alloc<uint32_t>((size_t)2 * S_COUNT * h->ncp, good);
    h->cobs = B.alloc<uint8_t>((size_t)OBS_PIX * h->nc, good);
    h->cboot = B.alloc<uint8_t>(h->nc, good);
    h->cx = B.alloc<int64_t>(h->nc, good); h->ct = B.alloc<int64_t>(h->nc, good);
    h->clives = B.alloc<int32_t>(h->nc, good); h->cdraws = B.alloc<int32_t>(h->nc, good);
    h->cframes = B.alloc<uint64_t>(h->nc, good); h->cinstr = B.alloc<uint64_t>(h->nc, good);
    h->cff = B.alloc<uint64_t>(h->nc, good);
    h->cbad = B.alloc<uint32_t>(h->nc, good);
    uint32_t* d_err = B.alloc<uint32_t>(1, good);
    if (!good) return fail();
    AreaTables T;
    area_tables(&T);
    if (!area_period_match(T)) { g_err = "INTER_AREA tables differ from the compiled-in periods"; return fail(); }
    // per-env words: level, RNG, lives = -1 (reset() installs the real start state)
    std::vector<uint32_t> ev((size_t)E_COUNT * h->np, 0);
    for (int i = 0; i < n; i++) {
        const size_t slot = (size_t)env_slot[i];
        auto w = [&](int k) -> uint32_t& { return ev[(size_t)k * h->np + slot]; };
        w(E_LEVEL) = (uint32_t)env_level[i];
        const uint64_t* r = rng + 6 * i;
        w(E_RNG_S3) = (uint32_t)(r[0] >> 32); w(E_RNG_S2) = (uint32_t)r[0];
        w(E_RNG_S1) = (uint32_t)(r[1] >> 32); w(E_RNG_S0) = (uint32_t)r[1];
        w(E_RNG_I3) = (uint32_t)(r[2] >> 32); w(E_RNG_I2) = (uint32_t)r[2];
        w(E_RNG_I1) = (uint32_t)(r[3] >> 32); w(E_RNG_I0) = (uint32_t)r[3];
        w(E_RNG_HAS32) = (uint32_t)r[4]; w(E_RNG_HALF) = (uint32_t)r[5];
        w(E_LIVES) = 0xffffffffu; w(E_SHOWS_BOOT) = 1; w(E_RESET_IDX) = 0xffffffffu;
    }
    if (!ok(hipMemcpy(d_rom, img.data(), img.size(), hipMemcpyHostToDevice), "upload rom") ||
        !ok(hipMemcpy(h->key_bank, key_bank.data(), key_bank.size(), hipMemcpyHostToDevice), "upload key banks") ||
        !ok(hipMemcpy(h->slot_env, slot_env.data(), slot_env.size() * 4, hipMemcpyHostToDevice), "upload slot map") ||
        !ok(hipMemcpy(d_lut, lut, 256, hipMemcpyHostToDevice), "upload lut") || !upload_records(d_recs, img) ||
        !ok(hipMemcpy(h->T, &T, sizeof(T), hipMemcpyHostToDevice), "upload tables") ||
        !ok(hipMemcpy(d_levels, lv.data(), lv.size() * sizeof(int), hipMemcpyHostToDevice), "upload levels") ||
        !ok(hipMemcpy(h->ev, ev.data(), ev.size() * 4, hipMemcpyHostToDevice), "upload env words"))
        return fail();
    if (h->queue) {   // the first step: every env in one bucket, in slot order
        std::vector<uint32_t> all(n);
        for (int i = 0; i < n; i++) all[i] = (uint32_t)i;
        StepQueue q{};
        q.next = h->queue_first;
        q.count[0][0] = (uint32_t)n;
        if (!ok(hipMemcpy(h->queue_list, all.data(), all.size() * 4, hipMemcpyHostToDevice), "upload step order") ||
            !ok(hipMemcpy(h->queue, &q, sizeof(q), hipMemcpyHostToDevice), "upload step queue"))
            return fail();
    }
    h->R.rom = d_rom; h->R.lut = d_lut; h->R.recs = d_recs; h->R.n_chr = n_roms;
    h->R.nt_bits = 0;
    for (int i = 0; i < 4; i++) h->R.nt_bits |= (nt[i] ? 1u : 0u) << i;
    // boot every level, build the reset cache
    const EmuLaunch lb = emu_launch(h->nl, h->cus), lc = emu_launch(h->nc, h->cus);
    BootArgs ba{h->R, h->nl, h->nlp, d_levels, h->key_bank, h->boot_mem, h->boot_sc, h->boot_gray, h->x0, h->t0, d_err};
    hipLaunchKernelGGL(k_boot, lb.grid, lb.block, 0, 0, ba);
    if (!ok(hipGetLastError(), "k_boot launch")) return fail();
    SmallObsArgs so{h->boot_gray, nullptr, nullptr, 1, h->boot_obs, h->nl, h->T};
    hipLaunchKernelGGL(k_small_obs, dim3((OBS_PIX + 255) / 256, h->nl), dim3(256), 0, 0, so);
    CacheArgs ca{h->R, h->cfg, h->key_bank, h->nl, h->nk, h->nc, h->nlp, h->ncp, h->boot_mem, h->boot_sc, h->x0, h->t0,
                 h->cmem, h->csc, h->cgray, h->csnap_mem, h->csnap_sc, h->cx, h->ct, h->clives, h->cdraws, h->cboot,
                 h->cframes, h->cinstr, h->cff, h->cbad};
    hipLaunchKernelGGL(k_cache, lc.grid, lc.block, 0, 0, ca);
    if (!ok(hipGetLastError(), "k_cache launch")) return fail();
    SmallObsArgs co{h->cgray, h->cboot, h->boot_obs, h->nk, h->cobs, h->nc, h->T};
    hipLaunchKernelGGL(k_small_obs, dim3((OBS_PIX + 255) / 256, h->nc), dim3(256), 0, 0, co);
    if (!ok(hipDeviceSynchronize(), "boot / reset cache")) return fail();
    uint32_t err = 0;
    if (!ok(hipMemcpy(&err, d_err, 4, hipMemcpyDeviceToHost), "boot status")) return fail();
    if (err) { g_err = "level boot did not finish (the ROM never started a level)"; return fail(); }
    return h;
}

// A buffer the kernels may write: device memory of the env's GPU or pinned host memory, aligned to `align`.
static bool kernel_writable(const MhEnv* h, const void* p, uintptr_t align, const char* name) {
    if (((uintptr_t)p & (align - 1)) != 0) {
        g_err = std::string(name) + ": not aligned to " + std::to_string(align) + " bytes";
        return false;
    }
    hipPointerAttribute_t at;
    const hipError_t e = hipPointerGetAttributes(&at, p);
    (void)hipGetLastError();   // a refused host pointer must not surface as the error of a later launch
    const bool dev = e == hipSuccess && at.type == hipMemoryTypeDevice && at.device == h->device;
    const bool pinned = e == hipSuccess && (at.type == hipMemoryTypeHost || at.type == hipMemoryTypeManaged);
    if (!dev && !pinned) {
        g_err = std::string(name) + ": neither device memory of GPU " + std::to_string(h->device) +
                " nor pinned host memory (pageable host memory cannot be written by the kernels)";
        return false;
    }
    return true;
}

int mh_set_buffers(MhEnv* h, uint8_t* obs, uint8_t* fin, float* rew, uint8_t* term, uint8_t* trunc,
                   int32_t* info, double* ep_ret, int32_t* ep_len) {
    if (!h || !obs || !fin || !rew || !term || !trunc || !info || !ep_ret || !ep_len) { g_err = "null buffer"; return -1; }
    if (!ok(hipSetDevice(h->device), "hipSetDevice")) return -1;
    if (!kernel_writable(h, obs, 4, "obs") || !kernel_writable(h, fin, 4, "final_obs") ||
        !kernel_writable(h, rew, 4, "rew") || !kernel_writable(h, term, 1, "term") ||
        !kernel_writable(h, trunc, 1, "trunc") || !kernel_writable(h, info, 4, "info") ||
        !kernel_writable(h, ep_ret, 8, "ep_ret") || !kernel_writable(h, ep_len, 4, "ep_len"))
        return -1;
    h->obs = obs; h->fin = fin; h->rew = rew; h->term = term; h->trunc = trunc; h->info = info;
    h->ep_ret = ep_ret; h->ep_len = ep_len;
    return 0;
}

int mh_reset(MhEnv* h, void* stream) {
    if (!h || !h->obs) { g_err = "buffers not set"; return -1; }
    CK(hipSetDevice(h->device));
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(k_reset, dim3(h->np / 64), dim3(64), 0, s, h->reset_args(1), (StepQueue*)nullptr, 0u);
    CK(hipGetLastError());
    launch_stack(h, s, 1);
    CK(hipGetLastError());
    return 0;
}

// Records event k of the current timed step (k = 0 .. MH_STAGES).
static int mark(MhEnv* h, hipStream_t s, int k) {
    if (!h->timing) return 0;
    size_t idx = h->timed_steps * (MH_STAGES + 1) + k;
    while (h->events.size() <= idx) {
        hipEvent_t e;
        CK(hipEventCreate(&e));
        h->events.push_back(e);
    }
    CK(hipEventRecord(h->events[idx], s));
    return 0;
}

int mh_step_async(MhEnv* h, const int64_t* d_actions, void* stream) {
    if (!h || !h->obs || !d_actions) { g_err = "buffers or actions not set"; return -1; }
    CK(hipSetDevice(h->device));
    hipStream_t s = (hipStream_t)stream;
    if (mark(h, s, 0)) return -1;
    StepArgs sa{h->R, h->cfg, h->n, h->np, h->mem, h->sc, h->ev, h->gray, h->snap_mem, h->snap_sc, d_actions,
                h->rew, h->term, h->trunc, h->info, h->ep_ret, h->ep_len, h->key_bank, h->slot_env, h->fresh,
                h->boot_obs};
    const EmuLaunch& ls = h->ls;
    hipLaunchKernelGGL(k_step, ls.grid, ls.block, 0, s, sa, h->queue, h->queue_list);
    CK(hipGetLastError());
    if (mark(h, s, 1)) return -1;
    if (mark(h, s, 2)) return -1;   // (a stage of its own until the observations moved into k_step: empty)
    hipLaunchKernelGGL(k_reset, dim3(h->np / 64), dim3(64), 0, s, h->reset_args(0), h->queue, h->queue_first);
    CK(hipGetLastError());
    if (mark(h, s, 3)) return -1;
    launch_stack(h, s, 0);
    CK(hipGetLastError());
    if (mark(h, s, 4)) return -1;
    if (h->timing) h->timed_steps++;
    return 0;
}

int mh_timing(MhEnv* h, int enable) {
    if (!h) return -1;
    h->timing = enable != 0;
    h->timed_steps = 0;
    // events for the first 128 timed steps now rather than inside the steps being timed: creating them
    // there cost ~1.5 ms per step of wall time in a 100-step run
    while (h->timing && h->events.size() < (size_t)128 * (MH_STAGES + 1)) {
        hipEvent_t e;
        CK(hipEventCreate(&e));
        h->events.push_back(e);
    }
    return 0;
}

int mh_timing_read(MhEnv* h, double* ms, int64_t* steps) {
    if (!h || !ms) return -1;
    CK(hipDeviceSynchronize());
    for (int k = 0; k < MH_STAGES; k++) ms[k] = 0.0;
    for (size_t t = 0; t < h->timed_steps; t++)
        for (int k = 0; k < MH_STAGES; k++) {
            float f = 0.f;
            CK(hipEventElapsedTime(&f, h->events[t * (MH_STAGES + 1) + k], h->events[t * (MH_STAGES + 1) + k + 1]));
            ms[k] += f;
        }
    if (steps) *steps = (int64_t)h->timed_steps;
    return 0;
}

int mh_step_wait(MhEnv* h, void* stream) {
    if (!h) return -1;
    CK(hipStreamSynchronize((hipStream_t)stream));
    return 0;
}

void mh_destroy(MhEnv* h) {
    if (!h) return;
    (void)hipSetDevice(h->device);
    (void)hipDeviceSynchronize();
    delete h;
}

static int64_t sum_words(const MhEnv* h, int lo_word, bool wide) {
    std::vector<uint32_t> lo(h->np), hi(h->np, 0);
    if (hipDeviceSynchronize() != hipSuccess) return -1;
    if (hipMemcpy(lo.data(), h->ev + (size_t)lo_word * h->np, h->np * 4, hipMemcpyDeviceToHost) != hipSuccess) return -1;
    if (wide && hipMemcpy(hi.data(), h->ev + (size_t)(lo_word + 1) * h->np, h->np * 4, hipMemcpyDeviceToHost) != hipSuccess) return -1;
    int64_t s = 0;
    for (int i = 0; i < h->n; i++) s += (int64_t)(lo[i] | ((uint64_t)hi[i] << 32));
    return s;
}
int64_t mh_frames(MhEnv* h) { return h ? sum_words(h, E_FRAMES_LO, true) : -1; }
int64_t mh_bad_ops(MhEnv* h) { return h ? sum_words(h, E_BAD, false) : -1; }
int64_t mh_instructions(MhEnv* h) { return h ? sum_words(h, E_INSTR_LO, true) : -1; }
int64_t mh_ff_instructions(MhEnv* h) { return h ? sum_words(h, E_FF_LO, true) : -1; }
int64_t mh_hack_redraws(MhEnv* h) { return h ? sum_words(h, E_HACK_REDRAWS, false) : -1; }
int mh_reemulations(MhEnv* h, int64_t* out) {
    if (!h || !out) { g_err = "null handle or buffer"; return -1; }
    for (int k = 0; k < 3; k++)
        if ((out[k] = sum_words(h, E_REEMU_ONE + k, false)) < 0) { g_err = "counter read failed"; return -1; }
    return 0;
}

int mh_env_ram(MhEnv* h, uint8_t* d_out, void* stream) {
    if (!h || !d_out) return -1;
    return launch_ram(h->mem, h->np, h->n, h->slot_env, d_out, (hipStream_t)stream);
}
int mh_env_canon(MhEnv* h, uint8_t* d_out, void* stream) {
    if (!h || !d_out) return -1;
    hipLaunchKernelGGL(k_canon, dim3(h->n), dim3(64), 0, (hipStream_t)stream, h->mem, h->sc, h->np, (const int32_t*)h->slot_env,
                       d_out);
    CK(hipGetLastError());
    return 0;
}
int mh_level_canon(MhEnv* h, uint8_t* d_out, void* stream) {
    if (!h || !d_out) return -1;
    hipLaunchKernelGGL(k_canon, dim3(h->nl), dim3(64), 0, (hipStream_t)stream, h->boot_mem, h->boot_sc, h->nlp, nullptr, d_out);
    CK(hipGetLastError());
    return 0;
}
int mh_level_obs(MhEnv* h, uint8_t* d_out, void* stream) {
    if (!h || !d_out) return -1;
    CK(hipMemcpyAsync(d_out, h->boot_obs, (size_t)OBS_PIX * h->nl, hipMemcpyDeviceToDevice, (hipStream_t)stream));
    return 0;
}
int mh_num_levels(MhEnv* h) { return h ? h->nl : -1; }

int64_t mh_state_bytes(void) { return (int64_t)MEM_ROWS + 4LL * S_COUNT; }
int64_t mh_env_bytes(MhEnv* h) {
    if (!h) return -1;
    int64_t per = 3LL * (MEM_ROWS + 4LL * S_COUNT) + 4LL * E_COUNT + 2LL * GRAY_PIX + OBS_PIX;
    if (h->queue) per += 2LL * WORK_BUCKETS * 4;
    return per * h->np / h->n;
}

MhRaw* mh_raw_create(const uint8_t* rom, int64_t rom_len, int n, int device) {
    g_err.clear();
    if (n < 1) { g_err = "invalid arguments"; return nullptr; }
    if ((uint32_t)n > MAX_ENVS) { g_err = "too many consoles (at most 979,648)"; return nullptr; }
    // (a wave runs one console whatever the variable says; an ill-formed value is an error, as it was)
    if (const char* f = getenv("MH_RAW_CONSOLES_PER_WAVE"); f && *f) {
        const int cpw = atoi(f);
        if (cpw != 1 && cpw != 2 && cpw != 4 && cpw != 8 && cpw != 16) {
            g_err = "MH_RAW_CONSOLES_PER_WAVE must be 1, 2, 4, 8 or 16";
            return nullptr;
        }
    }
    std::vector<uint8_t> img;
    uint16_t nt[4];
    if (!load_cart(rom, rom_len, img, nt)) return nullptr;
    CKN(hipSetDevice(device));
    MhRaw* h = new MhRaw();
    bool good = true;
    h->n = n; h->np = pad64(n); h->device = device; h->cus = device_cus(device);
    h->lr = emu_launch(n, h->cus);
    auto& B = h->B;
    uint8_t* d_rom = B.alloc<uint8_t>(0xa000, good);
    uint8_t* d_lut = B.alloc<uint8_t>(256, good);
    uint32_t* d_recs = B.alloc<uint32_t>(REC_COUNT, good);
    h->mem = B.alloc<uint8_t>((size_t)MEM_ROWS * h->np, good);
    h->bk_mem = B.alloc<uint8_t>((size_t)MEM_ROWS * h->np, good);
    h->sc = B.alloc<uint32_t>((size_t)S_COUNT * h->np, good);
    h->bk_sc = B.alloc<uint32_t>((size_t)S_COUNT * h->np, good);
    h->screen = B.alloc<uint8_t>((size_t)GRAY_PIX * h->np, good);
    h->bad = B.alloc<uint32_t>(h->np, good);
    h->instr = B.alloc<uint32_t>(h->np, good);
    h->ff = B.alloc<uint32_t>(h->np, good);
    if (!good) { delete h; return nullptr; }
    uint8_t ident[256];
    for (int i = 0; i < 256; i++) ident[i] = (uint8_t)i;
    if (!ok(hipMemcpy(d_rom, img.data(), 0xa000, hipMemcpyHostToDevice), "upload rom") ||
        !ok(hipMemcpy(d_lut, ident, 256, hipMemcpyHostToDevice), "upload lut") || !upload_records(d_recs, img)) {
        delete h;
        return nullptr;
    }
    h->R.rom = d_rom; h->R.lut = d_lut; h->R.recs = d_recs; h->R.n_chr = 1;
    h->R.nt_bits = 0;
    for (int i = 0; i < 4; i++) h->R.nt_bits |= (nt[i] ? 1u : 0u) << i;
    RawArgs ra{h->R, h->n, h->np, h->mem, h->sc, h->screen, nullptr, 0, h->bad, h->instr, h->ff, 1};
    hipLaunchKernelGGL(k_raw, h->lr.grid, h->lr.block, 0, 0, ra);
    if (!ok(hipDeviceSynchronize(), "raw power-on")) { delete h; return nullptr; }
    return h;
}
int mh_raw_frame(MhRaw* h, const uint8_t* d_buttons, int render, void* stream) {
    if (!h || !d_buttons) return -1;
    RawArgs ra{h->R, h->n, h->np, h->mem, h->sc, h->screen, d_buttons, render, h->bad, h->instr, h->ff, 0};
    hipLaunchKernelGGL(k_raw, h->lr.grid, h->lr.block, 0, (hipStream_t)stream, ra);
    CK(hipGetLastError());
    return 0;
}
int mh_raw_ram(MhRaw* h, uint8_t* d_out, void* stream) {
    if (!h || !d_out) return -1;
    return launch_ram(h->mem, h->np, h->n, nullptr, d_out, (hipStream_t)stream);
}
int mh_raw_screen(MhRaw* h, uint8_t* d_out, void* stream) {
    if (!h || !d_out) return -1;
    CK(hipMemcpyAsync(d_out, h->screen, (size_t)h->n * GRAY_PIX, hipMemcpyDeviceToDevice, (hipStream_t)stream));
    return 0;
}
int mh_raw_screen_rgb(MhRaw* h, const uint8_t* d_rgb64, uint8_t* d_out, void* stream) {
    if (!h || !d_rgb64 || !d_out) { g_err = "null handle or buffer"; return -1; }
    hipLaunchKernelGGL(k_frames_rgb, dim3(h->n, GRAY_PIX / 4 / RGB_WORDS), dim3(256), 0, (hipStream_t)stream, h->screen, d_rgb64,
                       d_out, (((uintptr_t)d_out) & 3) == 0);
    CK(hipGetLastError());
    return 0;
}
int mh_raw_canon(MhRaw* h, uint8_t* d_out, void* stream) {
    if (!h || !d_out) return -1;
    hipLaunchKernelGGL(k_canon, dim3(h->n), dim3(64), 0, (hipStream_t)stream, h->mem, h->sc, h->np, nullptr, d_out);
    CK(hipGetLastError());
    return 0;
}
int mh_raw_backup(MhRaw* h, void* stream) {
    if (!h) return -1;
    CK(hipMemcpyAsync(h->bk_mem, h->mem, (size_t)MEM_ROWS * h->np, hipMemcpyDeviceToDevice, (hipStream_t)stream));
    CK(hipMemcpyAsync(h->bk_sc, h->sc, (size_t)S_COUNT * h->np * 4, hipMemcpyDeviceToDevice, (hipStream_t)stream));
    return 0;
}
int mh_raw_restore(MhRaw* h, void* stream) {
    if (!h) return -1;
    CK(hipMemcpyAsync(h->mem, h->bk_mem, (size_t)MEM_ROWS * h->np, hipMemcpyDeviceToDevice, (hipStream_t)stream));
    CK(hipMemcpyAsync(h->sc, h->bk_sc, (size_t)S_COUNT * h->np * 4, hipMemcpyDeviceToDevice, (hipStream_t)stream));
    return 0;
}
static int64_t raw_sum(MhRaw* h, uint32_t* d) {
    std::vector<uint32_t> v(h->np);
    if (hipDeviceSynchronize() != hipSuccess) return -1;
    if (hipMemcpy(v.data(), d, h->np * 4, hipMemcpyDeviceToHost) != hipSuccess) return -1;
    int64_t s = 0;
    for (int i = 0; i < h->n; i++) s += v[i];
    return s;
}
int64_t mh_raw_bad_ops(MhRaw* h) { return h ? raw_sum(h, h->bad) : -1; }
int64_t mh_raw_instructions(MhRaw* h) { return h ? raw_sum(h, h->instr) : -1; }
int64_t mh_raw_ff_instructions(MhRaw* h) { return h ? raw_sum(h, h->ff) : -1; }
void mh_raw_destroy(MhRaw* h) {
    if (!h) return;
    (void)hipSetDevice(h->device);
    (void)hipDeviceSynchronize();
    delete h;
}

// mh_resize's tables: one copy per device, allocated on the device's first call and kept until the process ends.
static std::mutex g_tables_mu;
static std::map<int, AreaTables*> g_tables;

int mh_resize(const uint8_t* d_src, uint8_t* d_dst, int n, void* stream) {
    if (!d_src || !d_dst || n < 1 || n > MH_RESIZE_MAX_IMAGES) { g_err = "invalid arguments (n must be 1..65535)"; return -1; }
    int dev = 0;
    CK(hipGetDevice(&dev));
    AreaTables* d_T = nullptr;
    {
        std::lock_guard<std::mutex> lk(g_tables_mu);
        auto it = g_tables.find(dev);
        if (it == g_tables.end()) {
            AreaTables T;
            area_tables(&T);
            CK(hipMalloc(&d_T, sizeof(T)));
            if (!ok(hipMemcpy(d_T, &T, sizeof(T), hipMemcpyHostToDevice), "upload tables")) { (void)hipFree(d_T); return -1; }
            g_tables[dev] = d_T;
        } else {
            d_T = it->second;
        }
    }
    hipLaunchKernelGGL(k_resize_images, dim3((OBS_PIX + 255) / 256, n), dim3(256), 0, (hipStream_t)stream, d_src, d_dst, n, d_T);
    CK(hipGetLastError());
    return 0;
}

// The policy entry points' buffers: memory of the current GPU (device, or pinned host memory it maps); anything
// else (pageable host memory, another GPU's memory) is refused before a kernel could fault on it.
static bool on_gpu(const void* p, const char* name) {
    int dev = 0;
    if (!ok(hipGetDevice(&dev), "hipGetDevice")) return false;
    hipPointerAttribute_t at;
    const hipError_t e = hipPointerGetAttributes(&at, p);
    (void)hipGetLastError();   // a refused pointer must not surface as the error of a later launch
    const bool good = e == hipSuccess && ((at.type == hipMemoryTypeDevice && at.device == dev) ||
                                          at.type == hipMemoryTypeHost || at.type == hipMemoryTypeManaged);
    if (!good) g_err = std::string(name) + ": not memory of GPU " + std::to_string(dev);
    return good;
}

int mh_policy_conv1(const uint8_t* d_obs, const void* d_w, const void* d_b, void* d_out, int64_t n, void* stream) {
    if (!d_obs || !d_w || !d_b || !d_out || n < 1) { g_err = "invalid arguments (n >= 1)"; return -1; }
    if ((((uintptr_t)d_obs) & 3) || (((uintptr_t)d_w) & 15) || (((uintptr_t)d_out) & 1) || (((uintptr_t)d_b) & 1)) {
        g_err = "obs must be 4-byte, weight 16-byte and bias / out 2-byte aligned";
        return -1;
    }
    if (!on_gpu(d_obs, "obs") || !on_gpu(d_w, "weight") || !on_gpu(d_b, "bias") || !on_gpu(d_out, "out")) return -1;
    int dev = 0, cus = 0;
    CK(hipGetDevice(&dev));
    CK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const int64_t blocks = std::min<int64_t>(n, (int64_t)std::max(cus, 1) * 2);   // what a CU holds: 2
    hipLaunchKernelGGL(k_policy_conv1, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, d_obs,
                       (const uint16_t*)d_w, (const uint16_t*)d_b, (uint16_t*)d_out, n, (((uintptr_t)d_out) & 7) == 0);
    CK(hipGetLastError());
    return 0;
}

int mh_policy_conv(const void* d_x, const void* d_w, const void* d_b, void* d_out, int64_t n, int layer, void* stream) {
    if (!d_x || !d_w || !d_b || !d_out || n < 1 || (layer != 2 && layer != 3)) {
        g_err = "invalid arguments (n >= 1, layer 2 or 3)";
        return -1;
    }
    if ((((uintptr_t)d_x) & 15) || (((uintptr_t)d_w) & 15) || (((uintptr_t)d_out) & 1) || (((uintptr_t)d_b) & 1)) {
        g_err = "input and weight must be 16-byte, bias and out 2-byte aligned";
        return -1;
    }
    if (!on_gpu(d_x, "input") || !on_gpu(d_w, "weight") || !on_gpu(d_b, "bias") || !on_gpu(d_out, "out")) return -1;
    int dev = 0, cus = 0;
    CK(hipGetDevice(&dev));
    CK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    cus = std::max(cus, 1);
    hipStream_t s = (hipStream_t)stream;
    const uint16_t *x = (const uint16_t*)d_x, *w = (const uint16_t*)d_w, *b = (const uint16_t*)d_b;
    uint16_t* y = (uint16_t*)d_out;
    const int wide = (((uintptr_t)d_out) & 7) == 0;
    auto run = [&](auto kernel, int images) {   // 2 blocks a CU
        const int64_t blocks = std::min<int64_t>((n + images - 1) / images, (int64_t)cus * 2);
        hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), 0, s, x, w, b, y, n, wide);
    };
    if (layer == 2 && n >= (int64_t)cus * CONV2_IMGS) run(k_policy_conv<32, 4, 2, 20, 9, CONV2_IMGS>, CONV2_IMGS);
    else if (layer == 2) run(k_policy_conv<32, 4, 2, 20, 9, 1>, 1);
    else if (n >= (int64_t)cus * CONV3_IMGS) run(k_policy_conv<64, 3, 1, 9, 7, CONV3_IMGS>, CONV3_IMGS);
    else run(k_policy_conv<64, 3, 1, 9, 7, 1>, 1);
    CK(hipGetLastError());
    return 0;
}

int mh_policy_conv12(const uint8_t* d_obs, const void* d_w1, const void* d_b1, const void* d_w2, const void* d_b2, void* d_out,
                     int64_t n, void* stream) {
    if (!d_obs || !d_w1 || !d_b1 || !d_w2 || !d_b2 || !d_out || n < 1) { g_err = "invalid arguments (n >= 1)"; return -1; }
    if ((((uintptr_t)d_obs) & 3) || ((((uintptr_t)d_w1) | ((uintptr_t)d_w2)) & 15) || (((uintptr_t)d_out) & 7) ||
        ((((uintptr_t)d_b1) | ((uintptr_t)d_b2)) & 1)) {
        g_err = "obs must be 4-byte, weights 16-byte, out 8-byte and biases 2-byte aligned";
        return -1;
    }
    if (!on_gpu(d_obs, "obs") || !on_gpu(d_w1, "weight") || !on_gpu(d_b1, "bias") || !on_gpu(d_w2, "weight") ||
        !on_gpu(d_b2, "bias") || !on_gpu(d_out, "out"))
        return -1;
    int dev = 0, cus = 0;
    CK(hipGetDevice(&dev));
    CK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const int64_t blocks = std::min<int64_t>(n, std::max(cus, 1));   // a CU holds one (its LDS)
    hipLaunchKernelGGL(k_policy_conv12, dim3((unsigned)blocks), dim3(512), 0, (hipStream_t)stream, d_obs, (const uint16_t*)d_w1,
                       (const uint16_t*)d_b1, (const uint16_t*)d_w2, (const uint16_t*)d_b2, (uint16_t*)d_out, n);
    CK(hipGetLastError());
    return 0;
}

int mh_policy_pack(const float* const* params, const int64_t* strides, void* d_out, void* stream) {
    if (!params || !strides || !d_out) { g_err = "invalid arguments"; return -1; }
    if (((uintptr_t)d_out) & 15) { g_err = "out must be 16-byte aligned"; return -1; }
    PackArgs a{};
    for (int i = 0; i < 8; i++) {
        if (!params[i] || (((uintptr_t)params[i]) & 3)) { g_err = "a parameter is null or not 4-byte aligned"; return -1; }
        if (!on_gpu(params[i], "parameter")) return -1;
    }
    if (!on_gpu(d_out, "out")) return -1;
    for (int k = 0; k < 3; k++) {
        a.w[k] = params[2 * k];
        for (int d = 0; d < 4; d++) a.st[k][d] = strides[4 * k + d];
    }
    for (int k = 0; k < 4; k++) a.b[k] = params[2 * k + 1];
    a.fc = params[6];
    a.out = (uint16_t*)d_out;
    hipLaunchKernelGGL(k_policy_pack, dim3(FC_OUT + PACK_SMALL), dim3(256), 0, (hipStream_t)stream, a);
    CK(hipGetLastError());
    return 0;
}

int mh_policy_heads(const void* d_h, const float* w_pi, const float* b_pi, const float* w_vf, const float* b_vf, float* logits,
                    float* value, int64_t n, int actions, void* stream) {
    if (!d_h || !w_pi || !b_pi || !w_vf || !b_vf || !logits || !value || n < 1 || actions < 1 || actions > 1024) {
        g_err = "invalid arguments (n >= 1, 1 <= actions <= 1024)";
        return -1;
    }
    if (((uintptr_t)d_h) & 15) { g_err = "h must be 16-byte aligned"; return -1; }
    for (const void* p : {(const void*)w_pi, (const void*)b_pi, (const void*)w_vf, (const void*)b_vf, (const void*)logits, (const void*)value}) {
        if (((uintptr_t)p) & 3) { g_err = "parameters and outputs must be 4-byte aligned"; return -1; }
        if (!on_gpu(p, "parameter or output")) return -1;
    }
    if (!on_gpu(d_h, "h")) return -1;
    int dev = 0, cus = 0;
    CK(hipGetDevice(&dev));
    CK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const int64_t blocks = std::min<int64_t>((n + 3) / 4, (int64_t)std::max(cus, 1) * 8);
    hipLaunchKernelGGL(k_policy_heads, dim3((unsigned)blocks, (unsigned)(actions / 8 + 1)), dim3(256), 0, (hipStream_t)stream,
                       (const uint16_t*)d_h, w_pi, b_pi, w_vf, b_vf, logits, value, n, actions);
    CK(hipGetLastError());
    return 0;
}

int mh_gae(const float* rew, const float* val, const uint8_t* start, const float* next_val, const uint8_t* next_start,
           int64_t T, int64_t n, float gamma, float gamma_lam, float* adv, float* ret, void* stream) {
    if (!rew || !val || !start || !next_val || !next_start || !adv || !ret || T < 1 || n < 1 || n > ((int64_t)1 << 36)) {
        g_err = "invalid arguments (T >= 1, 1 <= n <= 2^36)";
        return -1;
    }
    for (const void* p : {(const void*)rew, (const void*)val, (const void*)next_val, (const void*)adv, (const void*)ret})
        if (((uintptr_t)p) & 3) { g_err = "the float rows must be 4-byte aligned"; return -1; }
    if (!on_gpu(rew, "rew") || !on_gpu(val, "val") || !on_gpu(start, "start") || !on_gpu(next_val, "next_val") ||
        !on_gpu(next_start, "next_start") || !on_gpu(adv, "adv") || !on_gpu(ret, "ret"))
        return -1;
    hipLaunchKernelGGL(k_gae, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, (hipStream_t)stream, rew, val, start, next_val,
                       next_start, T, n, gamma, gamma_lam, adv, ret);
    CK(hipGetLastError());
    return 0;
}

int mh_policy_input(const uint8_t* d_obs, void* d_out, int64_t n, int k, void* stream) {
    if (!d_obs || !d_out || n < 1 || (k != 1 && k != 2 && k != 4 && k != 8)) {
        g_err = "invalid arguments (n >= 1, k in 1, 2, 4, 8)";
        return -1;
    }
    if ((((uintptr_t)d_obs) & 3) || (((uintptr_t)d_out) & 3)) { g_err = "obs and out must be 4-byte aligned"; return -1; }
    if (!on_gpu(d_obs, "obs") || !on_gpu(d_out, "out")) return -1;
    const int64_t groups = n * (OBS_PIX / 4);
    const dim3 grid((unsigned)((groups + 255) / 256));
    hipStream_t s = (hipStream_t)stream;
    uint32_t* o = (uint32_t*)d_out;
    if (k == 1) {   // one channel: two pixels per 32-bit word
        hipLaunchKernelGGL(k_policy_input_k1, grid, dim3(256), 0, s, d_obs, o, groups);
    } else if (k == 2) {
        hipLaunchKernelGGL(k_policy_input<2>, grid, dim3(256), 0, s, d_obs, o, groups);
    } else if (k == 4) {
        hipLaunchKernelGGL(k_policy_input<4>, grid, dim3(256), 0, s, d_obs, o, groups);
    } else {
        hipLaunchKernelGGL(k_policy_input<8>, grid, dim3(256), 0, s, d_obs, o, groups);
    }
    CK(hipGetLastError());
    return 0;
}

// ---- the allocation-free resize (mh_resize_noalloc)
// Its filter tables live in `scratch`, a file-scope device array statically initialised with the tables the
// compiler computes (kAreaTables, area_taps's double operations at compile time): every GPU the library runs on
// holds one copy, loaded with the code object, at its own address, until the process ends. No kernel writes it
// and every call only reads it, so calls on one GPU never race over it and a first call under stream capture
// records nothing but the resize. The first call on a device looks up that device's address of the array
// (hipGetSymbolAddress; the array's name in host code is only a host-side stand-in, not a device address); the
// first call in the process checks once that the compile-time tables are, bit for bit, the run-time tables that
// mh_resize copies to the device (area_tables()).
static_assert(sizeof(AreaTables) == 8736, "the scratch array holds 8,736 B on every GPU");
static __device__ __align__(256) AreaTables scratch[1] = {kAreaTables};
constexpr int MH_MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static int g_scratch_checked;                          // 0 not yet, 1 the tables match, -1 they differ
static AreaTables* g_scratch_tables[MH_MAX_DEVICES];   // the device address of `scratch`, per device

static AreaTables* scratch_tables() {
    int dev = 0;
    if (!ok(hipGetDevice(&dev), "hipGetDevice")) return nullptr;
    if (dev < 0 || dev >= MH_MAX_DEVICES) { g_err = "device index beyond the allocation-free path's table"; return nullptr; }
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_checked) {
        AreaTables host;
        area_tables(&host);
        g_scratch_checked = area_tables_equal(host, kAreaTables) ? 1 : -1;
    }
    if (g_scratch_checked < 0) { g_err = "compile-time INTER_AREA tables differ from the run-time ones"; return nullptr; }
    if (!g_scratch_tables[dev]) {
        void* p = nullptr;
        if (!ok(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)")) return nullptr;
        g_scratch_tables[dev] = (AreaTables*)p;
    }
    return g_scratch_tables[dev];
}

int mh_resize_noalloc(const uint8_t* d_src, uint8_t* d_dst, int n, void* stream) {
    if (!d_src || !d_dst) { g_err = "null image buffer"; return -1; }
    if (n < 1 || n > MH_RESIZE_MAX_IMAGES) {
        g_err = "mh_resize_noalloc: n = " + std::to_string(n) + " images; one call takes 1 .. 65535";
        return -1;
    }
    hipStream_t s = (hipStream_t)stream;
    AreaTables* T = scratch_tables();
    if (!T) return -1;
    hipLaunchKernelGGL(k_resize_images, dim3((OBS_PIX + 255) / 256, n), dim3(256), 0, s, d_src, d_dst, n, (const AreaTables*)T);
    CK(hipGetLastError());
    return 0;
}

static bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

int mh_replay_add(uint8_t* frames, uint8_t* age, int16_t* act, float* rew, uint8_t* flags, int64_t* ptr,
                  uint8_t* new_ep, int n_envs, int capacity, int frame_bytes, int k, const uint8_t* obs,
                  const uint8_t* next_obs, const int64_t* action, const float* reward, const uint8_t* done,
                  const uint8_t* truncated, void* stream) {
    if (!frames || !age || !act || !rew || !flags || !ptr || !new_ep || !obs || !next_obs || !action || !reward ||
        !done || !truncated || n_envs < 1 || capacity < 2 || k < 1 || frame_bytes < 16 || frame_bytes % 16) {
        g_err = "invalid arguments"; return -1;
    }
    if (k > capacity) { g_err = "stack depth k exceeds the ring capacity"; return -1; }
    if (!aligned16(frames) || !aligned16(obs) || !aligned16(next_obs)) { g_err = "frame buffers must be 16-byte aligned"; return -1; }
    ReplayAddArgs A{ReplayRing{frames, age, act, rew, flags, ptr, new_ep, n_envs, capacity, (uint32_t)frame_bytes},
                    obs, next_obs, k, action, reward, done, truncated};
    hipLaunchKernelGGL(k_replay_add, dim3(n_envs), dim3(256), 0, (hipStream_t)stream, A);
    CK(hipGetLastError());
    return 0;
}

int mh_replay_candidates(const int64_t* ptr, int n_envs, int capacity, int k, int64_t n_step, int64_t* cand, int64_t* count,
                         void* stream) {
    if (!ptr || !cand || !count || n_envs < 1 || capacity < 2 || k < 1) { g_err = "invalid arguments"; return -1; }
    hipLaunchKernelGGL(k_replay_candidates, dim3(1), dim3(DRAW_THREADS), 0, (hipStream_t)stream, ptr, n_envs, capacity, k,
                       n_step, cand, count);
    CK(hipGetLastError());
    return 0;
}

int mh_replay_draw(const int64_t* ptr, const uint8_t* flags, int n_envs, int capacity, int k, int64_t n_step, const int64_t* cand,
                   const int64_t* pick, const double* u, const int64_t* rows, int64_t n, int64_t* env, int64_t* pos,
                   uint8_t* open, int64_t* rows_out, int64_t* count, void* stream) {
    if (!ptr || !flags || !cand || !pick || !u || !env || !pos || !open || !rows_out || !count || rows_out == rows ||
        n_envs < 1 || capacity < 2 || k < 1 || n < 1 || n > ((int64_t)1 << 38)) {
        g_err = "invalid arguments"; return -1;
    }
    DrawArgs A{ptr, flags, n_envs, capacity, k, n_step, cand, pick, u, rows, n, env, pos, open, rows_out, count};
    hipLaunchKernelGGL(k_replay_draw, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, A);
    hipLaunchKernelGGL(k_replay_open, dim3(1), dim3(DRAW_THREADS), 0, (hipStream_t)stream, A);
    CK(hipGetLastError());
    return 0;
}

int mh_replay_gather(const uint8_t* frames, const uint8_t* age, const int16_t* act, const float* rew,
                     const uint8_t* flags, int n_envs, int capacity, int frame_bytes, int k, const int64_t* env,
                     const int64_t* pos, int batch, int n_step, const float* gamma_pow, uint8_t* obs,
                     uint8_t* next_obs, int64_t* action, float* reward, float* discount, float* terminal,
                     int64_t* steps, int32_t* err, void* stream) {
    if (!frames || !age || !act || !rew || !flags || !env || !pos || !gamma_pow || !obs || !next_obs || !action ||
        !reward || !discount || !terminal || !steps || !err || n_envs < 1 || capacity < 2 || k < 1 ||
        frame_bytes < 16 || frame_bytes % 16 || batch < 0 || n_step < 0) {
        g_err = "invalid arguments"; return -1;
    }
    // a stack reaches k - 1 slots back from its newest one: deeper than the ring it would wrap onto itself
    if (k > capacity) { g_err = "stack depth k exceeds the ring capacity"; return -1; }
    if (!aligned16(frames) || !aligned16(obs) || !aligned16(next_obs)) { g_err = "frame buffers must be 16-byte aligned"; return -1; }
    if (batch == 0) return 0;
    ReplayGatherArgs A{ReplayRing{(uint8_t*)frames, (uint8_t*)age, (int16_t*)act, (float*)rew, (uint8_t*)flags,
                                  nullptr, nullptr, n_envs, capacity, (uint32_t)frame_bytes},
                       k, n_step, batch, env, pos, gamma_pow, obs, next_obs, action, reward, discount, terminal,
                       steps, err};
    hipLaunchKernelGGL(k_replay_gather, dim3(batch), dim3(REPLAY_GATHER_THREADS), 0, (hipStream_t)stream, A);
    CK(hipGetLastError());
    return 0;
}

}  // extern "C"
