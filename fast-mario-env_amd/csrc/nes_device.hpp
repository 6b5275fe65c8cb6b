// Device-side NES console for gfx950: one console per wave.
//
// A wave runs one console. Its whole state is wave-uniform, the memory (RAM, VRAM, OAM, palette) in LDS while a kernel
// runs, and every branch of the emulation is a scalar branch. The registers stay in one vector register, word k in
// lane k (struct File): frame() holds the CPU's in scalar registers and calls the PPU's catch-up, the register
// accesses and the rare whole instruction as functions, which take the words they need out of the file and put back
// what they change. (With all of them as variables of one inlined frame loop, the ~45 words and the copies where its
// paths join did not fit the scalar registers: a loop iteration took 1,700 cycles, most of them spill code.) The 64
// lanes work together where there is data to spread over them: the pixels of a batch of render lines, the sprite
// evaluation, the sprite-0 hit's pixels, and the copies of memory. Measured against 16 consoles per wave in lockstep
// (each on four lanes, state in vector registers, RAM in global memory): k_step in mario_hip.hip.
//
// Layout in HBM:
//   MEM[e * MEM_ROWS + row]  one byte per row: RAM 0..2047, VRAM 2048..4095, OAM 4096..4351, PAL 4352..4383.
//                            (The host build, tests/hostbuild, interleaves its consoles: MEM[row * NP + e].)
//   SC[word * NP + e]        32-bit scalar registers of the CPU / PPU / joypads (enum Scalar), NP = the env count
//                            rounded up to a multiple of 64.
// PRG (32 KB) and CHR (8 KB) are read-only and shared by every env: each workgroup stages them in LDS.
//
// The machine follows the reference's nes-py-exact model (csrc/nes_core.hpp): instruction-atomic CPU
// with skip cycles, catch-up PPU advanced only at PPU register accesses / the NMI point / frame end,
// exact sprite-0 hit, nes-py's flag layout and bus quirks. Counters are kept relative to the current
// frame start (32-bit) instead of the reference's absolute int64 values; the 64-bit iteration count at
// the frame start is only needed for the OAM-DMA odd/even cycle (nes_core.hpp:194).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// The host build of this code (tests/hostbuild) runs a console on one lane, with a one-lane wave's intrinsics.
#ifndef MH_LANES_PER_ENV
#define MH_LANES_PER_ENV 64
#endif
// Pointers through which wave-uniform addresses of read-only data are loaded with scalar loads (the constant
// address space): data in device memory which no kernel writes.
#ifndef MH_SCALAR_CONST
#define MH_SCALAR_CONST __attribute__((address_space(4)))
#endif

namespace mh {

constexpr int ROW_RAM = 0, ROW_VRAM = 2048, ROW_OAM = 4096, ROW_PAL = 4352, MEM_ROWS = 4384;
// Most envs (consoles) of one instance, a limit of the interface: MEM_ROWS * np, np the padded count (a multiple of 64),
// stays below 2^32, and so do the host build's offsets and the output kernels' indexes.
constexpr uint32_t MAX_ENVS = (uint32_t)((0xffffffffull / MEM_ROWS) & ~63ull);
static_assert(MAX_ENVS == 979648 && (uint64_t)MEM_ROWS * MAX_ENVS <= 0xffffffffull, "the interface's limit");
constexpr int LANES = MH_LANES_PER_ENV;
static_assert(LANES == 1 || LANES == 64, "a console runs on a wave's 64 lanes, or on the host's one");
constexpr bool ON_GPU = LANES == 64;
// Emulator launch shape: blocks of up to 16 waves, one console each, one block per CU: four waves per SIMD, so that
// a wave's scalar loads, LDS reads and branches are covered by the others' instructions (a SIMD issues one scalar
// instruction per 4 cycles, whichever wave it is from).
constexpr int WAVES_PER_BLOCK = 16;
constexpr int EMU_WAVES_PER_SIMD = WAVES_PER_BLOCK / 4;
constexpr int LDS_LANES = ON_GPU ? WAVES_PER_BLOCK : 1;        // consoles sharing one block's LDS
// A console's share of LDS: its memory, then the renderer's words: the gray palette, and the sprite entries (8 a line)
// of the DRAW_LINES lines drawn at once.
constexpr int LDS_SP_WORDS = MEM_ROWS / 4;
constexpr int DRAW_LINES = 4;
constexpr int GP_PALETTE = 0, GP_SPRITES = 8, LDS_GP_REGION = GP_SPRITES + 8 * DRAW_LINES;
constexpr int LDS_ENV_WORDS = LDS_SP_WORDS + LDS_GP_REGION;
constexpr int FRAME_ITERS = 29781;                 // CPU iterations per nes-py Emulator::step
constexpr int LINE_END = 341;
constexpr int GRAY_PIX = 256 * 240;
// Byte offset of row `row` of console e in a memory block of np consoles
__host__ __device__ __forceinline__ size_t mem_offset(uint32_t np, uint32_t e, uint32_t row) {
    return ON_GPU ? (size_t)e * MEM_ROWS + row : (size_t)row * np + e;
}
// Console::ppu_flags bits: PPUMASK (show / hide-edge, bits 0-3) and PPUCTRL (bits 4-8) settings
enum : uint32_t { PF_SHOW_BG = 1, PF_SHOW_SPR = 2, PF_HIDE_EDGE_BG = 4, PF_HIDE_EDGE_SPR = 8, PF_LONG_SPR = 16,
                  PF_NMI_EN = 32, PF_BG_PAGE = 64, PF_SPR_PAGE = 128, PF_INC32 = 256 };
enum : uint8_t { FN = 0x01, FV = 0x02, FONE = 0x04, FB = 0x08, FD = 0x10, FI = 0x20, FZ = 0x40, FC = 0x80 };
// Error flags or-ed into a console's bad-op counter (every parity check requires a zero count):
// ERR_HACK_LIMIT  the env layer's busy-state loop hit its frame limit.
constexpr uint32_t ERR_HACK_LIMIT = 1u << 24, ERR_FLAGS = ERR_HACK_LIMIT;
enum : uint8_t { ST_PRE = 0, ST_RENDER = 1, ST_POST = 2, ST_VBLANK = 3 };

// Scalar words of one console, interleaved as SC[w * NP + e].
enum Scalar : int {
    S_ITER_LO = 0, S_ITER_HI, S_EXEC_REL, S_PC, S_SP, S_A, S_X, S_Y, S_P, S_ZERO_SKIP,
    S_JOY_STROBE0, S_JOY_STROBE1, S_JOY_BUTTONS0, S_JOY_BUTTONS1, S_JOY_BITS0, S_JOY_BITS1,
    S_PSTATE, S_EVEN, S_VBLANK, S_S0HIT, S_FIRST_WRITE, S_DATA_BUFFER, S_OAM_ADDR, S_FINE_X,
    S_SHOW_BG, S_SHOW_SPR, S_HIDE_EDGE_BG, S_HIDE_EDGE_SPR, S_LONG_SPR, S_NMI_EN, S_BG_PAGE, S_SPR_PAGE,
    S_NSL, S_SL_LO, S_SL_HI, S_PCYC, S_SCANLINE, S_V, S_T, S_INC, S_COUNT,
    // words of a running console's register file beside them: the PPUCTRL / PPUMASK settings and the joypads packed, the
    // PPU's position (relative to the frame start), derived state, and the counters of the frame being run
    F_PPU_FLAGS = S_COUNT, F_JOY, F_JOY_STROBE, F_PPU_CALLS, F_NMI_THRESH, F_NMI_CALL, F_PEND_LINE, F_PAL_DIRTY,
    F_QUIET, F_BAD, F_INSTR, F_FF, F_COUNT
};

// Base cycles per opcode (data table of nes_core.hpp:42-51; 0 = not an official opcode).
constexpr uint8_t kCycleData[256] = {
    7, 6, 0, 0, 0, 3, 5, 0, 3, 2, 2, 0, 0, 4, 6, 0, 2, 5, 0, 0, 0, 4, 6, 0, 2, 4, 0, 0, 0, 4, 7, 0,
    6, 6, 0, 0, 3, 3, 5, 0, 4, 2, 2, 0, 4, 4, 6, 0, 2, 5, 0, 0, 0, 4, 6, 0, 2, 4, 0, 0, 0, 4, 7, 0,
    6, 6, 0, 0, 0, 3, 5, 0, 3, 2, 2, 0, 3, 4, 6, 0, 2, 5, 0, 0, 0, 4, 6, 0, 2, 4, 0, 0, 0, 4, 7, 0,
    6, 6, 0, 0, 0, 3, 5, 0, 4, 2, 2, 0, 5, 4, 6, 0, 2, 5, 0, 0, 0, 4, 6, 0, 2, 4, 0, 0, 0, 4, 7, 0,
    0, 6, 0, 0, 3, 3, 3, 0, 2, 0, 2, 0, 4, 4, 4, 0, 2, 6, 0, 0, 4, 4, 4, 0, 2, 5, 2, 0, 0, 5, 0, 0,
    2, 6, 2, 0, 3, 3, 3, 0, 2, 2, 2, 0, 4, 4, 4, 0, 2, 5, 0, 0, 4, 4, 4, 0, 2, 4, 2, 0, 4, 4, 4, 0,
    2, 6, 0, 0, 3, 3, 5, 0, 2, 2, 2, 0, 4, 4, 6, 0, 2, 5, 0, 0, 0, 4, 6, 0, 2, 4, 0, 0, 0, 4, 7, 0,
    2, 6, 0, 0, 3, 3, 5, 0, 2, 2, 2, 2, 4, 4, 6, 0, 2, 5, 0, 0, 0, 4, 6, 0, 2, 4, 0, 0, 0, 4, 7, 0,
};

// ---------------------------------------------------------------- decode table
// One word per opcode with everything the fast instruction path needs, generated from the
// reference's decode cascade (implied, branch, type 1, type 2, type 0; nes_core.hpp:619-1163):
// addressing mode, page-cross rule, data read, ALU operation, source and destination register,
// stack / control-flow operation, flag class and base cycles. Invalid opcodes keep their addressing
// (type 0 with an invalid operation still consumes its operand bytes and page-cross cycle).
namespace dec {
enum : uint32_t { M_NONE = 0, M_IMM, M_ZP, M_ZPX, M_ZPY, M_ABS, M_ABSX, M_ABSY, M_INDX, M_INDY };
enum : uint32_t { OP_PASS = 0, OP_ORA, OP_AND, OP_EOR, OP_ADC, OP_SBC, OP_CMP, OP_BIT, OP_ASL, OP_ROL, OP_LSR,
                  OP_ROR, OP_INC, OP_DEC, OP_FLAG, OP_NOP };
enum : uint32_t { R_M = 0, R_A, R_X, R_Y, R_SP };                       // R_M: the data operand
enum : uint32_t { D_NONE = 0, D_A, D_X, D_Y, D_SP, D_MEM };
enum : uint32_t { X_NONE = 0, X_BRK, X_JSR, X_RTS, X_RTI, X_PHA, X_PHP, X_PLA, X_PLP, X_JMP, X_JMPI, X_BRANCH };
enum : uint32_t { FL_NONE = 0, FL_NZ, FL_NZC, FL_NZCV, FL_BIT, FL_OP };
constexpr uint32_t PEN = 1u << 4, RD = 1u << 5, OK = 1u << 7;
constexpr int ALU_SH = 8, SRC_SH = 12, DST_SH = 15, X_SH = 18, FL_SH = 22, FOP_SH = 25, CYC_SH = 28;

constexpr uint32_t mk(uint32_t am, bool pen, bool rd, bool ok, uint32_t alu, uint32_t src, uint32_t dst,
                      uint32_t x, uint32_t fl, uint32_t fop = 0) {
    return am | (pen ? PEN : 0u) | (rd ? RD : 0u) | (ok ? OK : 0u) | alu << ALU_SH | src << SRC_SH |
           dst << DST_SH | x << X_SH | fl << FL_SH | fop << FOP_SH;
}
constexpr uint32_t entry(int op) {
    const int cc = op & 3, bbb = (op >> 2) & 7, fn = op >> 5;
    const uint32_t cyc = (uint32_t)kCycleData[op] << CYC_SH;
    switch (op) {   // the implied table (nes_core.hpp:630-690); flag ops: fop 0 CLC 1 SEC 2 CLI 3 SEI 4 CLV 5 CLD 6 SED
        case 0x00: return mk(M_NONE, false, false, true, OP_NOP, R_M, D_NONE, X_BRK, FL_NONE) | cyc;
        case 0x08: return mk(M_NONE, false, false, true, OP_NOP, R_M, D_NONE, X_PHP, FL_NONE) | cyc;
        case 0x18: return mk(M_NONE, false, false, true, OP_FLAG, R_M, D_NONE, X_NONE, FL_OP, 0) | cyc;
        case 0x20: return mk(M_ABS, false, false, true, OP_NOP, R_M, D_NONE, X_JSR, FL_NONE) | cyc;
        case 0x28: return mk(M_NONE, false, false, true, OP_NOP, R_M, D_NONE, X_PLP, FL_NONE) | cyc;
        case 0x38: return mk(M_NONE, false, false, true, OP_FLAG, R_M, D_NONE, X_NONE, FL_OP, 1) | cyc;
        case 0x40: return mk(M_NONE, false, false, true, OP_NOP, R_M, D_NONE, X_RTI, FL_NONE) | cyc;
        case 0x48: return mk(M_NONE, false, false, true, OP_NOP, R_M, D_NONE, X_PHA, FL_NONE) | cyc;
        case 0x4c: return mk(M_ABS, false, false, true, OP_NOP, R_M, D_NONE, X_JMP, FL_NONE) | cyc;
        case 0x58: return mk(M_NONE, false, false, true, OP_FLAG, R_M, D_NONE, X_NONE, FL_OP, 2) | cyc;
        case 0x60: return mk(M_NONE, false, false, true, OP_NOP, R_M, D_NONE, X_RTS, FL_NONE) | cyc;
        case 0x68: return mk(M_NONE, false, false, true, OP_NOP, R_M, D_NONE, X_PLA, FL_NONE) | cyc;
        case 0x6c: return mk(M_ABS, false, false, true, OP_NOP, R_M, D_NONE, X_JMPI, FL_NONE) | cyc;
        case 0x78: return mk(M_NONE, false, false, true, OP_FLAG, R_M, D_NONE, X_NONE, FL_OP, 3) | cyc;
        case 0x88: return mk(M_NONE, false, false, true, OP_DEC, R_Y, D_Y, X_NONE, FL_NZ) | cyc;
        case 0x8a: return mk(M_NONE, false, false, true, OP_PASS, R_X, D_A, X_NONE, FL_NZ) | cyc;
        case 0x98: return mk(M_NONE, false, false, true, OP_PASS, R_Y, D_A, X_NONE, FL_NZ) | cyc;
        case 0x9a: return mk(M_NONE, false, false, true, OP_PASS, R_X, D_SP, X_NONE, FL_NONE) | cyc;
        case 0xa8: return mk(M_NONE, false, false, true, OP_PASS, R_A, D_Y, X_NONE, FL_NZ) | cyc;
        case 0xaa: return mk(M_NONE, false, false, true, OP_PASS, R_A, D_X, X_NONE, FL_NZ) | cyc;
        case 0xb8: return mk(M_NONE, false, false, true, OP_FLAG, R_M, D_NONE, X_NONE, FL_OP, 4) | cyc;
        case 0xba: return mk(M_NONE, false, false, true, OP_PASS, R_SP, D_X, X_NONE, FL_NZ) | cyc;
        case 0xc8: return mk(M_NONE, false, false, true, OP_INC, R_Y, D_Y, X_NONE, FL_NZ) | cyc;
        case 0xca: return mk(M_NONE, false, false, true, OP_DEC, R_X, D_X, X_NONE, FL_NZ) | cyc;
        case 0xd8: return mk(M_NONE, false, false, true, OP_FLAG, R_M, D_NONE, X_NONE, FL_OP, 5) | cyc;
        case 0xe8: return mk(M_NONE, false, false, true, OP_INC, R_X, D_X, X_NONE, FL_NZ) | cyc;
        case 0xea: return mk(M_NONE, false, false, true, OP_NOP, R_M, D_NONE, X_NONE, FL_NONE) | cyc;
        case 0xf8: return mk(M_NONE, false, false, true, OP_FLAG, R_M, D_NONE, X_NONE, FL_OP, 6) | cyc;
        default: break;
    }
    if ((op & 0x1f) == 0x10) return mk(M_NONE, false, false, true, OP_NOP, R_M, D_NONE, X_BRANCH, FL_NONE) | cyc;
    if (cc == 1) {
        const uint32_t am = bbb == 0 ? M_INDX : bbb == 1 ? M_ZP : bbb == 2 ? M_IMM : bbb == 3 ? M_ABS
                          : bbb == 4 ? M_INDY : bbb == 5 ? M_ZPX : bbb == 6 ? M_ABSY : M_ABSX;
        const bool pen = fn != 4 && (bbb == 4 || bbb == 6 || bbb == 7);
        switch (fn) {
            case 0: return mk(am, pen, true, true, OP_ORA, R_A, D_A, X_NONE, FL_NZ) | cyc;
            case 1: return mk(am, pen, true, true, OP_AND, R_A, D_A, X_NONE, FL_NZ) | cyc;
            case 2: return mk(am, pen, true, true, OP_EOR, R_A, D_A, X_NONE, FL_NZ) | cyc;
            case 3: return mk(am, pen, true, true, OP_ADC, R_A, D_A, X_NONE, FL_NZCV) | cyc;
            case 4: return mk(am, pen, false, true, OP_PASS, R_A, D_MEM, X_NONE, FL_NONE) | cyc;
            case 5: return mk(am, pen, true, true, OP_PASS, R_M, D_A, X_NONE, FL_NZ) | cyc;
            case 6: return mk(am, pen, true, true, OP_CMP, R_A, D_NONE, X_NONE, FL_NZC) | cyc;
            default: return mk(am, pen, true, true, OP_SBC, R_A, D_A, X_NONE, FL_NZCV) | cyc;
        }
    }
    if (cc == 2 && bbb != 4 && bbb != 6) {
        const bool xy = fn == 4 || fn == 5;
        const uint32_t am = bbb == 0 ? M_IMM : bbb == 1 ? M_ZP : bbb == 2 ? M_NONE : bbb == 3 ? M_ABS
                          : bbb == 5 ? (xy ? M_ZPY : M_ZPX) : (xy ? M_ABSY : M_ABSX);
        const bool pen = bbb == 7, acc = bbb == 2;
        if (fn < 4) {
            const uint32_t alu = fn == 0 ? OP_ASL : fn == 1 ? OP_ROL : fn == 2 ? OP_LSR : OP_ROR;
            return (acc ? mk(am, pen, false, true, alu, R_A, D_A, X_NONE, FL_NZC)
                        : mk(am, pen, true, true, alu, R_M, D_MEM, X_NONE, FL_NZC)) | cyc;
        }
        switch (fn) {
            case 4: return mk(am, pen, false, true, OP_PASS, R_X, D_MEM, X_NONE, FL_NONE) | cyc;
            case 5: return mk(am, pen, true, true, OP_PASS, R_M, D_X, X_NONE, FL_NZ) | cyc;
            case 6: return mk(am, pen, true, true, OP_DEC, R_M, D_MEM, X_NONE, FL_NZ) | cyc;
            default: return mk(am, pen, true, true, OP_INC, R_M, D_MEM, X_NONE, FL_NZ) | cyc;
        }
    }
    if (cc == 0 && (bbb & 1 || bbb == 0)) {
        const uint32_t am = bbb == 0 ? M_IMM : bbb == 1 ? M_ZP : bbb == 3 ? M_ABS : bbb == 5 ? M_ZPX : M_ABSX;
        const bool pen = bbb == 7;
        switch (fn) {
            case 1: return mk(am, pen, true, true, OP_BIT, R_A, D_NONE, X_NONE, FL_BIT) | cyc;
            case 4: return mk(am, pen, false, true, OP_PASS, R_Y, D_MEM, X_NONE, FL_NONE) | cyc;
            case 5: return mk(am, pen, true, true, OP_PASS, R_M, D_Y, X_NONE, FL_NZ) | cyc;
            case 6: return mk(am, pen, true, true, OP_CMP, R_Y, D_NONE, X_NONE, FL_NZC) | cyc;
            case 7: return mk(am, pen, true, true, OP_CMP, R_X, D_NONE, X_NONE, FL_NZC) | cyc;
            default: return mk(am, pen, false, false, OP_NOP, R_M, D_NONE, X_NONE, FL_NONE) | cyc;
        }
    }
    return mk(M_NONE, false, false, false, OP_NOP, R_M, D_NONE, X_NONE, FL_NONE) | cyc;
}
struct Table {
    uint32_t w[256];
    constexpr Table() : w() {
        for (int i = 0; i < 256; i++) w[i] = entry(i);
    }
};
}  // namespace dec

__device__ __constant__ static const dec::Table kDecode{};

#if defined(__AMDGCN__)
// v_writelane_b32 (clang has no builtin for the intrinsic)
extern "C" __device__ int mh_writelane(int value, int lane, int old) __asm("llvm.amdgcn.writelane.i32");
#endif
// A wave-uniform value, in a scalar register
__device__ __forceinline__ uint32_t uni(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
// A wave-uniform 64-bit value (a pointer): the builtin returns a signed int, so each half is taken as unsigned
// before it is widened (else the low half's bit 31 would spread into the high half).
__device__ __forceinline__ uint64_t uni64(uint64_t v) { return (uint64_t)uni((uint32_t)v) | (uint64_t)uni((uint32_t)(v >> 32)) << 32; }

}  // namespace mh
#include "cpu_gfx950.hpp"
namespace mh {

// Memory in LDS, addressed as such
#ifndef MH_LDS
#if defined(__AMDGCN__)
#define MH_LDS __attribute__((address_space(3)))
#else
#define MH_LDS
#endif
#endif

struct Cart {
    const MH_LDS uint8_t* prg;   // 0x8000 bytes (16 KB images mirrored), in LDS
    const MH_LDS uint8_t* chr;   // 0x2000 bytes, in LDS
    const uint32_t* dec;     // decode words (kDecode)
    const uint32_t* recs;    // the program as records (cpu_gfx950.hpp; none on the host build, which decodes as it goes)
    uint32_t nt_bits;        // bit k set: name table k ($2000 + k * $400) maps to VRAM $400, else to $000
};

typedef uint32_t mh_u32x4 __attribute__((ext_vector_type(4)));

// A console's registers: word k (Scalar) in lane k of one vector register. (The host build: an array.)
struct File {
#if defined(__AMDGCN__)
    uint32_t r;
    __device__ __forceinline__ uint32_t get(int k) const { return (uint32_t)__builtin_amdgcn_readlane((int)r, k); }
    __device__ __forceinline__ void set(int k, uint32_t v) { r = (uint32_t)mh_writelane((int)uni(v), k, (int)r); }
#else
    uint32_t r[F_COUNT];
    uint32_t get(int k) const { return r[k]; }
    void set(int k, uint32_t v) { r[k] = v; }
#endif
};
static_assert(F_COUNT <= 64, "a word per lane");

// What a console's functions need beside its registers: LDS addresses, the program's records, the frame buffer. On the
// GPU the words of a second vector register, so that a call takes two.
struct Ctx {
#if defined(__AMDGCN__)
    File w;
    enum : int { M, GP, PRG, CHR, LUT, DEC_LO, DEC_HI, RECS_LO, RECS_HI, GRAY_LO, GRAY_HI, NT_BITS, NP, RENDER };
    __device__ __forceinline__ MH_LDS uint8_t* memory() const { return (MH_LDS uint8_t*)(uintptr_t)w.get(M); }
    __device__ __forceinline__ uint32_t name_tables() const { return w.get(NT_BITS); }
#else
    uint8_t* memory() const { return m; }
    uint32_t name_tables() const { return cart.nt_bits; }
    uint8_t* m; uint32_t* gp; Cart cart; uint8_t* gray; const uint8_t* lut; uint32_t np; bool render;
#endif
};

// The machine with its registers as variables, for the length of one function.
struct Core {
    // ---- memory views
    MH_LDS uint8_t* m;       // the console's memory in LDS: byte r is row r (ROW_*)
    MH_LDS uint32_t* gp;     // the renderer's words in LDS (GP_*)
    uint32_t np;             // envs of the memory block, padded: the host build's interleaved frame buffers
    const MH_LDS uint8_t* prg_;              // 0x8000 bytes (16 KB images mirrored)
    const MH_LDS uint8_t* chr;               // 0x2000 bytes
    const MH_LDS uint8_t* lut;               // palette value -> gray (256 entries)
    const uint32_t* dec;                     // decode words
    uint32_t nt_bits;
    uint8_t* gray;           // the env's frame buffer: pixels 4i..4i+3 in the 32-bit word at gray + 4 i gray_step()
    bool render;
    uint32_t lane;           // this lane of the wave: the only field that differs between the lanes
    // ---- CPU
    uint32_t pc, a, x, y, sp, p;
    int32_t exec_at, ppu_calls, nmi_thresh;  // relative to the current frame start
    uint32_t iter_lo;                        // low word of the iteration count at the frame start
    int32_t cur, skip;
    uint32_t zero_skip;
    // ---- joypads
    // both ports in one word (buttons 0 | buttons 1 << 8 | shift register 0 << 16 | shift register 1 << 24);
    // their strobes are bits 0 and 1 of joy_strobe
    uint32_t joy, joy_strobe;
    // ---- PPU
    uint32_t pstate, even, vblank, s0hit, first_write, fine_x, oam_addr, data_buffer, nsl;
    uint32_t ppu_flags;                      // the PPUCTRL / PPUMASK settings as PF_* bits
    uint32_t sl_lo, sl_hi;                   // sprite list: 8 indices packed in two words
    int32_t pcyc, scanline;
    uint32_t v, t;
    int32_t nmi_call;                        // the PPU call that raised an NMI in this catch-up (0: none)
    // ---- counters of this frame
    uint32_t bad_ops, instructions;          // instructions: retired, poll-loop fast-forwards included
    uint32_t ff_instructions;                // of those, the ones poll_skip fast-forwarded without executing
    // ---- derived state (not part of the machine state)
    int32_t pend_line;                       // scanline of a sprite evaluation not yet materialized (-1: the list is current)
    uint32_t pal_dirty;                      // the gray palette in LDS must be rebuilt

    // ------------------------------------------------------------ in and out of the register file
    __device__ __forceinline__ void attach(const Ctx& c) {
#if defined(__AMDGCN__)
        auto ptr = [&](int k) { return (uint64_t)c.w.get(k) | (uint64_t)c.w.get(k + 1) << 32; };
        m = (MH_LDS uint8_t*)(uintptr_t)c.w.get(Ctx::M); gp = (MH_LDS uint32_t*)(uintptr_t)c.w.get(Ctx::GP);
        prg_ = (const MH_LDS uint8_t*)(uintptr_t)c.w.get(Ctx::PRG); chr = (const MH_LDS uint8_t*)(uintptr_t)c.w.get(Ctx::CHR);
        lut = (const MH_LDS uint8_t*)(uintptr_t)c.w.get(Ctx::LUT); dec = (const uint32_t*)ptr(Ctx::DEC_LO);
        gray = (uint8_t*)ptr(Ctx::GRAY_LO); nt_bits = c.w.get(Ctx::NT_BITS); np = c.w.get(Ctx::NP);
        render = c.w.get(Ctx::RENDER) != 0; lane = __lane_id();
#else
        m = c.m; gp = c.gp; prg_ = c.cart.prg; chr = c.cart.chr; lut = c.lut; dec = c.cart.dec; gray = c.gray;
        nt_bits = c.cart.nt_bits; np = c.np; render = c.render; lane = 0;
#endif
    }
    __device__ __forceinline__ void open_ppu(const File& f) {
        pstate = f.get(S_PSTATE); even = f.get(S_EVEN); vblank = f.get(S_VBLANK); s0hit = f.get(S_S0HIT);
        fine_x = f.get(S_FINE_X); oam_addr = f.get(S_OAM_ADDR); nsl = f.get(S_NSL); ppu_flags = f.get(F_PPU_FLAGS);
        sl_lo = f.get(S_SL_LO); sl_hi = f.get(S_SL_HI); pcyc = (int32_t)f.get(S_PCYC); scanline = (int32_t)f.get(S_SCANLINE);
        v = f.get(S_V); t = f.get(S_T); ppu_calls = (int32_t)f.get(F_PPU_CALLS); nmi_thresh = (int32_t)f.get(F_NMI_THRESH);
        pend_line = (int32_t)f.get(F_PEND_LINE); pal_dirty = f.get(F_PAL_DIRTY);
    }
    __device__ __forceinline__ void close_ppu(File& f) const {   // what a catch-up changes
        f.set(S_PSTATE, pstate); f.set(S_EVEN, even); f.set(S_VBLANK, vblank); f.set(S_S0HIT, s0hit);
        f.set(S_PCYC, (uint32_t)pcyc); f.set(S_SCANLINE, (uint32_t)scanline); f.set(S_V, v);
        f.set(F_PPU_CALLS, (uint32_t)ppu_calls); f.set(F_NMI_THRESH, (uint32_t)nmi_thresh); f.set(F_NMI_CALL, (uint32_t)nmi_call);
        f.set(F_PEND_LINE, (uint32_t)pend_line); f.set(F_PAL_DIRTY, pal_dirty);
    }
    __device__ __forceinline__ void open_io(const File& f) {     // the registers behind the CPU's bus
        open_ppu(f);
        first_write = f.get(S_FIRST_WRITE); data_buffer = f.get(S_DATA_BUFFER); joy = f.get(F_JOY);
        joy_strobe = f.get(F_JOY_STROBE); iter_lo = f.get(S_ITER_LO);
    }
    __device__ __forceinline__ void close_io(File& f) const {    // what a register access changes
        f.set(S_VBLANK, vblank); f.set(S_FIRST_WRITE, first_write); f.set(S_DATA_BUFFER, data_buffer); f.set(F_JOY, joy);
        f.set(F_JOY_STROBE, joy_strobe); f.set(S_OAM_ADDR, oam_addr); f.set(S_FINE_X, fine_x); f.set(F_PPU_FLAGS, ppu_flags);
        f.set(S_V, v); f.set(S_T, t); close_sprites(f); f.set(F_PAL_DIRTY, pal_dirty);
    }
    __device__ __forceinline__ void close_sprites(File& f) const {
        f.set(S_NSL, nsl); f.set(S_SL_LO, sl_lo); f.set(S_SL_HI, sl_hi); f.set(F_PEND_LINE, (uint32_t)pend_line);
    }
    __device__ __forceinline__ void open_cpu(const File& f) {
        pc = f.get(S_PC); a = f.get(S_A); x = f.get(S_X); y = f.get(S_Y); sp = f.get(S_SP); p = f.get(S_P);
        exec_at = (int32_t)f.get(S_EXEC_REL); zero_skip = f.get(S_ZERO_SKIP);
        bad_ops = f.get(F_BAD); instructions = f.get(F_INSTR); ff_instructions = f.get(F_FF);
    }
    __device__ __forceinline__ void close_cpu(File& f) const {
        f.set(S_PC, pc); f.set(S_A, a); f.set(S_X, x); f.set(S_Y, y); f.set(S_SP, sp); f.set(S_P, p);
        f.set(S_EXEC_REL, (uint32_t)exec_at); f.set(S_ZERO_SKIP, zero_skip);
        f.set(F_BAD, bad_ops); f.set(F_INSTR, instructions); f.set(F_FF, ff_instructions);
    }

    // ------------------------------------------------------------ memory
    // The wave has stored to LDS (or to its own memory block) what its lanes read next: a wave's LDS accesses complete
    // in order, so only the compiler has to keep them so; memory accesses are waited for.
    __device__ __forceinline__ static void lds_sync() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    __device__ __forceinline__ static void mem_sync() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    }
    __device__ __forceinline__ uint32_t ram(uint32_t ad) const { return uni(m[ROW_RAM + (ad & 0x7ff)]); }
    __device__ __forceinline__ void set_ram(uint32_t ad, uint32_t val) { m[ROW_RAM + (ad & 0x7ff)] = (uint8_t)val; }
    __device__ __forceinline__ uint32_t oam(uint32_t i) const { return uni(m[ROW_OAM + (i & 0xff)]); }
    __device__ __forceinline__ void set_oam(uint32_t i, uint32_t val) { m[ROW_OAM + (i & 0xff)] = (uint8_t)val; }
    // sprite k's four OAM bytes: y | tile << 8 | attr << 16 | x << 24 (oam_word: of a lane's own sprite)
    __device__ __forceinline__ uint32_t oam_word(uint32_t k) const { return ((const MH_LDS uint32_t*)(m + ROW_OAM))[k]; }
    __device__ __forceinline__ uint32_t oam_sprite(uint32_t k) const { return uni(oam_word(k)); }
    __device__ __forceinline__ uint32_t sl(int k) const { return ((k < 4 ? sl_lo >> (8 * k) : sl_hi >> (8 * (k - 4))) & 0xffu); }
    __device__ __forceinline__ void set_sl(int k, uint32_t i) {
        if (k < 4) sl_lo = (sl_lo & ~(0xffu << (8 * k))) | (i << (8 * k));
        else sl_hi = (sl_hi & ~(0xffu << (8 * (k - 4)))) | (i << (8 * (k - 4)));
    }
    // words between a frame buffer's words: frames are whole on the GPU (a lane's 16 pixels are one 16-byte store),
    // interleaved by env on the host build
    __device__ __forceinline__ uint32_t gray_step() const { return ON_GPU ? 1u : np; }
    __device__ __forceinline__ uint32_t prg(uint32_t ad) const { return uni(prg_[ad & 0x7fff]); }
    // PPUCTRL / PPUMASK settings (0 or 1; inc(): the VRAM address increment, 1 or 32)
    __device__ __forceinline__ uint32_t show_bg() const { return ppu_flags & 1u; }
    __device__ __forceinline__ uint32_t show_spr() const { return (ppu_flags >> 1) & 1u; }
    __device__ __forceinline__ uint32_t hide_edge_bg() const { return (ppu_flags >> 2) & 1u; }
    __device__ __forceinline__ uint32_t hide_edge_spr() const { return (ppu_flags >> 3) & 1u; }
    __device__ __forceinline__ uint32_t long_spr() const { return (ppu_flags >> 4) & 1u; }
    __device__ __forceinline__ uint32_t nmi_en() const { return (ppu_flags >> 5) & 1u; }
    __device__ __forceinline__ uint32_t bg_page() const { return (ppu_flags >> 6) & 1u; }
    __device__ __forceinline__ uint32_t spr_page() const { return (ppu_flags >> 7) & 1u; }
    __device__ __forceinline__ uint32_t inc() const { return (ppu_flags & PF_INC32) ? 32 : 1; }
    // ------------------------------------------------------------ CPU bus (nes_core.hpp:150-208)
    // Accesses for which needs_sync() holds see the PPU caught up to 3 * (cur + 1): frame() syncs
    // before it issues them (the reference catches up inside the access; the target is the same).
    __device__ __forceinline__ static bool needs_sync(uint32_t ad, bool wr) {
        if ((ad & 0xe000) == 0x2000) return wr || (ad & 7) == 2 || (ad & 7) == 7;
        return wr && ad == 0x4014;
    }
    __device__ __forceinline__ uint32_t read(uint32_t ad) {
        if (ad >= 0x8000) return prg(ad);
        if (ad < 0x2000) return ram(ad);
        if (ad < 0x4000) {
            const uint32_t r = ad & 7;
            if (r == 2) return status_read();
            if (r == 7) return data_read();
            if (r == 4) return oam(oam_addr);
            return 0;
        }
        if (ad == 0x4016) return pad_read(0);
        if (ad == 0x4017) return pad_read(1);
        return 0;
    }
    __device__ __forceinline__ void write(uint32_t ad, uint32_t val) {
        if (ad < 0x2000) { set_ram(ad, val); return; }
        if (ad < 0x4000) {
            // a pending sprite evaluation is materialized before its inputs (OAM, oam_addr, sprite size) change
            const uint32_t r = ad & 7;
            if (r == 0 || r == 3 || r == 4) materialize_sprites();
            switch (r) {
                case 0: ctrl_write(val); break;
                case 1: mask_write(val); break;
                case 3: oam_addr = val; break;
                case 4: set_oam(oam_addr, val); oam_addr = (oam_addr + 1) & 0xffu; break;
                case 5: scroll_write(val); break;
                case 6: addr_write(val); break;
                case 7: data_write(val); break;
                default: break;
            }
            return;
        }
        if (ad == 0x4014) {  // OAM DMA: 513 cycles, +1 on an odd absolute cycle; copies from RAM pages only
            materialize_sprites();
            skip += 513 + (int)((iter_lo + (uint32_t)cur + 1u) & 1u);
            const uint32_t src = val << 8;
            if (src < 0x2000) {
                for (uint32_t i = lane; i < 256; i += LANES) m[ROW_OAM + ((oam_addr + i) & 0xff)] = m[ROW_RAM + ((src + i) & 0x7ff)];
                lds_sync();
            }
            return;
        }
        if (ad == 0x4016) {   // strobe both ports; its falling edge latches the buttons into the shift registers
            joy_strobe = (val & 1) ? 3 : 0;
            if (!(val & 1)) joy = (joy & 0xffffu) | (joy << 16);
        }
    }
    // port i: while strobed, button A; else the next bit of its shift register, which then shifts
    __device__ __forceinline__ uint32_t pad_read(int i) {
        const uint32_t sh = 16 + 8 * i;
        if ((joy_strobe >> i) & 1) return ((joy >> (8 * i)) & 1u) | 0x40u;
        const uint32_t bit = (joy >> sh) & 1u;
        joy = (joy & ~(0xffu << sh)) | ((((joy >> sh) & 0xffu) >> 1) << sh);
        return bit | 0x40u;
    }

    // ------------------------------------------------------------ PPU registers (nes_core.hpp:211-260)
    __device__ __forceinline__ void ctrl_write(uint32_t c) {
        ppu_flags = (ppu_flags & (PF_SHOW_BG | PF_SHOW_SPR | PF_HIDE_EDGE_BG | PF_HIDE_EDGE_SPR)) |
                    ((c >> 7) & 1 ? PF_NMI_EN : 0u) | ((c >> 5) & 1 ? PF_LONG_SPR : 0u) |
                    ((c >> 4) & 1 ? PF_BG_PAGE : 0u) | ((c >> 3) & 1 ? PF_SPR_PAGE : 0u) | ((c & 4) ? PF_INC32 : 0u);
        t = (t & 0xf3ff) | ((c & 3) << 10);
    }
    __device__ __forceinline__ void mask_write(uint32_t k) {
        ppu_flags = (ppu_flags & ~(PF_SHOW_BG | PF_SHOW_SPR | PF_HIDE_EDGE_BG | PF_HIDE_EDGE_SPR)) |
                    (!(k & 2) ? PF_HIDE_EDGE_BG : 0u) | (!(k & 4) ? PF_HIDE_EDGE_SPR : 0u) |
                    ((k >> 3) & 1 ? PF_SHOW_BG : 0u) | ((k >> 4) & 1 ? PF_SHOW_SPR : 0u);
    }
    __device__ __forceinline__ uint32_t status_read() {
        const uint32_t r = (s0hit << 6) | (vblank << 7);
        vblank = 0; first_write = 1;
        return r;
    }
    __device__ __forceinline__ void addr_write(uint32_t d) {
        if (first_write) { t = (t & 0x00ff) | ((d & 0x3f) << 8); first_write = 0; }
        else { t = (t & 0xff00) | d; v = t; first_write = 1; }
    }
    __device__ __forceinline__ uint32_t data_read() {
        uint32_t d = uni(vbus_read(v));
        v = (v + inc()) & 0xffffu;
        if (v < 0x3f00) { const uint32_t b = data_buffer; data_buffer = d; d = b; }
        return d;
    }
    __device__ __forceinline__ void data_write(uint32_t d) { vbus_write(v, d); v = (v + inc()) & 0xffffu; }
    __device__ __forceinline__ void scroll_write(uint32_t d) {
        if (first_write) { t = (t & ~0x1fu) | (d >> 3); fine_x = d & 7; first_write = 0; }
        else { t = (t & ~0x73e0u) | ((d & 7) << 12) | ((d & 0xf8) << 2); first_write = 1; }
    }

    // ------------------------------------------------------------ picture bus (nes_core.hpp:263-285)
    // (vbus_read and nametable take a lane's own address too)
    __device__ __forceinline__ uint32_t nt_row(uint32_t ad) const {
        const uint32_t k = ad < 0x2400 ? 0 : ad < 0x2800 ? 1 : ad < 0x2c00 ? 2 : 3;
        return (((nt_bits >> k) & 1u) << 10) | (ad & 0x3ffu);
    }
    __device__ __forceinline__ uint32_t vbus_read(uint32_t ad) const {
        if (ad < 0x2000) return chr[ad];
        if (ad < 0x3eff) return m[ROW_VRAM + nt_row(ad)];
        if (ad < 0x3fff) return m[ROW_PAL + (ad & 0x1f)];
        return 0;
    }
    __device__ __forceinline__ void vbus_write(uint32_t ad, uint32_t d) {
        if (ad < 0x2000) return;
        if (ad < 0x3eff) m[ROW_VRAM + nt_row(ad)] = (uint8_t)d;
        else if (ad < 0x3fff) { m[ROW_PAL + (ad == 0x3f10 ? 0 : (ad & 0x1f))] = (uint8_t)d; pal_dirty = 1; }
    }
    __device__ __forceinline__ uint32_t nametable(uint32_t ad) const {
        return m[ROW_VRAM + ((((nt_bits >> ((ad >> 10) & 3u)) & 1u) << 10) | (ad & 0x3ffu))];
    }

    // ------------------------------------------------------------ PPU timing (nes_core.hpp:289-308)
    __device__ __forceinline__ void nmi_threshold() {
        const int line = pstate == ST_PRE ? -1 : pstate == ST_POST ? 240 : scanline;
        const int32_t pos = (line + 1) * 341 + (pcyc - 1);
        const int32_t vbl = 242 * 341;
        const int32_t d = pos <= vbl ? vbl - pos + 1 : (262 * 341 - pos) + vbl + 1;
        nmi_thresh = ppu_calls + d - 8;
    }

    __device__ __forceinline__ static uint32_t coarse_x_added(uint32_t v, uint32_t n) {
        const uint32_t tot = (v & 0x1f) + n;
        return ((v & ~0x1fu) | (tot & 31)) ^ ((tot & 32) << 5);
    }
    __device__ __forceinline__ void coarse_x_add(int n) { v = coarse_x_added(v, (uint32_t)n); }
    __device__ __forceinline__ void fine_y_step() {
        if ((v & 0x7000) != 0x7000) { v = (v + 0x1000) & 0xffffu; return; }
        v &= ~0x7000u;
        uint32_t yy = (v >> 5) & 31;
        if (yy == 29) { yy = 0; v ^= 0x800; }
        else if (yy == 31) yy = 0;
        else yy++;
        v = (v & ~0x3e0u) | (yy << 5);
    }
    __device__ __forceinline__ void copy_h() { v = (v & ~0x41fu) | (t & 0x41f); }
    __device__ __forceinline__ void copy_v() { v = (v & ~0x7be0u) | (t & 0x7be0); }

    // Per-line sprite list from oam_addr/4 (nes_core.hpp:336-349). The PPU only records the scanline
    // of an evaluation; the list is computed from OAM when something needs it (a change of OAM / oam_addr / sprite
    // size, or the end of the kernel). Until then its inputs are unchanged, so the late evaluation gives the same
    // list; a line drawn meanwhile evaluates its own (draw_lines).
    // The sprites in range of an evaluation at scanline `line`, as a 64-bit mask (bit i: line - y_i in [0, h)), from
    // index oam_addr / 4 on: the list is its first (at most 8) set bits. Lane i tests sprite i.
    // `more`: lines before it, too.
    __device__ __forceinline__ uint64_t in_range(int line, uint32_t more = 0) const {
        const uint32_t h = (long_spr() ? 16u : 8u) + more;
        uint64_t b = 0;
        if constexpr (ON_GPU) {
            b = __ballot((uint32_t)(line - (int)(oam_word(lane) & 0xffu)) < h);
        } else {
            for (uint32_t i = 0; i < 64; i++) b |= (uint64_t)((uint32_t)(line - (int)(oam_word(i) & 0xffu)) < h) << i;
        }
        return b & (~0ull << (oam_addr >> 2));
    }
    __device__ __forceinline__ void materialize_sprites() {
        if (pend_line < 0) return;
        uint64_t b = in_range(pend_line);   // entries past the count keep their old values
        int n = 0;
        while (b && n < 8) {
            set_sl(n++, (uint32_t)__builtin_ctzll(b));
            b &= b - 1;
        }
        nsl = (uint32_t)n;
        pend_line = -1;
    }
    // "nsl > 0 && sl[0] == 0" without materializing: sprite 0 heads the list exactly when the
    // evaluation starts at index 0 and sprite 0 is in range.
    __device__ __forceinline__ bool sprite0_first() const {
        if (pend_line < 0) return nsl > 0 && sl(0) == 0;
        if (oam_addr >= 4) return false;
        const int d = pend_line - (int)(oam_sprite(0) & 0xffu);
        return d >= 0 && d < (long_spr() ? 16 : 8);
    }
    // the background pattern at pixel px, with v at its tile (a lane's own px and v)
    __device__ __forceinline__ uint32_t bg_pattern(int px, uint32_t v) const {
        const uint32_t xf = (fine_x + (uint32_t)px) & 7u;
        const uint32_t pa = ((nametable(0x2000 | (v & 0x0fff)) * 16) + ((v >> 12) & 7)) | (bg_page() << 12);
        return ((chr[pa] >> (7 ^ xf)) & 1u) | (((chr[pa + 8] >> (7 ^ xf)) & 1u) << 1);
    }
    // the picture-bus address of row py of the sprite with OAM word ow, with C++ int semantics for stale lists
    // (nes_core.hpp:369-391)
    __device__ __forceinline__ uint32_t sprite_row(uint32_t ow, int py) const {
        const int sy = (int)((ow + 1u) & 0xffu), h = long_spr() ? 16 : 8;
        const uint32_t tile = (ow >> 8) & 0xffu;
        int yo = (py - sy) % h;
        if (ow & 0x800000u) yo ^= (h - 1);
        if (!long_spr()) return (uint32_t)((int)tile * 16 + yo + (spr_page() ? 0x1000 : 0)) & 0xffffu;
        yo = (yo & 7) | ((yo & 8) << 1);
        return ((uint32_t)((int)(tile >> 1) * 32 + yo) & 0xffffu) | ((tile & 1) << 12);
    }
    // sprite 0's 2-bit pattern at (px, py)
    __device__ __forceinline__ uint32_t sprite0_pattern(uint32_t ow, int px, int py) const {
        int xs = (px - (int)(ow >> 24)) % 8;
        if (!(ow & 0x400000u)) xs ^= 7;
        const uint32_t ad = sprite_row(ow, py);
        return ((vbus_read(ad) >> xs) & 1u) | (((vbus_read((ad + 8) & 0xffffu) >> xs) & 1u) << 1);
    }

    // Visible dots [x0, x1): sprite-0 hit and the coarse-x increments of v (nes_core.hpp:394-413). The lanes test the
    // (at most 8) pixels under sprite 0 at once.
    __device__ __forceinline__ void dots_hit_scroll(int x0, int x1) {
        if (!show_bg()) return;
        if (!s0hit && show_spr() && sprite0_first()) {
            const uint32_t ow = oam_sprite(0);
            const int sx = (int)(ow >> 24);
            int lo = x0 > sx ? x0 : sx;
            const int hi = x1 < sx + 8 ? x1 : sx + 8;
            if (hide_edge_spr() && lo < 8) lo = 8;
            if (hide_edge_bg() && lo < 8) lo = 8;
            bool hit = false;
            for (int px = lo + (int)lane; px < hi; px += LANES) {
                const uint32_t vp = coarse_x_added(v, (uint32_t)inc_count(x0, px));
                hit |= bg_pattern(px, vp) && sprite0_pattern(ow, px, scanline);
            }
            if (__any(hit)) s0hit = 1;
        }
        coarse_x_add(inc_count(x0, x1));
    }
    __device__ __forceinline__ int inc_count(int lo, int hi) const {   // x in [lo, hi) with (fine_x + x) % 8 == 7
        const int r = (7 - (int)fine_x) & 7;
        return (hi - r + 7) / 8 - (lo - r + 7) / 8;
    }

    // bytes of the 8-byte value hi:lo picked by the selector bytes of sel (each 0..7)
    __device__ __forceinline__ static uint32_t byte_perm(uint32_t hi, uint32_t lo, uint32_t sel) {
        return __builtin_amdgcn_perm(hi, lo, sel);
    }

    // ---- the renderer
    // gray value of every palette address, lut[pal[i]]; rebuilt after palette writes
    __device__ __forceinline__ void build_gray_palette() {
        for (uint32_t i = lane; i < 32; i += LANES) ((MH_LDS uint8_t*)(gp + GP_PALETTE))[i] = lut[m[ROW_PAL + i]];
        lds_sync();
        pal_dirty = 0;
    }
    // v at the start of the i-th line after this one, both layers on: fine_y_step i times, and copy_h. (Coarse y
    // 30 and 31 wrap to 0 without the mirror switch that 29 makes.)
    __device__ __forceinline__ uint32_t v_lines_on(uint32_t i) const {
        uint32_t yy = ((v >> 5) & 31u) * 8u + ((v >> 12) & 7u), mirror = 0;   // i <= 240
        if (yy >= 240u) yy = (yy + i) & 255u;
        else {
            yy += i;
            if (yy >= 240u) { yy -= 240u; mirror = 0x800u; }
        }
        return (v & 0x8000u) | ((v ^ mirror) & 0x800u) | (t & 0x41fu) | (yy >> 3) << 5 | (yy & 7u) << 12;
    }
    // A sprite's row on line py as one word: x | the row's two planes, bit j pixel x + j, << 8 and << 16 | palette
    // (bits 24-25), behind the background (bit 29), bit 31 set.
    __device__ __forceinline__ uint32_t sprite_entry(uint32_t ow, int py) const {
        const uint32_t ad = sprite_row(ow, py);
        uint32_t lo = vbus_read(ad), hi = vbus_read((ad + 8) & 0xffffu);
        if (!(ow & 0x400000u)) {
            lo = __builtin_bitreverse32(lo) >> 24;
            hi = __builtin_bitreverse32(hi) >> 24;
        }
        return (ow >> 24) | lo << 8 | hi << 16 | ((ow >> 16) & 0x23u) << 24 | 0x80000000u;
    }

    // Pixels [x0, x1) of `count` lines from this one on: gray values into the frame buffer (nes_core.hpp:427-513), with v
    // as it is at x0 of this line, and at the later lines' starts as the scroll leaves it (v_lines_on; with the
    // background off v stays and does not matter). Whole lines (x0 = 0, x1 = 256) go four at a time, 16 lanes a line
    // and 16 pixels (two screen-aligned groups of 8, from three background tiles) a lane; a line that a catch-up cuts
    // goes alone.
    //
    // First the lines' sprites: lane i tests sprite i against each line (in_range's ballot); a sprite in range is the
    // line's entry number "sprites before it in the ballot" if that is below 8, and the lanes that hold one fetch
    // its pattern row at once and leave it as a word in LDS. Each lane then merges the line's entries that reach
    // its pixels, in list order: a byte takes the sprite only where no earlier one is opaque. Line i > 0 takes its
    // sprites from the evaluation at the line before it, this line from the pending one or the list.
    //
    // Four pixels are one 32-bit word, a byte each, and are computed together without branches: the
    // pattern bits of the four pixels are spread to the four bytes by a multiply, the background gray
    // value is a byte permute of the two tiles' gray tables, a sprite pixel's gray value is a byte
    // permute of the sprite palette's 16 gray values, and priority is a per-byte mask.
    __device__ __forceinline__ void draw_lines(uint32_t count, int x0, int x1) {
        if (pal_dirty) build_gray_palette();
        MH_LDS uint32_t* const ent = gp + GP_SPRITES;
        // any sprite on any of the lines? (the pending evaluation may be the last frame's, of line 239)
        bool some = false;
        if (show_spr()) {
            if (pend_line >= 0 && count > 1) some = (in_range(scanline + (int)count - 2, count) | in_range(pend_line)) != 0;
            else some = true;
        }
        for (uint32_t base = 0; base < count; base += DRAW_LINES) draw_batch(base, count, x0, x1, some, ent);
    }
    __device__ __forceinline__ void draw_batch(uint32_t base, uint32_t count, int x0, int x1, bool some, MH_LDS uint32_t* ent) {
        const uint32_t cnt = count - base < (uint32_t)DRAW_LINES ? count - base : (uint32_t)DRAW_LINES;
        uint32_t most = 0;                      // sprites of the line that has most
        if (some) {
            for (uint32_t i = lane; i < 8 * DRAW_LINES; i += LANES) ent[i] = 0;
            lds_sync();
            for (uint32_t li = 0; li < cnt; li++) {
                const int py = scanline + (int)(base + li);
                uint64_t b = 0;
                if (base + li > 0) b = in_range(py - 1);
                else if (pend_line >= 0) b = in_range(pend_line);
                else for (uint32_t k = 0; k < nsl; k++) b |= 1ull << sl((int)k);
                if (!b) continue;
#if defined(__AMDGCN__)
                const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0));
                if (((b >> lane) & 1u) && rank < 8u) ent[8 * li + rank] = sprite_entry(oam_word(lane), py);
#else
                for (uint32_t i = 0, rank = 0; i < 64 && rank < 8; i++)
                    if ((b >> i) & 1u) ent[8 * li + rank++] = sprite_entry(oam_word(i), py);
#endif
                const uint32_t n = (uint32_t)__popcll(b) < 8u ? (uint32_t)__popcll(b) : 8u;
                most = n > most ? n : most;
            }
            lds_sync();
        }
        const MH_LDS uint32_t* const pal = gp + GP_PALETTE;
        const uint32_t f = fine_x;
        // pixel bb of a group takes the second tile's gray table when f + bb >= 8: bytes bb >= 8 - f
        const uint64_t second = f ? (~0ull << (8 * (8 - f))) : 0ull;
        const uint32_t tsel0 = (uint32_t)second & 0x04040404u, tsel1 = (uint32_t)(second >> 32) & 0x04040404u;
        const uint32_t bg_on = show_bg() ? ~0u : 0u, gs = gray_step();
        for (uint32_t unit = lane; unit < 16 * cnt; unit += LANES) {
            const uint32_t li = unit >> 4, q = unit & 15u, i = base + li, py = (uint32_t)scanline + i;
            const uint32_t vl = i && show_bg() ? v_lines_on(i) : v, fy = (vl >> 12) & 7u, cy = (vl >> 5) & 31u;
            // the line's first tile: v addresses the tile of pixel x0, (f + x0) / 8 tiles into the line
            int c0 = (int)(vl & 31u) - (int)((f + (uint32_t)x0) >> 3);
            uint32_t nt = (vl >> 10) & 3u;
            if (c0 < 0) { c0 += 32; nt ^= 1u; }
            const uint32_t bp0 = pal[0], bp1 = pal[1], bp2 = pal[2], bp3 = pal[3];
            uint32_t lo[3], hi[3], gt[3];       // the three tiles' pattern rows and gray tables
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const uint32_t col = (uint32_t)c0 + 2 * q + (uint32_t)k, n2 = nt ^ ((col >> 5) & 1u), cx = col & 31u;
                const MH_LDS uint8_t* const row = m + ROW_VRAM + (((nt_bits >> n2) & 1u) << 10);
                const uint32_t tile = row[cy * 32 + cx], at8 = row[0x3c0 + (cy >> 2) * 8 + (cx >> 2)];
                const uint32_t at = (at8 >> (((cy & 2u) << 1) | (cx & 2u))) & 3u;
                const uint32_t pa = (tile * 16 + fy) | (bg_page() << 12);
                lo[k] = chr[pa] & bg_on;   // the background off: pattern 0, the universal background
                hi[k] = chr[pa + 8] & bg_on;
                // byte p: the gray value of background pattern p (0: palette address 0; else palette address 4 at + p)
                const uint32_t w01 = (at & 1u) ? bp1 : bp0, w23 = (at & 1u) ? bp3 : bp2;
                gt[k] = (((at & 2u) ? w23 : w01) & 0xffffff00u) | (bp0 & 0xffu);
            }
            // the line's sprites over these 16 pixels: a byte a pixel, the sprite palette entry (bits 0-3), in front
            // of the background (bit 6), bit 7 set (0: none)
            uint32_t sb[4] = {0, 0, 0, 0};
            for (uint32_t k = 0; k < most; k++) {
                const uint32_t en = ent[8 * li + k];
                const int off = (int)(en & 0xffu) - (int)(16 * q);
                if (!en || off <= -8 || off >= 16) continue;
                const uint32_t tag = 0x80u | ((en >> 22) & 0xcu) | ((en & 0x20000000u) ? 0u : 0x40u);
                uint32_t cw[2];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const uint32_t pat = (__umul24((en >> (8 + 4 * h)) & 0xfu, 0x204081u) & 0x01010101u) |
                                         ((__umul24((en >> (16 + 4 * h)) & 0xfu, 0x204081u) & 0x01010101u) << 1);
                    const uint32_t nz = (pat + 0x7f7f7f7fu) & 0x80808080u;
                    cw[h] = (pat | tag * 0x01010101u) & (nz | (nz - (nz >> 7)));
                }
                const uint64_t span = (uint64_t)cw[1] << 32 | cw[0];
                const uint32_t so = 8u * (uint32_t)(off < 0 ? -off : off & 7);
                const uint64_t s0 = off < 0 ? span >> so : span << so;                    // at byte 0 (or 8)
                const uint64_t s1 = off > 0 && (off & 7) ? span >> (64u - so) : 0ull;     // what it pushes out
                const uint64_t w0 = off < 8 ? s0 : 0ull, w1 = off < 8 ? (off < 0 ? 0ull : s1) : s0;
                const uint32_t c[4] = {(uint32_t)w0, (uint32_t)(w0 >> 32), (uint32_t)w1, (uint32_t)(w1 >> 32)};
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    const uint32_t occ = sb[b] & 0x80808080u;
                    sb[b] |= c[b] & ~(occ | (occ - (occ >> 7)));
                }
            }
            uint32_t out[4];
#pragma unroll
            for (int g = 0; g < 2; g++) {
                // pixel 8g + bb is bit 15 - bb of the window after the fine-scroll shift; reversed: bit 16 + bb
                const uint32_t rlo = __builtin_bitreverse32(((lo[g] << 8) | lo[g + 1]) << f);
                const uint32_t rhi = __builtin_bitreverse32(((hi[g] << 8) | hi[g + 1]) << f);
                const bool edge = q == 0 && g == 0;   // pixels 0-7 may hide either layer
                const uint32_t keep_bg = edge && hide_edge_bg() ? 0u : ~0u, keep_sp = edge && hide_edge_spr() ? 0u : ~0u;
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    // background pattern of the four pixels, one per byte (0..3)
                    const uint32_t nlo = (rlo >> (16 + 4 * h)) & 0xfu, nhi = (rhi >> (16 + 4 * h)) & 0xfu;
                    const uint32_t bgp = (((__umul24(nlo, 0x204081u) & 0x01010101u) |
                                           ((__umul24(nhi, 0x204081u) & 0x01010101u) << 1))) & keep_bg;
                    uint32_t word = byte_perm(gt[g + 1], gt[g], bgp | (h ? tsel1 : tsel0));
                    if (most) {
                        const uint32_t c = sb[2 * g + h];
                        const uint32_t opaque = (bgp + 0x7f7f7f7fu) & 0x80808080u;       // background pattern != 0
                        const uint32_t take = c & (~opaque | (c << 1)) & 0x80808080u & keep_sp;
                        const uint32_t tmask = take | (take - (take >> 7));
                        const uint32_t sel = c & 0x07070707u;
                        const uint32_t hi8 = (c << 4) & 0x80808080u;                    // entry 8..15
                        const uint32_t hmask = hi8 | (hi8 - (hi8 >> 7));
                        const uint32_t sg = (byte_perm(pal[7], pal[6], sel) & hmask) | (byte_perm(pal[5], pal[4], sel) & ~hmask);
                        word = (sg & tmask) | (word & ~tmask);
                    }
                    out[2 * g + h] = word;
                }
            }
            uint32_t* const w = (uint32_t*)gray + ((size_t)py * 64 + 4 * q) * gs;   // word of pixels 16q .. 16q+3
            const int xg = 16 * (int)q;
            if (xg >= x0 && xg + 16 <= x1) {
                // streaming stores: the frames are read once, after the frame loop
                if constexpr (ON_GPU) __builtin_nontemporal_store(mh_u32x4{out[0], out[1], out[2], out[3]}, (mh_u32x4*)w);
                else for (int b = 0; b < 4; b++) w[b * gs] = out[b];
            } else if (xg < x1 && xg + 16 > x0) {
                for (int b = 0; b < 16; b++)
                    if (xg + b >= x0 && xg + b < x1) ((uint8_t*)(w + (b >> 2) * gs))[b & 3] = (uint8_t)(out[b >> 2] >> (8 * (b & 3)));
            }
        }
    }

    // Of the n whole render lines from this one's start on, how many can go by at once: none that could raise the
    // sprite-0 hit (0: the first one could, or the scroll goes line by line because copy_h is off).
    __device__ __forceinline__ int plain_lines(int n) const {
        if (!show_bg()) return n;
        if (!show_spr()) return 0;
        if (s0hit) return n;
        if (sprite0_first()) return 0;
        if (oam_addr >= 4) return n;
        // the lists still to come: evaluated at the end of line s - 1 for line s, sprite 0 in range from y0 on
        const int y0 = (int)(oam_sprite(0) & 0xffu), h = long_spr() ? 16 : 8;
        const int first = y0 + 1 > scanline + 1 ? y0 + 1 : scanline + 1;
        if (first - 1 >= y0 + h) return n;
        const int k = first - scanline;
        return k < n ? k : n;
    }

    // advance the PPU by n calls (nes_core.hpp:539-616)
    __device__ __forceinline__ void ppu_run(int32_t n) {
        while (n > 0) {
            int c = pcyc;
            if (pstate == ST_RENDER) {
                if (c >= 1 && c <= 256) {
                    // whole lines, or a piece of one
                    const bool whole = c == 1 && n >= LINE_END;
                    int k = 0;
                    if (whole) {
                        const int left = 240 - scanline, due = n / LINE_END;
                        k = plain_lines(due < left ? due : left);
                    }
                    const int len = whole ? 256 : n < 257 - c ? n : 257 - c;
                    if (render) draw_lines(k > 0 ? (uint32_t)k : 1u, c - 1, c - 1 + len);
                    if (k == 0) {
                        dots_hit_scroll(c - 1, c - 1 + len);
                        if (whole) {
                            if (show_bg()) { fine_y_step(); if (show_spr()) copy_h(); }
                            k = 1;
                        }
                    } else if (show_bg()) {
                        v = v_lines_on((uint32_t)k);
                    }
                    if (k > 0) {
                        scanline += k;
                        ppu_calls += k * LINE_END; n -= k * LINE_END;
                        pend_line = scanline - 1;   // sprite evaluation for the next line (materialized lazily)
                        if (scanline >= 240) pstate = ST_POST;
                        continue;
                    }
                    pcyc += len; ppu_calls += len; n -= len;
                    c = pcyc;
                }
                if (n <= 0) {
                    // the calls ran out inside the visible dots
                } else if (c == 257) {
                    if (show_bg()) fine_y_step();
                    pcyc++; ppu_calls++; n--;
                } else if (c == 258) {
                    if (show_bg() && show_spr()) copy_h();
                    pcyc++; ppu_calls++; n--;
                } else if (c > 258 && c < LINE_END) {
                    const int k = n < LINE_END - c ? n : LINE_END - c;
                    pcyc += k; ppu_calls += k; n -= k;
                } else if (c >= LINE_END) {
                    pend_line = scanline;   // sprite evaluation for the next line (materialized lazily)
                    scanline++;
                    pcyc = 1; ppu_calls++; n--;
                    if (scanline >= 240) pstate = ST_POST;
                } else {
                    pcyc++; ppu_calls++; n--;
                }
            } else if (pstate == ST_PRE) {
                const bool on = show_bg() && show_spr();
                const int end = LINE_END - (!even && on);
                const int k = c >= end ? 1 : (n < end - c ? n : end - c);
                const int lo = c, hi = c + k;
                if (lo <= 1 && 1 < hi) vblank = s0hit = 0;
                if (on) {
                    if (lo <= 258 && 258 < hi) copy_h();
                    if (lo <= 304 && 281 < hi) copy_v();
                }
                ppu_calls += k; n -= k;
                if (hi - 1 >= end) { pstate = ST_RENDER; scanline = 0; pcyc = 1; }
                else pcyc = hi;
            } else if (pstate == ST_POST) {
                if (c >= LINE_END) { scanline++; pcyc = 1; pstate = ST_VBLANK; ppu_calls++; n--; }
                else { const int k = n < LINE_END - c ? n : LINE_END - c; pcyc += k; ppu_calls += k; n -= k; }
            } else {
                if (n >= LINE_END && scanline >= 241 && scanline < 260 && !(scanline == 241 && c <= 1) && c <= LINE_END) {
                    // whole lines of the vertical blank past its start, up to its last one, at the same dot
                    int k = n / LINE_END;
                    if (k > 260 - scanline) k = 260 - scanline;
                    scanline += k; ppu_calls += k * LINE_END; n -= k * LINE_END;
                } else if (c >= LINE_END) {
                    scanline++; pcyc = 1;
                    if (scanline >= 261) { pstate = ST_PRE; scanline = 0; even = !even; }
                    ppu_calls++; n--;
                } else if (c == 1 && scanline == 241) {
                    vblank = 1; ppu_calls++; n--; pcyc = 2;
                    if (nmi_en()) { nmi_call = ppu_calls; n = 0; }   // the caller raises it and goes on
                } else {
                    int lim = LINE_END - c;
                    if (scanline == 241 && c < 1) lim = 1 - c;
                    const int k = n < lim ? n : lim;
                    pcyc += k; ppu_calls += k; n -= k;
                }
            }
        }
    }

    // ------------------------------------------------------------ CPU (nes_core.hpp:619-899)
    __device__ __forceinline__ void set_nz(uint32_t r) { p = (p & ~(uint32_t)(FZ | FN)) | (r ? 0u : (uint32_t)FZ) | (r & 0x80 ? (uint32_t)FN : 0u); }
    __device__ __forceinline__ void push(uint32_t d) { set_ram(0x100 | sp, d); sp = (sp - 1) & 0xffu; }
    // NMI raised by PPU call `call` (1-based, frame-relative); nes_core.hpp:520-531
    __device__ __forceinline__ void nmi(int32_t call) {
        const int32_t it = (call - 1) / 3;
        push(pc >> 8); push(pc & 0xffu); push(p | 0x20);
        p |= FI;
        pc = prg(0xfffa) | prg(0xfffb) << 8;
        const int32_t d = (zero_skip && it == exec_at) ? 0 : (exec_at - it + 1);
        exec_at = it + d + 6;
        zero_skip = 0;
    }
#if defined(__AMDGCN__)
    // The CPU on the scalar unit from instruction j on, up to frame()'s stopping rules as one limit on the catch-up
    // point 3 (j + 1): at most 3 end (j < end), and no NMI check that needs a catch-up first (below nmi_thresh, or
    // already caught up to it). False if it ran nothing.
    __device__ __forceinline__ bool cpu_run(int32_t j, int32_t end, const uint32_t* recs) {
        int32_t lim = nmi_thresh - 1 > ppu_calls ? nmi_thresh - 1 : ppu_calls;
        lim = lim < 3 * end ? lim : 3 * end;
        const int32_t exlim = lim / 3 - 1;      // lim >= 3 (j + 1) > 0
        ScalarRegs r{a, x, y, sp, ((p & FN) ? 0x100u : 0u) | ((p & FZ) ? 0u : 1u), (p & FC) ? 1u : 0u, (p & FV) ? 0x80u : 0u,
                     p & ~(uint32_t)(FN | FV | FZ | FC), (uint32_t)(exlim - j) << 16, pc << 2};
        scalar_run(r, recs, (uint32_t)(uintptr_t)(m + ROW_RAM), (uint32_t)(uintptr_t)prg_);
        const uint32_t n = r.left & 0xffffu;
        if (!n) return false;
        a = r.a; x = r.x; y = r.y; sp = r.sp;
        p = r.p_rest | ((r.nz & 0x180u) ? (uint32_t)FN : 0u) | ((r.nz & 0xffu) ? 0u : (uint32_t)FZ) |
            (r.c ? (uint32_t)FC : 0u) | ((r.v & 0x80u) ? (uint32_t)FV : 0u);
        pc = (r.pc4 >> 2) & 0xffffu;
        exec_at = exlim - ((int32_t)r.left >> 16);
        zero_skip = 0;
        instructions += n;
        return true;
    }
#endif
    __device__ __forceinline__ void cross_penalty(uint32_t u, uint32_t w, int k) { if ((u ^ w) & 0xff00) skip += k; }

    // The data operation of decode word D: the result byte and the new flags, from the packed registers regs
    // (a | x << 8 | y << 16 | sp << 24), the data operand m (the first operand byte when nothing was read), the
    // flags p and whether a data operand was read. Every choice is a select on bits of the decode word (chains of equality
    // tests on one small field would be lowered to a branch tree).
    struct AluOut { uint32_t r8, p; };
    __device__ __forceinline__ static AluOut alu_op(uint32_t D, uint32_t regs, uint32_t m, uint32_t p, bool rd) {
        using namespace dec;
        const uint32_t alu = (D >> ALU_SH) & 15u, src = (D >> SRC_SH) & 7u, fl = (D >> FL_SH) & 7u;
        const uint32_t a = regs & 0xffu;
        const uint32_t rv = src ? (regs >> (8 * (src - 1))) & 0xffu : (uint32_t)m;   // R_A, R_X, R_Y, R_SP, or M
        const uint32_t sv = rd ? (uint32_t)m : rv;                // operand of the unary operations
        const uint32_t cin = (p & FC) ? 1u : 0u;
        const uint32_t sum = a + m + cin;                         // ADC
        const uint32_t dif = a - m - (1u - cin);                  // SBC
        const uint32_t cmp = rv - m;                              // CMP / CPX / CPY
        const bool u0 = alu & 1u, u1 = alu & 2u, u2 = alu & 4u, u3 = alu & 8u;
        const uint32_t rc = u0 ? cin : 0u;                        // ROL / ROR carry in
        // OP_ results by the bits of alu: PASS ORA AND EOR ADC SBC CMP BIT ASL ROL LSR ROR INC DEC FLAG NOP
        const uint32_t g0 = u0 ? (uint32_t)(a | m) : sv, g1 = u0 ? (uint32_t)(a ^ m) : (uint32_t)(a & m);
        const uint32_t g2 = u0 ? dif : sum, g3 = u0 ? sv : cmp;
        const uint32_t g4 = (sv << 1) | rc, g5 = (sv >> 1) | (rc << 7), g6 = u0 ? sv - 1 : sv + 1, g7 = sv;
        const uint32_t h0 = u1 ? g1 : g0, h1 = u1 ? g3 : g2, h2 = u1 ? g5 : g4, h3 = u1 ? g7 : g6;
        const uint32_t res = u3 ? (u2 ? h3 : h2) : (u2 ? h1 : h0);
        const uint32_t r8 = res & 0xffu;
        // carry: ADC bit 8 of the sum; SBC / CMP no borrow; ASL / ROL bit 7; LSR / ROR bit 0
        const uint32_t c_sub = ((res >> 8) & 1u) ^ 1u, c_adc = (sum >> 8) & 1u;
        const uint32_t carry = u3 ? (u1 ? (sv & 1u) : ((sv >> 7) & 1u)) : ((u0 | u1) ? c_sub : c_adc);
        const uint32_t ovf = u0 ? ((a ^ dif) & (~(uint32_t)m ^ dif) & 0x80u) : ((a ^ sum) & (m ^ sum) & 0x80u);
        // flag groups NONE NZ NZC NZCV BIT OP as masks of the bits they replace
        const uint32_t nzv = (r8 ? 0u : FZ) | (r8 >> 7);          // FN is bit 0
        const uint32_t fz = (a & m) ? 0u : FZ;
        const uint32_t bitv = fz | (m & 0x40 ? FV : 0u) | (m >> 7);
        const uint32_t fop = (D >> FOP_SH) & 7u;
        const uint32_t fm = fop < 2 ? FC : fop < 4 ? FI : fop == 4 ? FV : FD;   // CLC SEC CLI SEI CLV CLD SED
        const uint32_t fset = (fop == 1 || fop == 3 || fop == 6) ? fm : 0u;
        uint32_t keep = 0xffu, set = 0u;
        if ((0xeu >> fl) & 1u) { keep &= ~(uint32_t)(FZ | FN); set |= nzv; }             // NZ, NZC, NZCV
        if ((0xcu >> fl) & 1u) { keep &= ~(uint32_t)FC; set |= carry ? FC : 0u; }        // NZC, NZCV
        if (fl == FL_NZCV) { keep &= ~(uint32_t)FV; set |= ovf ? FV : 0u; }
        if (fl == FL_BIT) { keep &= ~(uint32_t)(FZ | FV | FN); set |= bitv; }
        if (fl == FL_OP) { keep &= ~fm; set |= fset; }
        return AluOut{r8, (p & keep) | set};
    }

    // One whole instruction from its decode word: addressing, at most one data read and one data
    // write through the bus, the ALU as register selects, and one small switch for the stack /
    // control-flow operations, in the reference's bus order (operand bytes, pointer, data read, data
    // write; JSR pushes before reading its operand; a branch reads its offset only when taken). It runs what
    // scalar_run leaves: invalid opcodes, code outside PRG, computed addresses of registers, BRK.
    // `pf`: the opcode and both following bytes are in PRG (pc <= 0xfffd); otherwise they are fetched through the bus,
    // with the PPU caught up first because a fetch may hit a PPU register. Returns false, with no effect, when the
    // PPU must be caught up to `tgt` first; the caller does that and starts the instruction again.
    __device__ __forceinline__ bool instruction(int32_t j, int32_t tgt) {
        using namespace dec;
        const bool pf = pc >= 0x8000u && pc <= 0xfffdu;
        if (!pf && ppu_calls < tgt) return false;
        uint32_t op, b1 = 0, b2 = 0, D;
        if (!pf) {
            op = read(pc);
            D = dec[op];
            const uint32_t xop0 = (D >> X_SH) & 15u;
            if (xop0 != X_JSR && xop0 != X_BRANCH) {   // JSR and branches fetch below, in their order
                const uint32_t am0 = D & 15u;
                if (am0 != M_NONE) b1 = read((pc + 1) & 0xffffu);
                if (am0 == M_ABS || am0 == M_ABSX || am0 == M_ABSY) b2 = read((pc + 2) & 0xffffu);
            }
        } else {
            op = prg(pc); b1 = prg(pc + 1); b2 = prg(pc + 2);
            D = dec[op];
        }
        const uint32_t am = D & 15u, xop = (D >> X_SH) & 15u, dst = (D >> DST_SH) & 7u;
        const bool rd = (D & RD) != 0, wr = dst == D_MEM;
        const uint32_t mb = 1u << am;
        constexpr uint32_t X_IDX = 1u << M_ZPX | 1u << M_ABSX, Y_IDX = 1u << M_ZPY | 1u << M_ABSY | 1u << M_INDY;
        constexpr uint32_t ZP_EA = 1u << M_ZP | 1u << M_ZPX | 1u << M_ZPY, IND = 1u << M_INDX | 1u << M_INDY;
        const uint32_t absv = b1 | b2 << 8;
        uint32_t base = absv;
        if (mb & IND) {   // pointer from the zero page
            const uint32_t z = am == M_INDX ? (b1 + x) & 0xffu : b1;
            base = ram(z) | ram((z + 1) & 0xffu) << 8;
        }
        const uint32_t idx = (mb & X_IDX) ? x : (mb & Y_IDX) ? y : 0u;
        const uint32_t ea = (mb & ZP_EA) ? (b1 + idx) & 0xffu : am == M_IMM ? (pc + 1) & 0xffffu : (base + idx) & 0xffffu;
        const uint32_t p2 = (absv & 0xff00) | ((absv + 1) & 0xff);   // JMP (ind): high byte, page wrap
        const bool sync = xop == X_JMPI ? (needs_sync(absv, false) || needs_sync(p2, false))
                                        : ((rd && needs_sync(ea, false)) || (wr && needs_sync(ea, true)));
        if (sync && ppu_calls < tgt) return false;   // only when pf: no bus access has happened yet
        cur = j;
        skip = 0;
        instructions++;
        if (D & PEN) cross_penalty(base, base + idx, 1);
        // data operand and ALU
        const uint32_t mv = rd && am != M_IMM ? read(ea) : b1;
        const AluOut ao = alu_op(D, a | x << 8 | y << 16 | sp << 24, mv, p, rd);
        p = ao.p;
        const uint32_t r8 = ao.r8;
        if (dst == D_A) a = r8;
        if (dst == D_X) x = r8;
        if (dst == D_Y) y = r8;
        if (dst == D_SP) sp = r8;
        if (wr) write(ea, r8);
        // control flow: the next pc by instruction length, branches and JMP
        constexpr uint32_t ABS3 = 1u << M_ABS | 1u << M_ABSX | 1u << M_ABSY;
        const uint32_t ret = (pc + 2) & 0xffffu;
        uint32_t npc = (pc + (am == M_NONE ? 1 : (mb & ABS3) ? 3 : 2)) & 0xffffu;
        switch (xop) {
            case X_BRANCH: {   // on N, V, C, Z (op bits 6-7) equal to op bit 5; 2 bytes; the offset is read only when taken
                const uint32_t fbit = (0x40800201u >> (8 * (op >> 6))) & 0xffu;   // FN FV FC FZ
                npc = ret;
                if (((p & fbit) != 0) == ((op & 0x20) != 0)) {
                    const uint32_t off = pf ? b1 : read((pc + 1) & 0xffffu);
                    npc = (ret + (uint32_t)(int32_t)(int8_t)off) & 0xffffu;
                    skip += ((ret ^ npc) & 0xff00) ? 3 : 1;
                }
                break;
            }
            case X_JMP: npc = absv; break;
            case X_BRK:
                push(ret >> 8); push(ret & 0xffu); push(p | 0x30);
                p |= FI; npc = prg(0xfffe) | prg(0xffff) << 8; skip += 7;
                break;
            case X_JSR:
                push(ret >> 8); push(ret & 0xffu);
                npc = absv;
                if (!pf) { const uint32_t lo = read((pc + 1) & 0xffffu); npc = lo | read((pc + 2) & 0xffffu) << 8; }
                break;
            case X_PHA: push(a); break;
            case X_PHP: push(p); break;
            case X_RTS: { const uint32_t lo = pull(); npc = ((lo | pull() << 8) + 1) & 0xffffu; break; }
            case X_RTI: { p = pull(); const uint32_t lo = pull(); npc = lo | pull() << 8; break; }
            case X_PLA: a = pull(); set_nz(a); break;
            case X_PLP: p = pull(); break;
            case X_JMPI: { const uint32_t lo = read(absv); npc = lo | read(p2) << 8; break; }
            default: break;
        }
        pc = npc;
        if (D & OK) skip += (int)((D >> CYC_SH) & 7u);
        else bad_ops++;
        exec_at = j + (skip >= 1 ? skip : 1);
        zero_skip = skip <= 0;
        return true;
    }
    __device__ __forceinline__ uint32_t pull() { sp = (sp + 1) & 0xffu; return ram(0x100 | sp); }

    // PPU calls from the current PPU position to (line, dot) on the frame timeline of
    // nmi_threshold() (pre-render line = -1, 262 x 341 calls); the one-dot-shorter odd pre-render
    // line is not modelled, so callers keep a margin. 0 means the very next call processes that dot.
    __device__ __forceinline__ int32_t calls_until(int line, int dot) const {
        const int now_line = pstate == ST_PRE ? -1 : pstate == ST_POST ? 240 : scanline;
        int32_t d = ((line + 1) * 341 + (dot - 1)) - ((now_line + 1) * 341 + (pcyc - 1));
        if (d < 0) d += 262 * 341;
        return d;
    }

    // PPU calls (a frame-relative count) up to which a catch-up moves nothing but the position: in the vertical blank,
    // past its start and up to the pre-render line, whose first dot clears the flags. -1 elsewhere.
    __device__ __forceinline__ int32_t quiet_until() const {
        return pstate == ST_VBLANK && !(scanline == 241 && pcyc <= 1) ? ppu_calls + calls_until(-1, 1) : -1;
    }

    // While sprite 0 heads the list of the line being drawn: PPU calls from now up to the one that raises the hit on
    // the rest of this line or the 7 lines after it (nothing writes to the PPU meanwhile), or else to the first dot past
    // them. Lane 8 i + k tests pixel k of the sprite on the i-th line. A wait loop read $2002 every 27 dots of these lines
    // before, with a catch-up, a piece of a line to draw and a status read each: k_step of 256 / 32,768 envs 0.87 -> 0.85 /
    // 7.75 -> 7.40 ms.
    __device__ __forceinline__ int32_t calls_to_hit() const {
        if (show_bg() && show_spr()) {
            const uint32_t ow = oam_sprite(0);
            const int sx = (int)(ow >> 24), y0 = (int)(ow & 0xffu), h = long_spr() ? 16 : 8;
            const int edge = hide_edge_spr() || hide_edge_bg() ? 8 : 0;
            auto hits = [&](int l) {
                const int i = l >> 3, px = sx + (l & 7), py = scanline + i, x0 = i ? 0 : pcyc - 1;
                // its later lists: evaluated at the end of the line before, from sprite 0 on
                const bool listed = i == 0 || (oam_addr < 4 && (uint32_t)(py - 1 - y0) < (uint32_t)h);
                if (!listed || py > 239 || px > 255 || px < x0 || px < edge) return false;
                // (past dot 257 v has stepped to the next line already)
                const uint32_t vl = i ? v_lines_on((uint32_t)(i - (pcyc > 257 ? 1 : 0))) : v;
                const uint32_t vp = coarse_x_added(vl, (uint32_t)inc_count(x0, px));
                return bg_pattern(px, vp) && sprite0_pattern(ow, px, py);
            };
            uint64_t b = 0;
            if constexpr (ON_GPU) b = __ballot(hits((int)lane));
            else for (int l = 63; l >= 0; l--) b = b << 1 | (uint64_t)hits(l);
            if (b) {
                const int l = __builtin_ctzll(b);
                return calls_until(scanline + (l >> 3), sx + (l & 7) + 1) + 1;
            }
        }
        return calls_until(scanline + 8 < 240 ? scanline + 8 : 240, 1);
    }

    // Exact fast-forward of the sprite-0 wait loops `LDA $2002 / AND #$40 / BEQ|BNE *-5` at pc (BEQ:
    // wait for the hit, BNE: wait for the clear at the pre-render line), with the PPU caught up to the
    // read of the first iteration (at j). Iterations whose $2002 reads provably return the same value
    // are not executed: they would only re-read an unchanged s0hit, clear an already clear vblank flag
    // and set first_write, and the PPU is caught up lazily anyway. The span ends before the first dot
    // where s0hit could change (the hit itself on a line that sprite 0 is on, its first line before that, or the
    // pre-render clear), before the NMI sync
    // point and inside the frame. Returns true if it advanced.
    __device__ __forceinline__ bool poll_skip(int32_t j, int32_t end, bool wait_hit) {
        if (wait_hit == (s0hit != 0)) return false;   // this read ends the loop: run it normally
        int32_t limit;                           // first PPU call count at which s0hit may differ
        if (wait_hit) {
            // A hit needs sprite 0 at the head of the list of the line being drawn. The list already
            // evaluated serves the current line (in RENDER) or line 0 of the next frame (elsewhere).
            // The lists still to come are evaluated at the ends of render lines m (the current one
            // onwards in RENDER, 0 onwards elsewhere) and serve line m + 1 (240: line 0 of the next
            // frame); with OAM, oam_addr and sprite size fixed (the loop writes nothing) sprite 0 can
            // head one only for y0 <= m < y0 + h.
            const int y0 = (int)(oam_sprite(0) & 0xffu), h = long_spr() ? 16 : 8;
            const int m = pstate == ST_RENDER && scanline > y0 ? scanline : y0;
            if (pstate == ST_RENDER && sprite0_first()) limit = ppu_calls + calls_to_hit();   // on the line being drawn
            else if (m <= 239 && m < y0 + h) limit = ppu_calls + calls_until(m + 1, 1) - 2;
            else if (y0 <= 238) limit = ppu_calls + calls_until(y0 + 1, 1) - 2;   // next frame
            else limit = 0x7fffffff;
            if (pstate != ST_RENDER && sprite0_first()) {
                const int32_t l0 = ppu_calls + calls_until(0, 1) - 2;
                if (l0 < limit) limit = l0;
            }
        } else {
            limit = ppu_calls + calls_until(-1, 1) - 2;
        }
        const int32_t c = 9 + ((((pc + 7) ^ pc) & 0xff00) ? 2 : 0);   // LDA 4 + AND 2 + taken branch 3 (+2)
        // start jl of the last skipped iteration: its three instructions start before the frame end
        // and below the NMI check, and its read precedes `limit`
        int32_t jl = end - 7;
        const int32_t by_nmi = (nmi_thresh - 1) / 3 - 7;
        const int32_t by_limit = (limit - 1) / 3 - 1;
        if (by_nmi < jl) jl = by_nmi;
        if (by_limit < jl) jl = by_limit;
        if (jl < j) return false;
        const int32_t k = (jl - j) / c + 1;
        vblank = 0;
        first_write = 1;
        a = s0hit ? 0x40 : 0x00;
        set_nz(a);
        exec_at = j + k * c;
        zero_skip = 0;
        instructions += 3 * (uint32_t)k;
        ff_instructions += 3 * (uint32_t)k;
        return true;
    }
};

// The functions of a console: registers in, registers out. Each is inlined at one place of run_frame(): only the file
// and the CPU's registers live across them. (As calls, every entry and return waited for the frame stores in flight.)
#if defined(__AMDGCN__)
#define MH_FN __device__ __attribute__((noinline))
#else
#define MH_FN inline
#endif
// The PPU caught up to `target` calls, or to the call that raises an NMI (F_NMI_CALL) if that comes before.
__device__ __forceinline__ File ppu_advance(File f, Ctx c, int32_t target) {
    Core k;
    k.attach(c);
    k.open_ppu(f);
    target = (int32_t)uni((uint32_t)target);
    k.nmi_call = 0;
    if (target > k.ppu_calls) {
        k.ppu_run(target - k.ppu_calls);
        k.nmi_threshold();
    }
    k.close_ppu(f);
    f.set(F_QUIET, (uint32_t)k.quiet_until());
    return f;
}
// An absolute access of instruction j to a register (record `rec`, REC_STORE of `val` or REC_LOAD). data: what was read;
// skip: the instruction's cycles.
struct IoResult { File f; uint32_t data; int32_t skip; };
__device__ __forceinline__ IoResult io_access(File f, Ctx c, uint32_t rec, uint32_t val, int32_t j) {
    rec = uni(rec); val = uni(val);
    const uint32_t ad = rec >> 16, r = ad & 7u;
    const bool st = (rec & 0xf0u) == REC_STORE;
    Core k;
    // the frequent ones open only the words they use (a word is a lane read, and a lane write where it changes)
    if (!st && ad >= 0x4000u) {                             // the joypads
        k.joy = f.get(F_JOY); k.joy_strobe = f.get(F_JOY_STROBE);
        const uint32_t d = k.pad_read((int)(ad & 1u));
        f.set(F_JOY, k.joy);
        return IoResult{f, d, 4};
    }
    if (st && ad < 0x4000u && r >= 5u) {                    // scroll, address, data
        k.v = f.get(S_V);
        if (r == 7u) {
            k.m = c.memory(); k.nt_bits = c.name_tables(); k.ppu_flags = f.get(F_PPU_FLAGS); k.pal_dirty = f.get(F_PAL_DIRTY);
            k.data_write(val);
            f.set(S_V, k.v); f.set(F_PAL_DIRTY, k.pal_dirty);
            return IoResult{f, 0, 4};
        }
        k.t = f.get(S_T); k.first_write = f.get(S_FIRST_WRITE);
        if (r == 6u) { k.addr_write(val); f.set(S_V, k.v); }
        else { k.fine_x = f.get(S_FINE_X); k.scroll_write(val); f.set(S_FINE_X, k.fine_x); }
        f.set(S_T, k.t); f.set(S_FIRST_WRITE, k.first_write);
        return IoResult{f, 0, 4};
    }
    if (!st && r == 2u) {
        k.s0hit = f.get(S_S0HIT); k.vblank = f.get(S_VBLANK);
        const uint32_t d = k.status_read();
        f.set(S_VBLANK, k.vblank); f.set(S_FIRST_WRITE, k.first_write);
        return IoResult{f, d, 4};
    }
    k.attach(c);
    k.open_io(f);
    k.cur = (int32_t)uni((uint32_t)j);
    k.skip = 4;
    uint32_t d = 0;
    if (st) k.write(ad, val);
    else d = k.read(ad);
    k.close_io(f);
    return IoResult{f, d, k.skip};
}
// poll_skip at instruction j; f's CPU words hold pc (in) and a, p, exec_at, zero_skip (out). F_NMI_CALL: 1 if it advanced.
__device__ __forceinline__ File poll_wait(File f, Ctx c, int32_t j, int32_t end, uint32_t wait_hit) {
    Core k;
    k.attach(c);
    k.open_ppu(f);
    k.open_cpu(f);
    k.first_write = f.get(S_FIRST_WRITE);
    const bool on = k.poll_skip((int32_t)uni((uint32_t)j), (int32_t)uni((uint32_t)end), uni(wait_hit) != 0);
    k.close_cpu(f);
    f.set(S_VBLANK, k.vblank);
    f.set(S_FIRST_WRITE, k.first_write);
    f.set(F_NMI_CALL, on ? 1u : 0u);
    return f;
}
// One whole instruction j, CPU words in f. F_NMI_CALL: 1 if the PPU must be caught up to `tgt` first (nothing done).
__device__ __forceinline__ File whole_instruction(File f, Ctx c, int32_t j, int32_t tgt) {
    Core k;
    k.attach(c);
    k.open_io(f);
    k.open_cpu(f);
    const bool done = k.instruction((int32_t)uni((uint32_t)j), (int32_t)uni((uint32_t)tgt));
    k.close_io(f);
    k.close_cpu(f);
    f.set(F_NMI_CALL, done ? 0u : 1u);
    return f;
}
// The sprite list of a pending evaluation, before the registers leave the kernel or its inputs change
MH_FN File sprites_listed(File f, Ctx c) {
    Core k;
    k.attach(c);
    k.open_ppu(f);
    k.materialize_sprites();
    k.close_sprites(f);
    return f;
}

// One nes-py Emulator::step (nes_core.hpp:1166-1204) with the exact `JMP *` idle fast-forward.
//
// The CPU runs ahead (scalar_run) until something needs the PPU or a rule of its own: the NMI point, an access to a
// PPU register (the catch-up point of instruction j is 3 (j + 1)), the frame end. The records say what an
// instruction that stops a run is; the common ones (the registers' absolute loads and stores, the idle loop, the
// sprite-0 wait) are handled here, the rest by instruction().
// While rendering is off (both PPUMASK show bits clear), the catch-up PPU neither moves v nor draws anything but
// the universal background colour, so the scroll and address writes and the $2007 writes to the pattern or name
// tables do not depend on where the PPU has been caught up to, and are made without a catch-up. ($2007 writes
// to the palette, $3EFF-$3FFE, change that colour.)
// Nor does any access from the start of the vertical blank to its end (quiet_until): what it reads and changes is then
// the same wherever the PPU stands in it. That is where a program's updates are: of the 31 register accesses of a
// frame (a level of the test cartridge) 28 had a catch-up of their own. Without those, and with the frequent registers
// opening only their own words in io_access(): k_step of 256 / 32,768 envs 1.03 -> 0.89 / 9.0 -> 8.2 ms.
MH_FN File run_frame(File f, Ctx c) {
    constexpr int32_t end = FRAME_ITERS, last_call = 3 * FRAME_ITERS;
    Core k;                                     // its CPU registers, memory and PPU position only
    k.attach(c);
    k.open_cpu(f);
    k.ppu_calls = (int32_t)f.get(F_PPU_CALLS); k.nmi_thresh = (int32_t)f.get(F_NMI_THRESH);
#if defined(__AMDGCN__)
    const MH_SCALAR_CONST uint32_t* const recs =
        (const MH_SCALAR_CONST uint32_t*)((uint64_t)c.w.get(Ctx::RECS_LO) | (uint64_t)c.w.get(Ctx::RECS_HI) << 32);
    auto record = [&](uint32_t ad) { return recs[ad]; };
#else
    // (the host build runs every instruction in C++)
    auto record = [&](uint32_t ad) { return decode_record(c.cart.prg, ad, c.cart.dec) & 0xffff00ffu; };
#endif
    int32_t want = -1;                          // catch the PPU up to here first
    int32_t quiet = -1;                         // accesses up to this call need no catch-up
    bool over = false;                          // the CPU is at the frame end
    for (;;) {
        if (want >= 0) {
            f = ppu_advance(f, c, want);
            quiet = (int32_t)f.get(F_QUIET);
            k.ppu_calls = (int32_t)f.get(F_PPU_CALLS); k.nmi_thresh = (int32_t)f.get(F_NMI_THRESH);
            const int32_t call = (int32_t)f.get(F_NMI_CALL);
            if (call) { k.nmi(call); if (k.ppu_calls < want) continue; }
            if (over) break;
            want = -1;
        }
        if (k.exec_at >= end) { want = last_call; over = true; continue; }
        const int32_t j = k.exec_at, tgt = 3 * (j + 1);
        if (tgt >= k.nmi_thresh && k.ppu_calls < tgt) { want = tgt; continue; }
        const uint32_t rec = record(k.pc), kind = rec & 0xf0u;
        if (rec & 0xff00u) {
#if defined(__AMDGCN__)
            if (k.cpu_run(j, end, (const uint32_t*)recs)) continue;
#endif
        } else if (kind == REC_IDLE) {
            const int32_t lim_end = end - j, lim_nmi = k.nmi_thresh - tgt;
            const int32_t k1 = lim_end > 0 ? (lim_end + 2) / 3 : 0;
            const int32_t k2 = lim_nmi > 0 ? (lim_nmi + 8) / 9 : 0;
            const int32_t kk = k1 < k2 ? k1 : k2;
            if (kk > 1) { k.exec_at = j + 3 * (kk - 1); k.zero_skip = 0; continue; }
        } else if (kind >= REC_STORE) {
            const uint32_t ad = rec >> 16, reg = rec >> 2 & 3u;
            const bool st = kind == REC_STORE;
            bool lazy = tgt <= quiet;
            if (!lazy && st && ad < 0x4000u && (ad & 7u) >= 5u && !(f.get(F_PPU_FLAGS) & (PF_SHOW_BG | PF_SHOW_SPR)))
                lazy = (ad & 7u) != 7u || f.get(S_V) - 0x3effu >= 0x100u;
            if (!lazy && k.ppu_calls < tgt && Core::needs_sync(ad, st)) { want = tgt; continue; }
            if (kind >= REC_POLL) {
                k.close_cpu(f);
                f = poll_wait(f, c, j, end, kind == REC_POLL_HIT);
                k.open_cpu(f);
                if (f.get(F_NMI_CALL)) continue;
            }
            const IoResult o = io_access(f, c, rec, reg == 0 ? k.a : reg == 1 ? k.x : k.y, j);
            f = o.f;
            if (!st) {
                const uint32_t d = uni(o.data);
                if (reg == 3u) {   // BIT
                    k.p = (k.p & ~(uint32_t)(FZ | FV | FN)) | ((k.a & d) ? 0u : (uint32_t)FZ) | ((d & 0x40u) ? (uint32_t)FV : 0u) | (d >> 7);
                } else {
                    if (reg == 0) k.a = d; else if (reg == 1) k.x = d; else k.y = d;
                    k.set_nz(d);
                }
            }
            k.instructions++;
            k.pc = (k.pc + 3) & 0xffffu;
            k.exec_at = j + (int32_t)uni((uint32_t)o.skip);
            k.zero_skip = 0;
            continue;
        }
        k.close_cpu(f);
        f = whole_instruction(f, c, j, tgt);
        k.open_cpu(f);
        if (f.get(F_NMI_CALL)) want = tgt;
    }
    // rebase the frame-relative counters on the new frame start
    k.exec_at -= FRAME_ITERS;
    k.close_cpu(f);
    f.set(F_PPU_CALLS, (uint32_t)(k.ppu_calls - 3 * FRAME_ITERS));
    f.set(F_NMI_THRESH, (uint32_t)(k.nmi_thresh - 3 * FRAME_ITERS));
    const uint32_t lo0 = f.get(S_ITER_LO), lo = lo0 + FRAME_ITERS;
    f.set(S_ITER_HI, f.get(S_ITER_HI) + (lo < lo0 ? 1u : 0u));
    f.set(S_ITER_LO, lo);
    return f;
}

// A console of the env layer and the kernels.
struct Console {
    MH_LDS uint8_t* m;       // its memory in LDS, between load() / power_on() and store()
    MH_LDS uint32_t* gp;
    Cart cart;
    const MH_LDS uint8_t* lut;
    uint32_t np;             // envs of the memory block, padded
    uint32_t lane;
    uint8_t* gray;           // the frame buffer frame() draws into, if `render`
    bool render;
    File f;
    uint32_t bad_ops, instructions, ff_instructions;
    uint32_t nframe;         // frame() calls since load(): the wave's issue priority in frame()

    __device__ __forceinline__ Ctx ctx() const {
        Ctx c;
#if defined(__AMDGCN__)
        c.w.r = 0;
        auto ptr = [&](int k, uint64_t p) { c.w.set(k, (uint32_t)p); c.w.set(k + 1, (uint32_t)(p >> 32)); };
        c.w.set(Ctx::M, (uint32_t)(uintptr_t)m); c.w.set(Ctx::GP, (uint32_t)(uintptr_t)gp);
        c.w.set(Ctx::PRG, (uint32_t)(uintptr_t)cart.prg); c.w.set(Ctx::CHR, (uint32_t)(uintptr_t)cart.chr);
        c.w.set(Ctx::LUT, (uint32_t)(uintptr_t)lut); ptr(Ctx::DEC_LO, (uint64_t)cart.dec); ptr(Ctx::RECS_LO, (uint64_t)cart.recs);
        ptr(Ctx::GRAY_LO, (uint64_t)gray); c.w.set(Ctx::NT_BITS, cart.nt_bits); c.w.set(Ctx::NP, np); c.w.set(Ctx::RENDER, render);
#else
        c.m = m; c.gp = gp; c.cart = cart; c.gray = gray; c.lut = lut; c.np = np; c.render = render;
#endif
        return c;
    }
    __device__ __forceinline__ uint32_t ram(uint32_t ad) const { return uni(m[ROW_RAM + (ad & 0x7ff)]); }
    __device__ __forceinline__ void set_ram(uint32_t ad, uint32_t val) { m[ROW_RAM + (ad & 0x7ff)] = (uint8_t)val; }
    // joypad port 0's buttons for the next frames (the env layer's action)
    __device__ __forceinline__ void set_buttons0(uint32_t b) { f.set(F_JOY, (f.get(F_JOY) & ~0xffu) | b); }
    __device__ __forceinline__ static void mem_sync() { Core::mem_sync(); }

    // ---- the register words of a block: lane k loads and stores word k
    __device__ __forceinline__ void load_regs(const uint32_t* sc, uint32_t e) {
#if defined(__AMDGCN__)
        f.r = sc[(size_t)(lane < S_COUNT ? lane : 0u) * np + e];
#else
        for (int k = 0; k < S_COUNT; k++) f.r[k] = sc[(size_t)k * np + e];
#endif
        auto w = [&](int k) { return f.get(k); };
        f.set(F_PPU_FLAGS, (w(S_SHOW_BG) ? PF_SHOW_BG : 0u) | (w(S_SHOW_SPR) ? PF_SHOW_SPR : 0u) |
                           (w(S_HIDE_EDGE_BG) ? PF_HIDE_EDGE_BG : 0u) | (w(S_HIDE_EDGE_SPR) ? PF_HIDE_EDGE_SPR : 0u) |
                           (w(S_LONG_SPR) ? PF_LONG_SPR : 0u) | (w(S_NMI_EN) ? PF_NMI_EN : 0u) |
                           (w(S_BG_PAGE) ? PF_BG_PAGE : 0u) | (w(S_SPR_PAGE) ? PF_SPR_PAGE : 0u) |
                           (w(S_INC) == 32 ? PF_INC32 : 0u));
        f.set(F_JOY, (w(S_JOY_BUTTONS0) & 0xffu) | (w(S_JOY_BUTTONS1) & 0xffu) << 8 | (w(S_JOY_BITS0) & 0xffu) << 16 |
                     (w(S_JOY_BITS1) & 0xffu) << 24);
        f.set(F_JOY_STROBE, (w(S_JOY_STROBE0) & 1u) | (w(S_JOY_STROBE1) & 1u) << 1);
        started();
    }
    __device__ __forceinline__ void started() {
        f.set(F_PEND_LINE, 0xffffffffu); f.set(F_PAL_DIRTY, 1); f.set(F_PPU_CALLS, 0); f.set(F_NMI_CALL, 0);
        f.set(F_BAD, 0); f.set(F_INSTR, 0); f.set(F_FF, 0);
        Core k;
        k.pstate = f.get(S_PSTATE); k.scanline = (int32_t)f.get(S_SCANLINE); k.pcyc = (int32_t)f.get(S_PCYC); k.ppu_calls = 0;
        k.nmi_threshold();
        f.set(F_NMI_THRESH, (uint32_t)k.nmi_thresh);
        nframe = 0;
    }
    __device__ __forceinline__ void store_regs(uint32_t* sc, uint32_t e) {
        f = sprites_listed(f, ctx());
        const uint32_t fl = f.get(F_PPU_FLAGS), joy = f.get(F_JOY), js = f.get(F_JOY_STROBE);
        auto w = [&](int k, uint32_t val) { f.set(k, val); };
        w(S_JOY_STROBE0, js & 1u); w(S_JOY_STROBE1, (js >> 1) & 1u);
        w(S_JOY_BUTTONS0, joy & 0xffu); w(S_JOY_BUTTONS1, (joy >> 8) & 0xffu);
        w(S_JOY_BITS0, (joy >> 16) & 0xffu); w(S_JOY_BITS1, joy >> 24);
        w(S_SHOW_BG, fl & PF_SHOW_BG ? 1u : 0u); w(S_SHOW_SPR, fl & PF_SHOW_SPR ? 1u : 0u);
        w(S_HIDE_EDGE_BG, fl & PF_HIDE_EDGE_BG ? 1u : 0u); w(S_HIDE_EDGE_SPR, fl & PF_HIDE_EDGE_SPR ? 1u : 0u);
        w(S_LONG_SPR, fl & PF_LONG_SPR ? 1u : 0u); w(S_NMI_EN, fl & PF_NMI_EN ? 1u : 0u);
        w(S_BG_PAGE, fl & PF_BG_PAGE ? 1u : 0u); w(S_SPR_PAGE, fl & PF_SPR_PAGE ? 1u : 0u);
        w(S_INC, fl & PF_INC32 ? 32u : 1u);
#if defined(__AMDGCN__)
        if (lane < S_COUNT) sc[(size_t)lane * np + e] = f.r;
#else
        for (int k = 0; k < S_COUNT; k++) sc[(size_t)k * np + e] = f.r[k];
#endif
    }
    // ---- the memory of console e of a block: to LDS, and back
    __device__ __forceinline__ void load_rows(const uint8_t* mem, uint32_t e) {
        if constexpr (ON_GPU) {
            const mh_u32x4* src = (const mh_u32x4*)(mem + mem_offset(np, e, 0));
#pragma unroll
            for (uint32_t i = lane; i < MEM_ROWS / 16; i += 64) ((MH_LDS mh_u32x4*)m)[i] = src[i];
            Core::lds_sync();
        } else {
            for (uint32_t r = 0; r < MEM_ROWS; r++) m[r] = mem[mem_offset(np, e, r)];
        }
    }
    __device__ __forceinline__ void store_rows(uint8_t* mem, uint32_t e) const {
        if constexpr (ON_GPU) {
            mh_u32x4* dst = (mh_u32x4*)(mem + mem_offset(np, e, 0));
#pragma unroll
            for (uint32_t i = lane; i < MEM_ROWS / 16; i += 64) dst[i] = ((const MH_LDS mh_u32x4*)m)[i];
        } else {
            for (uint32_t r = 0; r < MEM_ROWS; r++) mem[mem_offset(np, e, r)] = m[r];
        }
    }
    // the whole console e of a memory block and its register words
    __device__ __forceinline__ void load(const uint8_t* mem, const uint32_t* sc, uint32_t e) { load_regs(sc, e); load_rows(mem, e); }
    __device__ __forceinline__ void store(uint8_t* mem, uint32_t* sc, uint32_t e) { store_regs(sc, e); store_rows(mem, e); }

    // power-on: zeroed machine, then CPU and PPU reset (nes_core.hpp:123-147)
    __device__ __forceinline__ void power_on() {
        for (uint32_t i = lane; i < MEM_ROWS / 4; i += LANES) ((MH_LDS uint32_t*)m)[i] = 0;
        Core::lds_sync();
        auto prg = [&](uint32_t ad) { return uni(cart.prg[ad & 0x7fff]); };
        for (int k = 0; k < F_COUNT; k++) f.set(k, 0);
        f.set(S_P, 0x34); f.set(S_PC, prg(0xfffc) | prg(0xfffd) << 8); f.set(S_SP, 0xfd);
        f.set(F_JOY_STROBE, 3); f.set(S_EVEN, 1); f.set(F_PPU_FLAGS, PF_SHOW_BG | PF_SHOW_SPR); f.set(S_FIRST_WRITE, 1);
        f.set(S_PSTATE, ST_PRE);
        started();
    }
    __device__ __forceinline__ void frame() {
        // The kernel ends with its slowest wave, and the waves of a SIMD compete for its issue slots: a wave at an
        // earlier frame since its console's load issues first (frames 0 and 1 at priority 3, frame 2 at 2, later ones at 1;
        // the observations after the frame loop at 0; a snapshot taken back is a load too), so a wave that falls behind
        // takes the slots of a SIMD-mate that is ahead.
        const uint32_t n = nframe++;
        if (n < 2) __builtin_amdgcn_s_setprio(3);
        else if (n < 3) __builtin_amdgcn_s_setprio(2);
        else __builtin_amdgcn_s_setprio(1);
        f = run_frame(f, ctx());
        instructions += f.get(F_INSTR); ff_instructions += f.get(F_FF); bad_ops += f.get(F_BAD);
        f.set(F_INSTR, 0); f.set(F_FF, 0); f.set(F_BAD, 0);
    }
};

}  // namespace mh
