// The 6502 on the scalar unit: a console's instructions run one after another in gfx950 assembly, with the
// console's registers in scalar registers and its RAM in LDS.
//
// Why assembly: the time of a scalar 6502 instruction is its instruction count (one scalar instruction per 4 cycles
// of a wave) plus the latency of its branches (a taken branch 20 cycles, one not taken 13) and loads (36 cycles for
// a scalar load that hits, ~45 for LDS). A C++ switch on the opcode compiles to a balanced compare tree, 8 levels of
// compare and branch (~65 ns of the 183 ns an instruction took), and a flag byte that every operation masks and
// merges. Here an opcode's body starts at a fixed 256-byte slot, so that dispatch is one add and one s_setpc_b64
// (12 ns), the record of the next instruction is loaded while the current one works, and N and Z are the last
// result until something asks for the flag byte. Measured on the 256-env step: see k_step in mario_hip.hip.
//
// Records. decode_prg() lays the program out once per cartridge as a word per address:
//   bits 31-16  operand: the immediate or zero-page byte, the absolute RAM address (& $7FF) or index base, or the
//               target of a branch, JMP or JSR
//   bits 15-8   slot (the opcode, or a variant of it): the byte offset of the slot's code is bits 15-0 & $FF00
//   bits 7-0    for slot 0 only: what the instruction is (REC_*, a multiple of 4: slot 0 is a table of branches to
//               the end, so that it needs no mask), with its address as the operand, else 0
// Slot 0 ends the run before the instruction: what is not an official opcode, whose operands are not in PRG, whose
// static address is a register of the PPU, joypad or DMA, the idle loop `JMP *`, the sprite-0 wait, BRK. Addresses
// below $8000 have record 0, so a run ends when the program leaves PRG.
// A run also ends before the first instruction that may not start (s8 below), and before one whose computed address
// is neither RAM nor PRG (reads) or not known to ignore writes.
#pragma once
#include <stdint.h>

namespace mh {

constexpr uint32_t REC_COUNT = 0x10000 + 16;     // a run that walks off $FFFF reads records 0 there
constexpr uint32_t REC_IDLE = 0x10u;             // JMP *
constexpr uint32_t REC_STORE = 0x20u;            // | 4 * source (0 A, 1 X, 2 Y): an absolute store to a register
constexpr uint32_t REC_LOAD = 0x30u;             // | 4 * destination (0 A, 1 X, 2 Y, 3 BIT): an absolute load from one
// the sprite-0 wait: LDA $2002 / AND #$40 / BEQ|BNE back to the LDA (a REC_LOAD to A); REC_POLL_HIT: BEQ, waiting for the hit
constexpr uint32_t REC_POLL = 0x40u, REC_POLL_HIT = 0x50u;
// slots of opcode variants, at opcodes the 6502 does not have
constexpr uint32_t SLOT_BR_CROSS[8] = {0x12, 0x32, 0x52, 0x72, 0x92, 0xb2, 0xd2, 0xf2};   // branches that cross a page
constexpr uint32_t SLOT_STORE_IGNORED = 0x0b;    // a 4-cycle store to an address that ignores writes
constexpr uint32_t SLOT_JMP_CONST = 0x1b;        // JMP (ind) through a pointer in PRG
constexpr uint32_t SLOT_LDA_CONST = 0x2b, SLOT_LDX_CONST = 0x3b, SLOT_LDY_CONST = 0x4b;   // absolute loads from PRG

// Record of the instruction at pc of the 32 KB program image prg ($8000-$FFFF).
inline uint32_t decode_record(const uint8_t* prg, uint32_t pc, const uint32_t* dec_words) {
    using namespace dec;
    if (pc < 0x8000u || pc > 0xfffdu) return 0;
    const uint32_t op = prg[pc - 0x8000u], b1 = prg[pc - 0x7fffu], b2 = prg[pc - 0x7ffeu];
    const uint32_t D = dec_words[op], am = D & 15u, xop = (D >> X_SH) & 15u, absv = b1 | b2 << 8;
    const bool rd = (D & RD) != 0, wr = ((D >> DST_SH) & 7u) == D_MEM;
    if (!(D & OK) || !((D >> CYC_SH) & 7u)) return 0;   // invalid, or an opcode the cycle table gives 0 cycles
    auto rec = [](uint32_t slot, uint32_t operand) { return operand << 16 | slot << 8; };
    auto byte_at = [&](uint32_t ad) { return (uint32_t)prg[ad & 0x7fffu]; };
    if (xop == X_BRK) return 0;
    if (xop == X_BRANCH) {
        const uint32_t ret = pc + 2, to = (ret + (uint32_t)(int32_t)(int8_t)b1) & 0xffffu;
        return rec(((ret ^ to) & 0xff00u) ? SLOT_BR_CROSS[op >> 5] : op, to);
    }
    if (xop == X_JMP) return absv == pc ? REC_IDLE : rec(op, absv);
    if (xop == X_JSR) return rec(op, absv);
    if (xop == X_JMPI) {   // the pointer's high byte wraps in its page
        const uint32_t p2 = (absv & 0xff00u) | ((absv + 1u) & 0xffu);
        if (absv >= 0x8000u) return rec(SLOT_JMP_CONST, byte_at(absv) | byte_at(p2) << 8);
        return absv < 0x2000u && (absv & 0xffu) != 0xffu ? rec(op, absv & 0x7ffu) : 0;
    }
    switch (am) {
        case M_NONE: return rec(op, 0);
        case M_IMM: return rec(op, b1);
        case M_ZP: case M_ZPX: case M_ZPY: case M_INDX: return rec(op, b1);
        case M_INDY: return b1 == 0xffu ? 0 : rec(op, b1);   // the body reads the pointer's bytes at b1 and b1 + 1
        case M_ABSX: case M_ABSY: return rec(op, absv);
        default: break;   // M_ABS
    }
    if (absv < 0x2000u) return rec(op, absv & 0x7ffu);
    if (absv >= 0x8000u) {
        if (rd && !wr) {
            const uint32_t slot = op == 0xad ? SLOT_LDA_CONST : op == 0xae ? SLOT_LDX_CONST : op == 0xac ? SLOT_LDY_CONST : 0u;
            return slot ? rec(slot, byte_at(absv)) : 0;
        }
        return !rd && wr ? rec(SLOT_STORE_IGNORED, 0) : 0;
    }
    const bool joypad = absv == 0x4016u || absv == 0x4017u;
    if (rd) {
        if (wr || (absv >= 0x4000u && !joypad)) return 0;
        const uint32_t dst = op == 0xad ? 0u : op == 0xae ? 1u : op == 0xac ? 2u : op == 0x2c ? 3u : 4u;
        if (dst == 4u) return 0;
        if (op == 0xad && absv == 0x2002u && pc <= 0xfff8u) {
            const uint8_t* q = prg + (pc - 0x8000u);
            if (q[3] == 0x29 && q[4] == 0x40 && (q[5] == 0xf0 || q[5] == 0xd0) && q[6] == 0xf9)
                return absv << 16 | (q[5] == 0xf0 ? REC_POLL_HIT : REC_POLL);
        }
        return absv << 16 | REC_LOAD | 4u * dst;
    }
    if (!wr) return 0;
    if (absv >= 0x4000u && (absv & ~2u) != 0x4014u) return rec(SLOT_STORE_IGNORED, 0);
    return absv << 16 | REC_STORE | (op == 0x8d ? 0u : op == 0x8e ? 4u : 8u);
}
inline void decode_prg(const uint8_t* prg, const uint32_t* dec_words, uint32_t* out) {
    for (uint32_t pc = 0; pc < REC_COUNT; pc++) out[pc] = decode_record(prg, pc, dec_words);
}

// A run's registers, wave-uniform. `left`: how many CPU iterations past ex the next instruction may still start
// (exlim - ex, 0 .. 32767) in the high half, and the instructions run in the low half; taking an instruction's
// cycles from it borrows exactly when the next instruction may not start.
struct ScalarRegs {
    uint32_t a, x, y, sp;
    uint32_t nz;        // N: bits 7 or 8 set; Z: bits 7-0 zero
    uint32_t c;         // 0 or 1
    uint32_t v;         // bit 7
    uint32_t p_rest;    // the other flag bits (FI, FD, FB, FONE)
    uint32_t left;
    uint32_t pc4;       // pc << 2, with anything in bits 1-0 (scalar loads ignore them)
};

#if defined(__AMDGCN__)
// The code, once in the device library; scalar_run calls it.
// Registers: s0 A, s1 X, s2 Y, s3 SP, s4 nz, s5 c, s6 v, s7 p_rest, s8 left, s9 pc4, s10 record, s11 operand,
// s12 s13 scratch, s[14:15] target, s16 slot 0 (low half), s[18:19] records, s20 $10000, s22 $FF,
// s24 address, s25 $800, s26 ram, s27 prg - $8000 (LDS byte offsets), s28 s29 the words of 4 and 5 cycles, s[30:31] the
// return; v5 ram, v6 prg - $8000, v7 ram + $100.
// Hazards seen to: a VALU instruction never reads a scalar register that v_readfirstlane wrote last (scalar
// instructions stand between) and v_readfirstlane never a vector register that the VALU wrote last; every load is
// waited for before its register is used, at the end too.
// What bounds it with the chip full is scalar issue, so a body does its addresses on the vector unit (HDV takes the
// operand out of the record and adds the base in one v_mad_u32_u16), and dispatch is three scalar instructions and
// the jump: with the code 64 KB aligned, a slot's address is the record's low half under the code's high half. An
// LDA from the zero page is 5 scalar instructions and the jump; it was 10 with a mask, an add and a carry for the
// target. k_step of 256 / 32,768 envs by that: 0.89 -> 0.87 / 8.2 -> 7.75 ms, 121,000 -> 103,000 scalar
// instructions an env.
// Indexed addresses past $7FF are not RAM's first image: PRG has its own tail (FAR), a mirror is left to frame().
// (Device code has no file-scope assembly: the code stands in a function that nothing calls.)
__device__ __attribute__((used, noinline)) void cpu_code() {
    asm volatile(R"ASM(
.macro NX cyc                    // the next instruction, after one of cyc cycles
 s_sub_u32 s8, s8, ((\cyc)<<16)-1
 GO
.endm
.macro NXK                       // the same with the cycles' word in s13 (PEN)
 s_sub_u32 s8, s8, s13
 GO
.endm
.macro GO                        // to the record's slot, or the end if scc: the code is 64 KB aligned, slot 0 first
 s_waitcnt lgkmcnt(0)
 s_cselect_b32 s12, 0, s10
 s_pack_lh_b32_b16 s14, s12, s16
 s_setpc_b64 s[14:15]
.endm
.macro PEN cyc                   // s13: the cycles' word, one cycle more if s24 (address) is not in s11's (base) page
 s_xor_b32 s12, s11, s24
 s_bitcmp1_b32 s12, 8
.if \cyc == 4
 s_cselect_b32 s13, s29, s28
.elseif \cyc == 5
 s_cselect_b32 s13, (6<<16)-1, s29
.else
 s_cselect_b32 s13, s20, 0
 s_add_u32 s13, s13, ((\cyc)<<16)-1
.endif
.endm
.macro HD len                    // operand to s11; on to the next record
 s_lshr_b32 s11, s10, 16
 s_add_u32 s9, s9, 4*(\len)
 s_load_dword s10, s[18:19], s9
.endm
.macro HDV len                   // operand + RAM to v0; on to the next record
 v_mad_u32_u16 v0, s10, 1, v5 op_sel:[1,0,0,0]
 s_add_u32 s9, s9, 4*(\len)
 s_load_dword s10, s[18:19], s9
.endm
.macro GOTO                      // on to the record of the operand's address
 s_lshr_b32 s9, s10, 14
 s_load_dword s10, s[18:19], s9
.endm
.macro LDB                       // RAM byte s11 (0..$7FF)
 v_add_u32 v0, s11, v5
 ds_read_u8 v1, v0
.endm
.macro GETM
 s_waitcnt lgkmcnt(0)
 v_readfirstlane_b32 s11, v1
.endm
.macro IDXZ r                    // zero page, indexed
 s_add_u32 s11, s11, \r
 s_and_b32 s11, s11, s22
.endm
.macro PTRY len                  // (zp),Y: base to s11, address to s24
 HDV \len
 ds_read_u8 v1, v0
 ds_read_u8 v2, v0 offset:1
 s_waitcnt lgkmcnt(0)
 v_lshl_or_b32 v1, v2, 8, v1
 s_nop 0
 v_readfirstlane_b32 s11, v1
 s_add_u32 s24, s11, s2
.endm
.macro PTRX                      // (zp,X): address to s24
 s_add_u32 s11, s11, s1
 s_and_b32 s11, s11, s22
 s_add_u32 s12, s11, 1
 s_and_b32 s12, s12, s22
 v_add_u32 v0, s11, v5
 v_add_u32 v2, s12, v5
 ds_read_u8 v1, v0
 ds_read_u8 v2, v2
 s_waitcnt lgkmcnt(0)
 v_readfirstlane_b32 s12, v1
 v_readfirstlane_b32 s13, v2
 s_lshl_b32 s13, s13, 8
 s_or_b32 s24, s12, s13
.endm
// ---- operations on the operand in s11
.macro A_LDA
 s_mov_b32 s0, s11
 s_mov_b32 s4, s11
.endm
.macro A_LDX
 s_mov_b32 s1, s11
 s_mov_b32 s4, s11
.endm
.macro A_LDY
 s_mov_b32 s2, s11
 s_mov_b32 s4, s11
.endm
.macro A_AND
 s_and_b32 s0, s0, s11
 s_mov_b32 s4, s0
.endm
.macro A_ORA
 s_or_b32 s0, s0, s11
 s_mov_b32 s4, s0
.endm
.macro A_EOR
 s_xor_b32 s0, s0, s11
 s_mov_b32 s4, s0
.endm
.macro A_ADC
 s_add_u32 s12, s0, s11
 s_add_u32 s12, s12, s5
 s_xor_b32 s6, s0, s12
 s_xor_b32 s11, s11, s12
 s_and_b32 s6, s6, s11
 s_lshr_b32 s5, s12, 8
 s_and_b32 s0, s12, s22
 s_mov_b32 s4, s0
.endm
.macro A_SBC
 s_xor_b32 s11, s11, s22
 A_ADC
.endm
.macro CMPR r
 s_sub_u32 s4, \r, s11
 s_cselect_b32 s5, 0, 1
 s_and_b32 s4, s4, s22
.endm
.macro A_CMP
 CMPR s0
.endm
.macro A_CPX
 CMPR s1
.endm
.macro A_CPY
 CMPR s2
.endm
.macro A_BIT
 s_and_b32 s4, s0, s11
 s_lshl_b32 s6, s11, 1
 s_and_b32 s12, s6, 0x100
 s_or_b32 s4, s4, s12
.endm
.macro M_ASL r
 s_lshr_b32 s5, \r, 7
 s_lshl_b32 \r, \r, 1
 s_and_b32 \r, \r, s22
 s_mov_b32 s4, \r
.endm
.macro M_ROL r
 s_lshl_b32 s12, \r, 1
 s_or_b32 s12, s12, s5
 s_lshr_b32 s5, \r, 7
 s_and_b32 \r, s12, s22
 s_mov_b32 s4, \r
.endm
.macro M_LSR r
 s_and_b32 s5, \r, 1
 s_lshr_b32 \r, \r, 1
 s_mov_b32 s4, \r
.endm
.macro M_ROR r
 s_lshl_b32 s12, s5, 7
 s_and_b32 s5, \r, 1
 s_lshr_b32 \r, \r, 1
 s_or_b32 \r, \r, s12
 s_mov_b32 s4, \r
.endm
.macro M_INC r
 s_add_u32 \r, \r, 1
 s_and_b32 \r, \r, s22
 s_mov_b32 s4, \r
.endm
.macro M_DEC r
 s_sub_u32 \r, \r, 1
 s_and_b32 \r, \r, s22
 s_mov_b32 s4, \r
.endm
// ---- the same on the byte that is being read into v1
.macro L_LDA
 s_waitcnt lgkmcnt(0)
 v_readfirstlane_b32 s0, v1
 s_mov_b32 s4, s0
.endm
.macro L_LDX
 s_waitcnt lgkmcnt(0)
 v_readfirstlane_b32 s1, v1
 s_mov_b32 s4, s1
.endm
.macro L_LDY
 s_waitcnt lgkmcnt(0)
 v_readfirstlane_b32 s2, v1
 s_mov_b32 s4, s2
.endm
.macro L_ORA
 GETM
 A_ORA
.endm
.macro L_AND
 GETM
 A_AND
.endm
.macro L_EOR
 GETM
 A_EOR
.endm
.macro L_ADC
 GETM
 A_ADC
.endm
.macro L_SBC
 GETM
 A_SBC
.endm
.macro L_CMP
 GETM
 A_CMP
.endm
.macro L_CPX
 GETM
 A_CPX
.endm
.macro L_CPY
 GETM
 A_CPY
.endm
.macro L_BIT
 GETM
 A_BIT
.endm
// ---- read-modify-write of the byte in s11, result to s4
.macro W_ASL
 s_lshr_b32 s5, s11, 7
 s_lshl_b32 s11, s11, 1
 s_and_b32 s4, s11, s22
.endm
.macro W_ROL
 s_lshl_b32 s12, s11, 1
 s_or_b32 s12, s12, s5
 s_lshr_b32 s5, s11, 7
 s_and_b32 s4, s12, s22
.endm
.macro W_LSR
 s_and_b32 s5, s11, 1
 s_lshr_b32 s4, s11, 1
.endm
.macro W_ROR
 s_lshl_b32 s12, s5, 7
 s_and_b32 s5, s11, 1
 s_lshr_b32 s11, s11, 1
 s_or_b32 s4, s11, s12
.endm
.macro W_INC
 s_add_u32 s11, s11, 1
 s_and_b32 s4, s11, s22
.endm
.macro W_DEC
 s_sub_u32 s11, s11, 1
 s_and_b32 s4, s11, s22
.endm
// ---- slots (SLOT n: the code at byte offset 256 n; an overlong one fails to assemble)
.macro SLOT n
 .org .Lmh_slots + 256*(\n), 0
.endm
.macro STOP n
 SLOT \n
 s_branch .Lmh_exit
.endm
.macro IMM n, op
 SLOT \n
 HD 2
 A_\op
 NX 2
.endm
.macro LDI n, r                  // LDA, LDX, LDY immediate
 SLOT \n
 s_lshr_b32 \r, s10, 16
 s_add_u32 s9, s9, 8
 s_load_dword s10, s[18:19], s9
 s_mov_b32 s4, \r
 NX 2
.endm
.macro ZP n, op
 SLOT \n
 HDV 2
 ds_read_u8 v1, v0
 L_\op
 NX 3
.endm
.macro ZPI n, op, r
 SLOT \n
 HD 2
 IDXZ \r
 LDB
 L_\op
 NX 4
.endm
.macro ABS n, op
 SLOT \n
 HDV 3
 ds_read_u8 v1, v0
 L_\op
 NX 4
.endm
.macro ABSI n, op, r             // not RAM: .Lmh_far_n
 SLOT \n
 HD 3
 s_add_u32 s24, s11, \r
 s_cmp_ge_u32 s24, s25
 s_cbranch_scc1 .Lmh_far_\n
 v_add_u32 v0, s24, v5
 ds_read_u8 v1, v0
 PEN 4
 L_\op
 NXK
.endm
.macro INDY n, op
 SLOT \n
 PTRY 2
 s_cmp_ge_u32 s24, s25
 s_cbranch_scc1 .Lmh_far_\n
 v_add_u32 v0, s24, v5
 ds_read_u8 v1, v0
 PEN 5
 L_\op
 NXK
.endm
.macro INDX n, op
 SLOT \n
 HD 2
 PTRX
 s_cmp_ge_u32 s24, s25
 s_cbranch_scc1 .Lmh_far_\n
 v_add_u32 v0, s24, v5
 ds_read_u8 v1, v0
 L_\op
 NX 6
.endm
.macro FAR n, op, cyc, len       // the rest of ABSI / INDY for PRG
.Lmh_far_\n:
 s_bitcmp1_b32 s24, 15
 s_cbranch_scc0 .Lmh_ref_\len
 v_add_u32 v0, s24, v6
 ds_read_u8 v1, v0
 PEN \cyc
 L_\op
 NXK
.endm
.macro FARX n, op                // of INDX
.Lmh_far_\n:
 s_bitcmp1_b32 s24, 15
 s_cbranch_scc0 .Lmh_ref_2
 v_add_u32 v0, s24, v6
 ds_read_u8 v1, v0
 L_\op
 NX 6
.endm
.macro PUTV r                    // the byte at v0 = r
 v_mov_b32 v1, \r
 ds_write_b8 v0, v1
.endm
.macro PUT r                     // RAM byte s11 = r
 v_add_u32 v0, s11, v5
 PUTV \r
.endm
.macro STZP n, r
 SLOT \n
 HDV 2
 PUTV \r
 NX 3
.endm
.macro STZPI n, r, i
 SLOT \n
 HD 2
 IDXZ \i
 PUT \r
 NX 4
.endm
.macro STABS n, r
 SLOT \n
 HDV 3
 PUTV \r
 NX 4
.endm
.macro STORE_AT n, cyc           // A to the computed address s24
 s_cmp_ge_u32 s24, s25
 s_cbranch_scc1 .Lmh_far_\n
 v_add_u32 v0, s24, v5
 PUTV s0
 NX \cyc
.endm
.macro STABSI n, i
 SLOT \n
 HD 3
 s_add_u32 s24, s11, \i
 STORE_AT \n, 5
.endm
.macro FARST n, cyc, len         // a store past RAM: PRG and $4000-$7FFF but DMA and the joypad strobe ignore it
.Lmh_far_\n:
 s_cmp_ge_u32 s24, 0x10000
 s_cbranch_scc1 .Lmh_ref_\len
 s_cmp_lt_u32 s24, 0x4000
 s_cbranch_scc1 .Lmh_ref_\len
 s_and_b32 s12, s24, 0xfffd
 s_cmp_eq_u32 s12, 0x4014
 s_cbranch_scc1 .Lmh_ref_\len
 NX \cyc
.endm
.macro RMW_TAIL op, cyc
 GETM
 W_\op
 PUTV s4
 NX \cyc
.endm
.macro RMZP n, op
 SLOT \n
 HDV 2
 ds_read_u8 v1, v0
 RMW_TAIL \op, 5
.endm
.macro RMZPX n, op
 SLOT \n
 HD 2
 IDXZ s1
 LDB
 RMW_TAIL \op, 6
.endm
.macro RMABS n, op
 SLOT \n
 HDV 3
 ds_read_u8 v1, v0
 RMW_TAIL \op, 6
.endm
.macro RMABSX n, op
 SLOT \n
 HD 3
 s_add_u32 s24, s11, s1
 s_cmp_ge_u32 s24, s25
 s_cbranch_scc1 .Lmh_ref_3
 v_add_u32 v0, s24, v5
 ds_read_u8 v1, v0
 PEN 7
 GETM
 W_\op
 PUTV s4
 NXK
.endm
.macro ACC n, op
 SLOT \n
 HD 1
 M_\op s0
 NX 2
.endm
.macro REG n, op, r
 SLOT \n
 HD 1
 M_\op \r
 NX 2
.endm
.macro XFER n, to, from          // with N and Z
 SLOT \n
 HD 1
 s_mov_b32 \to, \from
 s_mov_b32 s4, \from
 NX 2
.endm
.macro SETF n, r, val
 SLOT \n
 HD 1
 s_mov_b32 \r, \val
 NX 2
.endm
.macro ORF n, mask
 SLOT \n
 HD 1
 s_or_b32 s7, s7, \mask
 NX 2
.endm
.macro CLRF n, mask
 SLOT \n
 HD 1
 s_andn2_b32 s7, s7, \mask
 NX 2
.endm
.macro BR_TAIL n, nt, cyc        // taken unless scc == nt
 s_cbranch_scc\nt .Lmh_nt_\n
 GOTO
 NX \cyc
.Lmh_nt_\n:
 s_add_u32 s9, s9, 8
 s_load_dword s10, s[18:19], s9
 NX 2
.endm
.macro BR_N n, nt, cyc
 SLOT \n
 s_and_b32 s12, s4, 0x180
 BR_TAIL \n, \nt, \cyc
.endm
.macro BR_V n, nt, cyc
 SLOT \n
 s_bitcmp1_b32 s6, 7
 BR_TAIL \n, \nt, \cyc
.endm
.macro BR_C n, nt, cyc
 SLOT \n
 s_cmp_lg_u32 s5, 0
 BR_TAIL \n, \nt, \cyc
.endm
.macro BR_NZ n, nt, cyc          // scc: Z clear
 SLOT \n
 s_and_b32 s12, s4, s22
 BR_TAIL \n, \nt, \cyc
.endm
.macro SPDN
 s_sub_u32 s3, s3, 1
 s_and_b32 s3, s3, s22
.endm
.macro PUSH r                    // RAM byte $100 + SP = r
 v_add_u32 v0, s3, v7
 v_mov_b32 v1, \r
 ds_write_b8 v0, v1
 SPDN
.endm
.macro SPUP
 s_add_u32 s3, s3, 1
 s_and_b32 s3, s3, s22
.endm
.macro UNPACK                    // flag byte s11 to its parts
 s_and_b32 s7, s11, 0x3c
 s_lshr_b32 s5, s11, 7
 s_lshl_b32 s6, s11, 6
 s_and_b32 s12, s11, 1
 s_lshl_b32 s12, s12, 8
 s_bitcmp0_b32 s11, 6
 s_cselect_b32 s4, 1, 0
 s_or_b32 s4, s4, s12
.endm

 .p2align 16
.Lmh_slots:
 .rept 64
 s_branch .Lmh_exit
 .endr
 INDX  0x01, ORA
 STOP  0x02
 STOP  0x03
 STOP  0x04
 ZP    0x05, ORA
 RMZP  0x06, ASL
 STOP  0x07
 SLOT  0x08                      // PHP
 HD 1
 s_and_b32 s12, s4, 0x180
 s_cselect_b32 s11, 1, 0
 s_or_b32 s11, s11, s7
 s_and_b32 s12, s4, s22
 s_cselect_b32 s12, 0, 64
 s_or_b32 s11, s11, s12
 s_lshl_b32 s12, s5, 7
 s_or_b32 s11, s11, s12
 s_lshr_b32 s12, s6, 6
 s_and_b32 s12, s12, 2
 s_or_b32 s11, s11, s12
 PUSH s11
 NX 3
 IMM   0x09, ORA
 ACC   0x0a, ASL
 SLOT  0x0b                      // a store that is ignored
 HD 3
 NX 4
 STOP  0x0c
 ABS   0x0d, ORA
 RMABS 0x0e, ASL
 STOP  0x0f
 BR_N  0x10, 1, 3
 INDY  0x11, ORA
 BR_N  0x12, 1, 5
 STOP  0x13
 STOP  0x14
 ZPI   0x15, ORA, s1
 RMZPX 0x16, ASL
 STOP  0x17
 SETF  0x18, s5, 0               // CLC
 ABSI  0x19, ORA, s2
 STOP  0x1a
 SLOT  0x1b                      // JMP (ind) through PRG
 GOTO
 NX 5
 STOP  0x1c
 ABSI  0x1d, ORA, s1
 RMABSX 0x1e, ASL
 STOP  0x1f
 SLOT  0x20                      // JSR
 s_lshr_b32 s12, s9, 2
 s_add_u32 s12, s12, 2
 GOTO
 v_mov_b32 v1, s12
 v_lshrrev_b32 v2, 8, v1
 v_add_u32 v0, s3, v7
 ds_write_b8 v0, v2
 SPDN
 v_add_u32 v0, s3, v7
 ds_write_b8 v0, v1
 SPDN
 NX 6
 INDX  0x21, AND
 STOP  0x22
 STOP  0x23
 ZP    0x24, BIT
 ZP    0x25, AND
 RMZP  0x26, ROL
 STOP  0x27
 SLOT  0x28                      // PLP
 HD 1
 SPUP
 v_add_u32 v0, s3, v7
 ds_read_u8 v1, v0
 GETM
 UNPACK
 NX 4
 IMM   0x29, AND
 ACC   0x2a, ROL
 SLOT  0x2b                      // LDA from PRG
 HD 3
 A_LDA
 NX 4
 ABS   0x2c, BIT
 ABS   0x2d, AND
 RMABS 0x2e, ROL
 STOP  0x2f
 BR_N  0x30, 0, 3
 INDY  0x31, AND
 BR_N  0x32, 0, 5
 STOP  0x33
 STOP  0x34
 ZPI   0x35, AND, s1
 RMZPX 0x36, ROL
 STOP  0x37
 SETF  0x38, s5, 1               // SEC
 ABSI  0x39, AND, s2
 STOP  0x3a
 SLOT  0x3b                      // LDX from PRG
 HD 3
 A_LDX
 NX 4
 STOP  0x3c
 ABSI  0x3d, AND, s1
 RMABSX 0x3e, ROL
 STOP  0x3f
 SLOT  0x40                      // RTI
 SPUP
 v_add_u32 v0, s3, v7
 SPUP
 v_add_u32 v2, s3, v7
 SPUP
 v_add_u32 v3, s3, v7
 ds_read_u8 v1, v0
 ds_read_u8 v2, v2
 ds_read_u8 v3, v3
 GETM
 v_readfirstlane_b32 s12, v2
 v_readfirstlane_b32 s13, v3
 s_lshl_b32 s13, s13, 8
 s_or_b32 s12, s12, s13
 s_lshl_b32 s9, s12, 2
 s_load_dword s10, s[18:19], s9
 UNPACK
 NX 6
 INDX  0x41, EOR
 STOP  0x42
 STOP  0x43
 STOP  0x44
 ZP    0x45, EOR
 RMZP  0x46, LSR
 STOP  0x47
 SLOT  0x48                      // PHA
 HD 1
 PUSH s0
 NX 3
 IMM   0x49, EOR
 ACC   0x4a, LSR
 SLOT  0x4b                      // LDY from PRG
 HD 3
 A_LDY
 NX 4
 SLOT  0x4c                      // JMP
 GOTO
 NX 3
 ABS   0x4d, EOR
 RMABS 0x4e, LSR
 STOP  0x4f
 BR_V  0x50, 1, 3
 INDY  0x51, EOR
 BR_V  0x52, 1, 5
 STOP  0x53
 STOP  0x54
 ZPI   0x55, EOR, s1
 RMZPX 0x56, LSR
 STOP  0x57
 CLRF  0x58, 0x20                // CLI
 ABSI  0x59, EOR, s2
 STOP  0x5a
 STOP  0x5b
 STOP  0x5c
 ABSI  0x5d, EOR, s1
 RMABSX 0x5e, LSR
 STOP  0x5f
 SLOT  0x60                      // RTS
 SPUP
 v_add_u32 v0, s3, v7
 SPUP
 v_add_u32 v2, s3, v7
 ds_read_u8 v1, v0
 ds_read_u8 v2, v2
 s_waitcnt lgkmcnt(0)
 v_lshl_or_b32 v1, v2, 8, v1
 s_nop 0
 v_readfirstlane_b32 s11, v1
 s_lshl2_add_u32 s9, s11, 4      // ($FFFF + 1: record 0 there, and its pc is 0)
 s_load_dword s10, s[18:19], s9
 NX 6
 INDX  0x61, ADC
 STOP  0x62
 STOP  0x63
 STOP  0x64
 ZP    0x65, ADC
 RMZP  0x66, ROR
 STOP  0x67
 SLOT  0x68                      // PLA
 HD 1
 SPUP
 v_add_u32 v0, s3, v7
 ds_read_u8 v1, v0
 L_LDA
 NX 4
 IMM   0x69, ADC
 ACC   0x6a, ROR
 STOP  0x6b
 SLOT  0x6c                      // JMP (ind) through RAM
 s_lshr_b32 s11, s10, 16
 v_add_u32 v0, s11, v5
 ds_read_u8 v1, v0
 ds_read_u8 v2, v0 offset:1
 s_waitcnt lgkmcnt(0)
 v_lshl_or_b32 v1, v2, 8, v1
 s_nop 0
 v_readfirstlane_b32 s11, v1
 s_lshl_b32 s9, s11, 2
 s_load_dword s10, s[18:19], s9
 NX 5
 ABS   0x6d, ADC
 RMABS 0x6e, ROR
 STOP  0x6f
 BR_V  0x70, 0, 3
 INDY  0x71, ADC
 BR_V  0x72, 0, 5
 STOP  0x73
 STOP  0x74
 ZPI   0x75, ADC, s1
 RMZPX 0x76, ROR
 STOP  0x77
 ORF   0x78, 0x20                // SEI
 ABSI  0x79, ADC, s2
 STOP  0x7a
 STOP  0x7b
 STOP  0x7c
 ABSI  0x7d, ADC, s1
 RMABSX 0x7e, ROR
 STOP  0x7f
 STOP  0x80
 SLOT  0x81                      // STA (zp,X)
 HD 2
 PTRX
 STORE_AT 0x81, 6
 STOP  0x82
 STOP  0x83
 STZP  0x84, s2
 STZP  0x85, s0
 STZP  0x86, s1
 STOP  0x87
 REG   0x88, DEC, s2             // DEY
 STOP  0x89
 XFER  0x8a, s0, s1              // TXA
 STOP  0x8b
 STABS 0x8c, s2
 STABS 0x8d, s0
 STABS 0x8e, s1
 STOP  0x8f
 BR_C  0x90, 1, 3
 SLOT  0x91                      // STA (zp),Y
 PTRY 2
 STORE_AT 0x91, 6
 BR_C  0x92, 1, 5
 STOP  0x93
 STZPI 0x94, s2, s1
 STZPI 0x95, s0, s1
 STZPI 0x96, s1, s2
 STOP  0x97
 XFER  0x98, s0, s2              // TYA
 STABSI 0x99, s2
 SLOT  0x9a                      // TXS
 HD 1
 s_mov_b32 s3, s1
 NX 2
 STOP  0x9b
 STOP  0x9c
 STABSI 0x9d, s1
 STOP  0x9e
 STOP  0x9f
 LDI   0xa0, s2
 INDX  0xa1, LDA
 LDI   0xa2, s1
 STOP  0xa3
 ZP    0xa4, LDY
 ZP    0xa5, LDA
 ZP    0xa6, LDX
 STOP  0xa7
 XFER  0xa8, s2, s0              // TAY
 LDI   0xa9, s0
 XFER  0xaa, s1, s0              // TAX
 STOP  0xab
 ABS   0xac, LDY
 ABS   0xad, LDA
 ABS   0xae, LDX
 STOP  0xaf
 BR_C  0xb0, 0, 3
 INDY  0xb1, LDA
 BR_C  0xb2, 0, 5
 STOP  0xb3
 ZPI   0xb4, LDY, s1
 ZPI   0xb5, LDA, s1
 ZPI   0xb6, LDX, s2
 STOP  0xb7
 SETF  0xb8, s6, 0               // CLV
 ABSI  0xb9, LDA, s2
 XFER  0xba, s1, s3              // TSX
 STOP  0xbb
 ABSI  0xbc, LDY, s1
 ABSI  0xbd, LDA, s1
 ABSI  0xbe, LDX, s2
 STOP  0xbf
 IMM   0xc0, CPY
 INDX  0xc1, CMP
 STOP  0xc2
 STOP  0xc3
 ZP    0xc4, CPY
 ZP    0xc5, CMP
 RMZP  0xc6, DEC
 STOP  0xc7
 REG   0xc8, INC, s2             // INY
 IMM   0xc9, CMP
 REG   0xca, DEC, s1             // DEX
 STOP  0xcb
 ABS   0xcc, CPY
 ABS   0xcd, CMP
 RMABS 0xce, DEC
 STOP  0xcf
 BR_NZ 0xd0, 0, 3
 INDY  0xd1, CMP
 BR_NZ 0xd2, 0, 5
 STOP  0xd3
 STOP  0xd4
 ZPI   0xd5, CMP, s1
 RMZPX 0xd6, DEC
 STOP  0xd7
 CLRF  0xd8, 0x10                // CLD
 ABSI  0xd9, CMP, s2
 STOP  0xda
 STOP  0xdb
 STOP  0xdc
 ABSI  0xdd, CMP, s1
 RMABSX 0xde, DEC
 STOP  0xdf
 IMM   0xe0, CPX
 INDX  0xe1, SBC
 STOP  0xe2
 STOP  0xe3
 ZP    0xe4, CPX
 ZP    0xe5, SBC
 RMZP  0xe6, INC
 STOP  0xe7
 REG   0xe8, INC, s1             // INX
 IMM   0xe9, SBC
 SLOT  0xea                      // NOP
 HD 1
 NX 2
 STOP  0xeb
 ABS   0xec, CPX
 ABS   0xed, SBC
 RMABS 0xee, INC
 STOP  0xef
 BR_NZ 0xf0, 1, 3
 INDY  0xf1, SBC
 BR_NZ 0xf2, 1, 5
 STOP  0xf3
 STOP  0xf4
 ZPI   0xf5, SBC, s1
 RMZPX 0xf6, INC
 STOP  0xf7
 ORF   0xf8, 0x10                // SED
 ABSI  0xf9, SBC, s2
 STOP  0xfa
 STOP  0xfb
 STOP  0xfc
 ABSI  0xfd, SBC, s1
 RMABSX 0xfe, INC
 STOP  0xff
 SLOT  0x100
// ---- the rest of the bodies whose address is not in RAM
 FARX 0x01, ORA
 FARX 0x21, AND
 FARX 0x41, EOR
 FARX 0x61, ADC
 FARX 0xa1, LDA
 FARX 0xc1, CMP
 FARX 0xe1, SBC
 FAR 0x11, ORA, 5, 2
 FAR 0x31, AND, 5, 2
 FAR 0x51, EOR, 5, 2
 FAR 0x71, ADC, 5, 2
 FAR 0xb1, LDA, 5, 2
 FAR 0xd1, CMP, 5, 2
 FAR 0xf1, SBC, 5, 2
 FAR 0x19, ORA, 4, 3
 FAR 0x39, AND, 4, 3
 FAR 0x59, EOR, 4, 3
 FAR 0x79, ADC, 4, 3
 FAR 0xb9, LDA, 4, 3
 FAR 0xd9, CMP, 4, 3
 FAR 0xf9, SBC, 4, 3
 FAR 0x1d, ORA, 4, 3
 FAR 0x3d, AND, 4, 3
 FAR 0x5d, EOR, 4, 3
 FAR 0x7d, ADC, 4, 3
 FAR 0xbd, LDA, 4, 3
 FAR 0xdd, CMP, 4, 3
 FAR 0xfd, SBC, 4, 3
 FAR 0xbc, LDY, 4, 3
 FAR 0xbe, LDX, 4, 3
 FARST 0x81, 6, 2
 FARST 0x91, 6, 2
 FARST 0x99, 5, 3
 FARST 0x9d, 5, 3
mh_cpu_run:
 s_mov_b64 exec, 1                 // one lane is enough
 s_mov_b32 s20, 0x10000
 s_movk_i32 s22, 0xff
 s_movk_i32 s25, 0x800
 s_mov_b32 s28, (4<<16)-1
 s_mov_b32 s29, (5<<16)-1
 s_load_dword s10, s[18:19], s9
 v_mov_b32 v5, s26
 v_mov_b32 v6, s27
 v_add_u32 v7, 0x100, v5
 s_getpc_b64 s[16:17]
.Lmh_here:
 s_sub_u32 s16, s16, .Lmh_here-.Lmh_slots
 s_subb_u32 s15, s17, 0
 s_and_b32 s12, s16, 0xffff        // (loaded out of line: nothing runs here, and frame() runs everything itself)
 s_cbranch_scc1 .Lmh_exit
 GO
.Lmh_ref_2:                          // left to frame(): back to the instruction
 s_sub_u32 s9, s9, 8
 s_branch .Lmh_exit
.Lmh_ref_3:
 s_sub_u32 s9, s9, 12
.Lmh_exit:
 s_waitcnt lgkmcnt(0)
 s_mov_b64 exec, -1
 s_setpc_b64 s[30:31]
)ASM");
}
// Runs at least one instruction unless its record is slot 0 (or it leaves its computed address to frame()). ram, prg:
// LDS byte offsets of the console's RAM and of the staged program. All lanes are active; lane 0 does the accesses.
__device__ __forceinline__ void scalar_run(ScalarRegs& r, const uint32_t* records, uint32_t ram, uint32_t prg) {
    records = (const uint32_t*)uni64((uint64_t)records);
    ram = uni(ram); prg = uni(prg);
    r.a = uni(r.a); r.x = uni(r.x); r.y = uni(r.y); r.sp = uni(r.sp); r.nz = uni(r.nz); r.c = uni(r.c); r.v = uni(r.v);
    r.p_rest = uni(r.p_rest); r.left = uni(r.left); r.pc4 = uni(r.pc4);
    asm volatile(" s_getpc_b64 s[14:15]\n"
                 " s_add_u32 s14, s14, mh_cpu_run@rel32@lo+4\n"
                 " s_addc_u32 s15, s15, mh_cpu_run@rel32@hi+12\n"
                 " s_swappc_b64 s[30:31], s[14:15]\n"
                 : "+{s0}"(r.a), "+{s1}"(r.x), "+{s2}"(r.y), "+{s3}"(r.sp), "+{s4}"(r.nz), "+{s5}"(r.c), "+{s6}"(r.v),
                   "+{s7}"(r.p_rest), "+{s8}"(r.left), "+{s9}"(r.pc4)
                 : "{s[18:19]}"(records), "{s26}"(ram), "{s27}"(prg - 0x8000u)
                 : "s10", "s11", "s12", "s13", "s14", "s15", "s16", "s17", "s20", "s22", "s24", "s25", "s28", "s29", "s30", "s31",
                   "v0", "v1", "v2", "v3", "v5", "v6", "v7", "scc", "memory");
}
#endif

}  // namespace mh
