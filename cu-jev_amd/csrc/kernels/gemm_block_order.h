/* The memory operations of gemm_block_kernel's K loop, in issue order, and the
 * waits that order them. The kernel issues from these functions, and a host
 * program that includes this file can walk the same order (no HIP in here).
 *
 * One pass of the loop is a unit of 32 k; unit u sits in slot S = u % 4. At
 * its top a wave waits until at most gb_vm() DMAs and gb_lgkm() LDS reads of
 * its own are outstanding and then passes a barrier. Inside it, one memory
 * operation may sit before MFMA (r, j), W row group r x token group j:
 *   READ_A  fragment `row` of the W ring's slot `slot`
 *   READ_B  fragment `row` of X for the unit in slot `slot` (buffer slot / 2)
 *   DMA_W   this wave's row group `row` of W unit u + 3 -> ring slot `slot`
 *   DMA_X   this wave's piece `row` of X stage u / 2 + 2 -> buffer `slot` / 2
 * A wave's LDS reads return in order and its DMAs complete in order, so a
 * count outstanding names the latest ones. */
#ifndef CUJEV_GEMM_BLOCK_ORDER_H
#define CUJEV_GEMM_BLOCK_ORDER_H

constexpr int GB_WU = 4; /* W units in the ring */
constexpr int GB_AD = 3; /* W fragments read ahead, in rows */

enum gb_kind { GB_NO_MEM, GB_READ_A, GB_READ_B, GB_DMA_W, GB_DMA_X };
struct gb_mem {
    gb_kind kind;
    int slot, row;
};

/* X fragments of the next unit that are read before the end of row group r */
constexpr int gb_b_upto(int r, int WN) { return r < 5 ? (r + 1) * WN / 5 : WN; }

/* what precedes MFMA (r, j) of the unit in slot S (nb is at most 1 for WN = 4,
 * whose rows end at j = 3) */
constexpr gb_mem gb_before(int S, int WN, int r, int j) {
    const int b0 = r > 0 ? gb_b_upto(r - 1, WN) : 0, nb = gb_b_upto(r, WN) - b0;
    if (j == 0) /* W, GB_AD rows ahead: the last ones are the next unit's */
        return {GB_READ_A, r + GB_AD < 8 ? S : (S + 1) & 3, (r + GB_AD) & 7};
    if (j == 1 && (S & 1) && r < WN)
        return {GB_DMA_X, S & 2, r};
    if (j == 2 && nb > 0)
        return {GB_READ_B, (S + 1) & 3, b0};
    if (j == 3 && r >= 4)
        return {GB_DMA_W, (S + 3) & 3, r - 4};
    if (j == 4 && nb > 1)
        return {GB_READ_B, (S + 1) & 3, b0 + 1};
    return {GB_NO_MEM, 0, 0};
}

/* DMAs that may be outstanding at the top of a unit: those of the unit before
 * it (4 W, and in odd units WN X pieces). What this unit reads was issued two
 * units back or earlier. */
constexpr int gb_vm(int S, int WN) { return (S & 1) ? 4 : 4 + WN; }

/* LDS reads that may be outstanding there. The unit's own DMAs overwrite the
 * ring slot whose last fragment is read at r = 4 of the unit before, which at
 * least four reads follow, and in odd units the X buffer whose last fragment
 * is also read at r = 4, which only the three W reads of r = 5, 6, 7 follow. */
constexpr int gb_lgkm(int S, int) { return (S & 1) ? 3 : 4; }

#endif
