// Packed logic-tree blocks on column-major words for gfx950: up to four complete blocks (8 taps,
// 4 -> 2 -> 1 gates, 2x2 pool as OR) of a frozen network run on one 32-sample column at a time,
// the column's activations held in LDS between the blocks.
//
// The row-major block (k_tree_packed) gives every lane one output row's words: tap rows are
// resolved per lane, 32 loads of 16 bytes each per pair of words.  Here a workgroup owns a whole
// column (one 32-bit word per feature), so a wave can take one output channel with a pooled
// position per lane: the channel's taps and gates are wave-uniform (scalar loads, scalar
// branches on the gate), a tap is one LDS read at lane base + channel offset, and neither the
// address arithmetic nor the gate choice costs vector instructions per word.  Between the
// blocks nothing leaves LDS.  9x32x32 -> 256 -> 512 channels at 2^20 samples: 1.75 ms and 0.48 ms
// for the rows turned to columns, where the row-major blocks took 3.30 + 0.60 ms and 0.40 ms for
// widening their input rows (shapes and sizes where they stay the faster ones: tree_columns_from
// in packed_net.py).  Bound by the instructions a SIMD issues, vector and scalar ones
// together (a column takes 32000 cycles: 22000 in the first block, 6500 in the second, the
// rest staging and barriers): every tap and gate evaluated 2.72 ms, only live ones with a
// branch per tap 2.13, a branch per subtree and unshared table words 1.75.
//
// LDS layout of a block's input: one plane per channel, zero halo included (a tap outside the
// image reads 0), rows of `pitch` words, a row's columns split by their phase modulo 2 * sw:
// neighbouring pooled positions then read neighbouring words.  The two conv rows of a pooling
// window are dy = sh * pitch words apart; with dy congruent to 4 modulo 16 the four pooled rows
// of a half-wave (8 x 8 positions) fall on distinct banks.
#include "common.h"

#include <algorithm>

namespace cl {
namespace {

constexpr int kTcThreads = 1024;
constexpr int kTcMaxBlocks = 4;
constexpr int kTcLdsWords = 40960;       // 160 KiB
constexpr int kTcDescWords = 32;         // words of a block's descriptor before the tables
constexpr int kTcTabWords = 20;          // table words per channel: 16 tap offsets, codes, opcodes
constexpr int kTcMaxIpt = 16;            // input words per thread
constexpr int kTcDy[] = {36, 68, 132};   // conv-row distances with two-word LDS reads

struct TreeColsBlock {
    int cin, h, w, cout, sh, sw, ph, pw;
    int kh, kw;
    int hr, wr;          // rows and columns of a padded plane that a tap can reach
    int wp, P;           // pooled width, pooled positions
    int pitch, cs, dy;   // plane row pitch, plane size, conv-row distance (words)
    int q, r;            // wr / (2 sw), wr % (2 sw): the phase split
    int base;            // LDS word of plane 0
    int uniform;         // a wave takes one channel (P % 64 == 0 and dy in kTcDy)
    int tab;             // first table word
    FastDiv div_p, div_wp, div_m;
};

static_assert(sizeof(TreeColsBlock) <= kTcDescWords * 4, "descriptor size");

struct TreeCols {
    int nb;
    int in_rows, in_words, out_words, lds_words;
};

__host__ __device__ __forceinline__ int phase_slot(const TreeColsBlock& g, int x) {
    const int m = 2 * g.sw;
    const int f = x % m;
    return f * g.q + (f < g.r ? f : g.r) + x / m;
}

__device__ __forceinline__ void exchange(uint32_t& a, uint32_t& b) {
    const uint32_t t = a;
    a = b;
    b = t;
}

// ------------------------------------------------------------------------------------------
// Tables of one block, a thread per channel: words 2k and 2k + 1 hold the LDS byte offsets of tap k
// at pooled position 0 for the two conv columns of the window, word 16 the gates as 4-bit codes
// for tree_block_uniform, word 17 the opcodes (nibbles) for tree_block_lanes, whose tap order is
// the block's own.
//
// Codes.  An opcode that is 1 at a = b = 0 is replaced by its complement and its reader's table
// turned round to match, which leaves one inversion at the root (bit 31 of word 16).  A gate
// that then ignores an operand, or reads one that is always 0, passes the other or is always 0
// itself; one that passes a, or is a & ~b, has its operands swapped: two taps, or two subtrees
// with all that hangs from them.  What is left is: pass b (code 0), a & b, ~a & b (bit 0, bit 2
// for the second), a ^ b, a | b (bit 1, bit 2 for the second).  Bit 3 marks a gate that reads
// both; bit 30 of word 16 a channel that is always 0.
// Taps and gates that no live gate reads are not evaluated: of random gates a quarter passes
// one operand and an eighth none, and 42 % of the taps are live.
// A channel with a tap on a channel past the input is all ones, as in the row-major block.
__global__ __launch_bounds__(256) void k_tree_cols_tables(const uint8_t* __restrict__ gates,
                                                          const int32_t* __restrict__ sel,
                                                          TreeColsBlock g,
                                                          TreeColsBlock* __restrict__ desc,
                                                          uint32_t* __restrict__ tab) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c == 0) *desc = g;  // read back through the scalar cache at a run-time block index
    if (c >= g.cout) return;
    uint32_t* t = tab + int64_t(c) * kTcTabWords;
    // LDS words of the taps, first | second << 16: in the order of the codes, in the block's own
    uint32_t tap[8], t0[8];
    bool bad = false;
#pragma unroll
    for (int k = 0; k < 8; ++k) bad |= ((sel[c * 8 + k] >> 16) & 0xFFFF) >= g.cin;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int s = sel[c * 8 + k];
        const int ch = (s >> 16) & 0xFFFF, ky = (s >> 8) & 0xFF, kx = s & 0xFF;
        // the caller answers for taps inside the kernel window; any other reads within plane 0
        const bool in = !bad && ky < g.kh && kx < g.kw;
        const int row = g.base + ch * g.cs + ky * g.pitch;
        const uint32_t o0 = in ? row + phase_slot(g, kx) : g.base;
        const uint32_t o1 = in ? row + phase_slot(g, kx + g.sw) : g.base;
        tap[k] = t0[k] = o0 | (o1 << 16);
    }
    uint32_t ops = 0, code[7], inv[7], kind[7];  // kind: 0 always 0, 1 passes b, 2 reads both
    uint32_t raw[7];
#pragma unroll
    for (int q = 0; q < 7; ++q) {
        uint32_t f = gates[c * 7 + q] & 15u;  // bits 3..0: (a, b) = 00, 01, 10, 11
        if (bad) f = 15u;
        raw[q] = f;
        ops |= f << (4 * q);
        const int l = 2 * (q - 4);
        const uint32_t ia = q < 4 ? 0u : q < 6 ? inv[l] : inv[4];
        const uint32_t ib = q < 4 ? 0u : q < 6 ? inv[l + 1] : inv[5];
        if (ia) f = ((f & 12u) >> 2) | ((f & 3u) << 2);
        if (ib) f = ((f & 10u) >> 1) | ((f & 5u) << 1);
        inv[q] = f >> 3;
        if (inv[q]) f ^= 15u;  // now the value at 00 is 0: bits 2..0 = 01, 10, 11
        const bool za = q >= 4 && kind[q < 6 ? l : 4] == 0u;      // an operand that is always 0
        const bool zb = q >= 4 && kind[q < 6 ? l + 1 : 5] == 0u;
        if (za) f = (f & 4u) ? 5u : 0u;          // f(0, b): b or 0
        if (zb) f = (f & 2u) && !za ? 3u : 0u;   // f(a, 0): a or 0
        const bool swap = f == 2u || f == 3u;    // a & ~b, a
        if (swap) f = f == 2u ? 4u : 5u;         // ~a & b, b
        kind[q] = f == 0u ? 0u : f == 5u ? 1u : 2u;
        //        ab           ~ab             a^b             a|b
        code[q] = f == 1u ? 9u : f == 4u ? 13u : f == 6u ? 10u : f == 7u ? 14u : 0u;
        if (swap) {
            if (q < 4) {
                exchange(tap[2 * q], tap[2 * q + 1]);
            } else if (q < 6) {
                exchange(code[l], code[l + 1]);
                exchange(kind[l], kind[l + 1]);
                exchange(tap[2 * l], tap[2 * l + 2]);
                exchange(tap[2 * l + 1], tap[2 * l + 3]);
            } else {
                exchange(code[4], code[5]);
                exchange(kind[4], kind[5]);
                exchange(code[0], code[2]);
                exchange(code[1], code[3]);
                exchange(kind[0], kind[2]);
                exchange(kind[1], kind[3]);
#pragma unroll
                for (int k = 0; k < 4; ++k) exchange(tap[k], tap[k + 4]);
            }
        }
    }
    // a gate is evaluated when its reader is: dead ones keep their codes, which nothing looks at
    uint32_t codes = (inv[6] << 31) | (kind[6] == 0u ? 1u << 30 : 0u);
#pragma unroll
    for (int q = 0; q < 7; ++q) codes |= code[q] << (4 * q);
    if (!g.uniform) {
        // the lanes read every tap: one whose value cannot reach the root goes to one shared
        // word, which costs no bank conflicts
        uint32_t need[7];
        need[6] = 1u;
#pragma unroll
        for (int q = 6; q >= 0; --q) {
            const uint32_t f = raw[q];
            const uint32_t na = need[q] && ((f ^ (f >> 2)) & 3u);
            const uint32_t nb = need[q] && ((f ^ (f >> 1)) & 5u);
            if (q == 6) need[4] = na, need[5] = nb;
            else if (q >= 4) need[2 * (q - 4)] = na, need[2 * (q - 4) + 1] = nb;
            else {
                tap[2 * q] = na ? t0[2 * q] : uint32_t(g.base) * 0x10001u;
                tap[2 * q + 1] = nb ? t0[2 * q + 1] : uint32_t(g.base) * 0x10001u;
            }
        }
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        t[2 * k] = 4u * (tap[k] & 0xffffu);
        t[2 * k + 1] = 4u * (tap[k] >> 16);
    }
    t[16] = codes;
    t[17] = ops;
    t[18] = t[19] = 0u;
}

// Four words of a node, one per conv position of a pooling window (named words, so that each
// stays a register of its own across the branches).
struct Win {
    uint32_t x, y, z, w;
};

// b = gate(a, b) from the code's low four bits (uniform): nothing for a gate that passes b, else
// one three-input operation per word with a scalar mask.  Truth-table immediates over (first,
// second, third) = 0xF0, 0xCC, 0xAA.
__device__ __forceinline__ void gate_coded(uint32_t code, const Win& a, Win& b) {
    const uint32_t m = uint32_t(__builtin_amdgcn_sbfe(int(code), 2, 1));
    if (code & 1u) {  // m ? ~a & b : a & b
        b.x = __builtin_amdgcn_bitop3_b32(a.x, b.x, m, 0x48);
        b.y = __builtin_amdgcn_bitop3_b32(a.y, b.y, m, 0x48);
        b.z = __builtin_amdgcn_bitop3_b32(a.z, b.z, m, 0x48);
        b.w = __builtin_amdgcn_bitop3_b32(a.w, b.w, m, 0x48);
        asm volatile("");  // a branch, not selects
    }
    if (code & 2u) {  // m ? a | b : a ^ b
        b.x = __builtin_amdgcn_bitop3_b32(a.x, b.x, m, 0xBC);
        b.y = __builtin_amdgcn_bitop3_b32(a.y, b.y, m, 0xBC);
        b.z = __builtin_amdgcn_bitop3_b32(a.z, b.z, m, 0xBC);
        b.w = __builtin_amdgcn_bitop3_b32(a.w, b.w, m, 0xBC);
        asm volatile("");
    }
}

__device__ __forceinline__ uint32_t gate_bits(uint32_t f, uint32_t a, uint32_t b) {
    const uint32_t f00 = uint32_t(__builtin_amdgcn_sbfe(int(f), 3, 1));
    const uint32_t f01 = uint32_t(__builtin_amdgcn_sbfe(int(f), 2, 1));
    const uint32_t f10 = uint32_t(__builtin_amdgcn_sbfe(int(f), 1, 1));
    const uint32_t f11 = uint32_t(__builtin_amdgcn_sbfe(int(f), 0, 1));
    const uint32_t hi = (a & f11) | (~a & f01);
    const uint32_t lo = (a & f10) | (~a & f00);
    return (b & hi) | (~b & lo);
}

// LDS word (relative to the block's plane of its channel) of pooled position p of a block whose
// output feeds `n`.
__device__ __forceinline__ int next_word(const TreeColsBlock& g, const TreeColsBlock& n, int p) {
    const int py = int(fast_div(uint32_t(p), g.div_wp)), px = p - py * g.wp;
    const int m = 2 * n.sw;
    const int x = px + n.pw;
    const int xq = int(fast_div(uint32_t(x), n.div_m)), f = x - xq * m;
    return (py + n.ph) * n.pitch + f * n.q + (f < n.r ? f : n.r) + xq;
}

// A block whose waves take one channel each (uniform taps and gates): lane = pooled position.
template <int DY>
__device__ __forceinline__ void tree_block_uniform(uint32_t* lds, const uint32_t* __restrict__ tab,
                                                   const TreeColsBlock& g, const TreeColsBlock* nx,
                                                   uint32_t* __restrict__ out) {
    const int lane = lane_id();
    const int kp = g.P / 64;
    for (int k0 = 0; k0 < kp; ++k0) {
        const int p = k0 * 64 + lane;
        const int py = int(fast_div(uint32_t(p), g.div_wp)), px = p - py * g.wp;
        const int posb = py * 2 * DY + px;
        // a position whose value is never read by the next block is not stored
        const int ow = nx ? next_word(g, *nx, p) : p;
        const bool keep = !nx || (py + nx->ph < nx->hr && px + nx->pw < nx->wr);
        uint32_t* dst_lds = lds + (nx ? nx->base + ow : 0);
        uint32_t* dst_out = out + ow;
        const int cs = nx ? nx->cs : g.P, cout = g.cout;
        const bool last = !nx;
        const uint32_t* src = lds + posb;
        const char* srcb = reinterpret_cast<const char*>(src);
        const uint32_t* t = tab + wave_id() * kTcTabWords;
        for (int c = wave_id(); c < cout; c += kTcThreads / 64, t += kTcThreads / 64 * kTcTabWords) {
            // The instruction count bounds this loop (vector and scalar ones together), so a
            // branch guards each subtree, not each tap.  The empty asm keeps the table's loads
            // ahead of the branches.
            uint32_t o[16], codes = t[16];
#pragma unroll
            for (int k = 0; k < 16; ++k) o[k] = t[k];
            asm volatile("" ::"s"(codes), "s"(o[0]), "s"(o[1]), "s"(o[2]), "s"(o[3]), "s"(o[4]),
                         "s"(o[5]), "s"(o[6]), "s"(o[7]), "s"(o[8]), "s"(o[9]), "s"(o[10]),
                         "s"(o[11]), "s"(o[12]), "s"(o[13]), "s"(o[14]), "s"(o[15]));
            Win v0, v1, v2, v3, v4, v5, v6, v7;
            auto tap = [&](uint32_t o0, uint32_t o1, Win& v) {
                const uint32_t* p0 = reinterpret_cast<const uint32_t*>(srcb + o0);
                const uint32_t* p1 = reinterpret_cast<const uint32_t*>(srcb + o1);
                v.x = p0[0];
                v.y = p0[DY];
                v.z = p1[0];
                v.w = p1[DY];
            };
            auto both = [&](int q) { return (codes & (8u << (4 * q))) != 0u; };
            if (both(6)) {
                if (both(4)) {
                    if (both(0)) tap(o[0], o[1], v0);
                    tap(o[2], o[3], v1);
                }
                if (both(1)) tap(o[4], o[5], v2);
                tap(o[6], o[7], v3);
            }
            if (both(5)) {
                if (both(2)) tap(o[8], o[9], v4);
                tap(o[10], o[11], v5);
            }
            if (both(3)) tap(o[12], o[13], v6);
            tap(o[14], o[15], v7);
            if (both(6)) {
                if (both(4)) gate_coded(codes, v0, v1);
                gate_coded(codes >> 4, v2, v3);
                gate_coded(codes >> 16, v1, v3);
            }
            if (both(5)) gate_coded(codes >> 8, v4, v5);
            gate_coded(codes >> 12, v6, v7);
            gate_coded(codes >> 20, v5, v7);
            gate_coded(codes >> 24, v3, v7);
            // pool: the OR of the four words, each inverted when the root is
            const uint32_t root = uint32_t(int(codes) >> 31);
            uint32_t r = root;
            if (!(codes & (1u << 30)))
                r = __builtin_amdgcn_bitop3_b32(v7.x, v7.y, root, 0x7E) |
                    __builtin_amdgcn_bitop3_b32(v7.z, v7.w, root, 0x7E);
            if (last) dst_out[c * cs] = r;
            else if (keep) dst_lds[c * cs] = r;
        }
    }
}

// Any block: a lane per (channel, pooled position), taps and opcodes per lane.
__device__ __forceinline__ void tree_block_lanes(uint32_t* lds, const uint32_t* __restrict__ tab,
                                                 const TreeColsBlock& g, const TreeColsBlock* nx,
                                                 uint32_t* __restrict__ out) {
    const int dy = g.dy;
    for (int item = threadIdx.x; item < g.cout * g.P; item += kTcThreads) {
        const int c = int(fast_div(uint32_t(item), g.div_p)), p = item - c * g.P;
        const int py = int(fast_div(uint32_t(p), g.div_wp)), px = p - py * g.wp;
        const int posb = py * 2 * dy + px;
        const uint4* t4 = reinterpret_cast<const uint4*>(tab + c * kTcTabWords);
        const uint32_t ops = tab[c * kTcTabWords + 17];
        const char* row0 = reinterpret_cast<const char*>(lds + posb);
        const char* row1 = row0 + 4 * dy;
        uint32_t v[8][4];
#pragma unroll
        for (int k = 0; k < 8; k += 2) {
            const uint4 o = t4[k / 2];  // two taps
            v[k][0] = *reinterpret_cast<const uint32_t*>(row0 + o.x);
            v[k][1] = *reinterpret_cast<const uint32_t*>(row0 + o.y);
            v[k][2] = *reinterpret_cast<const uint32_t*>(row1 + o.x);
            v[k][3] = *reinterpret_cast<const uint32_t*>(row1 + o.y);
            v[k + 1][0] = *reinterpret_cast<const uint32_t*>(row0 + o.z);
            v[k + 1][1] = *reinterpret_cast<const uint32_t*>(row0 + o.w);
            v[k + 1][2] = *reinterpret_cast<const uint32_t*>(row1 + o.z);
            v[k + 1][3] = *reinterpret_cast<const uint32_t*>(row1 + o.w);
        }
        uint32_t r = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t n[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) n[q] = gate_bits(ops >> (4 * q), v[2 * q][i], v[2 * q + 1][i]);
            r |= gate_bits(ops >> 24, gate_bits(ops >> 16, n[0], n[1]),
                           gate_bits(ops >> 20, n[2], n[3]));
        }
        if (nx) {
            if (py + nx->ph < nx->hr && px + nx->pw < nx->wr)
                lds[nx->base + c * nx->cs + next_word(g, *nx, p)] = r;
        } else {
            out[item] = r;
        }
    }
}

// Persistent workgroups, one column at a time: the next column's words are in flight while the
// blocks run, and go to the first block's planes as soon as that block is done with them.
template <int IPT>
__global__ __launch_bounds__(kTcThreads) void k_tree_cols(const uint32_t* __restrict__ x,
                                                          int64_t cols,
                                                          const TreeColsBlock* __restrict__ desc,
                                                          const uint32_t* __restrict__ tables,
                                                          TreeCols t, uint32_t* __restrict__ y) {
    extern __shared__ __align__(16) uint32_t lds[];
    const int tid = threadIdx.x;
    for (int i = tid; i < t.lds_words; i += kTcThreads) lds[i] = 0;  // the halos stay zero
    const TreeColsBlock& g0 = desc[0];
    // LDS words of input words tid + 1024 j, two to a register; 0xffff: no tap reaches it
    uint32_t dst[IPT / 2];
    {
        const int hw = g0.h * g0.w;
#pragma unroll
        for (int j = 0; j < IPT; ++j) {
            const int rr = tid + kTcThreads * j;
            const int ch = rr / hw, pix = rr - ch * hw;
            const int iy = pix / g0.w + g0.ph, ix = pix % g0.w + g0.pw;
            const bool in = rr < t.in_rows && iy < g0.hr && ix < g0.wr;
            const uint32_t d = in ? g0.base + ch * g0.cs + iy * g0.pitch + phase_slot(g0, ix)
                                  : 0xffffu;
            if (j % 2) dst[j / 2] |= d << 16;
            else dst[j / 2] = d;
        }
    }
    uint32_t in[IPT];
    auto fetch = [&](int64_t c) {
#pragma unroll
        for (int j = 0; j < IPT; ++j) {
            const int rr = tid + kTcThreads * j;
            in[j] = c < cols && rr < t.in_rows ? x[c * t.in_words + rr] : 0u;
        }
    };
    auto stage = [&]() {
#pragma unroll
        for (int j = 0; j < IPT; ++j) {
            const uint32_t d = (dst[j / 2] >> (16 * (j % 2))) & 0xffffu;
            if (d != 0xffffu) lds[d] = in[j];
        }
    };
    int64_t col = blockIdx.x;
    const int64_t step = gridDim.x;
    fetch(col);
    __syncthreads();
    stage();
    fetch(col + step);
    __syncthreads();
    for (; col < cols; col += step) {  // uniform: every thread meets every barrier
        for (int b = 0; b < t.nb; ++b) {
            const TreeColsBlock& g = desc[b];
            const TreeColsBlock* nx = b + 1 < t.nb ? desc + b + 1 : nullptr;
            const uint32_t* tab = tables + g.tab;
            uint32_t* out = y + col * t.out_words;
            if (g.uniform && g.dy == kTcDy[0]) tree_block_uniform<kTcDy[0]>(lds, tab, g, nx, out);
            else if (g.uniform && g.dy == kTcDy[1]) tree_block_uniform<kTcDy[1]>(lds, tab, g, nx, out);
            else if (g.uniform) tree_block_uniform<kTcDy[2]>(lds, tab, g, nx, out);
            else tree_block_lanes(lds, tab, g, nx, out);
            __syncthreads();  // this block's output is complete, its input is free
            if (b == 0) {
                stage();
                fetch(col + 2 * step);
                if (t.nb == 1) __syncthreads();
            }
        }
    }
}

// ------------------------------------------------------------------------------------------
// Rows of packed words to columns: y[c * out_words + r] = word c of row r.  A workgroup moves 64
// rows x 128 words through LDS (pitch 129: the column reads of a half-wave meet 32 banks);
// XCD x takes a contiguous range of column tiles, every row tile of one before the next, so a
// column's 256-byte runs are written close in time.
constexpr int kTrRows = 64, kTrWords = 128;

__global__ __launch_bounds__(256) void k_rows_to_columns(const uint32_t* __restrict__ x,
                                                         uint32_t* __restrict__ y, int64_t rows,
                                                         int64_t cols, int64_t out_words,
                                                         int64_t row_tiles,
                                                         int64_t tiles_per_xcd) {
    __shared__ uint32_t tile[kTrRows][kTrWords + 1];
    const int64_t i = blockIdx.x / 8;
    const int64_t ct = (blockIdx.x % 8) * tiles_per_xcd + i / row_tiles;
    const int64_t r0 = (i % row_tiles) * kTrRows, c0 = ct * kTrWords;
    if (c0 >= cols) return;  // uniform per workgroup
    const int w = wave_id(), lane = lane_id();
    uint32_t v[kTrRows / 4][2];
#pragma unroll
    for (int k = 0; k < kTrRows / 4; ++k) {
        const int64_t r = std::min(r0 + w * (kTrRows / 4) + k, rows - 1);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int64_t c = std::min(c0 + 64 * h + lane, cols - 1);
            v[k][h] = __builtin_nontemporal_load(x + r * cols + c);
        }
    }
#pragma unroll
    for (int k = 0; k < kTrRows / 4; ++k)
#pragma unroll
        for (int h = 0; h < 2; ++h) tile[w * (kTrRows / 4) + k][64 * h + lane] = v[k][h];
    __syncthreads();
#pragma unroll 4
    for (int j = w; j < kTrWords; j += 4) {
        const int64_t c = c0 + j, r = r0 + lane;
        if (c < cols && r < rows) y[c * out_words + r] = tile[lane][j];
    }
}

// Geometry of a chain of blocks, geom[b] = (cin, h, w, cout, sh, sw, ph, pw, kh, kw); false when
// the chain does not fit: more than four blocks, an input wider than 16 words per thread, planes
// beyond LDS, blocks that do not follow one another.
bool tree_cols_plan(const int64_t* geom, int64_t nb, TreeCols& t, TreeColsBlock* blocks) {
    if (nb < 1 || nb > kTcMaxBlocks) return false;
    t = TreeCols{};
    t.nb = int(nb);
    int64_t base = 0, tab = 0;
    for (int64_t b = 0; b < nb; ++b) {
        const int64_t* e = geom + 10 * b;
        for (int i = 0; i < 10; ++i)
            if (e[i] < (i == 6 || i == 7 ? 0 : 1) || e[i] > 65535) return false;
        TreeColsBlock& g = blocks[b];
        g = TreeColsBlock{};
        g.cin = int(e[0]), g.h = int(e[1]), g.w = int(e[2]), g.cout = int(e[3]);
        g.sh = int(e[4]), g.sw = int(e[5]), g.ph = int(e[6]), g.pw = int(e[7]);
        const int kh = g.kh = int(e[8]), kw = g.kw = int(e[9]);
        if (g.h + 2 * g.ph < kh || g.w + 2 * g.pw < kw || kh > 255 || kw > 255) return false;
        const int ho = (g.h + 2 * g.ph - kh) / g.sh + 1, wo = (g.w + 2 * g.pw - kw) / g.sw + 1;
        if (ho % 2 || wo % 2 || ho == 0 || wo == 0) return false;
        g.wp = wo / 2;
        g.P = (ho / 2) * g.wp;
        if (int64_t(g.cout) * g.P >= (int64_t(1) << 24)) return false;
        g.hr = (ho - 1) * g.sh + kh;
        g.wr = (wo - 1) * g.sw + kw;
        g.q = g.wr / (2 * g.sw);
        g.r = g.wr % (2 * g.sw);
        if (b > 0) {
            const TreeColsBlock& p = blocks[b - 1];
            if (g.cin != p.cout || g.h * g.w != p.P || g.w != p.wp) return false;
        } else {
            if (int64_t(g.cin) * g.h * g.w > int64_t(kTcMaxIpt) * kTcThreads) return false;
            t.in_rows = g.cin * g.h * g.w;
        }
        // pitch: the first conv-row distance with paired reads that holds a row, when a wave can
        // take one channel and the planes fit; else odd, which spreads the rows over the banks
        g.uniform = 0;
        g.pitch = g.wr | 1;
        if (g.P % 64 == 0)
            for (int dy : kTcDy)
                if (!g.uniform && dy % g.sh == 0 && dy / g.sh >= g.wr &&
                    base + int64_t(g.cin) * g.hr * (dy / g.sh) <= kTcLdsWords) {
                    g.uniform = 1;
                    g.pitch = dy / g.sh;
                }
        g.dy = g.sh * g.pitch;
        if (int64_t(g.hr) * g.pitch > kTcLdsWords) return false;
        g.cs = g.hr * g.pitch;
        g.base = int(base);
        base += int64_t(g.cin) * g.cs;
        if (base > kTcLdsWords) return false;
        g.tab = int(tab);
        tab += int64_t(g.cout) * kTcTabWords;
        g.div_p = make_fastdiv(uint32_t(g.P));
        g.div_wp = make_fastdiv(uint32_t(g.wp));
        g.div_m = make_fastdiv(uint32_t(2 * g.sw));
    }
    t.lds_words = int(base);
    return true;
}

}  // namespace
}  // namespace cl

using namespace cl;

extern "C" int cl_packed_rows_to_columns(const void* x, void* y, int64_t rows, int64_t row_bytes,
                                         int64_t out_words, void* stream) {
    clear_error();
    CL_ARG(rows >= 0 && row_bytes >= 0, "negative shape");
    CL_ARG(row_bytes % 4 == 0, "packed rows must be a multiple of 4 bytes");
    CL_ARG(out_words >= rows, "out_words (%lld) must be at least the %lld rows",
           (long long)out_words, (long long)rows);
    const int64_t cols = row_bytes / 4;
    if (rows == 0 || cols == 0) return CL_OK;
    CL_ARG(x && y, "null pointer argument");
    CL_ARG(aligned(x, 4) && aligned(y, 4), "misaligned buffers");
    const int64_t row_tiles = ceil_div(rows, kTrRows);
    const int64_t per_xcd = ceil_div(ceil_div(cols, kTrWords), 8);
    CL_ARG(8 * per_xcd * row_tiles < (int64_t(1) << 31), "too many words for one launch");
    k_rows_to_columns<<<unsigned(8 * per_xcd * row_tiles), 256, 0, as_stream(stream)>>>(
        static_cast<const uint32_t*>(x), static_cast<uint32_t*>(y), rows, cols, out_words,
        row_tiles, per_xcd);
    return check_launch("cl_packed_rows_to_columns");
}

extern "C" int cl_tree_columns_layout(const int64_t* geometry, int64_t num_blocks,
                                      int64_t* applies, int64_t* in_rows, int64_t* out_rows,
                                      int64_t* table_words) {
    clear_error();
    CL_ARG(geometry && applies && in_rows && out_rows && table_words, "null pointer argument");
    TreeCols t;
    TreeColsBlock blk[kTcMaxBlocks];
    *applies = *in_rows = *out_rows = *table_words = 0;
    if (!tree_cols_plan(geometry, num_blocks, t, blk)) return CL_OK;
    const TreeColsBlock& last = blk[t.nb - 1];
    *applies = 1;
    *in_rows = t.in_rows;
    *out_rows = int64_t(last.cout) * last.P;
    *table_words = int64_t(t.nb) * kTcDescWords + last.tab + int64_t(last.cout) * kTcTabWords;
    return CL_OK;
}

extern "C" int cl_tree_columns(const void* x, int64_t cols, int64_t in_words,
                               const int64_t* geometry, int64_t num_blocks,
                               const uint8_t* const* gates, const int32_t* const* selections,
                               void* tables, void* y, int64_t out_words, void* stream) {
    clear_error();
    TreeCols t;
    TreeColsBlock blk[kTcMaxBlocks];
    CL_ARG(geometry && gates && selections, "null pointer argument");
    CL_ARG(tree_cols_plan(geometry, num_blocks, t, blk),
           "the blocks do not fit the column pass (cl_tree_columns_layout)");
    const TreeColsBlock& last = blk[t.nb - 1];
    CL_ARG(cols >= 0 && cols < (int64_t(1) << 31), "bad column count");
    CL_ARG(in_words >= t.in_rows && in_words < (int64_t(1) << 31) &&
               out_words >= int64_t(last.cout) * last.P && out_words < (int64_t(1) << 31),
           "in_words or out_words too small");
    if (cols == 0) return CL_OK;
    CL_ARG(x && tables && y, "null pointer argument");
    CL_ARG(aligned(x, 4) && aligned(tables, 16) && aligned(y, 4), "misaligned buffers");
    t.in_words = int(in_words);
    t.out_words = int(out_words);
    hipStream_t s = as_stream(stream);
    static_assert(sizeof(TreeColsBlock) % 4 == 0, "descriptor size");
    auto* desc = static_cast<TreeColsBlock*>(tables);
    auto* tab = static_cast<uint32_t*>(tables) + t.nb * kTcDescWords;
    for (int b = 0; b < t.nb; ++b) {
        CL_ARG(gates[b] && selections[b], "null pointer argument");
        k_tree_cols_tables<<<unsigned(ceil_div(blk[b].cout, 256)), 256, 0, s>>>(
            gates[b], selections[b], blk[b], desc + b, tab + blk[b].tab);
    }
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
        set_error("cannot query the device");
        return CL_ERR_HIP;
    }
    const int lds = t.lds_words * 4;
    const unsigned grid = unsigned(std::min<int64_t>(cols, std::max(cus, 1)));
    auto go = [&](auto ipt) {
        auto* kern = &k_tree_cols<decltype(ipt)::value>;
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) {
            set_error("cannot reserve %d bytes of LDS for the column pass", lds);
            return int(CL_ERR_HIP);
        }
        kern<<<grid, kTcThreads, lds, s>>>(static_cast<const uint32_t*>(x), cols, desc, tab, t,
                                           static_cast<uint32_t*>(y));
        return check_launch("cl_tree_columns");
    };
    if (t.in_rows <= 4 * kTcThreads) return go(std::integral_constant<int, 4>{});
    if (t.in_rows <= 10 * kTcThreads) return go(std::integral_constant<int, 10>{});
    return go(std::integral_constant<int, kTcMaxIpt>{});
}
