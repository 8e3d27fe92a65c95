// A pruned packed network on columns for gfx950: the two-input gates that are left of a frozen
// network once constants, pass-through gates and gates that nothing reads are folded away
// (packed_circuit.py builds the tables), evaluated level by level in LDS, and the class counts.
//
// The fused passes in packed_net.hip evaluate every row of every layer.  Of a network with
// random gates a quarter of the gates pass an operand, an eighth are constant, and what reads
// a constant folds in turn: 22800 two-input gates are left of the 72000 of 784 -> 6 x 12000,
// 16700 of the 32000 of a 2 x 16000 tail.  A signal may be read by any later level, so rows do
// not live in per-layer buffers but in pages of 64 LDS words, handed out when a wave writes its
// 64 gates and reused once the last level that reads one of them is done: a whole network of two
// convolutions of 9 x 32 x 32 and 2 x 16000 (122600 rows, 28000 to 31000 gates left) fits.
// Against all rows: 784 -> 6 x 12000 for 4 M samples 1.51 ms (3.96), the tail 2 x 16000 of a
// logic-tree network for 1 M 0.38 (0.66), the convolutions and their tail for 1 M 1.29 (2.47):
// rows turned to columns 0.48, the circuit 0.80.  Where it is not the faster one:
// packed_circuit.pays.
//
// What bounds it: a workgroup has the CU's LDS to itself, so its phases follow one another.  Of
// 14000 cycles per column of 64 samples of the first, the gates take 7000 (22 pages per wave, six
// words each, 1.07 passes per read), waiting at the levels' barriers 2300, the class counts 4000
// (vector work on ten of sixteen waves) and staging 500; over the pass the vector units are 59 %
// busy and LDS 41 %.
//
// A thread holds its gates in registers for the whole launch (slot q: gate lane of the wave's
// q-th page): the LDS word addresses of both operands, 16 bits each, and the opcode.  A signal is
// two 32-bit words, 64 samples, in the two halves of its page, so one instruction reads or
// writes both (ds_read2st64 / ds_write2st64) and the address arithmetic of a gate serves 64
// samples.  A gate that is 1 for a = b = 0 is kept inverted by the builder, which leaves three
// opcode bits per gate.  Pages of one kind of gate, with a branch per page in
// place of the masks, took 2.09 ms where this form with the same counting took 1.65: scalar work
// in place of vector work, and two passes per read for want of freedom in placing the gates.
// The barriers order LDS alone, and the next column's input stays in flight across them (1.65 to
// 1.47 ms).  Words 64 apart in a page of their own, with the opcode beside the addresses, cost 2 %
// of that and let the circuit have all of LDS.
#include "common.h"

#include <algorithm>

namespace cl {
namespace {

constexpr int kPcThreads = 1024;
constexpr int kPageWords = 128;      // 64 signals: word 0 of each, then word 1
constexpr int kPcMaxPages = 320;     // all of LDS
constexpr int kPcMaxSlots = 48;
constexpr int kPcRound = 8;          // input pages per wave held in registers at most
constexpr int kPcMaxRounds = 2;
constexpr int kPcMaxSteps = 508;     // counted entries of a lane: below 2^9
constexpr uint32_t kNone = 0xffffu;

struct CircuitNet {
    const uint32_t* ent;     // [slots][1024] operand words, a | b << 16
    const uint32_t* ops;     // [slots / 8][1024] nibbles: the gate's values for ab = 01, 10, 11
    const uint32_t* dst;     // [16][max slots / 2] per wave: page words of slots 2i, 2i + 1
    const uint16_t* in;      // [in_pages][64] input row of a signal of pages 1, 2, ...
    const uint2* cnt;        // [groups][k][64] four LDS words
    const int32_t* ones;     // [k] added to every count
    uint32_t start;          // bit i: slots 2i, 2i + 1 begin a level
    int pairs, groups, groups_inv, in_pages, in_words, k;
};

typedef uint32_t word_pair __attribute__((ext_vector_type(2), aligned(4)));
using lds_word = __attribute__((address_space(3))) uint32_t;

// An LDS word (the pass has no static LDS: its pages begin at address 0).
__device__ __forceinline__ lds_word* lds_at(uint32_t word) {
    return reinterpret_cast<lds_word*>(word << 2);
}

// The LDS word in the low half of v: one instruction, where the compiler takes two.
__device__ __forceinline__ lds_word* lds_at_low(uint32_t v) {
    uint32_t byte;
    asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD "
        "src1_sel:WORD_0"
        : "=v"(byte)
        : "v"(2u), "v"(v));
    return reinterpret_cast<lds_word*>(byte);
}

// A barrier that orders LDS only: global loads and stores stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <uint32_t TABLE>
__device__ __forceinline__ uint32_t bitop(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_amdgcn_bitop3_b32(a, b, c, TABLE);
}

// a, return = sum and carry of a + x + y on bit planes; INV: of a + ~x + ~y.
template <bool INV>
__device__ __forceinline__ uint32_t plane_add(uint32_t& a, uint32_t x, uint32_t y) {
    constexpr uint32_t A = 0xF0, X = INV ? 0x33 : 0xCC, Y = INV ? 0x55 : 0xAA;
    const uint32_t carry = bitop<((A & X) | (A & Y) | (X & Y)) & 0xFF>(a, x, y);
    a = bitop<(A ^ X ^ Y) & 0xFF>(a, x, y);
    return carry;
}

// One stage of gathering a half-wave's bits of a sample in one lane: a 32 x 32 bit transpose
// (row = lane, column = sample) up to the order of the rows, which a popcount does not see.
// Lanes with bit K clear keep the columns with bit K clear.
template <int K>
__device__ __forceinline__ uint32_t gather_stage(uint32_t t, int lane) {
    const bool low = (lane & K) == 0;
    if constexpr (K == 16) {
        const auto p = __builtin_amdgcn_permlane16_swap(t, t, false, false);
        return __builtin_amdgcn_perm(p[1], p[0], low ? 0x05040100u : 0x07060302u);
    } else if constexpr (K == 8) {
        return __builtin_amdgcn_perm(dpp_move<0x128>(t), t, low ? 0x06020400u : 0x07030501u);
    } else {
        constexpr uint32_t m = K == 4 ? 0x0F0F0F0Fu : K == 2 ? 0x33333333u : 0x55555555u;
        // the partner of bit 2 is lane ^ 7 (row_half_mirror), of bits 1 and 0 a quad permutation
        const uint32_t p = dpp_move<K == 4 ? 0x141 : K == 2 ? 0x4E : 0xB1>(t);
        const uint32_t sh = __builtin_amdgcn_alignbit(p, p, low ? 32 - K : K);
        const uint32_t keep = low ? m : ~m;
        return (t & keep) | (sh & ~keep);
    }
}

// Adds a group of four entries per lane to the bit planes of both words.
template <int B, bool INV>
__device__ __forceinline__ void count_group(uint2 v, uint32_t (&p)[2][B]) {
    const lds_word* at[4] = {lds_at_low(v.x), lds_at(v.x >> 16), lds_at_low(v.y), lds_at(v.y >> 16)};
    uint32_t x[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i][0] = at[i][0], x[i][1] = at[i][64];
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        const uint32_t c0 = plane_add<INV>(p[w][0], x[0][w], x[1][w]);
        const uint32_t c1 = plane_add<INV>(p[w][0], x[2][w], x[3][w]);
        uint32_t c = plane_add<false>(p[w][1], c0, c1);
#pragma unroll
        for (int i = 2; i < B; ++i) {
            const uint32_t carry = p[w][i] & c;
            p[w][i] ^= c;
            c = carry;
        }
    }
}

// The count entries of a class, AHEAD groups of them.  Where the gates leave registers for them, a
// wave keeps the first of its first class for the whole launch.
template <int AHEAD>
struct Entries {
    uint2 v[AHEAD];
    int32_t ones;
    __device__ __forceinline__ void load(const CircuitNet& net, int c, int group) {
        const int last = net.groups + net.groups_inv - 1;
        ones = 0;
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) v[i] = make_uint2(0, 0);
        if (c < net.k) ones = net.ones[c];
        if (c < net.k && last >= 0)  // uniform; past the last group it is loaded again, unused
#pragma unroll
            for (int i = 0; i < AHEAD; ++i)
                v[i] = net.cnt[(size_t(min(group + i, last)) * net.k + c) * 64 + lane_id()];
        // waited for here, whichever of them are used: a load that may still be in flight at its
        // register's next use would have every gate of the next column wait for the input too
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) asm volatile("" : "+v"(v[i].x), "+v"(v[i].y));
        asm volatile("" : "+v"(ones));
    }
};

// Class counts of a column, one wave per class: every lane adds the words of its entries into B
// bit planes (a carry-save tree of four entries at a time; groups counted inverted come after
// the others, and the zero page pads both), the half-waves' planes are added with one word on
// each, and each plane's bits of a sample are gathered in one lane and summed by popcount.
template <int B, bool KEPT, int AHEAD>
__device__ __forceinline__ void circuit_counts(const CircuitNet& net, const Entries<AHEAD>& first,
                                               int64_t word, int64_t nsamples,
                                               int32_t* __restrict__ counts) {
    int lane = lane_id();
    asm volatile("" : "+v"(lane));  // the stages' lane constants are not worth registers elsewhere
    const int total = net.groups + net.groups_inv;
    for (int c = wave_id(); c < net.k; c += kPcThreads / 64) {  // uniform per wave
        Entries<AHEAD> e = first;
        if (!KEPT || c >= kPcThreads / 64) e.load(net, c, 0);
        uint32_t p[2][B], q[B + 1];
#pragma unroll
        for (int i = 0; i < B; ++i) p[0][i] = p[1][i] = 0;
        for (int g = 0; g < total; g += AHEAD) {
            if (g > 0) e.load(net, c, g);
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) {
                if (g + i < net.groups) count_group<B, false>(e.v[i], p);
                else if (g + i < total) count_group<B, true>(e.v[i], p);
            }
        }
        uint32_t carry = 0;
#pragma unroll
        for (int i = 0; i < B; ++i) {
            // lanes 0-31: word 0 of both half-waves; lanes 32-63: word 1
            const auto s = __builtin_amdgcn_permlane32_swap(p[0][i], p[1][i], false, false);
            q[i] = s[0];
            carry = plane_add<false>(q[i], s[1], carry);
        }
        q[B] = carry;
        int32_t n = e.ones;
#pragma unroll
        for (int b = 0; b <= B; ++b) {
            uint32_t t = gather_stage<16>(q[b], lane);
            t = gather_stage<8>(t, lane);
            t = gather_stage<4>(t, lane);
            t = gather_stage<2>(t, lane);
            t = gather_stage<1>(t, lane);
            n += int32_t(__builtin_popcount(t)) << b;
        }
        const int64_t sample = word * 32 + lane;
        if (sample < nsamples) counts[sample * net.k + c] = n;
    }
}

// Persistent workgroups: columns of two words, a contiguous range per XCD.  COLS: x is
// column-major, x[c * in_words + row]; else rows of `cols` words.  Pages of input are reused by
// gates but not by gates that the counts read, so the next column is staged while this one is
// counted: rounds of up to IPT pages per wave, the first loaded a column ahead.
template <int TG, int IPT, int B, bool COLS>
__global__ __launch_bounds__(kPcThreads) void k_packed_circuit(const uint32_t* __restrict__ x,
                                                               int64_t cols, int64_t nsamples,
                                                               CircuitNet net,
                                                               int32_t* __restrict__ counts) {
    const int tid = threadIdx.x, lane = lane_id(), wave = wave_id();
    uint32_t ent[TG], ops[TG / 8];
    const int slots = 2 * net.pairs;
#pragma unroll
    for (int q = 0; q < TG; ++q) ent[q] = q < slots ? net.ent[q * kPcThreads + tid] : 0u;
#pragma unroll
    for (int q = 0; q < TG / 8; ++q) ops[q] = 8 * q < slots ? net.ops[q * kPcThreads + tid] : 0u;
    constexpr int kRounds = IPT < kPcRound ? 1 : kPcMaxRounds;
    uint32_t src[kRounds][IPT];  // input rows; two share a register
#pragma unroll
    for (int r = 0; r < kRounds; ++r)
#pragma unroll
        for (int j = 0; j < IPT; ++j) {
            const int page = (r * IPT + j) * (kPcThreads / 64) + wave;
            src[r][j] = page < net.in_pages ? net.in[page * 64 + lane] : kNone;
        }
    uint32_t row[kRounds][(IPT + 1) / 2];
#pragma unroll
    for (int r = 0; r < kRounds; ++r)
#pragma unroll
        for (int j = 0; j < IPT; j += 2)
            row[r][j / 2] = src[r][j] | (j + 1 < IPT ? src[r][j + 1] << 16 : kNone << 16);
    if (tid < kPageWords) *lds_at(tid) = 0;  // page 0: zeros
    uint32_t dst[TG / 2];  // scalar registers
#pragma unroll
    for (int i = 0; i < TG / 2; ++i)
        dst[i] = __builtin_amdgcn_readfirstlane(net.dst[wave * (kPcMaxSlots / 2) + i]);
    const int64_t units = (cols + 1) / 2;
    const int64_t per = (units + 7) / 8;
    const int64_t nb8 = gridDim.x / 8;
    const int64_t u_first = (blockIdx.x % 8) * per + blockIdx.x / 8;
    const int64_t u_end = std::min(units, (blockIdx.x % 8 + 1) * per);
    uint32_t in[IPT][2];
    auto rows_of = [&](int r, int j) { return (row[r][j / 2] >> (16 * (j % 2))) & 0xffffu; };
    auto fetch = [&](int r, int64_t u) {
        const bool both = 2 * u + 1 < cols;
#pragma unroll
        for (int j = 0; j < IPT; ++j) {
            const uint32_t i = rows_of(r, j);
            in[j][0] = in[j][1] = 0;
            if (u < u_end && i != kNone) {
                const uint32_t* p = x + (COLS ? 2 * u * net.in_words + i : i * cols + 2 * u);
                if (COLS) {
                    in[j][0] = p[0];
                    if (both) in[j][1] = p[net.in_words];
                } else if (both) {  // one access for both words: every lane reads a line of its own
                    const word_pair v = *reinterpret_cast<const word_pair*>(p);
                    in[j][0] = v.x, in[j][1] = v.y;
                } else {
                    in[j][0] = p[0];
                }
            }
        }
    };
    auto stage = [&](int r) {
        int at = lane;
        asm volatile("" : "+v"(at));  // addresses are not worth registers from column to column
#pragma unroll
        for (int j = 0; j < IPT; ++j)
            if (rows_of(r, j) != kNone) {
                const int page = 1 + (r * IPT + j) * (kPcThreads / 64) + wave;
                lds_word* out = lds_at(page * kPageWords + at);
                out[0] = in[j][0];
                out[64] = in[j][1];
            }
    };
    constexpr int kPageRound = IPT * (kPcThreads / 64);
    // the rounds after the first of column u
    auto more = [&](int64_t u) {
#pragma unroll
        for (int r = 1; r < kRounds; ++r)
            if (r * kPageRound < net.in_pages) {  // uniform
                fetch(r, u);
                stage(r);
            }
    };
    fetch(0, u_first);
    stage(0);
    more(u_first);
    Entries<B == 5 ? 4 : 1> entries;
    constexpr bool kKept = TG <= 32;
    if (kKept) entries.load(net, wave, 0);
    __builtin_amdgcn_s_waitcnt(0);  // the tables are there: no wait for them in the loop
    fetch(0, u_first + nb8);
    lds_barrier();
    for (int64_t u = u_first; u < u_end; u += nb8) {
#pragma unroll
        for (int b = 0; b < TG / 4; ++b) {
            if (2 * b < net.pairs) {  // uniform
                // four slots' reads in flight; a level may begin with the second pair
                const bool split = (net.start >> (2 * b + 1)) & 1u;
                uint32_t va[4][2], vb[4][2], page[4];
                auto read = [&](int j0) {
#pragma unroll
                    for (int j = j0; j < j0 + 2; ++j) {
                        const int q = 4 * b + j;
                        page[j] = (dst[q / 2] >> (16 * (q % 2))) & 0xffffu;  // uniform per wave
                        if (page[j] != kNone) {
                            const lds_word* ra = lds_at_low(ent[q]);
                            const lds_word* rb = lds_at(ent[q] >> 16);
                            va[j][0] = ra[0], va[j][1] = ra[64];
                            vb[j][0] = rb[0], vb[j][1] = rb[64];
                        }
                    }
                };
                auto write = [&](int j0) {
#pragma unroll
                    for (int j = j0; j < j0 + 2; ++j) {
                        const int q = 4 * b + j;
                        if (page[j] != kNone) {
                            const int o = int(ops[q / 8]), at = 4 * (q % 8);
                            const uint32_t f01 = uint32_t(__builtin_amdgcn_sbfe(o, at, 1));
                            const uint32_t f10 = uint32_t(__builtin_amdgcn_sbfe(o, at + 1, 1));
                            const uint32_t f11 = uint32_t(__builtin_amdgcn_sbfe(o, at + 2, 1));
                            lds_word* out = lds_at(page[j] + lane);
#pragma unroll
                            for (int w = 0; w < 2; ++w) {
                                const uint32_t a = va[j][w], c = vb[j][w];
                                const uint32_t hi = (a & f11) | (~a & f01);  // b = 1
                                const uint32_t lo = a & f10;                 // b = 0
                                out[64 * w] = (c & hi) | (~c & lo);
                            }
                        }
                    }
                };
                if (b > 0 && (net.start >> (2 * b)) & 1u) lds_barrier();
                read(0);
                if (!split) read(2);
                write(0);
                if (split) {
                    lds_barrier();
                    read(2);
                }
                write(2);
            }
        }
        // the staged words are waited for here, not behind the stores of the counts
#pragma unroll
        for (int j = 0; j < IPT; ++j) asm volatile("" : "+v"(in[j][0]), "+v"(in[j][1]));
        lds_barrier();
        stage(0);
        more(u + nb8);
        circuit_counts<B, kKept>(net, entries, u * 2, nsamples, counts);
        // opaque per column: keeps the compiler from hoisting the addresses it derives from
        // them out of the column loop, three registers per gate, and has what the counts made
        // it spill back before the input is asked for: it would be waited for behind that
#pragma unroll
        for (int q = 0; q < TG; ++q) asm volatile("" : "+v"(ent[q]));
#pragma unroll
        for (int q = 0; q < TG / 8; ++q) asm volatile("" : "+v"(ops[q]));
#pragma unroll
        for (int i = 0; i < TG / 2; ++i) asm volatile("" : "+s"(dst[i]));
#pragma unroll
        for (int r = 0; r < kRounds; ++r)
#pragma unroll
            for (int j = 0; j < (IPT + 1) / 2; ++j) asm volatile("" : "+v"(row[r][j]));
        fetch(0, u + 2 * nb8);  // in flight through the next column's gates, not the counts
        lds_barrier();
    }
}

}  // namespace
}  // namespace cl

using namespace cl;

extern "C" int cl_packed_circuit_limits(int64_t* max_pages, int64_t* max_slots,
                                        int64_t* max_steps, int64_t* max_input_pages) {
    clear_error();
    CL_ARG(max_pages && max_slots && max_steps && max_input_pages, "null pointer argument");
    *max_pages = kPcMaxPages;
    *max_slots = kPcMaxSlots;
    *max_steps = kPcMaxSteps;
    *max_input_pages = kPcMaxRounds * kPcRound * (kPcThreads / 64);
    return CL_OK;
}

extern "C" int cl_packed_circuit(const void* x, int64_t cols, int64_t columns_major,
                                 int64_t in_words, int64_t nsamples, const int64_t* shape,
                                 const uint32_t* ent, const uint32_t* ops, const uint32_t* dst,
                                 const uint16_t* in, const uint32_t* cnt, const int32_t* ones,
                                 int32_t* counts, void* stream) {
    clear_error();
    CL_ARG(shape && cols >= 0, "bad arguments");
    const int64_t pairs = shape[0], start = shape[1], groups = shape[2], inv = shape[3],
                  in_pages = shape[4], k = shape[5], pages = shape[6];
    CL_ARG(pairs >= 0 && 2 * pairs <= kPcMaxSlots, "too many slots");
    CL_ARG(start >= 0 && start < (int64_t(1) << 32), "bad level mask");
    CL_ARG(groups >= 0 && inv >= 0 && 4 * (groups + inv) <= kPcMaxSteps, "bad step count");
    CL_ARG(pages >= 1 && pages <= kPcMaxPages && in_pages >= 0 && in_pages < pages &&
               in_pages <= kPcMaxRounds * kPcRound * (kPcThreads / 64), "bad page count");
    CL_ARG(k >= 1 && k <= (int64_t(1) << 16), "bad class count");
    CL_ARG(nsamples >= 0 && nsamples <= cols * 32, "more samples than packed bits");
    CL_ARG(!columns_major || (in_words >= 0 && in_words < (int64_t(1) << 31)), "bad arguments");
    if (nsamples == 0 || cols == 0) return CL_OK;
    CL_ARG(x && ent && ops && dst && in && cnt && ones && counts, "null pointer argument");
    CL_ARG(aligned(x, 4) && aligned(cnt, 8), "misaligned input");
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
        set_error("cannot query the device");
        return CL_ERR_HIP;
    }
    const CircuitNet net{ent, ops, dst, in, reinterpret_cast<const uint2*>(cnt), ones,
                         uint32_t(start), int(pairs), int(groups), int(inv), int(in_pages),
                         int(in_words), int(k)};
    const int64_t want = std::max<int64_t>(8, (int64_t(cus) / 8) * 8);
    int rc = CL_OK;
    auto go = [&](auto tc, auto ic, auto bc, auto cc) {
        auto* kern = &k_packed_circuit<decltype(tc)::value, decltype(ic)::value,
                                       decltype(bc)::value, decltype(cc)::value>;
        const int lds = int(pages) * kPageWords * 4;
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) {
            set_error("cannot reserve %d bytes of LDS for the circuit pass", lds);
            rc = CL_ERR_HIP;
            return;
        }
        const int64_t blocks = std::min<int64_t>(want, 8 * ceil_div(ceil_div(cols, 2), 8));
        kern<<<unsigned(blocks), kPcThreads, lds, as_stream(stream)>>>(
            static_cast<const uint32_t*>(x), cols, nsamples, net, counts);
    };
    using std::integral_constant;
    auto by_layout = [&](auto tc, auto ic, auto bc) {
        if (columns_major) go(tc, ic, bc, std::true_type{});
        else go(tc, ic, bc, std::false_type{});
    };
    auto by_input = [&](auto tc, auto bc) {
        if (in_pages <= kPcThreads / 64) by_layout(tc, integral_constant<int, 1>{}, bc);
        else if (in_pages <= 2 * kPcThreads / 64) by_layout(tc, integral_constant<int, 2>{}, bc);
        else if (in_pages <= 4 * kPcThreads / 64) by_layout(tc, integral_constant<int, 4>{}, bc);
        else by_layout(tc, integral_constant<int, kPcRound>{}, bc);
    };
    auto by_steps = [&](auto tc) {
        if (4 * (groups + inv) < 32) by_input(tc, integral_constant<int, 5>{});
        else by_input(tc, integral_constant<int, 9>{});
    };
    if (2 * pairs <= 32) by_steps(integral_constant<int, 32>{});
    else if (2 * pairs <= 40) by_steps(integral_constant<int, 40>{});
    else by_steps(integral_constant<int, kPcMaxSlots>{});
    if (rc) return rc;
    return check_launch("cl_packed_circuit");
}
