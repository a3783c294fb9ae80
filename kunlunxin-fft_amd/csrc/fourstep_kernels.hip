// fourstep_kernels.hip -- two-pass (Bailey 4-step) FFT for core lengths
// 2^8 .. 2^20, the MI355X form of the reference's hybrid path
// (src/xpu/adapter_hybrid.py:224-270, scripts/issue10_wp3_perf.py:428-461).
//
// N = N1*N2, n = n1*N2 + n2, k = k1 + N1*k2:
//   X[k1 + N1*k2] = sum_n2 W_N2^(n2*k2) * [ W_N^(n2*k1) * sum_n1 x[n1*N2+n2] W_N1^(n1*k1) ]
// Pass 1 (column pass): for each n2, an N1-point FFT down the column
//   x[n1*N2 + n2] (row stride N2), stored transposed as Z[n2*N1 + k1] -- one
//   contiguous run of N1 per column, so the store is unit-stride and the layout
//   hand-off costs no pass of its own (the reference's k_twiddle_fused idea,
//   issue10_wp3_perf.py:214-242).
// Pass 2 (row pass): for each k1, an N2-point FFT over W_N^(n2*k1) Z[k1 + N1*n2]
//   (stride N1), stored to X[k1 + N1*k2] -- the same addresses it read, so pass 2
//   runs in place on the output buffer and the plan needs no workspace.
// Both passes are one kernel template: a block owns C adjacent columns (lanes
// run along the columns, so every row access is a C*8-byte contiguous run),
// keeps them in LDS, and runs the same Stockham passes as the single-pass
// kernel on each column.  Inverse = conjugated roots; the norm scale is applied
// by pass 2's store.
// The twiddle W_N^(n2*k1) costs no product of its own: an N2-point FFT of
// inputs times w^n2, w = W_N^k1, is the same FFT network with other roots
// (its outputs are the input polynomial at w W_N2^k2 instead of W_N2^k2), so
// pass 2 takes it into the roots of its merged butterflies (dft_dit, PassRoots)
// and pass 1 stores plain column transforms.
// Where the passes already move their bytes at the rate of a copy, vector
// instructions are what is left to save: a timing-only build without butterflies and
// twiddles ran N = 2^20, B = 64 in 345 us against 380.  Multiplying pass 1's
// outputs by the twiddle and pass 2's inputs by pass twiddles took 3151 vector
// instructions per thread over the two passes at 1024 points and 32 elements;
// merged they take 2745.  N = 2^20, B = 64: 375 -> 364 us; 2^16, B = 256: 85.1
// -> 81.2; C2R 2^18, B = 256: 192 -> 179; R2C: 240 -> 236; 2^16, B = 32: 14.7 ->
// 14.0.
// Those roots are products of a Stockham root, from a per-pass table (rows
// W^k, W^2k, W^4k, ...) that both passes have, and of W_N^(2^t k1), t < log2
// N2, from one row per t of N1 entries: both loads are contiguous or shared
// across the lanes of a column group.
#include "mfft_device.hpp"
#include "mfft_internal.hpp"

namespace mfft {

// Elements per thread and column-group width for a pass of length 2^logl.
// 16 columns make every row access a 128-byte run (8 columns: 64-byte runs,
// which measured about 20% less HBM bandwidth for these strided reads).  From
// 512 points a thread holds 32 elements and the exchange is split into real
// and imaginary halves, which keeps a block of 16 columns within 70 KB of LDS
// and about 100 VGPRs, so two blocks share a CU.
constexpr int col_loge(int logl) { return logl >= 9 ? 5 : (logl >= 8 ? 4 : (logl >= 6 ? 3 : 2)); }
constexpr int col_logc(int) { return 4; }
// Schedule 3 (narrow groups, for a batch of one or a few transforms): 4
// columns per workgroup and at most 16 elements per thread (8 for passes of
// 256 and 512 points), so a launch has 4x the workgroups and every thread a
// shorter load-compute-store chain; its 32-byte row runs cost bandwidth that
// such a launch does not use anyway (N = 2^18-2^20, B = 1: 25-28% less time
// than schedule 0).  Measured per pass length: 8 elements beat 16 by 5-7% at
// 256 and 512 points and lose 2-3% at 1024; 2 columns per workgroup lose.
constexpr int col_loge_narrow(int logl) { return logl >= 10 ? 4 : (logl >= 8 ? 3 : col_loge(logl)); }
constexpr int kNarrowLogC = 2;
int fourstep_col_loge(int logl, int schedule) { return schedule == 3 ? col_loge_narrow(logl) : col_loge(logl); }

namespace {

__device__ __forceinline__ int pad(int i) { return i + (i >> 4); }
// pad(i + K) from pi = pad(i), for a compile-time K: when K is a multiple of
// 16 it is pi + K + K/16, a constant offset the LDS instruction encodes, so
// a run of accesses shares one address register.
template <int K>
__device__ __forceinline__ int pad_add(int pi, int i) {
    if constexpr (K % 16 == 0) return pi + K + K / 16;
    else return pad(i + K);
}
// the same with one slot per 32 elements (split exchange)
__device__ __forceinline__ int pad32(int i) { return i + (i >> 5); }
template <int K>
__device__ __forceinline__ int pad32_add(int pi, int i) {
    if constexpr (K % 32 == 0) return pi + K + K / 32;
    else return pad32(i + K);
}

// Whole transforms per XCD: within every full chunk of 8 x `groups` blocks,
// XCD x (physical blocks 8i + x) takes the `groups` column groups of
// transform x of the chunk, in order.  For the real passes, whose bin rows
// hold n/2 + 1 complex values, transform b's grid starts 8b bytes into a
// 128-byte line, so every column run straddles lines it shares with the
// neighbouring groups; with all groups of a transform on one XCD, dispatched
// together, those lines meet in one L2 (measured at N = 2^17: C2R pass-1
// fetch 298 -> 204 MiB, R2C pass-2 write 162 -> 129 MiB).  A bijection on
// every full chunk; the tail keeps its order.
__device__ __forceinline__ int xcd_row_block(int p, int total, int groups) {
    const int chunk = 8 * groups;
    if (p >= total - total % chunk) return p;
    const int local = p % chunk;
    return (p - local) + (local & 7) * groups + (local >> 3);
}

// Workgroups are dispatched to the 8 XCDs round-robin (block p -> XCD p % 8),
// and each XCD has its own L2.  A column group's rows are 128-byte runs at a
// power-of-two stride; in dispatch order XCD x would see only two of every 16
// adjacent column groups, so all its strided runs would sit in two of the 16
// 128-byte slots of each 2 KB of a row.  This map gives every XCD 16
// consecutive logical blocks (16 adjacent column groups) of each chunk of
// 128; measured 4-9% off the column passes at N = 2^16..2^19 against that
// pairing, results bit-identical.  A bijection on every full chunk; the tail
// keeps its order.
__device__ __forceinline__ int xcd_run_block(int p, int total) { return xcd_row_block(p, total, 16); }

template <int LOGL, int LOGE, int LOGC>
struct ColCfg {
    static_assert(LOGE < LOGL, "a column pass needs more than one thread per column");
    static constexpr int LOG_L = LOGL, LOG_E = LOGE;
    static constexpr int L = 1 << LOGL;
    static constexpr int E = 1 << LOGE;
    static constexpr int C = 1 << LOGC;
    static constexpr int T = L / E;  // threads per column
    static constexpr int WG = C * T;
    static constexpr int P = sched_passes(LOGL, LOGE);
    // Column pitch in float2 units, == 32/C (mod 32): a half-wave (32 lanes)
    // covers C columns x 32/C rows, and with this pitch the C columns start
    // 64/C dwords apart, tiling the 64 LDS banks without conflicts.
    static constexpr int PITCH0 = L + (L >> 4);
    static constexpr int PITCH = PITCH0 + ((32 / C - PITCH0 % 32) + 32) % 32;
    static constexpr int logr(int p) { return sched_logr(LOGL, LOGE, p); }
    static constexpr int lns(int p) { return sched_lns(LOGE, p); }
    // last pass: radix, butterflies per thread, span
    static constexpr int LR_LAST = sched_logr(LOGL, LOGE, P - 1);
    static constexpr int R_LAST = 1 << LR_LAST;
    static constexpr int NB_LAST = E / R_LAST;
    static constexpr int NS_LAST = L / R_LAST;
    static constexpr int TW_SIZE = sched_tw_size(LOGL, LOGE);  // pass twiddle table entries
    // 32 elements per thread exchange real and imaginary parts separately
    // through a float array (half the LDS of a float2 exchange), padded one
    // slot per 32 elements (pad32: the stride-32 writes of a radix-32 pass
    // then fall 33 floats apart).  Its column pitch, in floats, is == 64/C
    // (mod 64) for the same bank tiling.
    static constexpr bool SPLIT = LOGE == 5;
    static constexpr int PITCH0F = L + (L >> 5);
    static constexpr int PITCHF = PITCH0F + ((64 / C - PITCH0F % 64) + 64) % 64;
    // LDS floats: the exchange, and the float2 staging of the transposed
    // store (all C columns at once, or C/2 at a time when split)
    static constexpr int XCH_FLOATS = SPLIT ? C * PITCHF : 2 * C * PITCH;
    static constexpr int STORE_FLOATS = SPLIT ? C * PITCH : 2 * C * PITCH;
    static constexpr int LDS_FLOAT2 = ((XCH_FLOATS > STORE_FLOATS ? XCH_FLOATS : STORE_FLOATS) + 1) / 2;
};

// The value unchanged, but hidden from the optimizer: work derived from it
// (twiddle reads, products) stays inside the loop that uses it instead of
// being hoisted out and held in registers across the loop.
__device__ __forceinline__ int opaque(int x) {
    asm volatile("" : "+v"(x));
    return x;
}

// Roots of one pass's butterfly b (dft_dit's r: r[i] = w^(2^i)).  KIND 0, a
// plain column FFT: w = W_(NS R)^k, k = b mod NS, from the pass table tw.
// KIND 1, the column FFT of inputs times W_N^(col n): the pass combines inputs
// b + q L / R and carries the L / (NS R)-spaced powers that the passes before
// it left over, so w = W_N^(col L / (NS R)) W_(NS R)^k.  col_tw: the table of
// W_N^(2^t col), 2^log_s entries a row, at this column.
template <class C, int KIND>
struct PassRoots {
    const float2* tw;
    const float2* col_tw;  // KIND 1
    int log_s;             // KIND 1
    template <int p, int m, int NR>  // b = j + m T
    __device__ __forceinline__ void load(float2 (&r)[NR], int b) const {
        constexpr int LR = C::logr(p), LNS = C::lns(p);
        const int k = b & ((1 << LNS) - 1);
        static_for<0, LR>([&](auto i) {
            float2 w = make_float2(1.0f, 0.0f);
            if constexpr (KIND == 1) w = col_tw[(C::LOG_L - LNS - LR + i.value) << log_s];
            if constexpr (p > 0) {
                const float2 s = tw[sched_tw_off(C::LOG_L, C::LOG_E, p) + (i.value << LNS) + k];
                w = KIND == 1 ? cmul(w, s) : s;
            }
            r[i.value] = w;
        });
    }
};

// Pass-0 operands of one column group: s = the group's first element of the
// transform (wave-uniform), lane (c, j) reads rows j + m*T + q*L/R0 of column c.
// Every address is a wave-uniform row pointer (SGPRs) plus one lane offset
// shared by all rows, so the 2^LOGE loads hold one address VGPR, not one each.
// The loads are non-temporal: each pass reads its input once, and pass 1's
// reads of X would otherwise evict pass 1's output Z from the MALL before
// pass 2 reads it (measured: 8-11% off the whole transform at 2^16-2^20).
// One complex64 read coherent across the CUs of the device: an
// agent-scope relaxed atomic load, which the compiler issues with the sc1
// policy.  It never returns a line from this CU's L1 (which may be stale
// when another CU has rewritten it) but does hit in the XCD's L2.
__device__ __forceinline__ float2 load_agent(const float2* p) {
    const unsigned long long u = __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
    return __builtin_bit_cast(float2, u);
}

// AGENT: read with load_agent (data another CU wrote in this launch) instead
// of the non-temporal load.
template <class C, bool AGENT = false>
__device__ __forceinline__ void col_load(float2 (&v)[C::E], const float2* s, int c, int j, int log_s) {
    constexpr int R0 = 1 << C::logr(0);
    constexpr int NB0 = C::E / R0;
    const uint32_t lane = (uint32_t)(c + (j << log_s)) * 8u;
    static_for<0, NB0>([&](auto m) {
        static_for<0, R0>([&](auto q) {
            const int row = m.value * C::T + q.value * (C::L / R0);
            const float2* a = byte_off(s + ((int64_t)row << log_s), lane);
            v[m.value * R0 + q.value] = AGENT ? load_agent(a) : load_nt(a);
        });
    });
}

// The Stockham passes of one column group, in place in v.  Pass p > 0 reads
// its operands from this thread's column in LDS; every pass but the last
// writes its outputs back (float2 through `lds`, or, SPLIT, one component at
// a time through the same memory as floats).  The last pass leaves its
// outputs in registers.  roots.load gives the roots of a pass's
// butterflies when that pass starts; r0: those of pass 0 (KIND 1), which the
// caller loads ahead of the operands.  With BARRIER0 the first LDS write also
// waits for the previous group's LDS readers.
template <class C, int DIR, int KIND, bool BARRIER0, class RootsT>
__device__ __forceinline__ void col_passes(float2 (&v)[C::E], float2* lds, int c, int j, const float2 (&r0)[C::LOG_E],
                                           const RootsT& roots) {
    constexpr int L = C::L, E = C::E, T = C::T, P = C::P;
    float2* lt = lds + c * C::PITCH;
    float* ltf = reinterpret_cast<float*>(lds) + c * C::PITCHF;
    static_for<0, P>([&](auto pp) {
        constexpr int p = pp.value;
        constexpr int LR = C::logr(p);
        constexpr int R = 1 << LR;
        constexpr int NB = E / R;
        constexpr int LNS = C::lns(p);
        constexpr int NS = 1 << LNS;
        const int pj = pad(j), pj32 = pad32(j);
        if constexpr (p > 0 && !C::SPLIT) {
            static_for<0, NB>([&](auto m) {
                static_for<0, R>([&](auto q) {
                    v[m.value * R + q.value] = lt[pad_add<m.value * T + q.value * (L / R)>(pj, j)];
                });
            });
        }
        static_for<0, NB>([&](auto m) {
            if constexpr (p == 0) {
                dft_dit<R, DIR, m.value * R, KIND == 1>(v, r0);
            } else {
                float2 r[LR];
                roots.template load<p, m.value>(r, j + m.value * T);
                dft_dit<R, DIR, m.value * R, true>(v, r);
            }
        });
        if constexpr (p < P - 1 && !C::SPLIT) {
            if constexpr (p > 0 || BARRIER0) __syncthreads();
            static_for<0, NB>([&](auto m) {
                const int b = j + m.value * T;
                const int base_o = ((b >> LNS) << (LNS + LR)) + (b & (NS - 1));
                const int pb = pad(base_o);
                static_for<0, R>([&](auto q) { lt[pad_add<q.value * NS>(pb, base_o)] = v[m.value * R + q.value]; });
            });
            __syncthreads();
        }
        if constexpr (p < P - 1 && C::SPLIT) {
            // real parts out of v[].x (this pass's layout) and back into v[].x
            // (the next pass's layout) while v[].y still holds this pass's
            // imaginary parts; then the same for .y
            constexpr int R1 = 1 << C::logr(p + 1);
            constexpr int NB1 = E / R1;
            static_for<0, 2>([&](auto comp) {
                if constexpr (p > 0 || BARRIER0 || comp.value > 0) __syncthreads();
                static_for<0, NB>([&](auto m) {
                    const int b = j + m.value * T;
                    const int base_o = ((b >> LNS) << (LNS + LR)) + (b & (NS - 1));
                    const int pb = pad32(base_o);
                    static_for<0, R>([&](auto q) {
                        const float2 x = v[m.value * R + q.value];
                        ltf[pad32_add<q.value * NS>(pb, base_o)] = comp.value == 0 ? x.x : x.y;
                    });
                });
                __syncthreads();
                static_for<0, NB1>([&](auto m) {
                    static_for<0, R1>([&](auto q) {
                        const float x = ltf[pad32_add<m.value * T + q.value * (L / R1)>(pj32, j)];
                        if constexpr (comp.value == 0) v[m.value * R1 + q.value].x = x;
                        else v[m.value * R1 + q.value].y = x;
                    });
                });
            });
        }
    });
}

// KIND 0: Z[n2*N1 + k1] through LDS: the last-pass outputs (k1 = b + q*NS)
// are staged per column, then read back with the lanes along k1 inside one
// column, so every wave writes whole 128-byte lines (a direct store from the
// Stockham registers writes 512/C-byte runs and measured slower).  SPLIT
// stages half the columns at a time.  d = Z + c0*N1.
// KIND 1: X[k1 + N1*k2] from registers, in place; d = X + c0 (k1 = c0 + c).
// Real transforms over the four-step core pair every index k of the core
// with its mirror L - k.  On the (k1, k2) grid of pass 2 (k = k1 + N1 k2) the
// mirror of (k1, k2) is (N1 - k1, N2 - 1 - k2), and of (0, k2) it is
// (0, N2 - k2); on the (n1, n2) grid of pass 1 (n = n1 N2 + n2) the mirror of
// (n1, n2) is (N1 - 1 - n1, N2 - n2), and of (n1, 0) it is (N1 - n1, 0).  The
// columns pair up as (p, N - p) for p = 1 .. N/2 - 1, plus (0, N/2), both of
// which are their own mirror columns.  A workgroup of 2 CP lane columns takes
// CP pairs (8 or 16): lane column c < CP holds member 0 of pair CP g + c, and
// c ^ CP its partner, so every mirror value is in the same workgroup.
// Column (member c / CP of pair CP g + c mod CP) of an N-column grid:
template <int CP = 8>
__device__ __forceinline__ int pair_col(int g, int c, int n) {
    const int p = CP * g + (c & (CP - 1));
    return c < CP ? p : (p ? n - p : n >> 1);
}
// Thread layout of the real passes, so that the rows of thread j and of its
// mirror thread T - 1 - j sit in lanes l and l ^ 32 of one wave: with 16 lane
// columns (jj = tid >> 4) the four row sets of wave w are 2w, 2w + 1,
// T - 1 - 2w and T - 2 - 2w (mirror column c ^ 8: lane l ^ 40); with 32 lane
// columns (jj = tid >> 5) the two row sets are w and T - 1 - w (mirror
// column c ^ 16: lane l ^ 48).
template <int T, int LOGC = 4>
__device__ __forceinline__ int mirror_row_set(int jj) {
    if constexpr (LOGC == 4) {
        static_assert(T % 4 == 0, "a wave holds four 16-lane row sets");
        return (jj & 2) ? T - 1 - 2 * (jj >> 2) - (jj & 1) : 2 * (jj >> 2) + (jj & 1);
    } else {
        static_assert(LOGC == 5 && T % 2 == 0, "a wave holds two 32-lane row sets");
        return (jj & 1) ? T - 1 - (jj >> 1) : (jj >> 1);
    }
}
// x as held by the lane at byte address `from` (lane * 4) of this wave
__device__ __forceinline__ float2 lane_value(float2 x, int from) {
    return make_float2(__int_as_float(__builtin_amdgcn_ds_bpermute(from, __float_as_int(x.x))),
                       __int_as_float(__builtin_amdgcn_ds_bpermute(from, __float_as_int(x.y))));
}
// R2C: pass 1 stores Z with its k1 positions permuted so that position
// 2CP g + c holds k1 = pair_col<CP>(g, c, N1): pass 2 then reads CP mirror
// pairs as one aligned 2CP-column run.  k1 stored at position `pos`:
template <int N1, int CP = 8>
__device__ __forceinline__ int pair_k1(int pos) { return pair_col<CP>(pos / (2 * CP), pos % (2 * CP), N1); }

// MAP 0: column c of the group is column c0 + c (d = Z + c0 N1).  MAP 1 (R2C
// pass 1): the same columns, each stored with its k1 permuted (pair_k1, CP
// pairs per group of pass 2).
// MAP 2 (C2R pass 1): lane column c is column pair_col(g, c, 2^log_s) (d = Z).
// NTS (KIND 1): non-temporal stores, for output that nothing in this launch
// reads again (it then does not displace lines the launch still uses).
// WT: write-through stores (store_out) of whole lines; off for the fused
// schedule's Z ring, which is meant to stay in the XCD's L2.
template <class C, int KIND, int MAP = 0, bool NTS = false, int CP = 8, bool WT = true>
__device__ __forceinline__ void col_store(const float2 (&v)[C::E], float2* d, float2* lds, int tid, int c, int j,
                                          int log_s, float scale, int g = 0) {
    if constexpr (KIND == 0) {
        constexpr int HALVES = C::SPLIT ? 2 : 1;
        constexpr int CH = C::C / HALVES;  // columns staged per round
        static_for<0, HALVES>([&](auto h) {
            __syncthreads();  // every read of the previous LDS contents is done
            if (HALVES == 1 || c / CH == h.value) {
                float2* lt = lds + (c - h.value * CH) * C::PITCH;
                const int pj = pad(j);
                static_for<0, C::NB_LAST>([&](auto m) {
                    static_for<0, C::R_LAST>([&](auto q) {
                        lt[pad_add<m.value * C::T + q.value * C::NS_LAST>(pj, j)] = v[m.value * C::R_LAST + q.value];
                    });
                });
            }
            __syncthreads();
            float2* dh = d + ((int64_t)(h.value * CH) << C::LOG_L);
            static_for<0, C::E / HALVES>([&](auto r) {
                const int e = tid + r.value * C::WG;
                const int cc = e >> C::LOG_L;
                const int k1 = e & (C::L - 1);
                if constexpr (MAP == 2) {
                    const int col = pair_col<C::C / 2>(g, h.value * CH + cc, 1 << log_s);
                    store_out<WT>(d + ((int64_t)col << C::LOG_L) + k1, lds[cc * C::PITCH + pad(k1)]);
                } else {
                    store_out<WT>(byte_off(dh + r.value * C::WG, (uint32_t)tid * 8u),
                                  lds[cc * C::PITCH + pad(MAP == 1 ? pair_k1<C::L, CP>(k1) : k1)]);
                }
            });
        });
    } else {
        const uint32_t lane = (uint32_t)(c + (j << log_s)) * 8u;
        static_for<0, C::NB_LAST>([&](auto m) {
            static_for<0, C::R_LAST>([&](auto q) {
                const int row = m.value * C::T + q.value * C::NS_LAST;
                float2* a = byte_off(d + ((int64_t)row << log_s), lane);
                const float2 x = cscale(v[m.value * C::R_LAST + q.value], scale);
                // write-through where a row run is a whole 128-byte line (16
                // columns or more; the narrow groups' 32-byte runs, written
                // through, took the 2^20-point pass 2 from 7.4 to 9.8 us)
                if constexpr (NTS) store_nt(a, x);
                else store_out<(WT && C::C >= 16)>(a, x);
            });
        });
    }
}

// KIND 0: pass 1 (column FFTs of length L = N1 over S = N2 columns, transposed
//         store).  KIND 1: pass 2 (in place, L = N2, S = N1 columns, with the
//         twiddle in its roots).
// One column group per block: the C columns [c0, c0 + C) of one batch row.
// KIND 1 runs in place (src == dst): every element of the block's columns is
// in registers before the first barrier, all stores come after it, and no
// other block touches these columns.
template <int LOGL, int LOGE, int LOGC, int DIR, int KIND>
__global__ __launch_bounds__((ColCfg<LOGL, LOGE, LOGC>::WG)) void fourstep_pass_kernel(
    const float2* src, float2* dst, const float2* __restrict__ tw,
    const float2* __restrict__ tw_col, int logn, int log_s, float scale, int rev) {
    using C = ColCfg<LOGL, LOGE, LOGC>;
    __shared__ float2 lds[C::LDS_FLOAT2];
    const int groups = (1 << log_s) >> LOGC;  // column groups per transform
    const int bid = xcd_run_block((int)blockIdx.x, (int)gridDim.x);
    const int64_t row0 = bid / groups;
    const int c0 = (bid - (int)(row0 * groups)) << LOGC;
    // pass 2 in reverse row order (rev): the rows pass 1 wrote last, whose Z
    // is the most likely to be still in the MALL, go first
    const int64_t row = (KIND == 1 && rev) ? (int64_t)((int)gridDim.x / groups) - 1 - row0 : row0;
    const int tid = threadIdx.x;
    const int c = tid & (C::C - 1);
    const int j = tid >> LOGC;
    const int64_t base = row << logn;

    const PassRoots<C, KIND> roots{tw, tw_col + c0 + c, log_s};
    float2 v[C::E], r0[C::LOG_E];
    if constexpr (KIND == 1) roots.template load<0, 0>(r0, j);
    col_load<C>(v, src + base + c0, c, j, log_s);
    col_passes<C, DIR, KIND, false>(v, lds, c, j, r0, roots);
    col_store<C, KIND>(v, KIND == 0 ? dst + base + ((int64_t)c0 << LOGL) : dst + base + c0, lds, tid, c, j,
                       log_s, scale);
}

// R2C pass 1: the column pass of the half-length core (forward), with Z
// stored in the pair-permuted k1 order (MAP 1) for the stitching pass 2 and
// its CP mirror pairs per workgroup.
template <int LOGL, int LOGE, int LOGC, int CP = 8>
__global__ __launch_bounds__((ColCfg<LOGL, LOGE, LOGC>::WG)) void fourstep_r2c_pass1_kernel(
    const float2* src, float2* dst, const float2* __restrict__ tw, int logn, int log_s) {
    using C = ColCfg<LOGL, LOGE, LOGC>;
    __shared__ float2 lds[C::LDS_FLOAT2];
    const int groups = (1 << log_s) >> LOGC;
    const int bid = xcd_run_block((int)blockIdx.x, (int)gridDim.x);
    const int64_t row = bid / groups;
    const int c0 = (bid - (int)(row * groups)) << LOGC;
    const int tid = threadIdx.x;
    const int c = tid & (C::C - 1);
    const int j = tid >> LOGC;
    const int64_t base = row << logn;
    float2 v[C::E];
    const float2 r0[C::LOG_E] = {};  // pass 0 has no roots
    col_load<C>(v, src + base + c0, c, j, log_s);
    col_passes<C, -1, 0, false>(v, lds, c, j, r0, PassRoots<C, 0>{tw, nullptr, 0});
    col_store<C, 0, 1, false, CP>(v, dst + base + ((int64_t)c0 << LOGL), lds, tid, c, j, log_s, 1.0f);
}

// R2C pass 2 with the stitch (kernels.py:1127-1177 formula, r2c_bin): the
// row pass of the half-length core over one aligned run of 2 CP columns of
// the permuted Z (CP = 8 or 16 mirror pairs), then every output bin from its
// core value and its mirror's, written to the n/2 + 1 bins of the row.  After
// the last Stockham pass thread j holds k2 = j + m T + q NS (element
// e = m R + q); the mirror of (k1, k2) is (n1 - k1, N2 - 1 - k2): element
// E - 1 - e of thread T - 1 - j in lane column c ^ CP, which the thread layout
// (mirror_row_set) puts at lane ^ (32 + CP) of the same wave, one ds_bpermute
// per component away.  Two columns of group 0 mirror onto themselves:
// k1 = n1/2 (lane column CP; partner lane ^ 32) and k1 = 0 (lane column 0),
// whose k2 pairs with
// N2 - k2 of another wave: its lanes store their bins again from a copy of
// the column in LDS, and the thread holding k = 0 also writes bin n/2.
// The bin twiddle exp(-2 pi i k / n), k = k1 + n1 k2, is
// tw_a[k1] tw_b[j] exp(-2 pi i K / (2 N2)), K = k2 - j.
template <int LOGL, int LOGE, int LOGC>
__global__ __launch_bounds__((ColCfg<LOGL, LOGE, LOGC>::WG)) void fourstep_r2c_pass2_kernel(
    const float2* src, float2* dst, const float2* __restrict__ tw, const float2* __restrict__ tw_col,
    const float2* __restrict__ tw_a, const float2* __restrict__ tw_b, int logn, int log_s, float scale) {
    using C = ColCfg<LOGL, LOGE, LOGC>;
    static_assert(LOGC == 4 || LOGC == 5, "8 or 16 mirror pairs per workgroup");
    constexpr int CP = C::C / 2;  // mirror pairs per workgroup
    constexpr int N2 = C::L, E = C::E;
    __shared__ float2 lds[C::LDS_FLOAT2];
    const int n1 = 1 << log_s;
    const int groups = n1 >> LOGC;
    const int bid = xcd_row_block((int)blockIdx.x, (int)gridDim.x, groups);
    const int64_t row = bid / groups;
    const int g = bid - (int)(row * groups);
    const int tid = threadIdx.x;
    const int c = tid & (C::C - 1);
    const int j = mirror_row_set<C::T, LOGC>(tid >> LOGC);
    const int64_t np = (int64_t)1 << logn;  // core length L = n/2
    const int k1 = pair_col<CP>(g, c, n1);
    const PassRoots<C, 1> roots{tw, tw_col + k1, log_s};
    float2 v[E], r0[C::LOG_E];
    roots.template load<0, 0>(r0, j);
    col_load<C>(v, src + (row << logn) + (g << LOGC), c, j, log_s);
    col_passes<C, -1, 1, false>(v, lds, c, j, r0, roots);
    const bool col0 = g == 0 && c == 0;
    float2* xo = dst + row * (np + 1) + k1;
    // K = k2 - j of element e
    auto kof = [](int e) { return (e / C::R_LAST) * C::T + (e % C::R_LAST) * C::NS_LAST; };
    if (g == 0) {  // block-uniform: column 0's values to LDS
        __syncthreads();  // the last pass's LDS reads are done
        if (c == 0) {
            static_for<0, E>([&](auto e) { lds[j + kof(e.value)] = v[e.value]; });
        }
        __syncthreads();
    }
    const int from = ((tid & 63) ^ (g == 0 && c == CP ? 32 : 32 + CP)) << 2;
    const float2 tj = cmul(tw_a[k1], tw_b[j]);
    // every lane stitches with its partner's values, without branches (column
    // 0's lanes store bins that they overwrite below)
    static_for<0, E / 2>([&](auto h) {
        constexpr int e0 = h.value, e1 = E - 1 - h.value;
        constexpr int K0 = kof(e0), K1 = kof(e1);
        const float2 m0 = lane_value(v[e1], from);  // the partner's element e1: the mirror of this e0
        const float2 m1 = lane_value(v[e0], from);
        xo[(int64_t)n1 * (j + K0)] = r2c_bin(v[e0], m0, rot<2 * N2, K0, -1>(tj), scale, false);
        xo[(int64_t)n1 * (j + K1)] = r2c_bin(v[e1], m1, rot<2 * N2, K1, -1>(tj), scale, false);
    });
    if (col0) {
        // addresses from an opaque copy of j: shared with the loop above, all
        // of them would stay in registers across it
        const int jc = opaque(j);
        static_for<0, E>([&](auto e) {
            constexpr int K = kof(e.value);
            const int k2 = jc + K;
            xo[(int64_t)n1 * k2] = r2c_bin(v[e.value], lds[(N2 - k2) & (N2 - 1)], rot<2 * N2, K, -1>(tj), scale,
                                           K == 0 && jc == 0);
            __builtin_amdgcn_sched_barrier(0);  // one element's read at a time
        });
        if (j == 0) xo[np] = r2c_bin(v[0], v[0], cmul(tw_a[0], tw_b[N2]), scale, true);
    }
}

// C2R pass 1 with the pre-twiddle (kernels.py:1180-1229 formula,
// c2r_pre_bin): the workgroup loads CP = 8 or 16 columns of the n/2 + 1 bins
// and their CP mirror columns (pair_col; with 16, 128 B runs of the bin rows,
// which are not line-aligned, so fewer lines are shared with the neighbouring
// workgroups), turns every bin into its core input with its
// mirror's value, then runs the column pass of the half-length inverse core
// and stores Z in place of the output row (the row pass runs in place there).
// The mirror of bin (n1, n2) is (N1 - 1 - n1, N2 - n2), and thread j's rows
// j + m T + q N1/R0 (element e = m R0 + q) have their mirrors in element
// E - 1 - e of thread T - 1 - j, lane column c ^ CP.  Threads are laid out
// (mirror_row_set) so that partner is lane ^ (32 + CP) of the same wave and
// each mirror value is one ds_bpermute per component away: no LDS round and
// no copy of the mirror values in registers.  Two columns of group 0 mirror
// onto themselves: column N2/2 (lane column CP; partner lane ^ 32) and column 0
// (lane column 0), whose row n1 pairs with row N1 - n1 of another wave and
// goes through LDS; bin n/2, the mirror of bin 0, is loaded by the thread
// that holds bin 0, and the imaginary parts of both are ignored.
// The pre-twiddle root exp(-2 pi i n / n_real), n = n1 N2 + n2, is
// tw_a[n2] * tw_b[n1].
template <int LOGL, int LOGE, int LOGC>
__global__ __launch_bounds__((ColCfg<LOGL, LOGE, LOGC>::WG)) void fourstep_c2r_pass1_kernel(
    const float2* src, float2* dst, const float2* __restrict__ tw, const float2* __restrict__ tw_a,
    const float2* __restrict__ tw_b, int logn, int log_s) {
    using C = ColCfg<LOGL, LOGE, LOGC>;
    static_assert(LOGC == 4 || LOGC == 5, "8 or 16 mirror pairs per workgroup");
    constexpr int CP = C::C / 2;  // mirror pairs per workgroup
    constexpr int N1 = C::L;
    constexpr int R0 = 1 << C::logr(0);
    constexpr int NB0 = C::E / R0;
    constexpr int E = C::E;
    __shared__ float2 lds[C::LDS_FLOAT2];
    const int n2n = 1 << log_s;
    const int groups = n2n >> LOGC;
    const int bid = xcd_row_block((int)blockIdx.x, (int)gridDim.x, groups);
    const int64_t row = bid / groups;
    const int g = bid - (int)(row * groups);
    const int tid = threadIdx.x;
    const int c = tid & (C::C - 1);
    const int j = mirror_row_set<C::T, LOGC>(tid >> LOGC);
    const int64_t np = (int64_t)1 << logn;
    const int n2 = pair_col<CP>(g, c, n2n);
    const bool col0 = g == 0 && c == 0;  // n2 = 0: mirror rows N1 - n1 of its own column, bin n/2 for n1 = 0
    const float2* xr = src + row * (np + 1);
    float2 v[E];
    // pass-0 operand rows n1 = j + m T + q N1/R0 of column n2 (non-temporal:
    // each bin is read once)
    const uint32_t lane = (uint32_t)(n2 + (j << log_s)) * 8u;
    static_for<0, NB0>([&](auto m) {
        static_for<0, R0>([&](auto q) {
            const int r = m.value * C::T + q.value * (N1 / R0);
            v[m.value * R0 + q.value] = load_nt(byte_off(xr + ((int64_t)r << log_s), lane));
        });
    });
    const float2 xny = (col0 && j == 0) ? load_nt(xr + np) : make_float2(0.0f, 0.0f);
    // K of element e: its row is n1 = j + K
    auto kof = [](int e) { return (e / R0) * C::T + (e % R0) * (N1 / R0); };
    if (g == 0) {  // block-uniform: column 0's rows through LDS
        if (c == 0) {
            static_for<0, E>([&](auto e) { lds[j + kof(e.value)] = v[e.value]; });
        }
        __syncthreads();
    }
    const int from = ((tid & 63) ^ (g == 0 && c == CP ? 32 : 32 + CP)) << 2;
    // the root of row j + K is tw_a[n2] tw_b[j] exp(-2 pi i K / (2 N1)): one
    // table product per thread, then compile-time rotations (K = m T + q N1/R0)
    const float2 tj = cmul(tw_a[n2], tw_b[j]);
    // every lane from its partner's values, without branches (a branch per
    // pair lets the compiler sink each pair's arithmetic below the last one,
    // holding every mirror value at once) ...
    static_for<0, E / 2>([&](auto h) {
        constexpr int e0 = h.value, e1 = E - 1 - h.value;
        constexpr int k0 = kof(e0), k1 = kof(e1);
        const float2 m0 = lane_value(v[e1], from);  // the partner's element e1: the mirror of this e0
        const float2 m1 = lane_value(v[e0], from);
        v[e0] = c2r_pre_bin(v[e0], m0, rot<2 * N1, k0, -1>(tj));
        v[e1] = c2r_pre_bin(v[e1], m1, rot<2 * N1, k1, -1>(tj));
    });
    // ... then column 0 again, from the copy of its rows in LDS
    if (col0) {
        static_for<0, E>([&](auto e) {
            constexpr int k = kof(e.value);
            const int r = j + k;
            float2 x = lds[r];
            float2 m = lds[(N1 - r) & (N1 - 1)];
            if constexpr (k == 0) {
                if (j == 0) {  // bin 0 pairs with bin n/2; both imaginary parts ignored
                    m = make_float2(xny.x, 0.0f);
                    x.y = 0.0f;
                }
            }
            v[e.value] = c2r_pre_bin(x, m, rot<2 * N1, k, -1>(tj));
            __builtin_amdgcn_sched_barrier(0);  // one element's reads at a time
        });
    }
    const float2 r0[C::LOG_E] = {};  // pass 0 has no roots
    col_passes<C, 1, 0, true>(v, lds, c, j, r0, PassRoots<C, 0>{tw, nullptr, 0});
    col_store<C, 0, 2>(v, dst + (row << logn), lds, tid, c, j, log_s, 1.0f, g);
}

// Persistent form of the same pass: gridDim.x blocks, a multiple of the
// column groups per transform, walk the `tiles` column groups of the launch
// with stride gridDim.x, so a block keeps one column index c0 while the batch
// row advances.  While a group is transformed the next one is already loading
// into registers, so HBM traffic continues through the block's compute and LDS
// phases; the pass twiddle table and, for pass 2, the W_N^(2^t k1) of the
// block's columns sit in LDS, which keeps the only global loads in flight during
// the compute those of the next group.  (Pass 2's roots held in registers across
// the loop instead spilled 224-240 bytes a lane against 144-160 at 512 and 1024
// points and took up to 9% more past 2^24 points: N = 2^17, B = 256, n1 = 256: 296
// us against 264, 2^18, B = 32: 52.4 against 48.0.)
template <int LOGL, int LOGE, int LOGC, int DIR, int KIND>
__global__ __launch_bounds__((ColCfg<LOGL, LOGE, LOGC>::WG), 4) void fourstep_persist_kernel(
    const float2* src, float2* dst, const float2* __restrict__ tw,
    const float2* __restrict__ tw_col, int logn, int log_s, float scale, int64_t tiles, int rev) {
    using C = ColCfg<LOGL, LOGE, LOGC>;
    __shared__ float2 lds[C::LDS_FLOAT2];
    __shared__ float2 lds_tw[C::TW_SIZE > 0 ? C::TW_SIZE : 1];
    __shared__ float2 lds_col[KIND == 1 ? LOGL * C::C : 1];  // [t][column]: W_N^(2^t k1)
    const int tid = threadIdx.x;
    const int c = tid & (C::C - 1);
    const int j = tid >> LOGC;
    const int log_groups = log_s - LOGC;  // column groups per transform = 2^log_groups
    const int64_t stride = gridDim.x;
    const int64_t t0 = xcd_run_block((int)blockIdx.x, (int)gridDim.x);
    const int c0 = (int)(t0 & ((1 << log_groups) - 1)) << LOGC;
    // batch row of tile t; pass 2 walks the rows in reverse order with rev
    const int64_t last_row = (tiles >> log_groups) - 1;
    auto row_of = [&](int64_t t) { return (KIND == 1 && rev) ? last_row - (t >> log_groups) : (t >> log_groups); };

    for (int i = tid; i < C::TW_SIZE; i += C::WG) lds_tw[i] = tw[i];
    if constexpr (KIND == 1) {
        for (int i = tid; i < LOGL * C::C; i += C::WG)
            lds_col[i] = tw_col[((i >> LOGC) << log_s) + c0 + (i & (C::C - 1))];
    }
    float2 v[C::E];
    col_load<C>(v, src + (row_of(t0) << logn) + c0, c, j, log_s);
    __syncthreads();  // lds_tw, lds_col complete

    // one column group: transform v (group t) and store it.  Per-call copies
    // of the loop invariants: recomputing addresses and roots costs less than the
    // registers that holding them across the loop (next to the prefetched
    // group) would take.
    auto process = [&](int64_t t) {
        const int jl = opaque(j), cl = opaque(c), tl = opaque(tid);
        const PassRoots<C, KIND> roots{lds_tw, KIND == 1 ? lds_col + cl : nullptr, LOGC};
        float2 r0[C::LOG_E] = {};  // pass 1's pass 0 has no roots
        if constexpr (KIND == 1) roots.template load<0, 0>(r0, jl);
        col_passes<C, DIR, KIND, true>(v, lds, cl, jl, r0, roots);
        const int64_t base = row_of(t) << logn;
        col_store<C, KIND>(v, dst + opaque_uniform(KIND == 0 ? base + ((int64_t)c0 << LOGL) : base + c0), lds, tl, cl,
                           jl, log_s, scale);
    };
    int64_t t = t0;
    for (; t + stride < tiles; t += stride) {
        float2 vn[C::E];
        col_load<C>(vn, src + opaque_uniform((row_of(t + stride) << logn) + c0), opaque(c), opaque(j), log_s);
        process(t);
        static_for<0, C::E>([&](auto r) { v[r.value] = vn[r.value]; });
    }
    process(t);
}

// Fused schedule: both passes in one launch, with each transform's
// intermediate Z kept in the L2 of the XCD that runs the transform.
//
// The MI355X L2 does not allocate on a store miss: a store to a line that is
// not in L2 goes on to memory, and a later read of it misses.  A store that
// hits a line already in L2 stays there (write-back).  So Z does not go to
// the output rows, as in the two-pass schedule, but to a small ring of Z
// slots per XCD in the workspace, reused transform after transform: after a
// slot's first use its lines are in L2 (pass 2's reads brought them in), and
// from then on pass 1 writes them and pass 2 reads them there, so Z makes no
// HBM round trip.  Pass 2 writes the final output rows.
//
// Every block reads the XCD it runs on (hardware register XCC_ID) and takes
// work only from the queue of that XCD's slot, XCC_ID mod nslot (nslot = the
// device's XCD count, so a partitioned device with fewer XCDs still drains
// every queue): transform t belongs to slot t mod nslot, and its queue hands
// out pass-1 groups of the slot's transform k, then pass-2 groups of k - D
// (D = lag), and so on.  Transform k uses ring slot k mod R (R >= D + 1).
// Two waits, both on transforms earlier in the queue:
// * a pass-2 group of k waits until all pass-1 groups of k have stored Z;
// * a pass-1 group of k, before it stores Z, waits until all pass-2 groups of
//   k - R have read the ring slot it is about to overwrite.
// Those groups were handed out before the waiting one, to running blocks, and
// the earliest unfinished item never waits, so every wait ends whatever the
// residency; each is nevertheless bounded by `wait_ticks` of the
// constant-rate wall clock and by a trip count.  A wait that gives up adds
// one to *overrun (plan-owned) and sets the launch's failure word; from then
// on every pass-2 group of the launch writes NaN rather than a transform that
// may hold incomplete or overwritten data.
//
// Producer and consumer share one L2, and completed stores plus a counter in
// L2 are the handshake (no L2 write-back or invalidation).  A CU's L1 may
// still hold lines of a ring slot from the slot's previous use, so pass 2
// reads Z with agent-coherent loads (load_agent), which skip L1 and hit L2.
// Pass 1 reads its input and pass 2 writes its output non-temporally: with
// ordinary output stores the streaming output displaced the ring's dirty
// lines from L2 (measured).  The counters are touched with
// read-modify-write atomics, which execute where the producers' increments
// live; an atomic load would be issued system-coherent and read memory behind
// the L2, never seeing them.
//
// Every branch of the work loop is on a wave-uniform value: wave 0 does the
// queue and counter atomics with all of its lanes (lane 0 adds 1, the others
// 0), and only scalar-register values steer the loop.  (A per-thread
// `if (tid == 0)` beside the barriers let the compiler split the loop into an
// inner loop around the barriers that only thread 0 could leave.)  The loop
// also stops after `total + 1` trips: a block dequeues at most `total` items.
//
// sync (int32, zeroed before the launch): [0, kFusedSlots) next item per
// slot, [kFusedFail] the launch's failure word, [kFusedHead, + rows) pass-1
// groups done per transform (plus kFusedFailMark for a group that skipped its
// store), [kFusedHead + rows, + rows) pass-2 groups done per transform.
// ring: nslot * R slots of 2^(LL1 + LL2) complex values.
template <int LL1, int LE1, int LC1, int LL2, int LE2, int LC2, int DIR>
__global__ __launch_bounds__((ColCfg<LL1, LE1, LC1>::WG)) void fourstep_fused_kernel(
    const float2* src, float2* dst, float2* ring, const float2* __restrict__ tw1, const float2* __restrict__ tw2,
    const float2* __restrict__ tw_col, float scale, int rows, int nslot, int lag, int nring, int per_take, int* sync,
    int* overrun, long long wait_ticks) {
    using A = ColCfg<LL1, LE1, LC1>;
    using B = ColCfg<LL2, LE2, LC2>;
    static_assert(A::WG == B::WG, "both passes run with the same block size");
    constexpr int LDS_N = A::LDS_FLOAT2 > B::LDS_FLOAT2 ? A::LDS_FLOAT2 : B::LDS_FLOAT2;
    __shared__ float2 lds[LDS_N];
    __shared__ int item_s, fail_s;
    constexpr int LOGN = LL1 + LL2;
    constexpr int G1 = (1 << LL2) >> LC1;  // pass-1 column groups per transform (columns n2)
    constexpr int G2 = (1 << LL1) >> LC2;  // pass-2 column groups per transform (columns k1)
    constexpr int kMaxPolls = 1 << 22;     // a second bound on one wait, besides the clock
    const int tid = threadIdx.x;
    // HW_REG_XCC_ID (hwreg 20), bits [3:0]
    const int xcc = (int)__builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20) & 15;
    const int slot = __builtin_amdgcn_readfirstlane(xcc % nslot);
    const int nt = rows > slot ? (rows - slot + nslot - 1) / nslot : 0;  // this slot's transforms
    const int total = nt * (G1 + G2);
    const int D = lag < nt ? lag : nt;  // pass 1 runs D transforms ahead of pass 2
    int* done1 = sync + kFusedHead;
    int* done2 = done1 + rows;
    const bool lead = __builtin_amdgcn_readfirstlane(tid) < 64;  // wave 0
    const int one = tid == 0 ? 1 : 0;
    // wave 0: wait until *ctr >= want; returns 0 if the wait gave up
    auto wait_for = [&](int* ctr, int want) -> int {
        // an add of an opaque zero: a literal 0 would be turned into an
        // (L2-bypassing) atomic load by the compiler
        const int zero = opaque(0);
        const long long t_start = wall_clock64();
        for (int poll = 0; __builtin_amdgcn_readfirstlane(atomicAdd(ctr, zero)) < want; ++poll) {
            if (poll >= kMaxPolls || wall_clock64() - t_start > wait_ticks) {
                atomicAdd(overrun, one);
                atomicAdd(sync + kFusedFail, one);
                __builtin_amdgcn_s_waitcnt(0);
                return 0;
            }
            __builtin_amdgcn_s_sleep(2);
        }
        return 1;
    };
    for (int trip = 0; trip <= total; ++trip) {
        // take `per_take` consecutive items with one atomic (every block
        // hitting one counter per item serialises on that L2 address)
        if (lead) item_s = __builtin_amdgcn_readfirstlane(atomicAdd(sync + slot, one * per_take));
        __syncthreads();
        const int it0 = __builtin_amdgcn_readfirstlane(item_s);
        __syncthreads();  // every thread has read item_s before it is written again
        if (it0 >= total) break;
        const int it_end = it0 + per_take < total ? it0 + per_take : total;
        // items of a take run in queue order: an item only waits for items
        // earlier in the queue, so the earliest unfinished item never waits
        for (int it = it0; it < it_end; ++it) {
        // queue order, D = lag: P1(0) .. P1(D-1) | P1(D) P2(0) | P1(D+1) P2(1) |
        // ... | P2(nt-D) .. P2(nt-1): pass 2 of transform k is handed out
        // after pass 1 of k + D - 1, and pass 1 of k after pass 2 of k - D - 1
        int k, g;
        bool second;
        if (it < D * G1) {
            k = it / G1, g = it - k * G1, second = false;
        } else {
            const int u = it - D * G1, mid = (nt - D) * (G1 + G2);
            if (u < mid) {
                const int blk = u / (G1 + G2), r = u - blk * (G1 + G2);
                if (r < G1) k = D + blk, g = r, second = false;
                else k = blk, g = r - G1, second = true;
            } else {
                const int w = u - mid;
                k = nt - D + w / G2, g = w - (w / G2) * G2, second = true;
            }
        }
        const int t = slot + nslot * k;
        float2* zr = ring + ((int64_t)(slot * nring + k % nring) << LOGN);
        // the lane index, hidden from the optimizer per item, so lane
        // addresses are recomputed per item instead of held across the loop
        const int tl = opaque(tid);
        if (!second) {
            const int c = tl & (A::C - 1), j = tl >> LC1, c0 = g << LC1;
            float2 v[A::E];
            col_load<A>(v, src + ((int64_t)t << LOGN) + c0, c, j, LL2);
            const float2 r0[A::LOG_E] = {};  // pass 0 has no roots
            col_passes<A, DIR, 0, true>(v, lds, c, j, r0, PassRoots<A, 0>{tw1, nullptr, 0});
            // the ring slot is free once every pass-2 group of k - R has read it
            int ok = 1;
            if (k >= nring) {
                if (lead) fail_s = wait_for(done2 + (t - nslot * nring), G2) ? 0 : 1;
                __syncthreads();
                ok = 1 - __builtin_amdgcn_readfirstlane(fail_s);
            }
            if (ok) col_store<A, 0, 0, false, 8, false>(v, zr + ((int64_t)c0 << LL1), lds, tl, c, j, LL2, 1.0f);
            __builtin_amdgcn_s_waitcnt(0);  // this thread's Z stores have reached L2
            __syncthreads();
            if (lead) atomicAdd(done1 + t, one * (ok ? 1 : 1 + kFusedFailMark));
        } else {
            if (lead) {
                int bad = wait_for(done1 + t, G1) ? 0 : 1;
                bad |= __builtin_amdgcn_readfirstlane(atomicAdd(done1 + t, opaque(0))) >= kFusedFailMark;
                bad |= __builtin_amdgcn_readfirstlane(atomicAdd(sync + kFusedFail, opaque(0))) != 0;
                fail_s = bad;
            }
            __syncthreads();
            const int failed = __builtin_amdgcn_readfirstlane(fail_s);
            const int c = tl & (B::C - 1), j = tl >> LC2, c0 = g << LC2;
            const PassRoots<B, 1> roots{tw2, tw_col + c0 + c, LL1};
            float2 v[B::E], r0[B::LOG_E];
            roots.template load<0, 0>(r0, j);
            col_load<B, true>(v, zr + c0, c, j, LL1);
            col_passes<B, DIR, 1, true>(v, lds, c, j, r0, roots);
            // a failed launch writes NaN, not a transform of partial data
            col_store<B, 1, 0, true>(v, dst + ((int64_t)t << LOGN) + c0, lds, tl, c, j, LL1,
                                     failed ? __builtin_nanf("") : scale);
            __syncthreads();  // every wave's reads of the ring slot are done
            if (lead) atomicAdd(done2 + t, one);
        }
        }
    }
}

// clears a fused launch's counters: the queues, the failure word and the
// per-transform counts
__global__ void zero_sync(int* sync, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) sync[i] = 0;
}

// Blocks of the persistent kernel one CU holds at once (occupancy query,
// made once per kernel).
template <int LOGL, int LOGE, int LOGC, int DIR, int KIND>
int persist_blocks_per_cu() {
    static const int n = [] {
        int b = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, fourstep_persist_kernel<LOGL, LOGE, LOGC, DIR, KIND>,
                                                         ColCfg<LOGL, LOGE, LOGC>::WG, 0) != hipSuccess) {
            (void)hipGetLastError();
            b = 1;
        }
        return b > 0 ? b : 1;
    }();
    return n;
}

// schedule 3: the narrow column groups
template <int LOGL, int DIR, int KIND>
hipError_t launch_pass_narrow(const float2* src, float2* dst, const mfft_plan* p, int64_t rows, int log_s,
                              float scale, hipStream_t stream) {
    constexpr int LOGE = col_loge_narrow(LOGL);
    constexpr int LOGC = kNarrowLogC;
    using C = ColCfg<LOGL, LOGE, LOGC>;
    const int logn = ilog2((int)p->core_n);
    const int64_t tiles = rows * (((int64_t)1 << log_s) >> LOGC);
    if (!launch_fits(tiles, C::WG)) return hipErrorInvalidConfiguration;
    fourstep_pass_kernel<LOGL, LOGE, LOGC, DIR, KIND><<<(unsigned)tiles, C::WG, 0, stream>>>(
        src, dst, KIND == 0 ? p->tw_n1 : p->tw_n2, p->tw_col, logn, log_s, scale, p->pass2_rev);
    mark(stream);
    return hipGetLastError();
}

template <int LOGL, int DIR, int KIND>
hipError_t launch_pass(const float2* src, float2* dst, const mfft_plan* p, int64_t rows,
                       int log_s, float scale, hipStream_t stream) {
    if (p->schedule == 3) return launch_pass_narrow<LOGL, DIR, KIND>(src, dst, p, rows, log_s, scale, stream);
    constexpr int LOGE = col_loge(LOGL);
    constexpr int LOGC = col_logc(LOGL);
    using C = ColCfg<LOGL, LOGE, LOGC>;
    const int logn = ilog2((int)p->core_n);
    const int64_t groups = ((int64_t)1 << log_s) >> LOGC;
    const int64_t tiles = rows * groups;
    if (!launch_fits(tiles, C::WG)) return hipErrorInvalidConfiguration;
    const float2* tw = KIND == 0 ? p->tw_n1 : p->tw_n2;
    if (p->schedule == 1) {
        // a multiple of the column groups (fixed c0 per block) and of 16,
        // at most one resident wave of blocks
        const int64_t unit = groups > 16 ? groups : 16;
        int64_t g = (int64_t)persist_blocks_per_cu<LOGL, LOGE, LOGC, DIR, KIND>() * p->num_cus;
        g = g / unit * unit;
        if (g < unit) g = unit;
        if (g > tiles) g = tiles;
        fourstep_persist_kernel<LOGL, LOGE, LOGC, DIR, KIND><<<(unsigned)g, C::WG, 0, stream>>>(
            src, dst, tw, p->tw_col, logn, log_s, scale, tiles, p->pass2_rev);
    } else {
        fourstep_pass_kernel<LOGL, LOGE, LOGC, DIR, KIND><<<(unsigned)tiles, C::WG, 0, stream>>>(
            src, dst, tw, p->tw_col, logn, log_s, scale, p->pass2_rev);
    }
    mark(stream);
    return hipGetLastError();
}

// KIND 0: R2C pass 1 (permuted Z); 1: R2C pass 2 with the stitch; 2: C2R
// pass 1 with the pre-twiddle.  log_s: log2 of the columns of the pass.
template <int LOGL, int KIND>
hipError_t launch_real_pass(const float2* src, float2* dst, const mfft_plan* p, int64_t rows, int log_s,
                            float scale, hipStream_t stream) {
    constexpr int LOGE = col_loge(LOGL);
    constexpr int LOGC = col_logc(LOGL);
    using C = ColCfg<LOGL, LOGE, LOGC>;
    const int logn = ilog2((int)p->core_n);
    const int64_t tiles = rows * (((int64_t)1 << log_s) >> LOGC);
    // (the 32-column forms below run half the blocks at twice the threads)
    if (!launch_fits(tiles, C::WG)) return hipErrorInvalidConfiguration;
    // 16 mirror pairs per workgroup (128 B runs of the bins) where the grid of
    // bins has 32 columns or more and the mirror pass is at most 512 points
    // (at 1024 the doubled workgroup's LDS leaves one per CU); R2C's two
    // passes take the same choice, since pass 1 permutes Z for pass 2's pairs
    using C5 = ColCfg<LOGL, LOGE, 5>;
    if constexpr (KIND == 0) {
        if (LOGL >= 5 && log_s <= 9)
            fourstep_r2c_pass1_kernel<LOGL, LOGE, LOGC, 16><<<(unsigned)tiles, C::WG, 0, stream>>>(
                src, dst, p->tw_n1, logn, log_s);
        else
            fourstep_r2c_pass1_kernel<LOGL, LOGE, LOGC><<<(unsigned)tiles, C::WG, 0, stream>>>(
                src, dst, p->tw_n1, logn, log_s);
    } else if constexpr (KIND == 1) {
        bool pairs16 = false;
        if constexpr (LOGL <= 9) {
            if (log_s >= 5) {
                pairs16 = true;
                fourstep_r2c_pass2_kernel<LOGL, LOGE, 5><<<(unsigned)(tiles >> 1), C5::WG, 0, stream>>>(
                    src, dst, p->tw_n2, p->tw_col, p->tw_ra, p->tw_rb, logn, log_s, scale);
            }
        }
        if (!pairs16)
            fourstep_r2c_pass2_kernel<LOGL, LOGE, LOGC><<<(unsigned)tiles, C::WG, 0, stream>>>(
                src, dst, p->tw_n2, p->tw_col, p->tw_ra, p->tw_rb, logn, log_s, scale);
    } else {
        bool pairs16 = false;
        if constexpr (LOGL <= 9) {
            if (log_s >= 5) {
                pairs16 = true;
                fourstep_c2r_pass1_kernel<LOGL, LOGE, 5><<<(unsigned)(tiles >> 1), C5::WG, 0, stream>>>(
                    src, dst, p->tw_n1, p->tw_ra, p->tw_rb, logn, log_s);
            }
        }
        if (!pairs16)
            fourstep_c2r_pass1_kernel<LOGL, LOGE, LOGC><<<(unsigned)tiles, C::WG, 0, stream>>>(
                src, dst, p->tw_n1, p->tw_ra, p->tw_rb, logn, log_s);
    }
    mark(stream);
    return hipGetLastError();
}

template <int KIND>
hipError_t dispatch_real(int logl, const float2* src, float2* dst, const mfft_plan* p, int64_t rows, int log_s,
                         float scale, hipStream_t stream) {
    switch (logl) {
        case 4: return launch_real_pass<4, KIND>(src, dst, p, rows, log_s, scale, stream);
        case 5: return launch_real_pass<5, KIND>(src, dst, p, rows, log_s, scale, stream);
        case 6: return launch_real_pass<6, KIND>(src, dst, p, rows, log_s, scale, stream);
        case 7: return launch_real_pass<7, KIND>(src, dst, p, rows, log_s, scale, stream);
        case 8: return launch_real_pass<8, KIND>(src, dst, p, rows, log_s, scale, stream);
        case 9: return launch_real_pass<9, KIND>(src, dst, p, rows, log_s, scale, stream);
        case 10: return launch_real_pass<10, KIND>(src, dst, p, rows, log_s, scale, stream);
        default: return hipErrorInvalidValue;
    }
}

template <int DIR, int KIND>
hipError_t dispatch_len(int logl, const float2* src, float2* dst, const mfft_plan* p, int64_t rows,
                        int log_s, float scale, hipStream_t stream) {
    switch (logl) {
        case 4: return launch_pass<4, DIR, KIND>(src, dst, p, rows, log_s, scale, stream);
        case 5: return launch_pass<5, DIR, KIND>(src, dst, p, rows, log_s, scale, stream);
        case 6: return launch_pass<6, DIR, KIND>(src, dst, p, rows, log_s, scale, stream);
        case 7: return launch_pass<7, DIR, KIND>(src, dst, p, rows, log_s, scale, stream);
        case 8: return launch_pass<8, DIR, KIND>(src, dst, p, rows, log_s, scale, stream);
        case 9: return launch_pass<9, DIR, KIND>(src, dst, p, rows, log_s, scale, stream);
        case 10: return launch_pass<10, DIR, KIND>(src, dst, p, rows, log_s, scale, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

bool fourstep_supported(int log2n1, int log2n2) {
    // each pass length in [16, 1024]; the other factor must hold a full column group
    if (log2n1 < 4 || log2n1 > 10 || log2n2 < 4 || log2n2 > 10) return false;
    return log2n2 >= col_logc(log2n1) && log2n1 >= col_logc(log2n2);
}

void fourstep_default_split(int log2n, int* log2n1, int* log2n2) {
    *log2n1 = log2n / 2;
    *log2n2 = log2n - *log2n1;
}

namespace {

template <int L1, int L2, int DIR>
hipError_t launch_fused_one(const float2* src, float2* dst, char* fws, const mfft_plan* p, int64_t rows,
                            float scale, hipStream_t stream) {
    constexpr int E1 = col_loge(L1), C1 = col_logc(L1), E2 = col_loge(L2), C2 = col_logc(L2);
    using A = ColCfg<L1, E1, C1>;
    int* sync = reinterpret_cast<int*>(fws);
    float2* ring = reinterpret_cast<float2*>(fws + p->fused_ring_off);
    const int nsync = kFusedHead + 2 * (int)rows;
    zero_sync<<<(nsync + 255) / 256, 256, 0, stream>>>(sync, nsync);
    mark(stream);
    // grid, lag, ring and take were fixed at plan creation (one resident
    // wave of blocks, a multiple of the XCD count)
    fourstep_fused_kernel<L1, E1, C1, L2, E2, C2, DIR><<<p->fused_grid, A::WG, 0, stream>>>(
        src, dst, ring, p->tw_n1, p->tw_n2, p->tw_col, scale, (int)rows, p->num_xcc,
        p->fused_lag, p->fused_ring, p->fused_take, sync, p->overrun, (long long)kFusedWaitMs * p->clock_khz);
    mark(stream);
    return hipGetLastError();
}

template <int L1, int L2>
int fused_occupancy_of() {
    constexpr int E1 = col_loge(L1), C1 = col_logc(L1), E2 = col_loge(L2), C2 = col_logc(L2);
    int b = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, fourstep_fused_kernel<L1, E1, C1, L2, E2, C2, -1>,
                                                     ColCfg<L1, E1, C1>::WG, 0) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return b;
}

#define MFFT_FUSED_SHAPES(X) X(7, 7) X(7, 8) X(8, 7) X(8, 8) X(8, 9) X(9, 8) X(9, 9)

hipError_t launch_fused(int dir, const float2* src, float2* dst, char* fws, const mfft_plan* p, int64_t rows,
                        float scale, hipStream_t stream) {
    if constexpr (!kFusedScheduleEnabled) {
        // switched off (plan creation rejects schedule 2); not instantiated
        (void)dir, (void)src, (void)dst, (void)fws, (void)p, (void)rows, (void)scale, (void)stream;
        return hipErrorNotSupported;
    } else {
        if (!fws) return hipErrorInvalidValue;
        const int l1 = ilog2((int)p->n1), l2 = ilog2((int)p->n2);
#define MFFT_FUSED_CASE(A, B)                                                                    \
        if (l1 == A && l2 == B)                                                                  \
            return dir < 0 ? launch_fused_one<A, B, -1>(src, dst, fws, p, rows, scale, stream)   \
                           : launch_fused_one<A, B, 1>(src, dst, fws, p, rows, scale, stream);
        MFFT_FUSED_SHAPES(MFFT_FUSED_CASE)
#undef MFFT_FUSED_CASE
        return hipErrorInvalidValue;
    }
}

}  // namespace

bool fourstep_fused_supported(int l1, int l2) {
    return l1 >= 7 && l1 <= 9 && l2 >= 7 && l2 <= 9 && l1 - l2 <= 1 && l2 - l1 <= 1;
}

int fourstep_fused_occupancy(int l1, int l2) {
#define MFFT_FUSED_OCC(A, B) \
    if (l1 == A && l2 == B) return fused_occupancy_of<A, B>();
    MFFT_FUSED_SHAPES(MFFT_FUSED_OCC)
#undef MFFT_FUSED_OCC
    return 0;
}

hipError_t launch_fourstep_real(const float2* src, float2* dst, float2* work, const mfft_plan* p, float scale,
                                hipStream_t stream) {
    const int l1 = ilog2((int)p->n1), l2 = ilog2((int)p->n2);
    const int64_t rows = p->batch;
    const int64_t chunk = p->chunk_rows > 0 ? p->chunk_rows : rows;
    const int64_t np = p->core_n;
    for (int64_t r0 = 0; r0 < rows; r0 += chunk) {
        const int64_t rc = rows - r0 < chunk ? rows - r0 : chunk;
        hipError_t e;
        if (p->transform_type == MFFT_R2C) {
            // x (n reals = np complex per row) -> permuted Z in `work` -> n/2 + 1 bins
            e = dispatch_real<0>(l1, src + r0 * np, work + r0 * np, p, rc, l2, 1.0f, stream);
            if (e == hipSuccess)
                e = dispatch_real<1>(l2, work + r0 * np, dst + r0 * (np + 1), p, rc, l1, scale, stream);
        } else {
            // n/2 + 1 bins -> pre-twiddled column pass into the output rows -> row pass in place
            e = dispatch_real<2>(l1, src + r0 * (np + 1), dst + r0 * np, p, rc, l2, 1.0f, stream);
            if (e == hipSuccess)
                e = dispatch_len<1, 1>(l2, dst + r0 * np, dst + r0 * np, p, rc, l1, scale, stream);
        }
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_fourstep(int dir, const float2* src, float2* dst, char* fws, const mfft_plan* p, int64_t rows,
                           float scale, hipStream_t stream, int* launches) {
    const int l1 = ilog2((int)p->n1), l2 = ilog2((int)p->n2);
    const int64_t chunk = p->chunk_rows > 0 ? p->chunk_rows : rows;
    const int64_t n = p->core_n;
    int count = 0;
    for (int64_t r0 = 0; r0 < rows; r0 += chunk) {
        const int64_t rc = rows - r0 < chunk ? rows - r0 : chunk;
        const float2* s = src + r0 * n;
        float2* d = dst + r0 * n;
        hipError_t e;
        if (p->schedule == 2) {
            e = launch_fused(dir, s, d, fws, p, rc, scale, stream);
            if (e != hipSuccess) return e;
            count += 2;
            continue;
        }
        e = dir < 0 ? dispatch_len<-1, 0>(l1, s, d, p, rc, l2, 1.0f, stream)
                    : dispatch_len<1, 0>(l1, s, d, p, rc, l2, 1.0f, stream);
        if (e != hipSuccess) return e;
        e = dir < 0 ? dispatch_len<-1, 1>(l2, d, d, p, rc, l1, scale, stream)
                    : dispatch_len<1, 1>(l2, d, d, p, rc, l1, scale, stream);
        if (e != hipSuccess) return e;
        count += 2;
    }
    if (launches) *launches = count;
    return hipSuccess;
}

}  // namespace mfft
