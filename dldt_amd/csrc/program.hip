// The single-launch form of a plan (program.h says what it is for and why it is shaped like this).
//
// Convolution tiles use v_mfma_i32_16x16x64_i8 with the pixels as rows and the output channels as columns: a lane holds
// four pixels of ONE channel per accumulator, so the epilogue's per-channel constants are one register each for the whole
// tile.  (With channels as rows, as in the per-layer kernels, every lane needs four channels' constants per accumulator:
// through LDS or as 16-byte loads they cost more than the arithmetic when a tile is this small.)  The A accumulators of a
// tile hold neighbouring channels (the weights' packing sees to it), so a lane stores A bytes of a pixel at once, 16 lanes
// its 16 A channels.  Both operands come from memory straight into operand registers: the weights of a tile are packed in
// fragment order (1 KB per load), a pixel fragment is 64 contiguous bytes of 16 pixels.  Waves of a workgroup split a
// tile's K (`ks`) where there are fewer tiles than waves: no byte is then loaded twice inside a workgroup, and the partial
// sums meet in LDS.  Where a pixel's window starts and where its results go is a table (four words a pixel): decoding them
// cost 200 instructions a tile, a sixth of a step.
// Reference semantics: as conv_kernel.h, dwconv.hip, pool.hip, fq.hip, glue.hip and attention.hip - the arithmetic of every
// step is the same sequence of f32 operations as in the per-step kernels, so the results are the same bits.
#include "program.h"

#include <chrono>

#include "div2.h"
#include "step_barrier.h"

struct hipie_fq;

namespace hipie {
namespace {

constexpr int kPartBytes = 128 * 1024;       // partial sums of eight waves x 16 fragments
constexpr int kKoffBytes = 16 * 1024;        // K offsets of the step's convolutions
constexpr int kMaxPieces = kKoffBytes / 4 / 2;
constexpr int kPlainAt = kPartBytes + kKoffBytes + 64;        // 16 i at entry i: the K offsets of a step whose K pieces lie one behind the other
constexpr int kLdsBytes = kPlainAt + kMaxPieces * 4;
// How long a launch waits for its last workgroup: 1 ms of the 100 MHz clock.  Alone it is complete in a few microseconds, behind
// the kernels of another request in the time these take; what holds compute units longer (another process's launch that
// waits for the same units) does not let go, and the steps need less than that beside it.
constexpr uint32_t kRollCallTicks = 100000, kMaxRollCallTicks = 10000000;
constexpr uint64_t kBarrierTicks = 200000000;

typedef __attribute__((address_space(3))) int8_t* lds_ptr;
typedef __attribute__((address_space(3))) v4i* lds_v4i;
typedef __attribute__((address_space(3))) int32_t* lds_i32;

struct ProgArgs {
    const int32_t* steps;
    void* bases[1 + kProgramIo];             // the arena, the call's inputs and outputs (ProgRef::base)
    uint32_t* control;
    uint32_t* report;
    int32_t n_steps, workgroups;
    uint32_t launch, roll_call_ticks;
};

// (addresses made from integers are told to be global memory: as generic pointers their loads would be FLAT, which the
// compiler waits for on the LDS counter as well)
#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(1))) uint8_t* GlobalBytes;
#else
typedef uint8_t* GlobalBytes;
#endif

// control words: a counter per XCD, 128 bytes apart
constexpr int kXcdWords = 32;
constexpr uint32_t kGivenUp = 1u << 26;      // added to a counter that was not complete when the roll call's time was up (a launch counts far less)

__device__ __forceinline__ int lane_index() { return static_cast<int>(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u))); }

// Everything that was asked of memory and LDS has come (or, of LDS only).  As instructions the compiler knows: behind a wait in inline
// assembly it goes on counting what was in flight in front of it, and waits for all of it, the barrier's own addition included,
// where a register of those loads is used again (0.5 us of a step's preparation).
__device__ __forceinline__ void wait_memory() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070);      // vmcnt(0) lgkmcnt(0)
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ void wait_lds() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);      // lgkmcnt(0)
    asm volatile("" ::: "memory");
}
// a barrier of the workgroup in front of which only LDS is waited for
__device__ __forceinline__ void meet() {
    wait_lds();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
struct Ctx {
    int rank, n_wg, wg_shift;                // neighbouring ranks share an XCD; n_wg = 1 << wg_shift
    int tid, lane, wave;
    const int32_t* steps;
    uint32_t words;                          // lane i: word i of the descriptor of the step that is run or prepared
    uint32_t words2;                         // ... word 64 + i
    uint32_t bases;                          // lanes 2 b, 2 b + 1: where operands of base b are (ProgArgs::bases)
    uint32_t *xcds, *own;                    // the eight counters, the one this workgroup counts at
    uint32_t target;                         // what each of them holds when the barrier that comes next is complete
    bool started, dead;                      // between the roll call and the first step's wait; after a wait that was given up
    lds_i32 flag;

    __device__ __forceinline__ uint32_t load_words(int step, int half) const { return static_cast<uint32_t>(steps[step * kProgramStepWords + half * (kProgramStepWords / 2) + lane]); }
    // an operand's address (of an absent one: the arena's, which nothing uses)
    __device__ __forceinline__ uint8_t* place(ProgRef r) const {
        const int b = 2 * max(r.base, 0);
        const uint64_t base = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(bases), b)) |
                              (static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(bases), b + 1))) << 32);
        return (uint8_t*)(GlobalBytes)(base + ((static_cast<uint64_t>(r.hi) << 32) | r.lo));
    }
    // The barrier between two steps comes in halves: every workgroup arrives with its stores acknowledged, then prepares the
    // next step - descriptor, tile, weights, constants: nothing the step before it wrote - and only then waits.
    // A workgroup counts at its XCD's counter and reads all eight: 32 additions to one address is what 256 workgroups take
    // (an address serves one every 10 ns: at a single one they took 4.1 us, at four a XCD the readers' traffic cost more than
    // it gave), and no second addition stands between the last arrival and its readers.  An empty barrier with the wait for a
    // store in front, us with 64 / 128 / 256 workgroups: 1.3 / 1.5 / 1.6; by way of a root counter that the last of an XCD
    // adds to 2.1 / 2.3 / 2.6, all at one counter 1.5 / 2.3 / 4.1, a flag per workgroup that everybody reads 1.4 / 1.6 / 1.8.
    // (One way between two workgroups, store to sight, takes 0.5 - 0.6 us, the wait for a store 0.36.)  In the program a step without
    // work, a copy of no bytes, takes 1.5 / 1.6 / 1.8 us; with the root counter and descriptors by scalar loads 3.6 / 4.1 / 4.2.
    __device__ __forceinline__ void arrive(int next_step) {
        words = load_words(next_step, 0);
        words2 = load_words(next_step, 1);
        arrive_at(*this);
    }
    __device__ __forceinline__ int32_t verdict() const { return flag[0]; }      // of the wait before: 0 if it was given up
    __device__ __forceinline__ bool lost(int32_t held) const { return __builtin_amdgcn_readfirstlane(held) == 0; }
    __device__ __forceinline__ void lose() const { flag[0] = 0; }
    __device__ __forceinline__ void settle() {
        wait_memory();
        __builtin_amdgcn_s_barrier();
        target += n_wg / 8;
    }
    __device__ __forceinline__ void count(bool held) const {
        // (not the wave that looks at the counters: its loads would come back behind the addition)
        if (held && tid == kProgramThreads - 64) (void)__hip_atomic_fetch_add(own, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ __forceinline__ void wait() {
        if (wave == 0 && !started) {
            const uint32_t* c = xcds + kXcdWords * (lane & 7);
            uint64_t t0 = 0;
            for (uint32_t n = 1;; ++n) {
                const uint32_t v = __hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (__builtin_amdgcn_ballot_w64(static_cast<int32_t>(v - target) < 0) == 0) break;
                if ((n & 255) != 0) continue;
                if (t0 == 0) t0 = wall_clock64();
                if (wall_clock64() - t0 > kBarrierTicks) {
                    if (lane == 0) give_up(*this);
                    break;
                }
            }
        }
        started = false;
        meet();
    }
    // Every workgroup has arrived behind the last step: the first one tells the host in the page-locked word that it looks at
    // (report_done).  All results were stored with device scope and acknowledged, so they are in memory.
    __device__ __forceinline__ void finish() {
        if (rank != 0) return;
        lane = lane_index();
        wait();
        if (wave == 0 && lane == 0) report(*this);
    }
    // (lane 0 of the first wave)
    __device__ __forceinline__ void tell(uint32_t what) const {
#if defined(__HIP_DEVICE_COMPILE__)
        typedef uint32_t* Word;
        const Word w = *(const __attribute__((address_space(4))) Word*)((const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr() + offsetof(ProgArgs, report));
        __hip_atomic_store(w, what, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
#endif
    }
    // Everybody is resident, or nobody starts.  A workgroup whose time is up adds kGivenUp to a counter that it has seen short
    // and that has not moved since: from then on that counter never holds what completes the roll call.  So "all eight have
    // been complete" and "one was given up" exclude each other, neither is ever taken back, and all workgroups find the same.
    __device__ __forceinline__ bool roll_call(uint32_t ticks) {
        if (wave == 0) {
            uint32_t* c = xcds + kXcdWords * (lane & 7);
            // (no time at all: given up before it can be complete)
            if (lane == 0) (void)__hip_atomic_fetch_add(own, ticks == 0 && rank == 0 ? 1u + kGivenUp : 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const uint64_t t0 = wall_clock64();
            bool all = false;
            for (;;) {
                const uint32_t v = __hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const int32_t beyond = static_cast<int32_t>(v - target);
                if (__builtin_amdgcn_ballot_w64(beyond >= static_cast<int32_t>(kGivenUp / 2)) != 0) break;
                const uint64_t missing = __builtin_amdgcn_ballot_w64(beyond < 0);
                all = missing == 0;
                if (all) break;
                if (wall_clock64() - t0 > ticks && lane == __builtin_ctzll(missing)) {
                    uint32_t expect = v;
                    (void)__hip_atomic_compare_exchange_strong(c, &expect, v + kGivenUp, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            if (lane == 0) {
                if (!all) tell(kReportCancelled);
                flag[0] = all ? 1 : 0;
            }
        }
        __syncthreads();
        return flag[0] != 0;
    }
};

// The steps that are not convolutions read their descriptor through the constant address space: scalar loads.
#if defined(__HIP_DEVICE_COMPILE__)
#define PROG_CONSTANT const __attribute__((address_space(4)))
#else
#define PROG_CONSTANT const
#endif
typedef PROG_CONSTANT int32_t* StepPtr;
__device__ __forceinline__ StepPtr step_ptr(const int32_t* steps, int s) {
    return (StepPtr)(reinterpret_cast<uintptr_t>(steps) + static_cast<uintptr_t>(s) * (kProgramStepWords * 4));
}
template <typename T>
__device__ __forceinline__ T unpack(StepPtr p) {
    constexpr int n = static_cast<int>(sizeof(T) / 4);
    int32_t w[n];
#pragma unroll
    for (int i = 0; i < n; ++i) w[i] = p[i];
    T t;
    __builtin_memcpy(&t, w, sizeof(T));
    return t;
}
// an operand's address: its base comes from the kernel's arguments by a scalar load
__device__ __forceinline__ uint8_t* resolve(int32_t base, uint32_t lo, uint32_t hi) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef uint8_t* BasePtr;
    typedef const __attribute__((address_space(4))) BasePtr* Bases;
    Bases b = (Bases)((const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr() + offsetof(ProgArgs, bases));
    return (uint8_t*)(GlobalBytes)(reinterpret_cast<uintptr_t>(b[base]) + ((static_cast<uint64_t>(hi) << 32) | lo));
#else
    return nullptr;
#endif
}
#define PROG_REF(x, r) resolve((r).base, (r).lo, (r).hi)
#define PROG_TABLE(T, p) reinterpret_cast<const T*>((const uint8_t*)(GlobalBytes)((static_cast<uint64_t>((p).hi) << 32) | (p).lo))


constexpr int kBeyond = 0x7ffffff0;          // a buffer offset no buffer reaches: loads give zero, stores nothing
#if defined(__HIP_DEVICE_COMPILE__)
constexpr int kDeviceScope = 16;             // sc1: what another XCD wrote, or will read
typedef __amdgpu_buffer_rsrc_t Buffer;
__device__ __forceinline__ Buffer make_buffer(const void* p) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, kBeyond, 0x00020000); }
template <int AUX> __device__ __forceinline__ v4i load16(Buffer b, uint32_t o, int imm = 0) { return __builtin_amdgcn_raw_buffer_load_b128(b, static_cast<int>(o), imm, AUX); }
__device__ __forceinline__ v4i shared16(Buffer b, uint32_t o) { return load16<kDeviceScope>(b, o); }
__device__ __forceinline__ uint32_t shared4(Buffer b, uint32_t o) { return static_cast<uint32_t>(__builtin_amdgcn_raw_buffer_load_b32(b, static_cast<int>(o), 0, kDeviceScope)); }
__device__ __forceinline__ uint32_t shared2(Buffer b, uint32_t o) { return static_cast<uint16_t>(__builtin_amdgcn_raw_buffer_load_b16(b, static_cast<int>(o), 0, kDeviceScope)); }
__device__ __forceinline__ uint32_t shared1(Buffer b, uint32_t o) { return static_cast<uint8_t>(__builtin_amdgcn_raw_buffer_load_b8(b, static_cast<int>(o), 0, kDeviceScope)); }
typedef int v2i __attribute__((ext_vector_type(2)));
__device__ __forceinline__ v2i shared8(Buffer b, uint32_t o) { return __builtin_amdgcn_raw_buffer_load_b64(b, static_cast<int>(o), 0, kDeviceScope); }
__device__ __forceinline__ void publish16(Buffer b, uint32_t o, v4i v) { __builtin_amdgcn_raw_buffer_store_b128(v, b, static_cast<int>(o), 0, kDeviceScope); }
__device__ __forceinline__ void publish8(Buffer b, uint32_t o, v2i v) { __builtin_amdgcn_raw_buffer_store_b64(v, b, static_cast<int>(o), 0, kDeviceScope); }
__device__ __forceinline__ void publish4(Buffer b, uint32_t o, uint32_t v) { __builtin_amdgcn_raw_buffer_store_b32(static_cast<int>(v), b, static_cast<int>(o), 0, kDeviceScope); }
__device__ __forceinline__ void publish2(Buffer b, uint32_t o, uint32_t v) { __builtin_amdgcn_raw_buffer_store_b16(static_cast<short>(v), b, static_cast<int>(o), 0, kDeviceScope); }
__device__ __forceinline__ void publish1(Buffer b, uint32_t o, uint32_t v) { __builtin_amdgcn_raw_buffer_store_b8(static_cast<char>(v), b, static_cast<int>(o), 0, kDeviceScope); }
#else
typedef const void* Buffer;
typedef int v2i __attribute__((ext_vector_type(2)));
__device__ __forceinline__ Buffer make_buffer(const void* p) { return p; }
template <int AUX> __device__ __forceinline__ v4i load16(Buffer, uint32_t, int = 0) { return v4i{0, 0, 0, 0}; }
__device__ __forceinline__ v4i shared16(Buffer, uint32_t) { return v4i{0, 0, 0, 0}; }
__device__ __forceinline__ v2i shared8(Buffer, uint32_t) { return v2i{0, 0}; }
__device__ __forceinline__ uint32_t shared4(Buffer, uint32_t) { return 0; }
__device__ __forceinline__ uint32_t shared2(Buffer, uint32_t) { return 0; }
__device__ __forceinline__ uint32_t shared1(Buffer, uint32_t) { return 0; }
__device__ __forceinline__ void publish16(Buffer, uint32_t, v4i) {}
__device__ __forceinline__ void publish8(Buffer, uint32_t, v2i) {}
__device__ __forceinline__ void publish4(Buffer, uint32_t, uint32_t) {}
__device__ __forceinline__ void publish2(Buffer, uint32_t, uint32_t) {}
__device__ __forceinline__ void publish1(Buffer, uint32_t, uint32_t) {}
#endif
__device__ __forceinline__ float4 shared16f(Buffer b, uint32_t o) {
    const v4i v = shared16(b, o);
    return make_float4(__int_as_float(v.x), __int_as_float(v.y), __int_as_float(v.z), __int_as_float(v.w));
}
__device__ __forceinline__ void publish16f(Buffer b, uint32_t o, const float4& v) {
    publish16(b, o, v4i{__float_as_int(v.x), __float_as_int(v.y), __float_as_int(v.z), __float_as_int(v.w)});
}

// ---- convolution --------------------------------------------------------------------------------------------------------

// Operand registers of a tile: D K steps in flight.  The L2 is 600 - 1000 clocks away and a wave's share of K is a handful
// of steps, so what counts is that all of them are requested at once, without a branch between two loads (behind a branch
// the compiler waits for every load in flight): the ring is always filled, and a step behind the end is a buffer load out
// of range (by its per-lane offset), which asks memory for nothing and adds zeros.
template <int A, int B> constexpr int ring_depth() { return A * B >= 16 ? 2 : (A * B >= 8 ? 4 : 6); }
template <int A, int B>
struct Ring {
    static constexpr int D = ring_depth<A, B>();
    v4i w[D][A], p[D][B];
};

// where a wave's tile finds its K steps
struct KSource {
    Buffer w, in;
    lds_i32 koff;
    int kk, ks, nk;                          // the steps kk, kk + ks, .. of nk
};

template <int A, int B>
__device__ __forceinline__ void load_weights(Ring<A, B>& g, const KSource& s, int d, int k, int lane) {
    const uint32_t o = static_cast<uint32_t>(lane * 16) + static_cast<uint32_t>(k < s.nk ? k * (A * 1024) : kBeyond);
#pragma unroll
    for (int a = 0; a < A; ++a) g.w[d][a] = load16<0>(s.w, o, a * 1024);
}
template <int A, int B>
__device__ __forceinline__ void load_pixels(Ring<A, B>& g, const KSource& s, const uint32_t (&off)[B], int d, int k, int lane) {
    // (the K-offset table is read at the last step where k lies behind the end: what LDS holds there, added to kBeyond, could
    // wrap round to an offset in range.  Contiguous K pieces come from a table too: a second form of the loop costs registers)
    const uint32_t o = static_cast<uint32_t>(s.koff[4 * min(k, s.nk - 1) + (lane >> 4)]) + (k < s.nk ? 0u : static_cast<uint32_t>(kBeyond));
#pragma unroll
    for (int b = 0; b < B; ++b) g.p[d][b] = shared16(s.in, off[b] + o);
}
template <int A, int B>
__device__ __forceinline__ void first_weights(Ring<A, B>& g, const KSource& s, int lane) {
#pragma unroll
    for (int d = 0; d < Ring<A, B>::D; ++d) load_weights<A, B>(g, s, d, s.kk + d * s.ks, lane);
}

template <int A, int B>
__device__ __forceinline__ void first_pixels(Ring<A, B>& g, const KSource& s, const uint32_t (&off)[B], int lane) {
#pragma unroll
    for (int d = 0; d < Ring<A, B>::D; ++d) load_pixels<A, B>(g, s, off, d, s.kk + d * s.ks, lane);
}

// acc += the wave's K steps; the first D steps' operands are already on their way (first_weights, first_pixels)
template <int A, int B>
__device__ __forceinline__ void k_loop(Ring<A, B>& g, const KSource& s, const uint32_t (&off)[B], int lane, v4i (&acc)[A][B]) {
    constexpr int D = Ring<A, B>::D;
    auto multiply = [&](int d) {
#pragma unroll
        for (int a = 0; a < A; ++a)
#pragma unroll
            for (int b = 0; b < B; ++b) acc[a][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(g.p[d][b], g.w[d][a], acc[a][b], 0, 0, 0);
    };
    int k = s.kk;
    while (k + D * s.ks < s.nk) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            multiply(d);
            load_weights<A, B>(g, s, d, k + (d + D) * s.ks, lane);
            load_pixels<A, B>(g, s, off, d, k + (d + D) * s.ks, lane);
        }
        k += D * s.ks;
    }
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (d == 0 || k + d * s.ks < s.nk) multiply(d);
}

// ---- a step's descriptor in a vector register: lane i holds word i (ProgConv has fewer than 64) -----------------------------
// Scalar loads cost 90 ns each where they stand one behind the other, hits included, and a step's preparation was a chain of
// fourteen of them; a word of this register costs an instruction.  It is loaded beside the wait for the step's stores.
__device__ __forceinline__ uint32_t word_of(uint32_t words, int i) { return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(words), i)); }
template <typename T>
__device__ __forceinline__ T words_of(uint32_t words, int i) {
    static_assert(sizeof(T) % 4 == 0, "words");
    uint32_t w[sizeof(T) / 4];
#pragma unroll
    for (int k = 0; k < static_cast<int>(sizeof(T) / 4); ++k) w[k] = word_of(words, i + k);
    T t;
    __builtin_memcpy(&t, w, sizeof(T));
    return t;
}
static_assert(sizeof(ProgConv) <= 64 * 4, "a lane per word");
#define PROG_FIELD(words, f) words_of<decltype(ProgConv::f)>(words, static_cast<int>(offsetof(ProgConv, f) / 4))
#define PROG_PLACE(x, f) (x).place(PROG_FIELD((x).words, f))
#define PROG_TABLE_OF(T, words, f) table_at<T>(PROG_FIELD(words, f))
template <typename T> __device__ __forceinline__ const T* table_at(ProgPtr p) { return PROG_TABLE(T, p); }

template <int A>
struct ChannelConstants {
    int32_t corr[A];
    float bias[A], scale[A], rmul[A], il[A], ih[A], r[A];
    float r2[A];                             // the second word of the two-operation division, else the divisor
};

template <int A, typename T>
__device__ __forceinline__ void load_channels(const T* p, T (&v)[A]) {
    if constexpr (A == 4) {
        const uint4 t = *reinterpret_cast<const uint4*>(p);
        v[0] = __builtin_bit_cast(T, t.x); v[1] = __builtin_bit_cast(T, t.y); v[2] = __builtin_bit_cast(T, t.z); v[3] = __builtin_bit_cast(T, t.w);
    } else if constexpr (A == 2) {
        const uint2 t = *reinterpret_cast<const uint2*>(p);
        v[0] = __builtin_bit_cast(T, t.x); v[1] = __builtin_bit_cast(T, t.y);
    } else v[0] = p[0];
}

// The tables a step uses, one row of OCp words each, behind one another in this order (ProgBuilder::constants)
template <int A>
__device__ __forceinline__ void load_constants(uint32_t fl, const uint8_t* table, int pitch, int oc, ChannelConstants<A>& k) {
    const uint8_t* row = table + oc * 4;
    auto next = [&](auto& v) {
        typedef std::remove_reference_t<decltype(v[0])> T;
        load_channels<A>(reinterpret_cast<const T*>(row), v);
        row += pitch;
    };
    next(k.corr);
    if (fl & CF_BIAS) next(k.bias);
    if (fl & CF_SCALE) next(k.scale);
    if (fl & CF_RES_MUL) next(k.rmul);
    if (fl & CF_OUT_FQ) {
        next(k.r);
        next(k.r2);
        if (!(fl & CF_FQ_SAT)) next(k.ih);
        if (!(fl & CF_FQ_IL0)) next(k.il);
    }
}

// what the chain behind a sum needs besides the channels' constants: the step's, the same for all lanes
struct StepConstants {
    uint32_t flags;
    Buffer out, res;
    float lm1, clamp_lo, clamp_hi;
    uint32_t off_bytes;                      // the level offset, four times
    int out_limit, res_limit;
    uint32_t plane;                          // bytes between the planes of f32 results; 0: channels innermost
};
template <bool DENSE>
__device__ __forceinline__ StepConstants step_constants(const Ctx& x, uint32_t words) {
    StepConstants s;
    s.flags = PROG_FIELD(words, flags);
    s.out = make_buffer(x.place(PROG_FIELD(words, out)));
    s.res = make_buffer(x.place(PROG_FIELD(words, res)));
    s.lm1 = PROG_FIELD(words, lm1);
    s.clamp_lo = PROG_FIELD(words, clamp_lo);
    s.clamp_hi = PROG_FIELD(words, clamp_hi);
    s.off_bytes = PROG_FIELD(words, off_bytes);
    s.out_limit = PROG_FIELD(words, out_limit);
    s.res_limit = PROG_FIELD(words, res_limit);
    s.plane = DENSE ? static_cast<uint32_t>(PROG_FIELD(words, out_sn)) : 0u;
    return s;
}

// up to four pixels of the output: byte offsets in the output and residual tensors (kBeyond: not there), and their residual values
template <int A>
struct Pixels {
    uint32_t out[4], res[4];
    static constexpr int kRaw = A == 4 ? 1 : A;
    uint32_t raw[4][kRaw];                   // A bytes in raw[.][0], or A f32 values (A = 4: those are loaded where they are used)
};
template <int A, int R>
__device__ __forceinline__ void load_residual(const StepConstants& s, int oc, Pixels<A>& q) {
    if (!(s.flags & CF_RES) || (s.flags & CF_RES_GEMM)) return;
    const bool f32 = s.flags & CF_RES_F32;
    const uint32_t o = oc < s.res_limit ? static_cast<uint32_t>(f32 ? 4 * oc : oc) : static_cast<uint32_t>(kBeyond);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (f32) {
            if constexpr (A == 2) {
                const v2i v = shared8(s.res, q.res[r] + o);
                q.raw[r][0] = v.x; q.raw[r][1] = v.y;
            } else if constexpr (A == 1) q.raw[r][0] = shared4(s.res, q.res[r] + o);
        } else {
            if constexpr (A == 4) q.raw[r][0] = shared4(s.res, q.res[r] + o);
            else if constexpr (A == 2) q.raw[r][0] = shared2(s.res, q.res[r] + o);
            else q.raw[r][0] = shared1(s.res, q.res[r] + o);
        }
    }
}

// the fused f32 chain (conv_epilogue.h) on A neighbouring channels of R pixels, up to the FakeQuantize
template <bool GELU, int A, int R, bool PAIR = false>
__device__ __forceinline__ void chain(const StepConstants& c, const ChannelConstants<A>& k, const int32_t (&sum)[A][R], const float (&rgemm)[A][R], const Pixels<A>& q, int oc,
                                      float (&x)[A][R]) {
    const uint32_t fl = c.flags;
#define PROG_EACH for (int a = 0; a < A; ++a) for (int r = 0; r < R; ++r)
#pragma unroll
    PROG_EACH x[a][r] = static_cast<float>(sum[a][r]);
    if (fl & CF_BIAS) {
#pragma unroll
        PROG_EACH x[a][r] = x[a][r] + k.bias[a];
    }
    if (fl & CF_SCALE) {
#pragma unroll
        PROG_EACH x[a][r] = x[a][r] * k.scale[a];
    }
    if (fl & CF_RES) {
        float rv[A][R];
        if constexpr (PAIR) {
#pragma unroll
            PROG_EACH rv[a][r] = rgemm[a][r];
        } else if (fl & CF_RES_F32) {
            if constexpr (A == 4) {
                const uint32_t o = oc < c.res_limit ? static_cast<uint32_t>(4 * oc) : static_cast<uint32_t>(kBeyond);
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const float4 v = shared16f(c.res, q.res[r] + o);
                    rv[0][r] = v.x; rv[1][r] = v.y; rv[2][r] = v.z; rv[3][r] = v.w;
                }
            } else {
#pragma unroll
                PROG_EACH rv[a][r] = __uint_as_float(q.raw[r][a]);
            }
        } else if (fl & CF_RES_U8B) {
#pragma unroll
            PROG_EACH rv[a][r] = res_byte_to_float<true>(q.raw[r][0], a);
        } else {
#pragma unroll
            PROG_EACH rv[a][r] = res_byte_to_float<false>(q.raw[r][0], a);
        }
        if (fl & CF_RES_MUL) {
#pragma unroll
            PROG_EACH rv[a][r] = rv[a][r] * k.rmul[a];
        }
#pragma unroll
        PROG_EACH x[a][r] = x[a][r] + rv[a][r];
    }
    if (fl & CF_RELU) {
#pragma unroll
        PROG_EACH x[a][r] = x[a][r] > 0.0f ? x[a][r] : 0.0f;
    }
    if (fl & CF_CLAMP) {
        if (fl & CF_OUT_FQ) {
#pragma unroll
            PROG_EACH x[a][r] = __builtin_amdgcn_fmed3f(x[a][r], c.clamp_lo, c.clamp_hi);
        } else {
#pragma unroll
            PROG_EACH x[a][r] = x[a][r] < c.clamp_lo ? c.clamp_lo : (x[a][r] > c.clamp_hi ? c.clamp_hi : x[a][r]);
        }
    }
    if constexpr (GELU && A != 1)            // (choose_tile)
        if (fl & CF_GELU) {
#pragma unroll
            PROG_EACH x[a][r] = gelu_one(x[a][r]);
        }
}

// the stored bytes of A neighbouring channels of R pixels; x is used up
template <int A, int R>
__device__ __forceinline__ void levels(const StepConstants& c, const ChannelConstants<A>& k, float (&x)[A][R], uint32_t (&bytes)[R]) {
    const uint32_t fl = c.flags;
    // level index: as fq_level_fast, operation by operation
    const bool il0 = (fl & CF_FQ_IL0) != 0;
    if (!(fl & CF_FQ_SAT)) {
#pragma unroll
        PROG_EACH x[a][r] = __builtin_amdgcn_fmed3f(x[a][r], il0 ? 0.f : k.il[a], k.ih[a]);
    }
    if (!il0) {
#pragma unroll
        PROG_EACH x[a][r] = x[a][r] - k.il[a];
    }
    if (fl & CF_FQ_DIV2) {
#pragma unroll
        PROG_EACH x[a][r] = fmaf(x[a][r], k.r[a], x[a][r] * k.r2[a]) * c.lm1;
    } else {                                 // CF_FQ_RCP: the builder takes no layer whose ranges need the dividing form
#pragma unroll
        PROG_EACH {
            const float n = x[a][r], d = k.r2[a];
            const float q0 = n * k.r[a];
            const float e0 = fmaf(-d, q0, n);
            const float q1 = fmaf(e0, k.r[a], q0);
            const float e1 = fmaf(-d, q1, n);
            x[a][r] = fmaf(e1, k.r[a], q1) * c.lm1;
        }
    }
    const uint32_t xmask = (fl & CF_OUT_XOR) ? 0x80808080u : 0u;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        uint32_t w = 0;
#pragma unroll
        for (int a = 0; a < A; ++a) w = __builtin_amdgcn_cvt_pk_u8_f32(x[a][r], a, w);
        if (fl & CF_OUT_ADD) w = add_bytes(w, c.off_bytes);
        bytes[r] = w ^ xmask;
    }
}

// the chain and the store of its values
template <bool GELU, int A, int R, bool PAIR = false>
__device__ __forceinline__ void finish(const StepConstants& c, const ChannelConstants<A>& k, const int32_t (&sum)[A][R], const float (&rgemm)[A][R], const Pixels<A>& q, int oc) {
    const uint32_t fl = c.flags;
    float x[A][R];
    chain<GELU, A, R, PAIR>(c, k, sum, rgemm, q, oc, x);
    if (!(fl & CF_OUT_FQ) && c.plane != 0) {
#pragma unroll
        for (int a = 0; a < A; ++a) {
            const uint32_t o = oc + a < c.out_limit ? static_cast<uint32_t>(oc + a) * c.plane : static_cast<uint32_t>(kBeyond);
#pragma unroll
            for (int r = 0; r < R; ++r) publish4(c.out, q.out[r] + o, __float_as_uint(x[a][r] + 0.f));
        }
        return;
    }
    if (!(fl & CF_OUT_FQ)) {
        const uint32_t o = oc < c.out_limit ? static_cast<uint32_t>(4 * oc) : static_cast<uint32_t>(kBeyond);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if constexpr (A == 4) publish16f(c.out, q.out[r] + o, make_float4(x[0][r], x[1][r], x[2][r], x[3][r]));
            else if constexpr (A == 2) publish8(c.out, q.out[r] + o, v2i{__float_as_int(x[0][r]), __float_as_int(x[1][r])});
            else publish4(c.out, q.out[r] + o, __float_as_uint(x[0][r]));
        }
        return;
    }
    uint32_t w[R];
    levels<A, R>(c, k, x, w);
    const uint32_t o = oc < c.out_limit ? static_cast<uint32_t>(oc) : static_cast<uint32_t>(kBeyond);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if constexpr (A == 4) publish4(c.out, q.out[r] + o, w[r]);
        else if constexpr (A == 2) publish2(c.out, q.out[r] + o, w[r]);
        else publish1(c.out, q.out[r] + o, w[r]);
    }
#undef PROG_EACH
}

// A step's K offsets into LDS.  A thread's first entry is requested here and stored by the caller, behind the tile's other
// requests (`first`); only a K of more than 512 pieces is waited for.  Every lane takes part in every round (those behind the
// end repeat the last entry): no lane is masked off here.
__device__ __forceinline__ int32_t request_offsets(lds_i32 to, const int32_t* from, int n, int tid) {
    for (int base = kProgramThreads; base < n; base += kProgramThreads) {
        const int i = min(base + tid, n - 1);
        to[i] = from[i];
    }
    return from[min(tid, n - 1)];
}

// four consecutive entries of a pixel table, from any of them (the table has room behind its last row)
typedef uint32_t Words4 __attribute__((ext_vector_type(4), aligned(4)));
template <int A>
__device__ __forceinline__ void place_pixels(const uint32_t* pix, int M, int at, Pixels<A>& q) {
    const Words4 po = *reinterpret_cast<const Words4*>(pix + M + at), pr = *reinterpret_cast<const Words4*>(pix + 2 * M + at);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        q.out[r] = po[r];
        q.res[r] = pr[r];
    }
}

// pixels r0 .. r0 + R - 1 of the quads of one column: the partial sums of the ks waves that share the tile, and the chain
template <bool GELU, int A, int B, int R, bool PAIR>
__device__ __forceinline__ void finish_column(const StepConstants& sc, const ChannelConstants<A>& k, const ChannelConstants<A>& k2, lds_v4i mine, lds_v4i mine2, int ks,
                                              int b, int r0, const Pixels<A>& q, int oc) {
    auto total = [&](lds_v4i from, const int32_t (&corr)[A], int32_t (&sum)[A][R]) {
#pragma unroll
        for (int a = 0; a < A; ++a)
#pragma unroll
            for (int r = 0; r < R; ++r) sum[a][r] = corr[a];                     // a sum starts from the channel's integer correction
        const lds_i32 w = (lds_i32)(from + b * A * 64) + r0;
        for (int s = 0; s < ks; ++s)
#pragma unroll
            for (int a = 0; a < A; ++a) {
                const lds_i32 v = w + (s * (A * B) + a) * 256;
                if constexpr (R == 4) {
                    const v4i t = *(lds_v4i)v;
#pragma unroll
                    for (int r = 0; r < 4; ++r) sum[a][r] += t[r];
                } else {
#pragma unroll
                    for (int r = 0; r < R; ++r) sum[a][r] += v[r];
                }
            }
    };
    int32_t sum[A][R];
    float rg[A][R] = {};
    total(mine, k.corr, sum);
    if constexpr (PAIR) {
        int32_t s2[A][R];
        total(mine2, k2.corr, s2);
#pragma unroll
        for (int a = 0; a < A; ++a)
#pragma unroll
            for (int r = 0; r < R; ++r) rg[a][r] = (static_cast<float>(s2[a][r]) + k2.bias[a]) * k2.scale[a];
    }
    finish<GELU, A, R, PAIR>(sc, k, sum, rg, q, oc);
}

template <bool GELU, int A, int B, bool PAIR = false>     // PAIR: a projection shortcut as a second product (F <= 8: room for two sets of partial sums)
__device__ __forceinline__ void conv_tiles(Ctx& x, lds_ptr lds) {
    constexpr int F = A * B;                  // fragments of a tile
    constexpr bool kLate = F >= 16;           // the largest tile has no registers for the channels' constants before its sums are done
    KSource src, src2{};
    const int shift = PROG_FIELD(x.words, ks_shift);
    src.ks = 1 << shift;
    const int per = 8 >> shift, sub = x.wave >> shift;       // tiles a workgroup works on at once; the wave's
    src.kk = x.wave & (src.ks - 1);
    src.nk = PROG_FIELD(x.words, nk);
    src.in = make_buffer(PROG_PLACE(x, in));
    const bool plain = PROG_FIELD(x.words, koff).hi == 0;
    const lds_i32 koff = (lds_i32)(lds + kPartBytes);
    src.koff = plain ? (lds_i32)(lds + kPlainAt) : koff;
    int32_t staged = 0, staged2 = 0;
    if (!plain) staged = request_offsets(koff, PROG_TABLE_OF(int32_t, x.words, koff), 4 * src.nk, x.tid);
    if constexpr (PAIR) {
        src2 = src;
        src2.nk = PROG_FIELD(x.words, nk2);
        src2.in = make_buffer(PROG_PLACE(x, in2));
        if (!plain) {
            src2.koff = koff + kMaxPieces;
            staged2 = request_offsets(koff + kMaxPieces, PROG_TABLE_OF(int32_t, x.words, koff2), 4 * src2.nk, x.tid);
        }
    }
    const uint32_t tiles = static_cast<uint32_t>(PROG_FIELD(x.words, tiles));
    const int t0 = static_cast<int>((static_cast<uint32_t>(x.rank) * tiles) >> x.wg_shift), t1 = static_cast<int>((static_cast<uint32_t>(x.rank + 1) * tiles) >> x.wg_shift);
    const int M = PROG_FIELD(x.words, M);
    const uint32_t* pix = PROG_TABLE_OF(uint32_t, x.words, pixels);
    const lds_v4i part = (lds_v4i)lds + x.wave * (F * 64) + x.lane;
    const lds_v4i part2 = (lds_v4i)(lds + kPartBytes / 2) + x.wave * (F * 64) + x.lane;
    const lds_v4i mine = (lds_v4i)lds + sub * src.ks * (F * 64) + x.lane, mine2 = (lds_v4i)(lds + kPartBytes / 2) + sub * src.ks * (F * 64) + x.lane;
    // The waves that share a tile's K share its chain as well: whole columns of pixels, or one of a quad's four pixels.  (The chain on
    // one wave's eight values is 0.3 us of a step; the others of its tile would only wait for it.  Two of the four pixels was a third
    // form: 8 KB of the kernel.  Every form counts: steps whose code does not fit the 64 KB that a pair of units' instruction cache
    // holds cost a ResNet-50 of batch 1 3 %, six times the misses, with a ring of its own for short K sums, for instance.)
    const int kk = src.kk, rows = (4 * B) >> shift <= 1 ? 1 : 4;      // (four columns and eight waves to a tile: choose_tile does not)
    const int col0 = rows == 4 ? kk & (B - 1) : min(kk >> 2, B - 1), r0 = rows == 4 ? 0 : kk & 3;
    const bool finishes = rows == 4 ? kk < B : kk < 4 * B;
    // Gelu's chain is long and its largest tiles are few: five on eight waves with 3072 channels of 1536 tokens and 256 workgroups, two of
    // them on one SIMD.  Where that takes fewer columns one behind the other every wave takes every eighth of the columns of all tiles:
    // an encoder of 6 layers x 3 x 512 tokens 566 us without, 552 with it.  With all eight waves busy (64 workgroups) it does not, and
    // would be slower (1243 and 1300: constants and places of another tile are fetched behind the product).  For the smaller tiles, as
    // quarters of columns, the code cost 12 layers x 128 tokens 10 % and gave it nothing.
    constexpr bool kSpreads = GELU && B == 4 && !PAIR;
    bool first = true;
    int base = t0;
    do {
        const int tile = base + sub;
        const bool on = tile < t1;
        ChannelConstants<A> k;
        ChannelConstants<A> k2;
        Ring<A, B> ring;
        uint32_t off[B], off2[B];
        Pixels<A> q;
        int lane = x.lane;
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile("" : "+v"(lane));       // (its functions are not kept in registers around the loop)
#endif
        const int lane16 = lane & 15, quad = lane >> 4;
        int ot, pt;
        fast_divmod(on ? tile : 0, PROG_FIELD(x.words, p_tiles), PROG_FIELD(x.words, inv_p_tiles), ot, pt);
        ot = __builtin_amdgcn_readfirstlane(ot);
        pt = __builtin_amdgcn_readfirstlane(pt);
        const int mt = pt * (16 * B), oc = ot * (16 * A) + A * lane16;
        bool spread = false, fin = on && finishes;
        int fmt = mt, fot = ot, column = sub * B + kk, columns = (sub + 1) * B;      // (kSpreads) whose column comes next, the first that is not the wave's
        auto take = [&] {
            int fpt;
            fast_divmod(base + column / B, PROG_FIELD(x.words, p_tiles), PROG_FIELD(x.words, inv_p_tiles), fot, fpt);
            fot = __builtin_amdgcn_readfirstlane(fot);
            fmt = __builtin_amdgcn_readfirstlane(fpt) * (16 * B);
        };
        if constexpr (kSpreads) {
            const int all = min(per, t1 - base) * B;
            spread = (PROG_FIELD(x.words, flags) & CF_GELU) && (all + 7) / 8 < (B + src.ks - 1) >> shift;
            if (spread) {
                column = x.wave;
                columns = all;
                fin = column < all;
                if (fin) take();
            }
        }
        src.w = make_buffer(PROG_TABLE_OF(int8_t, x.words, wgt) + static_cast<int64_t>(ot) * src.nk * (A * 1024));
        if constexpr (PAIR) src2.w = make_buffer(PROG_TABLE_OF(int8_t, x.words, wgt2) + static_cast<int64_t>(ot) * src2.nk * (A * 1024));
        // All that the step in front does not write is on its way before the wait: operands, constants, where the results go and, from
        // an older step, the residual.  Loads come back in order and a branch hides from the compiler how many there were behind it:
        // nothing that is loaded under a condition stands behind the pixels, which are the first to be waited for.
        if constexpr (kSpreads) {
            if (fin) place_pixels<A>(pix, M, fmt + 16 * (column & (B - 1)) + 4 * quad, q);
        }
        if (on) {
#pragma unroll
            for (int b = 0; b < B; ++b) off[b] = pix[mt + 16 * b + lane16];
            if (!kSpreads && finishes) place_pixels<A>(pix, M, mt + 16 * col0 + 4 * quad + r0, q);      // the first column this wave finishes
            if constexpr (PAIR) {
#pragma unroll
                for (int b = 0; b < B; ++b) off2[b] = pix[3 * M + mt + 16 * b + lane16];
            }
        }
        if (on) {
            if constexpr (PAIR) first_weights<A, B>(ring, src2, x.lane);
            else first_weights<A, B>(ring, src, x.lane);
            if (!kSpreads && finishes) {
                const int pitch = PROG_FIELD(x.words, OCp) * 4;
                if constexpr (PAIR) {
                    const uint8_t* t2 = PROG_TABLE_OF(uint8_t, x.words, constants2) + oc * 4;
                    load_channels<A>(reinterpret_cast<const int32_t*>(t2), k2.corr);
                    load_channels<A>(reinterpret_cast<const float*>(t2 + pitch), k2.bias);
                    load_channels<A>(reinterpret_cast<const float*>(t2 + 2 * pitch), k2.scale);
                }
                if constexpr (!kLate) load_constants<A>(PROG_FIELD(x.words, flags), PROG_TABLE_OF(uint8_t, x.words, constants), pitch, oc, k);
                StepConstants r{};
                r.flags = PROG_FIELD(x.words, flags);
                r.res = make_buffer(PROG_PLACE(x, res));
                r.res_limit = PROG_FIELD(x.words, res_limit);
                if (rows == 4) load_residual<A, 4>(r, oc, q);
                    else load_residual<A, 1>(r, oc, q);
            }
        }
        if (first) {
            if (!plain) {
                koff[min(x.tid, 4 * src.nk - 1)] = staged;
                if constexpr (PAIR) koff[kMaxPieces + min(x.tid, 4 * src2.nk - 1)] = staged2;
            }
            x.wait();
            first = false;
        }
        if (on) {
            if constexpr (PAIR) first_pixels<A, B>(ring, src2, off2, x.lane);
            else first_pixels<A, B>(ring, src, off, x.lane);
        }
        uint32_t words = x.words;
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile("" : "+v"(words));      // (what only the end needs is read here, not in front of the loop)
#endif
        const StepConstants sc = step_constants<true>(x, words);
        v4i acc[A][B];
        auto start = [&] {
#pragma unroll
            for (int a = 0; a < A; ++a)
#pragma unroll
                for (int b = 0; b < B; ++b) acc[a][b] = v4i{0, 0, 0, 0};
        };
        auto put = [&](lds_v4i to) {
#pragma unroll
            for (int a = 0; a < A; ++a)
#pragma unroll
                for (int b = 0; b < B; ++b) to[(b * A + a) * 64] = acc[a][b];
        };
        if (on) {
            if constexpr (PAIR) {
                start();
                k_loop<A, B>(ring, src2, off2, x.lane, acc);
                first_weights<A, B>(ring, src, x.lane);
                first_pixels<A, B>(ring, src, off, x.lane);
                put(part2);
            }
            start();
            k_loop<A, B>(ring, src, off, x.lane, acc);
            if constexpr (kLate && !kSpreads) load_constants<A>(sc.flags, PROG_TABLE_OF(uint8_t, words, constants), PROG_FIELD(words, OCp) * 4, oc, k);
            if constexpr (!kSpreads) put(part);
        }
        if constexpr (kSpreads) {
            const int foc = fot * (16 * A) + A * lane16;
            if (fin) {
                load_constants<A>(sc.flags, PROG_TABLE_OF(uint8_t, words, constants), PROG_FIELD(words, OCp) * 4, foc, k);
                load_residual<A, 4>(sc, foc, q);
            }
            if (on) put(part);
        }
        if (src.ks > 1 || spread) meet();
        if constexpr (kSpreads) {
            while (fin) {
                const int foc = fot * (16 * A) + A * lane16;
                finish_column<GELU, A, B, 4, PAIR>(sc, k, k2, (lds_v4i)lds + column / B * src.ks * (F * 64) + x.lane, mine2, src.ks, column & (B - 1), 0, q, foc);
                column += spread ? 8 : src.ks;
                if (column >= columns) break;
                const int held = fot;
                if (spread) take();
                if (fot != held) load_constants<A>(sc.flags, PROG_TABLE_OF(uint8_t, words, constants), PROG_FIELD(words, OCp) * 4, fot * (16 * A) + A * lane16, k);
                place_pixels<A>(pix, M, fmt + 16 * (column & (B - 1)) + 4 * quad, q);
                load_residual<A, 4>(sc, fot * (16 * A) + A * lane16, q);
            }
        } else if (on && finishes) {
            if (B == 4 || rows == 4) {
                for (int b = kk;;) {
                    finish_column<GELU, A, B, 4, PAIR>(sc, k, k2, mine, mine2, src.ks, b, 0, q, oc);
                    b += src.ks;
                    if (b >= B) break;
                    place_pixels<A>(pix, M, mt + 16 * b + 4 * quad, q);
                    load_residual<A, 4>(sc, oc, q);
                }
            } else if constexpr (B < 4) {
                finish_column<GELU, A, B, 1, PAIR>(sc, k, k2, mine, mine2, src.ks, col0, r0, q, oc);
            }
        }
        base += per;
        if ((src.ks > 1 || spread) && base < t1) meet();
    } while (base < t1);
}

// ---- depthwise 3 x 3 ----------------------------------------------------------------------------------------------------
// A lane owns four channels of G output pixels of a row: its columns of three input rows, byte transposes (v_perm) and
// v_dot4_i32_i8 as in dwconv.hip; consecutive lanes take consecutive channels.  G = 4 does the fewest operations per value,
// G = 1 a quarter of the work per lane: where a step's values are no more than the launch's lanes at one pixel each, what a
// lane does is what the step takes (ProgBuilder::conv).
template <int STRIDE, int G>
__device__ __forceinline__ void dw_items(Ctx& x) {
    constexpr int COLS = G == 1 ? 3 : 3 + 3 * STRIDE;
    const int OH = PROG_FIELD(x.words, OH), OW = PROG_FIELD(x.words, OW), items = PROG_FIELD(x.words, items), stride = 8 * x.n_wg * 64;
    const int c4s = PROG_FIELD(x.words, c4), quads = PROG_FIELD(x.words, quads), OCp = PROG_FIELD(x.words, OCp);
    const int in_sn = PROG_FIELD(x.words, in_sn), in_sh = PROG_FIELD(x.words, in_sh), in_sw = PROG_FIELD(x.words, in_sw), row_sh = PROG_FIELD(x.words, row_sh);
    const int out_sn = PROG_FIELD(x.words, out_sn), out_sh = PROG_FIELD(x.words, out_sh), out_sw = PROG_FIELD(x.words, out_sw);
    const int res_sn = PROG_FIELD(x.words, res_sn), res_sh = PROG_FIELD(x.words, res_sh), res_sw = PROG_FIELD(x.words, res_sw);
    const float inv_c4 = PROG_FIELD(x.words, inv_c4), inv_quads = PROG_FIELD(x.words, inv_quads), inv_OH = PROG_FIELD(x.words, inv_OH);
    const Buffer in = make_buffer(PROG_PLACE(x, in));
    const StepConstants sc = step_constants<false>(x, x.words);
    const int8_t* wgt = PROG_TABLE_OF(int8_t, x.words, wgt);
    const uint8_t* constants = PROG_TABLE_OF(uint8_t, x.words, constants);
    const bool f32 = sc.flags & CF_RES_F32, fo = !(sc.flags & CF_OUT_FQ);
    const int last_col = (OW - 1) * STRIDE + 2;
    bool first = true;
    int i0 = (x.wave * x.n_wg + x.rank) * 64;
    do {
        const int item = min(i0 + x.lane, items - 1);
        const bool on = i0 + x.lane < items;
        int q, c4, row, quad, n, oh;
        fast_divmod(item, c4s, inv_c4, q, c4);
        fast_divmod(q, quads, inv_quads, row, quad);
        fast_divmod(row, OH, inv_OH, n, oh);
        const int oc = 4 * c4, ow0 = G * quad;
        const uint32_t p = static_cast<uint32_t>(n * in_sn + oh * in_sh + oc);
        uint32_t v[3][COLS];
        uint4 wr[3];
#pragma unroll
        for (int r = 0; r < 3; ++r) wr[r] = *reinterpret_cast<const uint4*>(wgt + (static_cast<int64_t>(r) * OCp + oc) * 4);
        ChannelConstants<4> k;
        load_constants<4>(sc.flags, constants, OCp * 4, oc, k);
        uint32_t col[COLS];
#pragma unroll
        for (int j = 0; j < COLS; ++j) col[j] = p + static_cast<uint32_t>((G == 1 ? ow0 * STRIDE + j : min(ow0 * STRIDE + j, last_col)) * in_sw);
        Pixels<4> pq;
        {
            const uint32_t o = static_cast<uint32_t>(n * out_sn + oh * out_sh), s = static_cast<uint32_t>(n * res_sn + oh * res_sh);
#pragma unroll
            for (int r = 0; r < G; ++r) {
                const int ow = min(ow0 + r, OW - 1);
                pq.out[r] = on && ow0 + r < OW ? (o + ow * out_sw) << (fo ? 2 : 0) : static_cast<uint32_t>(kBeyond);
                pq.res[r] = (s + ow * res_sw) << (f32 ? 2 : 0);
            }
        }
        if (first) {
            x.wait();
            first = false;
        }
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int j = 0; j < COLS; ++j) v[r][j] = shared4(in, col[j] + static_cast<uint32_t>(r * row_sh));
        load_residual<4, G>(sc, oc, pq);
        int32_t acc[4][G];                    // [channel][pixel]
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int r = 0; r < G; ++r) acc[a][r] = k.corr[a];
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            const uint32_t w[4] = {wr[r].x, wr[r].y, wr[r].z, wr[r].w};
            if constexpr (STRIDE == 1 && G == 4) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    uint32_t t[4];
                    transpose_bytes(v[r][2 * h], v[r][2 * h + 1], v[r][2 * h + 2], v[r][2 * h + 3], t);
#pragma unroll
                    for (int a = 0; a < 4; ++a) {
                        acc[a][2 * h] = __builtin_amdgcn_sdot4(static_cast<int>(t[a]), static_cast<int>(w[a]), acc[a][2 * h], false);
                        acc[a][2 * h + 1] = __builtin_amdgcn_sdot4(static_cast<int>(t[a]), static_cast<int>(w[a] << 8), acc[a][2 * h + 1], false);
                    }
                }
            } else {
#pragma unroll
                for (int h = 0; h < G; ++h) {
                    uint32_t t[4];
                    transpose_bytes(v[r][2 * h], v[r][2 * h + 1], v[r][2 * h + 2], v[r][2 * h + 2], t);
#pragma unroll
                    for (int a = 0; a < 4; ++a) acc[a][h] = __builtin_amdgcn_sdot4(static_cast<int>(t[a]), static_cast<int>(w[a]), acc[a][h], false);
                }
            }
        }
        const float none[4][G] = {};
        finish<false, 4, G>(sc, k, acc, none, pq, oc);
        i0 += stride;
    } while (i0 < items);
}

// ---- expansion and depthwise 3 x 3 in one step ------------------------------------------------------------------------------
// A convolution whose only reader is the depthwise layer behind it (the first two layers of an inverted residual block): a
// workgroup computes 16 A channels of the input rows under a band of R output rows, requantised, into a patch in LDS - the rows
// between two bands by both - and the depthwise layer from there.  The tensor between the layers does not exist, and the block
// is two steps instead of three: a step of a network at batch 1 takes 3 - 4 us whatever it does (barrier, preparation, first
// operands, stores), a row computed twice a matrix instruction and a chain on four values a lane.  MobileNetV2 at batch 1, us:
// 197 with the layers apart, 182 with this, 170 with a fragment's pixels requested while the one before is multiplied, 168 with
// the second layer's constants requested behind the wait instead of in front of it (the preparation, 2.2 us, was longer than
// the barrier; 1.6 now).  What is left of such a step: 1.5 preparation and barrier, 1.2 - 2.3 first layer, 0.6 - 1.0 second.
// The descriptor's first half is the convolution with the geometry of both (ProgExpand), its second half the depthwise layer.
constexpr int kExpandSteps = 4;               // K steps of the convolution, held in registers

template <int A>
__device__ __forceinline__ void expand_depthwise(Ctx& x, lds_ptr lds) {
    // (what only the layers' ends need is read and requested behind the wait, while the first pixels are on their way: before it,
    // it stands between this step and the one before)
    const int nk = PROG_FIELD(x.words, nk), S = PROG_FIELD(x.words, expand.stride), R = PROG_FIELD(x.words, expand.rows), W = PROG_FIELD(x.words, expand.W);
    const int H = PROG_FIELD(x.words, expand.H), bands = PROG_FIELD(x.words, expand.bands), all_bands = PROG_FIELD(x.words, expand.all_bands);
    const int PW = PROG_FIELD(x.words, expand.patch_w), pad_t = PROG_FIELD(x.words, expand.pad_top), OH = PROG_FIELD(x.words, expand.OH);
    const bool plain = PROG_FIELD(x.words, koff).hi == 0;
    const lds_i32 staged_to = (lds_i32)(lds + kPartBytes), koff = plain ? (lds_i32)(lds + kPlainAt) : staged_to;
    int32_t staged = 0;
    if (!plain) staged = request_offsets(staged_to, PROG_TABLE_OF(int32_t, x.words, koff), 4 * nk, x.tid);
    const uint32_t units = static_cast<uint32_t>(PROG_FIELD(x.words, tiles));
    const int t0 = static_cast<int>((static_cast<uint32_t>(x.rank) * units) >> x.wg_shift), t1 = static_cast<int>((static_cast<uint32_t>(x.rank + 1) * units) >> x.wg_shift);
    if (t0 >= t1) {
        x.wait();
        return;
    }
    const uint32_t* pix = PROG_TABLE_OF(uint32_t, x.words, pixels);
    const int lane16 = x.lane & 15, quad = x.lane >> 4, c4 = x.tid & (4 * A - 1);
    int unit = t0;
    do {
        int ct, nb, n, band;
        fast_divmod(unit, all_bands, PROG_FIELD(x.words, expand.inv_all_bands), ct, nb);
        ct = __builtin_amdgcn_readfirstlane(ct);
        nb = __builtin_amdgcn_readfirstlane(nb);
        fast_divmod(nb, bands, PROG_FIELD(x.words, expand.inv_bands), n, band);
        n = __builtin_amdgcn_readfirstlane(n);
        band = __builtin_amdgcn_readfirstlane(band);
        const int oy0 = band * R, rows = min(R, OH - oy0), iy0 = oy0 * S - pad_t, patch_rows = (rows - 1) * S + 3;
        const int y0 = max(iy0, 0), y1 = min(iy0 + patch_rows, H), count = (y1 - y0) * W, m0 = (n * H + y0) * W;
        const int oc = ct * (16 * A) + A * lane16, oc4 = ct * (16 * A) + 4 * c4;
        const Buffer wb = make_buffer(PROG_TABLE_OF(int8_t, x.words, wgt) + static_cast<int64_t>(ct) * nk * (A * 1024));
        v4i wt[kExpandSteps][A];
#pragma unroll
        for (int k = 0; k < kExpandSteps; ++k)
#pragma unroll
            for (int a = 0; a < A; ++a) wt[k][a] = load16<0>(wb, static_cast<uint32_t>(x.lane * 16) + static_cast<uint32_t>(k < nk ? k * (A * 1024) : kBeyond), a * 1024);
        ChannelConstants<A> k1;
        load_constants<A>(PROG_FIELD(x.words, flags), PROG_TABLE_OF(uint8_t, x.words, constants), PROG_FIELD(x.words, OCp) * 4, oc, k1);
        int f = x.wave;
        uint32_t off = pix[m0 + min(16 * f + lane16, count - 1)];
        // the patch at the level of the padding (every lane takes part, those behind the end repeat the last piece)
        const int pieces = patch_rows * PW * A, fill = PROG_FIELD(x.words, expand.fill);
        for (int base = 0; base < pieces; base += kProgramThreads) ((lds_v4i)lds)[min(base + x.tid, pieces - 1)] = v4i{fill, fill, fill, fill};
        if (unit == t0) {
            if (!plain) staged_to[min(x.tid, 4 * nk - 1)] = staged;
            x.wait();
        } else meet();
        // the convolution: a wave's fragments of 16 pixels, eight apart
        const Buffer in = make_buffer(PROG_PLACE(x, in));
        const int frags = (count + 15) / 16;
        v4i p[kExpandSteps], next[kExpandSteps];
        auto request = [&](v4i (&to)[kExpandSteps]) {
#pragma unroll
            for (int k = 0; k < kExpandSteps; ++k)
                to[k] = shared16(in, off + static_cast<uint32_t>(koff[4 * min(k, nk - 1) + quad]) + (k < nk ? 0u : static_cast<uint32_t>(kBeyond)));
        };
        request(p);
        off = pix[m0 + min(16 * f + 128 + lane16, count - 1)];
        const StepConstants c1 = step_constants<false>(x, x.words), c2 = step_constants<false>(x, x.words2);
        const int OCp2 = PROG_FIELD(x.words2, OCp), pad_l = PROG_FIELD(x.words, expand.pad_left);
        const float inv_W = PROG_FIELD(x.words, expand.inv_W);
        uint4 wr[3];
#pragma unroll
        for (int r = 0; r < 3; ++r) wr[r] = *reinterpret_cast<const uint4*>(PROG_TABLE_OF(int8_t, x.words2, wgt) + (static_cast<int64_t>(r) * OCp2 + oc4) * 4);
        ChannelConstants<4> k2;
        load_constants<4>(c2.flags, PROG_TABLE_OF(uint8_t, x.words2, constants), OCp2 * 4, oc4, k2);
        while (f < frags) {
            const int j0 = 16 * f + 4 * quad;
            f += 8;
            request(next);                       // (those behind the last one read its pixels)
            off = pix[m0 + min(16 * f + 128 + lane16, count - 1)];
            v4i acc[A];
#pragma unroll
            for (int a = 0; a < A; ++a) acc[a] = v4i{k1.corr[a], k1.corr[a], k1.corr[a], k1.corr[a]};
#pragma unroll
            for (int k = 0; k < kExpandSteps; ++k)
                if (k == 0 || k < nk)
#pragma unroll
                    for (int a = 0; a < A; ++a) acc[a] = __builtin_amdgcn_mfma_i32_16x16x64_i8(p[k], wt[k][a], acc[a], 0, 0, 0);
            int32_t sum[A][4];
            const float none[A][4] = {};
            float v[A][4];
            uint32_t bytes[4];
#pragma unroll
            for (int a = 0; a < A; ++a)
#pragma unroll
                for (int r = 0; r < 4; ++r) sum[a][r] = acc[a][r];
            const Pixels<A> nowhere{};
            chain<false, A, 4>(c1, k1, sum, none, nowhere, oc, v);
            levels<A, 4>(c1, k1, v, bytes);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                int row, col;
                fast_divmod(min(j0 + r, count - 1), W, inv_W, row, col);        // (pixels behind the last one hold its values)
                const lds_ptr at = lds + ((y0 - iy0 + row) * PW + col + pad_l) * (16 * A) + A * lane16;
                if constexpr (A == 1) *at = static_cast<int8_t>(bytes[r]);
                else *(__attribute__((address_space(3))) uint16_t*)at = static_cast<uint16_t>(bytes[r]);
            }
#pragma unroll
            for (int k = 0; k < kExpandSteps; ++k) p[k] = next[k];
        }
        meet();
        // the depthwise layer: four channels of a pixel per lane
        const int OW = PROG_FIELD(x.words, expand.OW), items = rows * OW * (4 * A);
        const int out_sn = PROG_FIELD(x.words2, out_sn), out_sh = PROG_FIELD(x.words2, out_sh), out_sw = PROG_FIELD(x.words2, out_sw);
        const float inv_OW = PROG_FIELD(x.words, expand.inv_OW);
        for (int base = 0; base < items; base += kProgramThreads) {
            const bool on = base + x.tid < items;
            int oy, ox;
            fast_divmod(min(base + x.tid, items - 1) / (4 * A), OW, inv_OW, oy, ox);
            const lds_ptr at = lds + (oy * S * PW + ox * S) * (16 * A) + 4 * c4;
            int32_t acc[4][1];
#pragma unroll
            for (int a = 0; a < 4; ++a) acc[a][0] = k2.corr[a];
            uint32_t v[3][3];
#pragma unroll
            for (int r = 0; r < 3; ++r)
#pragma unroll
                for (int j = 0; j < 3; ++j) v[r][j] = *(const __attribute__((address_space(3))) uint32_t*)(at + (r * PW + j) * (16 * A));
#pragma unroll
            for (int r = 0; r < 3; ++r) {
                const uint32_t w[4] = {wr[r].x, wr[r].y, wr[r].z, wr[r].w};
                uint32_t t[4];
                transpose_bytes(v[r][0], v[r][1], v[r][2], v[r][2], t);
#pragma unroll
                for (int a = 0; a < 4; ++a) acc[a][0] = __builtin_amdgcn_sdot4(static_cast<int>(t[a]), static_cast<int>(w[a]), acc[a][0], false);
            }
            Pixels<4> q;
            q.out[0] = on ? static_cast<uint32_t>(n * out_sn + (oy0 + oy) * out_sh + ox * out_sw) : static_cast<uint32_t>(kBeyond);
            q.res[0] = 0;
            const float none[4][1] = {};
            finish<false, 4, 1>(c2, k2, acc, none, q, oc4);
        }
        ++unit;
        if (unit < t1) meet();
    } while (unit < t1);
}

// ---- entry, pooling, exit ---------------------------------------------------------------------------------------------------
__device__ __forceinline__ uint32_t level_bytes(const FqChannel& f, float lm1, float off, float v) {
    return static_cast<uint32_t>(static_cast<int>(fq_level_clamped<true>(f, lm1, v) + off)) & 0xffu;
}

__device__ __forceinline__ void entry_items(const ProgEntry& e, const Ctx& x) {
    const uint8_t* in = PROG_REF(x, e.in);
    const Buffer out = make_buffer(PROG_REF(x, e.out));
    const FqChannel* tab = PROG_TABLE(FqChannel, e.tab);
    const int groups = e.cs / 4, waves_per_plane = (e.HW + 63) / 64;       // four channels of 64 pixels of one image
    const int items = e.N * groups * waves_per_plane;
    for (int i = x.wave * x.n_wg + x.rank; i < items; i += 8 * x.n_wg) {
        const int pw = i % waves_per_plane, np = i / waves_per_plane, g = np % groups, n = np / groups;
        const int p = pw * 64 + x.lane;
        const bool on = p < e.HW;
        int h, w;
        fast_divmod(on ? p : 0, e.W, e.inv_W, h, w);
        const int64_t src = (static_cast<int64_t>(n) * e.C + 4 * g) * e.HW + (on ? p : 0);
        float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (4 * g + j < e.C) {
                const int64_t o = src + static_cast<int64_t>(j) * e.HW;
                v[j] = e.u8_in ? static_cast<float>(in[o]) : reinterpret_cast<const float*>(in)[o];
            }
        uint32_t dw = (static_cast<uint32_t>(static_cast<int>(e.off)) & 0xffu) * 0x01010101u;     // level 0 in the channels that do not exist
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (4 * g + j < e.C) dw = (dw & ~(0xffu << (8 * j))) | (level_bytes(tab[4 * g + j], e.lm1, e.off, v[j]) << (8 * j));
        publish4(out, on ? static_cast<uint32_t>(n * e.out_sn + h * e.out_sh + static_cast<int64_t>(w) * e.cs + 4 * g) : static_cast<uint32_t>(kBeyond), dw);
    }
}

// bytewise running maxima in the order-preserving unsigned domain, as pool.hip
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void max_take(uint32_t stored, uint32_t& even, uint32_t& odd) {
    const uint32_t v = stored ^ 0x80808080u;
    even = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, even), __builtin_bit_cast(u16x2, v & 0x00ff00ffu)));
    odd = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, odd), __builtin_bit_cast(u16x2, v & 0xff00ff00u)));
}

__device__ __forceinline__ void max_pool_items(const ProgPool& s, const Ctx& x) {
    const PoolArgs& a = s.a;
    const int cg = a.cs / 4;
    const Buffer in = make_buffer(PROG_REF(x, s.in)), out = make_buffer(PROG_REF(x, s.out));
    for (int i0 = (x.wave * x.n_wg + x.rank) * 64; i0 < s.items; i0 += 8 * x.n_wg * 64) {
        const int t = i0 + x.lane;
        if (t >= s.items) continue;
        const int m = t / cg, c = (t - m * cg) * 4;
        const int n = m / a.OHOW, rem = m - n * a.OHOW, oh = rem / a.OW, ow = rem - oh * a.OW;
        const int y0 = oh * a.sh - a.pt, x0 = ow * a.sw - a.pl;
        const uint32_t base = static_cast<uint32_t>(n * a.in_sn + c);
        uint32_t even = 0, odd = 0;
        if (s.k3) {
            uint32_t v[9];
#pragma unroll
            for (int j = 0; j < 9; ++j) {
                const int yy = min(max(y0 + j / 3, 0), a.H - 1), xx = min(max(x0 + j % 3, 0), a.W - 1);
                v[j] = shared4(in, base + static_cast<uint32_t>(yy * a.in_sh + xx * a.in_sw));
            }
#pragma unroll
            for (int j = 0; j < 9; ++j) max_take(v[j], even, odd);
        } else {
            const int ya = max(y0, 0), xa = max(x0, 0);
            const int yb = min(min(y0 + a.kh, a.H + a.pb), a.H), xb = min(min(x0 + a.kw, a.W + a.pr), a.W);
            for (int yy = ya; yy < yb; ++yy)
                for (int xx = xa; xx < xb; ++xx) max_take(shared4(in, base + static_cast<uint32_t>(yy * a.in_sh + xx * a.in_sw)), even, odd);
        }
        publish4(out, static_cast<uint32_t>(n * a.out_sn + oh * a.out_sh + ow * a.out_sw + c), (even | odd) ^ 0x80808080u);
    }
}

// Average pool: sixteen lanes share a window (a lane sums every sixteenth cell of four channels), so that a global pool of
// one image - a few hundred outputs of 49 cells - still has all of the group's waves loading.
__device__ __forceinline__ void avg_pool_items(const ProgPool& s, const Ctx& x) {
    const PoolArgs& a = s.a;
    const int cg = a.cs / 4, items = s.items;
    const Buffer in = make_buffer(PROG_REF(x, s.in)), out = make_buffer(PROG_REF(x, s.out));
    const int share = x.lane >> 2;            // lanes 4 q + j of a wave: share q of item j
    for (int i0 = (x.wave * x.n_wg + x.rank) * 4; i0 < items; i0 += 8 * x.n_wg * 4) {
        const int t = min(i0 + (x.lane & 3), items - 1);
        const int m = t / cg, c = (t - m * cg) * 4;
        const int n = m / a.OHOW, rem = m - n * a.OHOW, oh = rem / a.OW, ow = rem - oh * a.OW;
        const int y0 = oh * a.sh - a.pt, x0 = ow * a.sw - a.pl;
        const int y1 = min(y0 + a.kh, a.H + a.pb), x1 = min(x0 + a.kw, a.W + a.pr);
        const bool padding_present = a.pt || a.pl || a.pb || a.pr;
        const int ya = max(y0, 0), yb = min(y1, a.H), xa = max(x0, 0), xb = min(x1, a.W);
        const int wx = max(xb - xa, 0), cells = max(yb - ya, 0) * wx;
        int count = padding_present ? cells : (y1 - y0) * (x1 - x0);
        const uint32_t base = static_cast<uint32_t>(n * a.in_sn + c);
        int sum[4] = {0, 0, 0, 0};
        for (int j = share; j < cells; j += 64) {
            uint32_t v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int jj = min(j + 16 * u, cells - 1), yy = jj / wx, xx = jj - yy * wx;
                v[u] = shared4(in, base + static_cast<uint32_t>((ya + yy) * a.in_sh + (xa + xx) * a.in_sw));
                if (j + 16 * u >= cells) v[u] = 0;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int b = 0; b < 4; ++b) sum[b] += static_cast<int8_t>(v[u] >> (8 * b));
        }
#pragma unroll
        for (int o = 4; o < 64; o <<= 1)
#pragma unroll
            for (int b = 0; b < 4; ++b) sum[b] += __shfl_xor(sum[b], o, 64);
        if (share != 0 || i0 + (x.lane & 3) >= items) continue;
        if (a.include_pad && padding_present) count = a.kh * a.kw;
        const float nf = static_cast<float>(count);
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float t4 = static_cast<float>(sum[j] + a.in_bias * cells) / nf;
            if (a.mul) t4 = t4 * a.mul[c + j];
            v[j] = t4;
        }
        const uint32_t o = static_cast<uint32_t>(n * a.out_sn + oh * a.out_sh + ow * a.out_sw + c);
        if (a.preserve) {
            uint32_t packed = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int total = sum[j] + a.in_bias * cells;
                const int r = a.preserve == 1 ? (total & 0xff) : static_cast<int>(static_cast<int8_t>(total & 0xff));
                const int level = static_cast<int>(__builtin_rintf(static_cast<float>(r) / nf));
                packed |= (static_cast<uint32_t>(level - (a.preserve == 1 ? 128 : 0)) & 0xffu) << (8 * j);
            }
            publish4(out, o, packed);
        } else if (a.fq_il) {
            uint32_t packed = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                FqChannel p;
                p.il = a.fq_il[c + j]; p.ih = a.fq_ih[c + j]; p.d = a.fq_d[c + j]; p.r = a.fq_r[c + j];
                packed |= level_bytes(p, a.lm1, a.out_off, v[j]) << (8 * j);
            }
            publish4(out, o, packed);
        } else {
            publish16f(out, 4 * o, make_float4(v[0], v[1], v[2], v[3]));
        }
    }
}

// (the caller's output buffer, which can be larger than a buffer descriptor reaches: nothing in the launch reads it, the host does)
template <typename TIn>
__device__ __forceinline__ void exit_items(const ProgExit& s, const Ctx& x) {
    const ExitArgs& a = s.a;
    const Buffer in = make_buffer(PROG_REF(x, s.in));
    uint8_t* out = PROG_REF(x, s.out);
    auto one = [&](const TIn raw, int n, int c, int p) {
        float v = static_cast<float>(raw) + a.in_bias;
        if (a.sub) v = v - a.sub[c];
        if (a.mul) v = v * a.mul[c];
        const int64_t o = (static_cast<int64_t>(n) * a.C + c) * a.HW + p;
        if (a.out_u8) __hip_atomic_store(out + o, static_cast<uint8_t>(static_cast<int>(v)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else __hip_atomic_store(reinterpret_cast<float*>(out) + o, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    if (a.HW >= 16) {                        // lanes along the pixels, four channels each (a pixel's channels are padded to four)
        const int waves = (a.HW + 63) / 64, cg = (a.C + 3) / 4, items = a.N * cg * waves;
        for (int i = x.wave * x.n_wg + x.rank; i < items; i += 8 * x.n_wg) {
            const int pw = i % waves, ng = i / waves, g = ng % cg, n = ng / cg, p = pw * 64 + x.lane;
            if (p >= a.HW) continue;
            const int h = p / a.W, w = p - h * a.W;
            const uint32_t q = static_cast<uint32_t>(n * a.in_sn + h * a.in_sh + w * a.in_sw + 4 * g) * sizeof(TIn);
            TIn raw[4];
            if constexpr (sizeof(TIn) == 4) {
                const v4i t = shared16(in, q);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int32_t word = t[j];
                    raw[j] = __builtin_bit_cast(TIn, word);
                }
            } else {
                const uint32_t t = shared4(in, q);
#pragma unroll
                for (int j = 0; j < 4; ++j) raw[j] = static_cast<TIn>(t >> (8 * j));
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (4 * g + j < a.C) one(raw[j], n, 4 * g + j, p);
        }
    } else {
        const int items = a.N * a.HW * a.C;
        for (int i0 = (x.wave * x.n_wg + x.rank) * 64; i0 < items; i0 += 8 * x.n_wg * 64) {
            const int i = i0 + x.lane;
            if (i >= items) continue;
            const int np = i / a.C, c = i - np * a.C, n = np / a.HW, p = np - n * a.HW;
            const int h = p / a.W, w = p - h * a.W;
            const uint32_t q = static_cast<uint32_t>(n * a.in_sn + h * a.in_sh + w * a.in_sw + c);
            TIn raw;
            if constexpr (sizeof(TIn) == 4) {
                const uint32_t word = shared4(in, 4 * q);
                raw = __builtin_bit_cast(TIn, word);
            } else raw = static_cast<TIn>(shared1(in, q));
            one(raw, n, c, p);
        }
    }
}

// ---- rows of an encoder -----------------------------------------------------------------------------------------------------
// v summed over the wave as a butterfly, lanes 32 apart first: the pairs and the order of __shfl_xor by 32, 16 .. 1.  Lanes 32 and
// 16 apart come together by a swap of rows, and behind those the value repeats every 16, 8, 4 lanes, so that a rotation by
// 8 and by 4 of a row's lanes and two permutations of its quads find the same partners: an instruction each, where a shuffle
// by way of LDS takes 0.05 us (twelve of them were 0.7 us of a LayerNorm step).
__device__ __forceinline__ float wave_total(float v) {
#if defined(__HIP_DEVICE_COMPILE__)
    const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(h[0]) + __uint_as_float(h[1]);
    const auto q = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(q[0]) + __uint_as_float(q[1]);
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, true));      // row_ror:8
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xf, 0xf, true));      // row_ror:4
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4e, 0xf, 0xf, true));       // quad_perm 2 3 0 1
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xb1, 0xf, 0xf, true));       // quad_perm 1 0 3 2
#endif
    return v;
}

__device__ __forceinline__ uint32_t levels4(const Requant& f, const float4& v) {
    return level_bytes(f.p, f.lm1, f.p.ol, v.x) | (level_bytes(f.p, f.lm1, f.p.ol, v.y) << 8) | (level_bytes(f.p, f.lm1, f.p.ol, v.z) << 16) |
           (level_bytes(f.p, f.lm1, f.p.ol, v.w) << 24);
}

__device__ __forceinline__ void embed_rows(const ProgEmbed& e, const Ctx& x) {
    const int32_t* ids = reinterpret_cast<const int32_t*>(PROG_REF(x, e.ids));
    const Buffer out = make_buffer(PROG_REF(x, e.out));
    const float *tab = PROG_TABLE(float, e.table), *add0 = PROG_TABLE(float, e.add0), *add1 = PROG_TABLE(float, e.add1);
    for (int t = x.wave * x.n_wg + x.rank; t < e.tokens; t += 8 * x.n_wg) {
        int64_t idx = ids[t];
        if (idx < 0) idx += e.vocab;
        idx = idx < 0 ? 0 : (idx >= e.vocab ? e.vocab - 1 : idx);
        const int64_t p = t % e.seq;
        const float* src = tab + idx * e.hidden;
        const float* a0 = add0 ? add0 + (e.pos0 ? p * e.hidden : 0) : nullptr;
        const float* a1 = add1 ? add1 + (e.pos1 ? p * e.hidden : 0) : nullptr;
        for (int i = 4 * x.lane; i < e.hidden; i += 256) {
            float4 v = ld4f(src + i);
            if (a0) { const float4 a = ld4f(a0 + i); v.x = v.x + a.x; v.y = v.y + a.y; v.z = v.z + a.z; v.w = v.w + a.w; }
            if (a1) { const float4 a = ld4f(a1 + i); v.x = v.x + a.x; v.y = v.y + a.y; v.z = v.z + a.z; v.w = v.w + a.w; }
            publish16f(out, 4u * static_cast<uint32_t>(t * e.hidden + i), v);
        }
    }
}

constexpr int kMvnChunks = 4;                 // rows of up to 1024 values
__device__ __forceinline__ void mvn_rows(const ProgMvn& s, Ctx& x) {
    const Buffer in = make_buffer(x.place(s.in)), yb = make_buffer(x.place(s.out)), qb = make_buffer(x.place(s.outq));
    const bool y = s.out.base >= 0, q = s.outq.base >= 0;
    const float *gamma = PROG_TABLE(float, s.gamma), *beta = PROG_TABLE(float, s.beta);
    const int axis = s.axis;
    int row = x.wave * x.n_wg + x.rank;
    // the affine part of a lane's columns, the same for all its rows, while the step before comes to its end
    float4 g[kMvnChunks], b[kMvnChunks];
#pragma unroll
    for (int j = 0; j < kMvnChunks; ++j) {
        const int i = min(256 * j + 4 * x.lane, axis - 4);
        if (gamma) g[j] = ld4f(gamma + i);
        if (beta) b[j] = ld4f(beta + i);
    }
    x.wait();
    for (; row < s.rows; row += 8 * x.n_wg) {
        const uint32_t p = static_cast<uint32_t>(row * axis);
        float4 v[kMvnChunks];
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < kMvnChunks; ++j) {
            const int i = 256 * j + 4 * x.lane;
            v[j] = shared16f(in, i < axis ? 4u * (p + i) : static_cast<uint32_t>(kBeyond));
        }
#pragma unroll
        for (int j = 0; j < kMvnChunks; ++j) sum += (v[j].x + v[j].y) + (v[j].z + v[j].w);
        const float mean = wave_total(sum) / static_cast<float>(axis);
        float sq = 0.f;
#pragma unroll
        for (int j = 0; j < kMvnChunks; ++j) {
            const int i = 256 * j + 4 * x.lane;
            v[j].x -= mean; v[j].y -= mean; v[j].z -= mean; v[j].w -= mean;
            if (i < axis) sq += (v[j].x * v[j].x + v[j].y * v[j].y) + (v[j].z * v[j].z + v[j].w * v[j].w);
        }
        float denom = 1.f;
        if (s.normalize) {
            const float var = wave_total(sq) / static_cast<float>(axis);
            denom = s.eps_inside ? sqrtf(var + s.eps) : sqrtf(var) + s.eps;
        }
#pragma unroll
        for (int j = 0; j < kMvnChunks; ++j) {
            const int i = 256 * j + 4 * x.lane;
            if (i >= axis) continue;
            float4 o = v[j];
            if (s.normalize) { o.x = o.x / denom; o.y = o.y / denom; o.z = o.z / denom; o.w = o.w / denom; }
            if (gamma) { o.x = o.x * g[j].x; o.y = o.y * g[j].y; o.z = o.z * g[j].z; o.w = o.w * g[j].w; }
            if (beta) { o.x = o.x + b[j].x; o.y = o.y + b[j].y; o.z = o.z + b[j].z; o.w = o.w + b[j].w; }
            if (y) publish16f(yb, 4u * (p + i), o);
            if (q) publish4(qb, p + i, levels4(s.fq, o));
        }
    }
}

__device__ __forceinline__ void fq_items(const ProgRows& s, const Ctx& x) {
    const Buffer in = make_buffer(PROG_REF(x, s.in)), out = make_buffer(PROG_REF(x, s.out));
    for (int i = 4 * ((x.wave * x.n_wg + x.rank) * 64 + x.lane); i < s.n; i += 4 * 8 * x.n_wg * 64) {
        const float4 v = shared16f(in, 4u * static_cast<uint32_t>(i));
        const float t[4] = {v.x, v.y, v.z, v.w};
        uint32_t w = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) w |= level_bytes(s.p, s.lm1, s.off, t[j]) << (8 * j);
        publish4(out, static_cast<uint32_t>(i), w);
    }
}

__device__ __forceinline__ void copy_items(const ProgRows& s, const Ctx& x) {
    const Buffer in = make_buffer(PROG_REF(x, s.in)), out = make_buffer(PROG_REF(x, s.out));
    for (int i = 16 * ((x.wave * x.n_wg + x.rank) * 64 + x.lane); i < s.n; i += 16 * 8 * x.n_wg * 64)
        publish16(out, static_cast<uint32_t>(i), shared16(in, static_cast<uint32_t>(i)));
}

// ---- attention --------------------------------------------------------------------------------------------------------------
// The core of attention.hip with the sequence length at run time: K and V^T of one (element, head) in LDS.  32 queries are the
// work of `split` waves: each takes every split-th tile of 32 keys - its scores stay in registers, up to kMostTiles of them -
// and the waves meet for the maximum, for the sum and for the integer sums of the context.  What bounds a step is the chain of
// exponentials and levels of one wave (1 us for a tile of 32 x 32), so the fewer tiles a wave has the better while there are
// compute units: the step of one sequence of 128 tokens, 12 heads, barrier included, took 11.2 us with a wave for 32 queries, 48
// waves in all, that multiplied the scores out three times, and takes 7.2 with four.  The sum keeps its order - a lane's keys one behind the
// other - so one wave adds the exponentials of all.  They take K's place in LDS, and the context's partial sums theirs.
constexpr int kMostTiles = 4;                 // of a wave
constexpr int kMostSplit = 8;
// LDS: V^T; K, then exponentials, then partial sums of the context; the mask, the maxima and the sums of the waves' rows
__host__ __device__ constexpr int attention_exchange(int S, int split) {
    const int k = S * 64, ctx = 64 * 1024, e = split > 1 ? kMostSplit / split * (S / 32) * 4096 : 0;
    return k > ctx ? (k > e ? k : e) : (ctx > e ? ctx : e);
}
__host__ __device__ constexpr int attention_lds(int S, int split) { return 64 * (S + 16) + attention_exchange(S, split) + 4 * S + 8 * 32 * 4 + 8 * 64 * 4; }
template <int PFORM>
__device__ __forceinline__ void attention_units(const ProgAttention& s, Ctx& x, lds_ptr lds) {
    typedef __attribute__((address_space(3))) float* lds_f32;
    typedef float v4f __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) v4f* lds_v4f;
    const AttentionArgs& a = s.a;
    const int S = s.S, nt = S / 32, vt_ld = S + 16, split = 1 << s.split_shift, w = x.wave & (split - 1), block = x.wave >> s.split_shift, blocks = kMostSplit >> s.split_shift;
    const int l32 = x.lane & 31, h = x.lane >> 5;
    const lds_ptr sVT = lds, sK = lds + 64 * vt_ld;
    const lds_v4i sCtx = (lds_v4i)sK;                                   // [wave][8 groups of 4 registers][64]
    const lds_f32 sMask = (lds_f32)(sK + attention_exchange(S, split)), sMax = sMask + S, sSum = sMax + 8 * 32 + block * 64 + x.lane;
    const Buffer qb = make_buffer(x.place(s.q)), kb = make_buffer(x.place(s.k)), vb = make_buffer(x.place(s.v)), out = make_buffer(x.place(s.out));
    const float* mask = s.has_mask ? reinterpret_cast<const float*>(x.place(s.mask)) : nullptr;
    constexpr float kLog2e = 1.4426950408889634f;
    bool first = true;
    int u = x.rank;
    do {
        const int eh = min(u, s.units - 1) / s.parts, part = u - eh * s.parts, n = eh / s.heads, hd = eh - n * s.heads;
        const uint32_t kp = static_cast<uint32_t>(n * a.ok + hd * a.sk), vp = static_cast<uint32_t>(n * a.ov + hd * a.sv);
        const int q0 = 32 * (part * blocks + block);
        const bool on = q0 < S && block < blocks;
        const uint32_t qbase = static_cast<uint32_t>(n * a.oq + hd * a.sq), obase = static_cast<uint32_t>(n * a.oo + hd * a.so);
        const int q_row = min(q0, S - 32) + l32;
        const float mk1 = mask ? mask[n * a.mask_outer + hd * a.mask_inner + min(x.tid, S - 1)] : 0.f;
        if (first) x.wait();
        first = false;
        if (u >= s.units) return;
        // K into LDS, V transposed into LDS: everything is requested before any of it is used
        constexpr int kRounds = kPlainSoftmax * 4 / kProgramThreads;      // S * 4 pieces of K, as many groups of 4 keys x 4 d of V, by 512 threads
        v4i kx[kRounds];
        uint32_t vw[kRounds][4];
#pragma unroll
        for (int j = 0; j < kRounds; ++j) {
            if (j * kProgramThreads >= S * 4) continue;
            const int i = min(x.tid + j * kProgramThreads, S * 4 - 1), r = i >> 2, c = i & 3;      // (threads behind the end repeat the last piece)
            kx[j] = shared16(kb, kp + static_cast<uint32_t>(r * a.ldk + c * 16));
        }
#pragma unroll
        for (int j = 0; j < kRounds; ++j) {
            if (j * kProgramThreads >= S * 4) continue;
            const int i = min(x.tid + j * kProgramThreads, S * 4 - 1), d4 = i & 15, kq = i >> 4;
#pragma unroll
            for (int q = 0; q < 4; ++q) vw[j][q] = shared4(vb, vp + static_cast<uint32_t>((4 * kq + q) * a.ldv + 4 * d4));
        }
        const uint32_t qrow = qbase + static_cast<uint32_t>(q_row * a.ldq);
        const v4i qf[2] = {shared16(qb, qrow + 16 * h), shared16(qb, qrow + 32 + 16 * h)};
        if (mask) sMask[min(x.tid, S - 1)] = mk1;
#pragma unroll
        for (int j = 0; j < kRounds; ++j) {
            if (j * kProgramThreads >= S * 4) continue;
            const int i = min(x.tid + j * kProgramThreads, S * 4 - 1), r = i >> 2, c = i & 3;
            *(lds_v4i)(sK + r * 64 + ((c ^ ((r >> 2) & 3)) * 16)) = kx[j];
        }
#pragma unroll
        for (int j = 0; j < kRounds; ++j) {
            if (j * kProgramThreads >= S * 4) continue;
            const int i = min(x.tid + j * kProgramThreads, S * 4 - 1), d4 = i & 15, kq = i >> 4;
            uint32_t t[4];
            transpose_bytes(vw[j][0], vw[j][1], vw[j][2], vw[j][3], t);
            const int key = 4 * kq, tile = key >> 5, in = key & 31;
            const int col = tile * 32 + ((in >> 2) & 1) * 16 + (in >> 3) * 4;
#pragma unroll
            for (int q = 0; q < 4; ++q) *(__attribute__((address_space(3))) uint32_t*)(sVT + (4 * d4 + q) * vt_ld + col) = t[q];
        }
        meet();
        // the scores of this wave's tiles and their maximum
        float v[kMostTiles][16];
        float m = -INFINITY;
        const int slot[2] = {((0 + h) ^ ((l32 >> 2) & 3)) * 16, ((2 + h) ^ ((l32 >> 2) & 3)) * 16};
#pragma unroll
        for (int j = 0; j < kMostTiles; ++j) {
            const int t = w + (j << s.split_shift);
            if (!on || t >= nt) continue;
            v16i acc = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(*(lds_v4i)(sK + (32 * t + l32) * 64 + slot[ks]), qf[ks], acc, 0, 0, 0);
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                v4f mk = {0.f, 0.f, 0.f, 0.f};
                if (s.has_mask) mk = *(lds_v4f)(sMask + 32 * t + 8 * g + 4 * h);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float y = static_cast<float>(acc[4 * g + r]) * a.scale1;
                    if (s.has_mask) y = y + mk[r];
                    v[j][4 * g + r] = y;
                    m = fmaxf(m, y);
                }
            }
        }
        m = fmaxf(m, __shfl_xor(m, 32, 64));
        if (split > 1) {
            sMax[x.wave * 32 + l32] = m;            // (the same in both halves of the wave)
            meet();
            for (int k = 0; k < split; ++k) m = fmaxf(m, sMax[(block * split + k) * 32 + l32]);
        }
        // exponentials, and their sum: a lane's one behind the other
        const float mL = -m * kLog2e;
        const lds_v4f sE = (lds_v4f)sK + block * nt * 4 * 64 + x.lane;   // [tile][group of four][64]
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < kMostTiles; ++j) {
            const int t = w + (j << s.split_shift);
            if (!on || t >= nt) continue;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
#pragma unroll
                for (int r = 4 * g; r < 4 * g + 4; ++r) {
                    v[j][r] = __builtin_amdgcn_exp2f(fmaf(v[j][r], kLog2e, mL));
                    sum += v[j][r];
                }
                if (split > 1) sE[(4 * t + g) * 64] = v4f{v[j][4 * g], v[j][4 * g + 1], v[j][4 * g + 2], v[j][4 * g + 3]};
            }
        }
        if (split > 1) {
            meet();
            if (on && w == 0) {
                sum = 0.f;
                for (int t = 0; t < nt; ++t)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const v4f e = sE[(4 * t + g) * 64];
                        sum += e.x; sum += e.y; sum += e.z; sum += e.w;
                    }
                sSum[0] = sum;
            }
            meet();
            sum = sSum[0];
        } else meet();                          // (K's last readers are through)
        sum += __shfl_xor(sum, 32, 64);
        const float inv = 1.0f / sum;
        // probabilities -> levels -> this wave's part of the second product
        v16i ctx[2] = {{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}, {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}};
#pragma unroll
        for (int j = 0; j < kMostTiles; ++j) {
            const int t = w + (j << s.split_shift);
            if (!on || t >= nt) continue;
            v4i pf = {0, 0, 0, 0};
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                float p[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) p[r] = v[j][4 * g + r] * inv;
                pf[g] = static_cast<int>(prob_levels4<true, PFORM>(a, p[0], p[1], p[2], p[3]));
            }
            // u8 probabilities q are stored as q - 128: the 128 that is missing from each, as twice 64
            const int n64 = a.p_bias ? 0x40404040 : 0;
            const v4i bias = {n64, n64, n64, n64};
#pragma unroll
            for (int db = 0; db < 2; ++db) {
                const v4i vf = *(lds_v4i)(sVT + (32 * db + l32) * vt_ld + 32 * t + 16 * h);
                ctx[db] = __builtin_amdgcn_mfma_i32_32x32x32_i8(vf, pf, ctx[db], 0, 0, 0);
                if (a.p_bias) {
                    ctx[db] = __builtin_amdgcn_mfma_i32_32x32x32_i8(vf, bias, ctx[db], 0, 0, 0);
                    ctx[db] = __builtin_amdgcn_mfma_i32_32x32x32_i8(vf, bias, ctx[db], 0, 0, 0);
                }
            }
        }
        // the waves' integer sums meet; each finishes 8 / split groups of four registers
#pragma unroll
        for (int i = 0; i < 8; ++i)
            sCtx[(x.wave * 8 + i) * 64 + x.lane] = v4i{ctx[i >> 2][4 * (i & 3)], ctx[i >> 2][4 * (i & 3) + 1], ctx[i >> 2][4 * (i & 3) + 2], ctx[i >> 2][4 * (i & 3) + 3]};
        meet();
        if (on) {
            const uint32_t orow = obase + static_cast<uint32_t>(q_row * a.ldo);
            for (int i = w; i < 8; i += split) {
                v4i c = {0, 0, 0, 0};
                for (int k = 0; k < split; ++k) c += sCtx[((block * split + k) * 8 + i) * 64 + x.lane];
                const int d = 32 * (i >> 2) + 8 * (i & 3) + 4 * h;
                const float4 o = make_float4(static_cast<float>(c.x) * a.scale2, static_cast<float>(c.y) * a.scale2, static_cast<float>(c.z) * a.scale2,
                                             static_cast<float>(c.w) * a.scale2);
                if (a.fq_o.levels) publish4(out, orow + d, levels4(a.fq_o, o));
                else publish16f(out, 4u * (orow + d), o);
            }
        }
        u += x.n_wg;
        if (u < s.units) meet();
    } while (u < s.units);
}

// Softmax of rows longer than kPlainSoftmax: eight waves for 32 queries, up to two tiles of keys a wave.  A tile's keys are the operand
// of one wave, so they come straight from memory, and its values go through LDS of the wave's own for their transposition: nothing
// of either is waited for together.  A workgroup's units lie one behind the other, so that most of them find keys and values where
// the unit before left them, and their queries are requested a unit ahead.  (With keys and values of a head in LDS for all waves,
// requested by all of them for every unit, staging was 2.3 of a unit's 8.4 us at 512 keys, and the waves met six times, now three:
// an encoder of 6 layers x 3 x 512 tokens took 592 us with 256 workgroups and 1387 with 64, and takes 563 and 1248.  At 128 keys, where
// a workgroup has one unit and half of its waves a tile, staging by all eight is the faster: 7.0 us a step, 7.8 so.)
__device__ __forceinline__ void attention_long(const ProgAttention& s, Ctx& x, lds_ptr lds) {
    typedef __attribute__((address_space(3))) float* lds_f32;
    typedef float v4f __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) v4f* lds_v4f;
    constexpr int kTiles = 2, kPitch = 32 * kTiles + 16, kValues = 64 * kPitch + 32;      // of a wave: values, transposed
    constexpr int kMaskAt = 8 * kValues, kMaxAt = kMaskAt + 8 * kTiles * 128, kSumAt = kMaxAt + 8 * 128, kCtxAt = kSumAt + 8 * 1024;
    static_assert(kCtxAt + 64 * 1024 <= kPartBytes + kKoffBytes, "LDS");
    const AttentionArgs& a = s.a;
    const int S = s.S, nt = S / 32, w = x.wave;
    const lds_ptr sVT = lds + w * kValues;                              // (every 16 rows 16 bytes on: no two of a wave's words in one bank)
    const lds_f32 sMask = (lds_f32)(lds + kMaskAt) + w * 32 * kTiles, sMax = (lds_f32)(lds + kMaxAt);
    const lds_v4i sCtx = (lds_v4i)(lds + kCtxAt);                       // [wave][8 groups of 4 registers][64]
    const Buffer qb = make_buffer(x.place(s.q)), kb = make_buffer(x.place(s.k)), vb = make_buffer(x.place(s.v)), out = make_buffer(x.place(s.out));
    const float* mask = s.has_mask ? reinterpret_cast<const float*>(x.place(s.mask)) : nullptr;
    const uint32_t units = static_cast<uint32_t>(s.units);
    int u = static_cast<int>((static_cast<uint32_t>(x.rank) * units) >> x.wg_shift);
    const int end = static_cast<int>((static_cast<uint32_t>(x.rank + 1) * units) >> x.wg_shift);
    v4i kf[kTiles][2], qf[2];
    // (element, head, first query) of a unit: divisions, so they are done a unit ahead
    auto place = [&](int unit, int& eh, int& n, int& hd, int& q0) {
        eh = unit / s.parts;
        n = eh / s.heads;
        hd = eh - n * s.heads;
        q0 = 32 * (unit - eh * s.parts);
    };
    int eh, n, hd, q0, have = -1;             // (have: whose keys and values are held)
    place(min(u, s.units - 1), eh, n, hd, q0);
    do {
        int lane = x.lane;
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile("" : "+v"(lane));       // (its functions are not kept in registers around the loop)
#endif
        const int l32 = lane & 31, h = lane >> 5;
        auto load_queries = [&] {
            const uint32_t row = static_cast<uint32_t>(n * a.oq + hd * a.sq) + static_cast<uint32_t>((q0 + l32) * a.ldq + 16 * h);
#pragma unroll
            for (int i = 0; i < 2; ++i) qf[i] = shared16(qb, row + 32 * i);
        };
        const bool fresh = eh != have;
        const uint32_t orow = static_cast<uint32_t>(n * a.oo + hd * a.so) + static_cast<uint32_t>((q0 + l32) * a.ldo);
        const uint32_t krow = static_cast<uint32_t>(n * a.ok + hd * a.sk) + static_cast<uint32_t>(l32 * a.ldk + 16 * h);
        const uint32_t vrow = static_cast<uint32_t>(n * a.ov + hd * a.sv) + static_cast<uint32_t>(8 * (lane >> 4) * a.ldv + 4 * (lane & 15));
        float mk = 0.f;
        if (fresh && mask) mk = mask[n * a.mask_outer + hd * a.mask_inner + min(32 * (w + 8 * h) + l32, S - 1)];
        if (have < 0) {
            x.wait();
            if (u >= end) return;
            load_queries();
        }
        have = eh;
        // a tile's keys, and its values as 4 keys x 4 d: everything is requested before any of it is used
        uint32_t vw[kTiles][2][4];
        if (fresh) {
#pragma unroll
            for (int j = 0; j < kTiles; ++j) {
                const int t = w + 8 * j;
                if (t >= nt) continue;
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) kf[j][ks] = shared16(kb, krow + static_cast<uint32_t>(32 * t * a.ldk + 32 * ks));
            }
#pragma unroll
            for (int j = 0; j < kTiles; ++j) {
                const int t = w + 8 * j;
                if (t >= nt) continue;
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        vw[j][i][q] = shared4(vb, vrow + static_cast<uint32_t>((32 * t + 4 * i + q) * a.ldv));
            }
            if (mask) sMask[32 * h + l32] = mk;
        }
        // the scores of this wave's tiles and their maximum
        float v[kTiles][16];
        float m = -INFINITY;
#pragma unroll
        for (int j = 0; j < kTiles; ++j) {
            const int t = w + 8 * j;
            if (t >= nt) continue;
            v16i acc = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf[j][ks], qf[ks], acc, 0, 0, 0);
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                v4f mg = {0.f, 0.f, 0.f, 0.f};
                if (s.has_mask) mg = *(lds_v4f)(sMask + 32 * j + 8 * g + 4 * h);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float y = static_cast<float>(acc[4 * g + r]) * a.scale1;
                    if (s.has_mask) y = y + mg[r];
                    v[j][4 * g + r] = y;
                    m = fmaxf(m, y);
                }
            }
        }
        if (u + 1 < end) {
            place(u + 1, eh, n, hd, q0);
            load_queries();
        }
        if (fresh) {
#pragma unroll
            for (int j = 0; j < kTiles; ++j) {
                if (w + 8 * j >= nt) continue;
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    uint32_t t[4];
                    transpose_bytes(vw[j][i][0], vw[j][i][1], vw[j][i][2], vw[j][i][3], t);
                    const int d = 4 * (lane & 15);      // (keys in the order in which their scores leave the matrix unit)
#pragma unroll
                    for (int q = 0; q < 4; ++q) *(lds_i32)(sVT + (d + q) * kPitch + 16 * (d >> 4) + 32 * j + 16 * i + 4 * (lane >> 4)) = static_cast<int32_t>(t[q]);
                }
            }
        }
        m = fmaxf(m, __shfl_xor(m, 32, 64));
        sMax[w * 32 + l32] = m;                     // (the same in both halves of the wave)
        meet();
#pragma unroll
        for (int k = 0; k < 8; ++k) m = fmaxf(m, sMax[k * 32 + l32]);
        // exponentials, their sums of four, and the tree over them of the stand-alone Softmax, whose first level, tiles t and t + 8, is
        // within a wave
        float e4[kTiles][4] = {};
#pragma unroll
        for (int j = 0; j < kTiles; ++j) {
            if (w + 8 * j >= nt) continue;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
#pragma unroll
                for (int r = 4 * g; r < 4 * g + 4; ++r) v[j][r] = expf(v[j][r] - m);
                e4[j][g] = (v[j][4 * g] + v[j][4 * g + 1]) + (v[j][4 * g + 2] + v[j][4 * g + 3]);
            }
        }
        const lds_v4f sSum = (lds_v4f)(lds + kSumAt) + lane;
        v4f p8[8];
        sSum[w * 64] = v4f{e4[0][0] + e4[1][0], e4[0][1] + e4[1][1], e4[0][2] + e4[1][2], e4[0][3] + e4[1][3]};
        meet();
#pragma unroll
        for (int t = 0; t < 8; ++t) p8[t] = sSum[t * 64];
#pragma unroll
        for (int o = 4; o > 0; o >>= 1)
#pragma unroll
            for (int t = 0; t < o; ++t)
#pragma unroll
                for (int g = 0; g < 4; ++g) p8[t][g] = p8[t][g] + p8[t + o][g];
        float sum = (p8[0][0] + p8[0][2]) + (p8[0][1] + p8[0][3]);
        sum += __shfl_xor(sum, 32, 64);
        const float inv = 1.0f / sum;
        // probabilities -> levels -> this wave's part of the second product
        v16i ctx[2] = {{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}, {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}};
#pragma unroll
        for (int j = 0; j < kTiles; ++j) {
            const int t = w + 8 * j;
            if (t >= nt) continue;
            v4i pf = {0, 0, 0, 0};
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                float p[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) p[r] = quotient(v[j][4 * g + r], sum, inv);
                pf[g] = static_cast<int>(prob_levels4<true, 0>(a, p[0], p[1], p[2], p[3]));
            }
            // u8 probabilities q are stored as q - 128: the 128 that is missing from each, as twice 64
            const int n64 = a.p_bias ? 0x40404040 : 0;
            const v4i bias = {n64, n64, n64, n64};
#pragma unroll
            for (int db = 0; db < 2; ++db) {
                const v4i vf = *(lds_v4i)(sVT + (32 * db + l32) * kPitch + 16 * (2 * db + (l32 >> 4)) + 32 * j + 16 * h);
                ctx[db] = __builtin_amdgcn_mfma_i32_32x32x32_i8(vf, pf, ctx[db], 0, 0, 0);
                if (a.p_bias) {
                    ctx[db] = __builtin_amdgcn_mfma_i32_32x32x32_i8(vf, bias, ctx[db], 0, 0, 0);
                    ctx[db] = __builtin_amdgcn_mfma_i32_32x32x32_i8(vf, bias, ctx[db], 0, 0, 0);
                }
            }
        }
        // the waves' integer sums meet; each finishes one of eight groups of four registers
#pragma unroll
        for (int i = 0; i < 8; ++i)
            sCtx[(w * 8 + i) * 64 + lane] = v4i{ctx[i >> 2][4 * (i & 3)], ctx[i >> 2][4 * (i & 3) + 1], ctx[i >> 2][4 * (i & 3) + 2], ctx[i >> 2][4 * (i & 3) + 3]};
        meet();
        v4i c = {0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < 8; ++k) c += sCtx[(k * 8 + w) * 64 + lane];
        const int d = 32 * (w >> 2) + 8 * (w & 3) + 4 * h;
        const float4 o = make_float4(static_cast<float>(c.x) * a.scale2, static_cast<float>(c.y) * a.scale2, static_cast<float>(c.z) * a.scale2,
                                     static_cast<float>(c.w) * a.scale2);
        if (a.fq_o.levels) publish4(out, orow + d, levels4(a.fq_o, o));
        else publish16f(out, 4u * (orow + d), o);
        // (the next unit's maxima, sums and partial sums are written behind meetings that the readers of this one's have passed as well)
    } while (++u < end);
}

// ---- the program ------------------------------------------------------------------------------------------------------------
// Three kernels, for networks over feature maps, for encoders, and for graphs with steps of both: every kind of step adds to the
// registers of all others.  The 4 x 4 tiles ask for 250 and more vector registers, none is spilled to memory; 309, 278 and 556
// scalar registers of the many step kinds are kept in lanes of vector registers.  The kernel with all kinds has no registers left for
// 4 x 4 tiles (with them it spills); its convolutions take smaller ones (an encoder layer of 96 tokens beside a ResNet-50 of width
// 16 at 64 x 64: 244 us, 467 by steps; beside a MobileNetV2 of 2 x 96 x 96 208 and 512).  A new step kind belongs into a kernel of its own where it
// needs more than they have.
template <bool MAPS, bool ROWS>
__global__ __launch_bounds__(kProgramThreads, 1) void program_kernel(const ProgArgs g) {
    extern __shared__ __attribute__((aligned(16))) int8_t smem[];
    lds_ptr lds = (lds_ptr)smem;
    lds_i32 flag = (lds_i32)(lds + kPartBytes + kKoffBytes);
    Ctx x;
    x.tid = threadIdx.x;
    x.lane = x.tid & 63;
    x.wave = __builtin_amdgcn_readfirstlane(x.tid >> 6);
    x.n_wg = g.workgroups;
    x.wg_shift = __builtin_ctz(x.n_wg);
    x.steps = g.steps;
    x.words = x.load_words(0, 0);
    x.words2 = x.load_words(0, 1);
    x.bases = reinterpret_cast<const uint32_t*>(g.bases)[min(x.lane, 2 * (1 + kProgramIo) - 1)];
    for (int i = x.tid; i < kMaxPieces; i += kProgramThreads) ((lds_i32)(lds + kPlainAt))[i] = 16 * i;
    x.rank = static_cast<int>(blockIdx.x % 8) * (x.n_wg / 8) + static_cast<int>(blockIdx.x / 8);
    x.xcds = g.control;
    x.own = x.xcds + kXcdWords * (blockIdx.x % 8);
    x.target = (g.launch * static_cast<uint32_t>(g.n_steps + 1) + 1) * static_cast<uint32_t>(x.n_wg / 8);      // a launch: the roll call and n_steps arrivals
    x.started = true;
    x.dead = false;
    x.flag = flag;
    if (!x.roll_call(g.roll_call_ticks)) return;
    for (int step = 0; step < g.n_steps; ++step) {
        // the thread's place is derived again in every step: as loop invariants its many functions (row, piece, quad ... of every
        // kind of step) would live in registers across all of them, and be moved out of the way and back around the large tiles
        int lane = lane_index();
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile("" : "+v"(lane));
#endif
        x.lane = lane;
        x.tid = 64 * x.wave + lane;
        const StepPtr words = step_ptr(g.steps, step);
        const int kind = static_cast<int>(word_of(x.words, 0));
        if (kind != PK_CONV && kind != PK_DW && kind != PK_EXPAND_DW && kind != PK_MVN && kind != PK_ATTENTION) x.wait();      // (those wait when they have prepared)
        switch (kind) {
        case PK_CONV: {
            switch (PROG_FIELD(x.words, a) * 8 + PROG_FIELD(x.words, b) + (PROG_FIELD(x.words, nk2) ? 64 : 0)) {
            case 8 + 1: conv_tiles<ROWS, 1, 1>(x, lds); break;
            case 16 + 1: conv_tiles<ROWS, 2, 1>(x, lds); break;
            case 16 + 2: conv_tiles<ROWS, 2, 2>(x, lds); break;
            case 32 + 2: conv_tiles<ROWS, 4, 2>(x, lds); break;
            case 64 + 16 + 2:
                if constexpr (MAPS) conv_tiles<ROWS, 2, 2, true>(x, lds);
                break;
            case 64 + 16 + 4:
                if constexpr (MAPS) conv_tiles<ROWS, 2, 4, true>(x, lds);
                break;
            default:
                if constexpr (!(MAPS && ROWS)) conv_tiles<ROWS, 4, 4>(x, lds);      // (choose_tile)
                break;
            }
            break;
        }
        case PK_ENTRY: entry_items(unpack<ProgEntry>(words), x); break;
        case PK_EXIT: {
            const ProgExit e = unpack<ProgExit>(words);
            if (e.in_dtype == HIPIE_F32) exit_items<float>(e, x);
            else if (e.in_dtype == HIPIE_I32) exit_items<int32_t>(e, x);
            else exit_items<int8_t>(e, x);
            break;
        }
        case PK_FQROWS: fq_items(unpack<ProgRows>(words), x); break;
        case PK_COPY: copy_items(unpack<ProgRows>(words), x); break;
        default:
            if constexpr (ROWS) {
                if (kind == PK_EMBED) embed_rows(unpack<ProgEmbed>(words), x);
                else if (kind == PK_MVN) mvn_rows(unpack<ProgMvn>(words), x);
                else if (!MAPS || kind == PK_ATTENTION) {
                    const ProgAttention t = unpack<ProgAttention>(words);
                    if (t.S > kPlainSoftmax) attention_long(t, x, lds);
                    else if (t.pform == 2) attention_units<2>(t, x, lds);
                    else attention_units<0>(t, x, lds);
                }
            }
            if constexpr (!MAPS) break;
            else if (kind == PK_DW) {
                switch (PROG_FIELD(x.words, stride) * 8 + PROG_FIELD(x.words, group)) {
                case 8 + 1: dw_items<1, 1>(x); break;
                case 8 + 4: dw_items<1, 4>(x); break;
                case 16 + 1: dw_items<2, 1>(x); break;
                default: dw_items<2, 4>(x); break;
                }
            } else if (kind == PK_EXPAND_DW) {
                if (PROG_FIELD(x.words, a) == 1) expand_depthwise<1>(x, lds);
                else expand_depthwise<2>(x, lds);
            } else if (kind == PK_MAXPOOL) max_pool_items(unpack<ProgPool>(words), x);
            else if (!ROWS || kind == PK_AVGPOOL) avg_pool_items(unpack<ProgPool>(words), x);
        }
        const int next = min(step + 1, g.n_steps - 1);       // (behind the last step nothing is prepared)
        {   // the next step's descriptor into the scalar cache: its eight lines asked for together, beside the stores' way to memory
            // (one behind the other they took 0.7 us of every step)
            const StepPtr n = step_ptr(g.steps, next);
            static_assert(kProgramStepWords == 128, "eight lines of 64 bytes");
            asm volatile("" ::"s"(n[0]), "s"(n[16]), "s"(n[32]), "s"(n[48]), "s"(n[64]), "s"(n[80]), "s"(n[96]), "s"(n[112]));
        }
        x.arrive(next);
        if (x.dead) return;
    }
    x.finish();
}

// constant weights [OCp][Kp] in the per-layer kernels' row order -> fragments of the tile kernel: for every tile of 16 A
// channels and every K step of 64 bytes A fragments, lane l's 16 bytes = channel 16 A tile + A (l % 16) + a, K bytes 16 (l / 16) on
__global__ __launch_bounds__(256) void pack_fragments_kernel(const int8_t* __restrict__ w, int8_t* __restrict__ f, int A, int OCp, int Kp, int64_t pieces) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= pieces) return;
    const int l = static_cast<int>(i & 63), nk = Kp / 64;
    const int64_t fr = i >> 6;
    const int a = static_cast<int>(fr % A), k = static_cast<int>(fr / A % nk), ot = static_cast<int>(fr / A / nk);
    const int oc = ot * 16 * A + A * (l & 15) + a;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (oc < OCp) {
        const int e = oc & 63;
        const int row = (oc & ~63) + 32 * ((e >> 4) & 1) + 8 * ((e >> 2) & 3) + 4 * (e >> 5) + (e & 3);
        v = *reinterpret_cast<const uint4*>(w + static_cast<int64_t>(row) * Kp + 64 * k + 16 * (l >> 4));
    }
    reinterpret_cast<uint4*>(f)[i] = v;
}

__global__ void clear_words(uint32_t* p, int n) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) p[i] = 0;
}

// Tile shape of a convolution step, by the clocks its busiest compute unit takes.  The constants are fitted, not derived: to
// the time of whole networks with one class of layers at a time in each of the shapes (ResNet-50, MobileNetV2, encoders and the
// convolution block, at 64, 128 and 256 workgroups), so that the choice loses as little as possible against the best shape of
// every class: summed over a network's classes, 167 in all, 0 - 5 % of its time, most of which is what the best of many noisy
// medians lies too low (the kernel as it is; the columns of Gelu that all waves share are not in the model).  Of the other shapes that were measured (1 x 2, 1 x 4, 2 x 4 of fragments) none is the best of a class by
// more than the runs differ.
// What the terms stand for: a load of 1 KB on a unit's path, a matrix instruction, a round trip to memory per filled ring, the
// f32 chain per value, a store instruction, the partial sums of the waves that share a K in LDS.  Rounds are tiles a wave takes
// one after another.
struct TileChoice { int a, b, ks; };
TileChoice choose_tile(int workgroups, int oc, int64_t pixels, int nk, int nk2, bool gelu, bool mixed) {
    static constexpr int kShapes[6][2] = {{4, 4}, {4, 2}, {2, 2}, {2, 1}, {1, 1}, {2, 4}};
    TileChoice best{4, 2, 1};
    double best_t = 1e30;
    for (const auto& shape : kShapes)
        for (int ks : {1, 2, 4, 8}) {
            const int a = shape[0], b = shape[1];
            if ((nk2 && (a != 2 || b < 2)) || (gelu && a == 1) || (b == 4 && (ks == 8 || (a == 2 && !nk2) || (a == 4 && mixed)))) continue;
            const int depth = a * b >= 16 ? 2 : (a * b >= 8 ? 4 : 6);
            const int64_t tiles = ceil_div(oc, 16 * a) * ceil_div(pixels, 16 * b), per_wg = ceil_div(tiles, workgroups);
            const int64_t rounds = ceil_div(per_wg, 8 / ks);
            const double waves = std::min<double>(8.0, static_cast<double>(per_wg) * ks / static_cast<double>(rounds));   // of a workgroup, busy
            auto loop = [&](int steps) {
                const double n = static_cast<double>(ceil_div(steps, ks));
                const double rate = std::max(waves * (a + b) * 11.4, std::max(1.0, waves / 4.0) * a * b * 14.6 + 2.7);
                return std::max(n * rate, std::ceil(n / depth) * 431.0) + 1368.0;
            };
            // a wave finishes whole columns of four pixels a lane, or one of the four
            const double rows = 4 * b <= ks ? 1.0 : 4.0, columns = std::max(1.0, std::ceil(static_cast<double>(b) / ks));
            const double writers = waves / ks * std::min(ks, rows == 1.0 ? 4 * b : b);
            const double chain = (gelu ? 74.3 : 2.6) * rows * a + 376.0;
            const double epi = columns * (chain * std::max(5.8, writers) + rows * 10.6 * writers);
            const double meet = ks > 1 ? 354.0 + 67.6 * (waves * a * b / 8.0 + ks * a * columns * rows / 4.0) : 0.0;
            const double t = static_cast<double>(rounds) * (loop(nk) + (nk2 ? loop(nk2) : 0.0) + epi + meet + 1224.0) + 248.0 * static_cast<double>(rounds - 1);
            if (t < best_t) {
                best_t = t;
                best = {a, b, ks};
            }
        }
    return best;
}

// What is in flight on a device, of all plans: how many requests were started and not yet waited for, and how many compute
// units their programs hold.
struct DeviceLoad {
    std::mutex lock;
    int requests = 0, units = 0;
    int together = 0, hold = 0;      // the most requests in flight when one of the last kHold was started
    static constexpr int kHold = 16;
};
DeviceLoad& device_load(int device) {
    static DeviceLoad loads[64];
    return loads[device & 63];
}

}  // namespace

ProgRef ProgBuilder::ref(const void* p) {
    const uint64_t v = reinterpret_cast<uintptr_t>(p), io = uint64_t(1) << 44, ar = uint64_t(1) << 32;
    int32_t base = 0;
    uint64_t off = v - ar;
    if (v >= io - (uint64_t(1) << 39)) {
        const uint64_t k = (v - io + (uint64_t(1) << 39)) >> 40;
        base = 1 + static_cast<int32_t>(k);
        off = v - io - (k << 40);
    }
    return {base, static_cast<uint32_t>(off), static_cast<uint32_t>(off >> 32)};
}

namespace {
// the bytes from a tensor's first element to behind its last
int64_t span_of(const hipie_tensor& t) {
    const int64_t esize = t.dtype == HIPIE_F32 || t.dtype == HIPIE_I32 ? 4 : 1;
    return ((t.n - 1) * t.stride_n + (t.h - 1) * t.stride_h + (t.w - 1) * t.stride_w + t.c) * esize;
}
}  // namespace

void ProgBuilder::writes(const void* p, int64_t bytes) { writing.push_back({static_cast<const uint8_t*>(p), bytes}); }

bool ProgBuilder::was_just_written(const void* p, const hipie_tensor& t) const {
    const uint8_t* at = static_cast<const uint8_t*>(p);
    const int64_t bytes = span_of(t);
    for (const auto& w : written)
        if (at < w.first + w.second && w.first < at + bytes) return true;
    return false;
}

ProgPtr ProgBuilder::keep(const void* host, size_t bytes) {
    owned.emplace_back();
    owned.back().upload(device, host, bytes);
    return ptr(owned.back().ptr);
}

// the channel tables that a layer's flags ask for, in load_constants' order
ProgPtr ProgBuilder::constants(const ConvArgs& a) {
    const uint32_t fl = a.flags;
    std::vector<const void*> rows{a.corr};
    if (fl & CF_BIAS) rows.push_back(a.bias);
    if (fl & CF_SCALE) rows.push_back(a.scale);
    if (fl & CF_RES_MUL) rows.push_back(a.res_mul);
    if (fl & CF_OUT_FQ) {
        rows.push_back(a.fq_r);
        rows.push_back((fl & CF_FQ_DIV2) ? a.fq_r2 : a.fq_d);
        if (!(fl & CF_FQ_SAT)) rows.push_back(a.fq_ih);
        if (!(fl & CF_FQ_IL0)) rows.push_back(a.fq_il);
    }
    return gather(rows, static_cast<size_t>(a.OCp) * 4);
}

ProgPtr ProgBuilder::fragments(const int8_t* w, int o_tiles, int A, int OCp, int Kp) {
    owned.emplace_back();
    const int64_t pieces = static_cast<int64_t>(o_tiles) * A * Kp;        // 16 A x Kp bytes per tile, 16 bytes a piece
    owned.back().alloc(device, static_cast<size_t>(pieces) * 16);
    hipLaunchKernelGGL(pack_fragments_kernel, dim3(static_cast<uint32_t>(ceil_div(pieces, 256))), dim3(256), 0, nullptr, w, owned.back().as<int8_t>(), A, OCp, Kp, pieces);
    HIPIE_CHECK_HIP(hipGetLastError());
    return ptr(owned.back().ptr);
}

// a depthwise layer's own fields; false: not a 3 x 3 layer that the kernel takes
bool ProgBuilder::depthwise(const ConvLaunch& l, ProgConv& c) {
    const ConvArgs& a = l.a;
    c.OH = a.OHOW / a.OW;
    c.OW = a.OW;
    if (l.kh != 3 || l.kw != 3 || l.dil_h != 1 || l.dil_w != 1 || a.conv_sh != a.conv_sw || a.conv_sh > 2 || !a.wgt2 || a.in_sw < a.out_sw) return false;
    c.kind = PK_DW;
    map_kinds = true;
    c.stride = a.conv_sh;
    c.wgt = ptr(a.wgt2);
    c.in_sn = a.in_sn; c.in_sh = a.in_sh * a.conv_sh; c.in_sw = a.in_sw; c.row_sh = a.in_sh;
    c.out_sn = a.out_sn; c.out_sh = a.out_sh; c.out_sw = a.out_sw;
    c.res_sn = a.res_sn; c.res_sh = a.res_sh; c.res_sw = a.res_sw;
    c.c4 = a.out_sw / 4;
    return true;
}

// what convolutions and depthwise layers have in common; false: the kernel does not take the layer
bool ProgBuilder::layer(const ConvArgs& a, const hipie_tensor& out, ProgConv& c) {
    if (a.M > (1 << 20) || a.koff_tile || (a.flags & CF_OUT_I32) || ((a.flags & CF_OUT_FQ) && !(a.flags & CF_FQ_RCP)) || (a.flags & (CF_RES_SUB | CF_POST_SCALE)))
        return false;
    const bool f32_out = !(a.flags & CF_OUT_FQ), f32_res = (a.flags & CF_RES_F32) != 0;
    for (int64_t bytes : {static_cast<int64_t>(out.n) * a.out_sn * (f32_out ? 4 : 1), static_cast<int64_t>(out.n) * a.res_sn * (f32_res ? 4 : 1)})
        if (bytes >= kBeyond) return false;
    c.in = ref(a.in + a.in_origin);
    c.out = ref(a.out);
    c.res = a.res ? ref(a.res) : ProgRef{-2, 0, 0};
    c.in2 = ProgRef{-2, 0, 0};
    c.out_limit = a.out_plane ? a.OC : a.out_sw;       // channels that the output holds
    c.res_limit = a.res_sw;
    c.constants = constants(a);
    c.flags = a.flags; c.lm1 = a.lm1; c.off_bytes = (static_cast<uint32_t>(static_cast<int>(a.out_off)) & 0xffu) * 0x01010101u; c.clamp_lo = a.clamp_lo; c.clamp_hi = a.clamp_hi;
    c.OCp = a.OCp;
    return true;
}

// Two layers as one step (expand_depthwise in this file), or false: they are two.  Where the kernel takes both layers one step is
// always the faster form (MobileNetV2 at batch 1, 2 and 4: 199, 207 and 221 us by two steps, 171, 183 and 204 by one).
// Channels per tile and rows per band are what gives a workgroup the fewest clocks; the times above move by less than 1 us where
// any of these constants is doubled or halved, as long as the units fit the workgroups in one round.
bool ProgBuilder::expand_depthwise(const hipie_conv* first, const hipie_tensor& in, const hipie_tensor& mid, const hipie_conv* second, const hipie_tensor& out, int fill) {
    ConvLaunch l1, l2;
    if (!conv_launch_arguments(first, in, nullptr, mid, l1) || !conv_launch_arguments(second, mid, nullptr, out, l2)) return false;
    const ConvArgs &a1 = l1.a, &a2 = l2.a;
    if (l1.depthwise || !l2.depthwise || a1.nk > kExpandSteps || !(a1.flags & CF_OUT_FQ) || !(a2.flags & CF_OUT_FQ) || ((a1.flags | a2.flags) & (CF_RES | CF_GELU))) return false;
    const int N = mid.n, H = mid.h, W = mid.w, OH = a2.OHOW / a2.OW, OW = a2.OW, S = a2.conv_sh;
    const int pw = std::max((OW - 1) * S + 3, W + l2.pad_left), channels = std::min(a1.out_sw, a2.out_sw);
    if (l2.pad_top > 2 || (OH - 1) * S - l2.pad_top >= H || channels % 16 != 0) return false;      // (every band has an input row)
    int best_a = 0, best_r = 0;
    double best = 1e30;
    for (int A : {1, 2})
        for (int R = 1; R <= OH; ++R) {
            const int64_t rows = (R - 1) * S + 3;
            if (rows * pw * 16 * A > kPartBytes) break;
            const int64_t units = ceil_div(channels, 16 * A) * N * ceil_div(OH, R), rounds = ceil_div(units, workgroups);
            const double frags = static_cast<double>(ceil_div(ceil_div(std::min<int64_t>(rows, H) * W, 16), 8)), items = static_cast<double>(ceil_div(R * OW * 4 * A, kProgramThreads));
            const double t = static_cast<double>(rounds) * (2500.0 + frags * (500.0 + 100.0 * A + 60.0 * A * a1.nk) + items * 1200.0);
            if (t < best) {
                best = t;
                best_a = A;
                best_r = R;
            }
        }
    if (!best_a) return false;
    ProgConv c{}, d{};
    if (!layer(a1, mid, c) || !layer(a2, out, d) || !depthwise(l2, d)) return false;
    const int64_t bands = ceil_div(OH, best_r), cts = ceil_div(channels, 16 * best_a), units = cts * N * bands;
    if (units * workgroups >= (1ll << 31) || units >= (1 << 24)) return false;
    c.kind = PK_EXPAND_DW;
    c.a = best_a;
    c.b = 1;
    c.tiles = static_cast<int32_t>(units);
    c.nk = a1.nk;
    if (!a1.k_linear) c.koff = ptr(a1.koff);
    c.wgt = fragments(a1.wgt, static_cast<int>(cts), best_a, a1.OCp, a1.Kp);
    std::vector<uint32_t> pix(static_cast<size_t>(a1.M));
    for (int64_t m = 0; m < a1.M; ++m) {
        const int64_t n = m / a1.OHOW, rem = m - n * a1.OHOW, y = rem / a1.OW, xx = rem - y * a1.OW;
        pix[static_cast<size_t>(m)] = static_cast<uint32_t>(n * a1.in_sn + y * a1.in_sh * a1.conv_sh + xx * a1.in_sw * a1.conv_sw);
    }
    c.pixels = keep(pix.data(), pix.size() * 4);
    ProgExpand& e = c.expand;
    e.stride = S; e.pad_top = l2.pad_top; e.pad_left = l2.pad_left;
    e.H = H; e.W = W; e.OH = OH; e.OW = OW;
    e.rows = best_r; e.bands = static_cast<int32_t>(bands); e.all_bands = static_cast<int32_t>(N * bands);
    e.patch_w = pw;
    e.fill = static_cast<int32_t>((static_cast<uint32_t>(fill) & 0xffu) * 0x01010101u);
    e.inv_W = 1.0f / static_cast<float>(W);
    e.inv_OW = 1.0f / static_cast<float>(OW);
    e.inv_bands = 1.0f / static_cast<float>(bands);
    e.inv_all_bands = 1.0f / static_cast<float>(N * bands);
    std::array<int32_t, kProgramStepWords> w{};
    std::memcpy(w.data(), &c, sizeof c);
    std::memcpy(w.data() + kProgramStepWords / 2, &d, sizeof d);
    writes(out.data, span_of(out));
    push(w);
    return true;
}

bool ProgBuilder::conv(const hipie_conv* conv, const hipie_tensor& in, const hipie_tensor* residual, const hipie_tensor& out, void* planes) {
    ConvLaunch l;
    if (!conv_launch_arguments(conv, in, residual, out, l)) return false;
    if (planes) planes_arguments(l.a, planes);
    const ConvArgs& a = l.a;
    const int64_t M = a.M;
    const bool f32_out = !(a.flags & CF_OUT_FQ), f32_res = (a.flags & CF_RES_F32) != 0;
    ProgConv c{};
    if (!layer(a, out, c)) return false;
    if (l.depthwise) {
        if (!depthwise(l, c)) return false;
        // four pixels a lane where a step has more values than that leaves lanes idle
        c.group = static_cast<int64_t>(out.n) * c.OH * a.OW * c.c4 <= static_cast<int64_t>(workgroups) * kProgramThreads ? 1 : 4;
        c.quads = static_cast<int32_t>(ceil_div(a.OW, c.group));
        const int64_t items = static_cast<int64_t>(out.n) * c.OH * c.quads * c.c4;
        if (items >= (1 << 24)) return false;
        c.items = static_cast<int32_t>(items);
        c.inv_c4 = 1.0f / static_cast<float>(c.c4);
        c.inv_quads = 1.0f / static_cast<float>(c.quads);
        c.inv_OH = 1.0f / static_cast<float>(c.OH);
        writes(out.data, span_of(out));
        add(c);
        return true;
    }
    c.kind = PK_CONV;
    // (a residual is loaded before the wait, so the step in front must not be the one that writes it: a step of no work goes between)
    if (a.res != nullptr && !(a.flags & CF_RES_GEMM) && was_just_written(a.res, *residual)) {
        ProgRows none{};
        none.kind = PK_COPY;
        none.in = none.out = ProgRef{0, 0, 0};
        add(none);
    }
    if (planes) c.out_sn = 4 * a.out_plane;
    c.nk = a.nk;
    const bool pair = (a.flags & CF_RES_GEMM) != 0;
    if (a.flags & CF_GELU) rows_kinds = true;
    if (pair) map_kinds = true;
    if (4 * a.nk > kMaxPieces || (pair && 4 * a.nk2 > kMaxPieces)) return false;
    const TileChoice t = choose_tile(workgroups, a.OC, M, a.nk, pair ? a.nk2 : 0, (a.flags & CF_GELU) != 0, mixed);
    c.a = t.a; c.b = t.b; c.ks_shift = __builtin_ctz(static_cast<unsigned>(t.ks));
    // (the channels the tensor is padded with are written too)
    const int o_tiles = static_cast<int>(ceil_div(std::min(c.out_limit, a.OCp), 16 * t.a));
    c.p_tiles = static_cast<int32_t>(ceil_div(M, 16 * t.b));
    c.inv_p_tiles = 1.0f / static_cast<float>(c.p_tiles);
    const int64_t tiles = static_cast<int64_t>(c.p_tiles) * o_tiles;
    if (tiles * workgroups >= (1ll << 31) || tiles >= (1 << 24) || static_cast<int64_t>(a.nk) * t.a * 1024 >= kBeyond) return false;
    c.tiles = static_cast<int32_t>(tiles);
    if (!(a.k_linear && (!pair || a.k_linear2))) c.koff = ptr(a.koff);       // (0: the kernel's own table, 16 i)
    c.wgt = fragments(a.wgt, o_tiles, t.a, a.OCp, a.Kp);
    if (pair) {
        c.in2 = ref(a.in2 + a.in2_origin);
        c.wgt2 = fragments(a.wgt2, o_tiles, t.a, a.OCp, a.Kp2);
        c.koff2 = ptr(a.koff2);
        c.nk2 = a.nk2;
        c.constants2 = gather({a.corr2, a.bias2, a.scale2}, static_cast<size_t>(a.OCp) * 4);
    }
    // where every pixel's window and results are; pixels behind the last one read where it does and store nowhere
    const int64_t pitch = static_cast<int64_t>(c.p_tiles) * 16 * t.b;
    c.M = static_cast<int32_t>(pitch);
    std::vector<uint32_t> pix(static_cast<size_t>(4 * pitch + 4));       // (a wave reads four entries from any of them)
    for (int64_t i = 0; i < pitch; ++i) {
        const int64_t m = std::min(i, M - 1), n = m / a.OHOW, rem = m - n * a.OHOW, oh = rem / a.OW, ow = rem - oh * a.OW;
        auto at = [&](int sn, int sh, int sw) { return static_cast<uint32_t>(n * sn + oh * sh + ow * sw); };
        pix[static_cast<size_t>(i)] = at(a.in_sn, a.in_sh * a.conv_sh, a.in_sw * a.conv_sw);
        pix[static_cast<size_t>(pitch + i)] = i < M ? at(a.out_sn, a.out_sh, a.out_sw) * (f32_out ? 4u : 1u) : static_cast<uint32_t>(kBeyond);
        pix[static_cast<size_t>(2 * pitch + i)] = at(a.res_sn, a.res_sh, a.res_sw) * (f32_res ? 4u : 1u);
        pix[static_cast<size_t>(3 * pitch + i)] = pair ? at(a.in2_sn, a.in2_sh * a.conv2_sh, a.in2_sw * a.conv2_sw) : 0u;
    }
    c.pixels = keep(pix.data(), pix.size() * 4);
    writes(out.data, span_of(out));
    add(c);
    return true;
}

// tables of `pitch` bytes behind one another in a buffer of the program's own
ProgPtr ProgBuilder::gather(const std::vector<const void*>& rows, size_t pitch) {
    owned.emplace_back();
    owned.back().alloc(device, rows.size() * pitch);
    for (size_t i = 0; i < rows.size(); ++i)
        HIPIE_CHECK_HIP(hipMemcpyAsync(owned.back().as<uint8_t>() + i * pitch, rows[i], pitch, hipMemcpyDeviceToDevice, nullptr));
    return ptr(owned.back().ptr);
}

bool ProgBuilder::entry(const hipie_fq* fq, bool u8_in, const void* in, const hipie_tensor& out) {
    FqLaunch f;
    if (!fq_launch_arguments(fq, out.dtype, f) || !f.rcp || out.c != f.channels) return false;
    const int64_t hw = static_cast<int64_t>(out.h) * out.w;
    if (hw >= (1 << 24) || out.stride_w % 4 != 0 || (out.stride_w > 4 && out.stride_w % 16 != 0) || static_cast<int64_t>(out.n) * out.stride_n >= kBeyond || out.n * hw * out.stride_w >= (1ll << 30)) return false;
    ProgEntry e{};
    e.kind = PK_ENTRY;
    e.N = out.n;
    e.u8_in = u8_in;
    e.C = out.c;
    e.cs = static_cast<int32_t>(out.stride_w);
    e.HW = static_cast<int32_t>(hw);
    e.W = out.w;
    e.inv_W = 1.0f / static_cast<float>(out.w);
    e.lm1 = f.lm1;
    e.off = f.off;
    e.out_sn = out.stride_n;
    e.out_sh = out.stride_h;
    e.in = ref(in);
    e.out = ref(out.data);
    e.tab = ptr(f.table);
    writes(out.data, span_of(out));
    add(e);
    return true;
}

bool ProgBuilder::pool(const PoolArgs& a, bool avg, bool rcp) {
    const int64_t span = static_cast<int64_t>(a.M / a.OHOW) * std::max<int64_t>(a.in_sn, 4ll * a.out_sn);
    if ((a.fq_il && !rcp) || static_cast<int64_t>(a.M) * a.cs >= (1ll << 30) || a.cs % 4 != 0 || span >= kBeyond) return false;
    ProgPool p{};
    p.kind = avg ? PK_AVGPOOL : PK_MAXPOOL;
    map_kinds = true;
    p.items = a.M * (a.cs / 4);
    const int OH = a.OHOW / a.OW;
    p.k3 = a.kh == 3 && a.kw == 3 && (OH - 1) * a.sh - a.pt + 3 <= a.H + a.pb && (a.OW - 1) * a.sw - a.pl + 3 <= a.W + a.pr;
    p.in = ref(a.in);
    p.out = ref(a.out);
    p.a = a;
    writes(a.out, static_cast<int64_t>(a.M / a.OHOW) * 4 * a.out_sn);
    add(p);
    return true;
}

bool ProgBuilder::exit(const ExitArgs& a, int in_dtype) {
    if (static_cast<int64_t>(a.N) * a.HW * a.C >= (1ll << 30) || static_cast<int64_t>(a.N) * a.in_sn * 4 >= kBeyond || a.in_sw % 4 != 0) return false;
    ProgExit e{};
    e.kind = PK_EXIT;
    e.in_dtype = in_dtype;
    e.in = ref(a.in);
    e.out = ref(a.out);
    e.a = a;
    add(e);
    return true;
}

bool ProgBuilder::embed(const float* table, int64_t vocab, int64_t hidden, const void* ids, int64_t tokens, int64_t seq, const float* add0, bool pos0,
                       const float* add1, bool pos1, void* out) {
    if (hidden % 4 != 0 || tokens * hidden * 4 >= kBeyond || seq >= (1 << 24)) return false;
    ProgEmbed e{};
    e.kind = PK_EMBED;
    rows_kinds = true;
    e.hidden = static_cast<int32_t>(hidden);
    e.seq = static_cast<int32_t>(seq);
    e.pos0 = pos0;
    e.pos1 = pos1;
    e.tokens = static_cast<int32_t>(tokens);
    e.vocab = vocab;
    e.ids = ref(ids);
    e.out = ref(out);
    e.table = ptr(table);
    e.add0 = ptr(add0);
    e.add1 = ptr(add1);
    writes(out, tokens * hidden * 4);
    add(e);
    return true;
}

bool ProgBuilder::mvn(const void* in, void* out, void* outq, int64_t rows, int64_t axis, bool normalize, float eps, bool eps_inside, const float* gamma,
                     const float* beta, const hipie_requant* rq) {
    if (rows * axis * 4 >= kBeyond || axis % 4 != 0 || axis > 256 * kMvnChunks) return false;
    ProgMvn m{};
    m.kind = PK_MVN;
    rows_kinds = true;
    m.axis = static_cast<int32_t>(axis);
    m.rows = static_cast<int32_t>(rows);
    m.normalize = normalize;
    m.eps_inside = eps_inside;
    m.eps = eps;
    m.in = ref(in);
    m.out = out ? ref(out) : ProgRef{-2, 0, 0};
    m.outq = outq ? ref(outq) : ProgRef{-2, 0, 0};
    m.gamma = ptr(gamma);
    m.beta = ptr(beta);
    if (outq) m.fq = make_requant(rq, "single-launch program");
    if (outq && !m.fq.rcp) return false;
    if (out) writes(out, rows * axis * 4);
    if (outq) writes(outq, rows * axis);
    add(m);
    return true;
}

bool ProgBuilder::attention(const hipie_attention* att, const void* const (&qkv)[3], const int64_t (&ld)[3], const int64_t (&inner)[3],
                           const int64_t (&outer)[3], void* out, int64_t ldo, int64_t so, int64_t oo, int batch, int batch_outer, const void* mask) {
    const AttentionArgs& proto = attention_prototype(att);
    if (!proto.p_div2 || (proto.fq_o.levels && !proto.fq_o.rcp)) return false;
    for (int i = 0; i < 3; ++i)
        if (batch_outer * outer[i] + batch * inner[i] + proto.S * ld[i] >= kBeyond) return false;
    if (4 * (batch_outer * oo + batch * so + proto.S * ldo) >= kBeyond) return false;
    if (proto.S > 512 || proto.S % 32 != 0 || proto.S < 32) return false;
    ProgAttention s{};
    s.kind = PK_ATTENTION;
    rows_kinds = true;
    s.S = proto.S;
    s.heads = batch;
    s.q = ref(qkv[0]); s.k = ref(qkv[1]); s.v = ref(qkv[2]);
    s.out = ref(out);
    s.has_mask = mask != nullptr;
    s.mask = mask ? ref(mask) : ProgRef{-2, 0, 0};
    s.pform = proto.p_sat ? 2 : 0;
    s.a = proto;
    s.a.ldq = ld[0]; s.a.sq = inner[0]; s.a.oq = outer[0];
    s.a.ldk = ld[1]; s.a.sk = inner[1]; s.a.ok = outer[1];
    s.a.ldv = ld[2]; s.a.sv = inner[2]; s.a.ov = outer[2];
    s.a.ldo = ldo; s.a.so = so; s.a.oo = oo;
    s.a.mask_inner = 0;
    s.a.mask_outer = proto.S;
    // Waves per 32 queries, by the clocks of a workgroup's round: staging, and the chain of a wave's tiles (from five waves on two
    // share a SIMD).  Against the best of the four splits the choice costs an encoder of two layers 0 - 2 % of its time (1 to 4
    // sequences of 32 to 384 keys, 64 and 256 workgroups; 6 % for 32 keys and 256, where one tile leaves nothing to share).  Longer
    // rows always take all eight (attention_long).
    const int qt = proto.S / 32;
    const int64_t elements = static_cast<int64_t>(batch_outer) * batch;
    double best = 1e30;
    if (proto.S > kPlainSoftmax) {
        best = 0.0;
        s.split_shift = 3;
        s.parts = qt;
        s.units = static_cast<int32_t>(elements * qt);
    } else for (int shift = 0; (1 << shift) <= kMostSplit; ++shift) {
        const int split = 1 << shift, blocks = std::min(kMostSplit / split, qt);
        const int64_t tiles = ceil_div(qt, split), parts = ceil_div(qt, kMostSplit / split), rounds = ceil_div(elements * parts, workgroups);
        if (tiles > kMostTiles || attention_lds(proto.S, split) > kPartBytes + kKoffBytes) continue;
        const double waves = static_cast<double>(blocks * std::min(split, qt));
        const double t = static_cast<double>(rounds) * (5000.0 + 4.0 * proto.S + std::max(1.0, waves / 5.0) * static_cast<double>(tiles) * 2400.0);
        if (t < best) {
            best = t;
            s.split_shift = shift;
            s.parts = static_cast<int32_t>(parts);
            s.units = static_cast<int32_t>(elements * parts);
        }
    }
    if (best >= 1e30) return false;
    writes(out, 4 * (batch_outer * oo + batch * so + proto.S * ldo));
    add(s);
    return true;
}

bool ProgBuilder::fq_rows(const hipie_fq* fq, const void* in, void* out, int out_dtype, int64_t n) {
    FqLaunch f;
    if (!fq_launch_arguments(fq, out_dtype, f) || !f.rcp || f.channels != 1 || n % 4 != 0 || 4 * n >= kBeyond / 2) return false;
    ProgRows r{};
    r.kind = PK_FQROWS;
    r.n = n;
    r.in = ref(in);
    r.out = ref(out);
    r.p = f.first;
    r.lm1 = f.lm1;
    r.off = f.off;
    writes(out, n);
    add(r);
    return true;
}

bool ProgBuilder::copy(const void* in, void* out, int64_t bytes) {
    if (bytes % 16 != 0 || bytes >= kBeyond / 2) return false;
    ProgRows r{};
    r.kind = PK_COPY;
    r.n = bytes;
    r.in = ref(in);
    r.out = ref(out);
    writes(out, bytes);
    add(r);
    return true;
}

Program::~Program() {
    if (report) (void)hipHostFree(report);
}

int Program::take_slot() {
    std::lock_guard<std::mutex> g(lock);
    for (int i = 0; i < kSlots; ++i)
        if (!((taken >> i) & 1)) {
            taken |= uint64_t(1) << i;
            report[16 * i] = 0;
            return i;
        }
    return -1;
}

void Program::give_slot(int slot) {
    std::lock_guard<std::mutex> g(lock);
    taken &= ~(uint64_t(1) << slot);
}

void Program::count(bool ran) {
    std::lock_guard<std::mutex> g(lock);
    if (ran) {
        ++done;
        penalty /= 2;
    } else {
        ++cancelled;
        penalty = std::min(4 * penalty + 4, kMostSkipped);
        skip = penalty;
    }
}

void Program::reset_counts() {
    std::lock_guard<std::mutex> g(lock);
    done = cancelled = 0;
    skip = penalty = 0;
}

std::string Program::counts() {
    std::lock_guard<std::mutex> g(lock);
    return std::to_string(done) + " " + std::to_string(cancelled);
}

size_t Program::device_bytes() const {
    size_t n = 0;
    for (const ProgramForm* f : {lone.get(), shared == lone ? nullptr : shared.get()})
        if (f) {
            n += f->steps.bytes;
            for (const auto& b : f->owned) n += b.bytes;
        }
    return n;
}

std::shared_ptr<ProgramForm> make_program_form(ProgBuilder&& b) {
    auto f = std::make_shared<ProgramForm>();
    f->workgroups = b.workgroups;
    f->n_steps = static_cast<int>(b.steps.size());
    f->maps = b.map_kinds;
    f->rows = b.rows_kinds;
    f->steps.upload(b.device, b.steps.data(), b.steps.size() * kProgramStepWords * 4);
    f->owned = std::move(b.owned);
    DeviceGuard g(b.device);
    HIPIE_CHECK_HIP(hipStreamSynchronize(nullptr));      // the repacking kernels
    return f;
}

std::shared_ptr<Program> make_program(int device) {
    auto p = std::make_shared<Program>();
    p->device = device;
    p->roll_call_ticks = kRollCallTicks;
    if (const char* ticks = std::getenv("HIPIE_ROLL_CALL_TICKS")) {      // (0: every launch is given up and runs again by steps)
        char* end = nullptr;
        const unsigned long n = std::strtoul(ticks, &end, 10);
        if (end != ticks && *end == 0) p->roll_call_ticks = static_cast<uint32_t>(std::min<unsigned long>(n, kMaxRollCallTicks));
    }
    HIPIE_CHECK_HIP(hipDeviceGetAttribute(&p->units, hipDeviceAttributeMultiprocessorCount, device));
    DeviceGuard g(device);
    HIPIE_CHECK_HIP(hipHostMalloc(reinterpret_cast<void**>(&p->report), Program::kSlots * 64, hipHostMallocDefault));
    std::memset(p->report, 0, Program::kSlots * 64);
    for (auto kernel : {&program_kernel<true, false>, &program_kernel<false, true>, &program_kernel<true, true>})
        HIPIE_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    return p;
}

int request_enters(int device) {
    DeviceLoad& d = device_load(device);
    std::lock_guard<std::mutex> g(d.lock);
    ++d.requests;
    if (d.requests >= d.together || --d.hold <= 0) {
        d.together = d.requests;
        d.hold = DeviceLoad::kHold;
    }
    return d.together;
}

void request_leaves(int device) {
    DeviceLoad& d = device_load(device);
    std::lock_guard<std::mutex> g(d.lock);
    --d.requests;
}

// A lone request takes the form that was fastest alone.  Beside others it takes the smaller one, if units are left for it
// (never more workgroups than compute units, so that all of them find a place), and else the steps, whose kernels share the
// device.  ResNet-50, batch 1, us a request with 2 and 4 in flight, two of the four on one hardware queue: steps 251 and 242, 64
// workgroups side by side 144 and 136 (alone: steps 493, 64 workgroups 274, 256 222).  With more than twice as many requests as find
// a place the ones by steps wait for the others: batch 3 with 128 workgroups, 4 in flight: 217, steps 254; 6 in flight: 242, steps
// 174 (batch 1, 64 workgroups beside others, 6 in flight: 118, steps 163).
const ProgramForm* Program::choose(int together) {
    const ProgramForm* f = together > 1 ? shared.get() : lone.get();
    if (!f || (lone != shared && together > 1 && together * f->workgroups > 2 * units)) return nullptr;
    std::lock_guard<std::mutex> g(lock);
    if (skip > 0) {
        --skip;
        return nullptr;
    }
    DeviceLoad& d = device_load(device);
    std::lock_guard<std::mutex> hold(d.lock);
    if (d.units + f->workgroups > units) return nullptr;
    d.units += f->workgroups;
    return f;
}

void Program::leave(const ProgramForm* f) {
    DeviceLoad& d = device_load(device);
    std::lock_guard<std::mutex> g(d.lock);
    d.units -= f->workgroups;
}

void launch_program(const Program& p, const ProgramForm& f, uint8_t* arena, void* const* io, int n_io, uint32_t* control, uint32_t launch, int slot,
                    hipStream_t s) {
    ProgArgs a{};
    a.steps = f.steps.as<int32_t>();
    a.bases[0] = arena;
    for (int i = 0; i < n_io; ++i) a.bases[1 + i] = io[i];
    a.control = control;
    a.report = p.report + 16 * slot;
    a.n_steps = f.n_steps;
    a.workgroups = f.workgroups;
    a.launch = launch;
    a.roll_call_ticks = p.roll_call_ticks;
    p.report[16 * slot] = 0;
    auto kernel = &program_kernel<true, false>;
    if (f.rows) kernel = f.maps ? &program_kernel<true, true> : &program_kernel<false, true>;
    hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(f.workgroups)), dim3(kProgramThreads), kLdsBytes, s, a);
    HIPIE_CHECK_HIP(hipGetLastError());
}

// The word is there 4.4 us before hipStreamSynchronize returns (a kernel of 64 workgroups that takes 10 us, launch to answer: 17.4 and
// 21.8 us), which waits for the kernel's end, its caches' write-back and a signal.  A launch that takes longer than kMostPolled is
// left to the runtime: the core has better things to do, and errors of the device are found there.
bool report_done(const Program& p, int slot) {
    constexpr auto kMostPolled = std::chrono::milliseconds(5);
    const uint32_t* word = p.report + 16 * slot;
    const auto t0 = std::chrono::steady_clock::now();
    for (uint32_t n = 1;; ++n) {
        const uint32_t v = __atomic_load_n(word, __ATOMIC_ACQUIRE);
        if (v != 0) return v == kReportDone;
        if (n % 256 == 0 && std::chrono::steady_clock::now() - t0 > kMostPolled) return false;
        __builtin_ia32_pause();
    }
}

bool program_failed(const Program& p, int slot, uint32_t* control, hipStream_t s) {
    const uint32_t v = __atomic_load_n(p.report + 16 * slot, __ATOMIC_ACQUIRE);
    if (v == kReportDone) return false;
    hipLaunchKernelGGL(clear_words, dim3(1), dim3(256), 0, s, control, static_cast<int>(kProgramControlBytes / 4));
    HIPIE_CHECK_HIP(hipGetLastError());
    return true;
}

}  // namespace hipie
