// A whole plan as ONE persistent kernel.
//
// What this is for: a request that somebody waits for.  As separate launches a batch-1 ResNet-50 is 54 dependent kernels
// at about 9 us each: 2.4 us of launch, then a cold start (arguments, descriptors, tables, operands from the memory-side
// cache - an XCD's L2 is written back and invalidated between kernels) in front of 1 - 2 us of work.  Here the workgroups
// stay, and a step ends in a barrier among them (Ctx::arrive; a step that only stores a dword a lane takes 1.8 us with 64
// workgroups, 1.9 with 128, 2.1 with 256).  The cold start disappears behind it, because a workgroup that has arrived prepares
// its next tile (offsets, weights, constants) before it waits, and the descriptor of the next step comes beside the stores.
//
// Coherence: the eight XCDs' L2 caches are not coherent with each other.  Every result is stored write-through with device
// scope (sc1), is awaited (s_waitcnt vmcnt(0)) in front of the barrier, and is loaded with device scope behind it; fences,
// which write back or invalidate a whole L2 each, are not needed.  Weights, tables and the caller's inputs, which nothing
// writes during the launch, are ordinary cached loads.
//
// Termination: a barrier needs every workgroup resident.  The roll call in front of the first step has a deadline: if the
// launch is not complete in time (other work holds the compute units), it is cancelled by compare-and-swap before it has
// written anything, the kernel drains, and the host runs the inference step by step, as it does with a growing number of the
// requests behind it (Program::count).  Later waits are bounded as well (all workgroups are resident by then, so they end; a
// bound that is hit ends the kernel and the host falls back the same way).  So the outputs are there when the host has waited,
// not before: the form is for inferences whose outputs nothing on the device reads earlier (plan.hip, start_request).
// Programs in flight together never ask for more compute units than there are (Program::choose).
#pragma once
#include <array>
#include <memory>
#include <mutex>
#include <string>

#include "attention.h"
#include "conv.h"
#include "pool.h"
#include "requant.h"

namespace hipie {

constexpr int kProgramThreads = 512;
constexpr int kProgramIo = 6;            // graph inputs + outputs a program can address
constexpr int kProgramStepWords = 128;

enum ProgKind : int32_t { PK_CONV, PK_DW, PK_ENTRY, PK_MAXPOOL, PK_AVGPOOL, PK_EXIT, PK_EMBED, PK_MVN, PK_ATTENTION, PK_FQROWS, PK_COPY, PK_EXPAND_DW };

// where an operand is: base 0 an arena offset, 1 + k an offset in the k-th input / output buffer of the call; < 0 absent
struct ProgRef {
    int32_t base;
    uint32_t lo, hi;
};
struct ProgPtr { uint32_t lo, hi; };   // a load-time buffer

// a convolution and the depthwise layer behind it: the map between them and the bands it is computed in
struct ProgExpand {
    int32_t stride, pad_top, pad_left;        // of the depthwise layer
    int32_t H, W, OH, OW;                     // of the map between the layers, of the result
    int32_t rows, bands, all_bands;           // result rows of a band, bands of an image, of all images
    int32_t patch_w, fill;                    // pixels of a patch row; four bytes of the padding's level
    float inv_W, inv_OW, inv_bands, inv_all_bands;
};
// convolution, weight MatMul (1 x 1 over rows) and depthwise 3 x 3
struct ProgConv {
    int32_t kind, a, b, ks_shift;     // oc fragments, pixel fragments of a wave's tile; log2 of the waves that share a tile's K
    int32_t p_tiles, tiles;           // pixel tiles; all tiles of the step
    float inv_p_tiles;
    ProgRef in, out, res, in2;         // `in` already moved to the first window's origin
    ProgPtr wgt, koff, constants;      
    ProgPtr wgt2, koff2, constants2;
    ProgPtr pixels;                    // four words a pixel: byte offsets of its window in `in` and `in2`, of itself in `out` and `res`
    int32_t nk, nk2, OCp, M;
    int32_t out_limit, res_limit;     // channels the tensors hold
    uint32_t flags;
    float lm1;
    uint32_t off_bytes;                // the level offset in every byte
    float clamp_lo, clamp_hi;
    union {
        struct {                       // depthwise
            int32_t stride, group, c4, quads, OH, OW, items;
            int32_t in_sn, in_sh, in_sw, row_sh, out_sn, out_sh, out_sw, res_sn, res_sh, res_sw;      // (dense: out_sn = bytes between the planes of f32 results, 0: channels innermost)
            float inv_c4, inv_quads, inv_OH;
        };
        ProgExpand expand;             // PK_EXPAND_DW, whose depthwise layer is a descriptor of its own behind this one
    };
};
struct ProgEntry {
    int32_t kind, u8_in, N, C, cs, HW, W;
    float inv_W, lm1, off;
    int64_t out_sn, out_sh;
    ProgRef in, out;
    ProgPtr tab;
};
struct ProgPool {
    int32_t kind, k3, items;
    ProgRef in, out;
    PoolArgs a;
};
struct ProgExit {
    int32_t kind, in_dtype;
    ProgRef in, out;
    ExitArgs a;
};
struct ProgEmbed {
    int32_t kind, hidden, seq, pos0, pos1, tokens;
    int64_t vocab;
    ProgRef ids, out;
    ProgPtr table, add0, add1;
};
struct ProgMvn {
    int32_t kind, axis, rows, normalize, eps_inside;
    float eps;
    ProgRef in, out, outq;             // base < 0: absent
    ProgPtr gamma, beta;
    Requant fq;
};
struct ProgAttention {
    int32_t kind, S, heads, units, split_shift, parts;   // log2 of the waves that share 32 queries, workgroups per (element, head)
    ProgRef q, k, v, out, mask;
    int32_t has_mask, pform;
    AttentionArgs a;
};
struct ProgRows {
    int32_t kind;
    int64_t n;                        // elements (PK_FQROWS) or bytes (PK_COPY), a multiple of 16 bytes read
    ProgRef in, out;
    FqChannel p;
    float lm1, off;
};

// Builds the step list while a plan is compiled.  Every method returns false when the single-launch form does not take
// the step (the plan then has no program).
struct ProgBuilder {
    int device = 0;
    int workgroups = 256;
    std::vector<std::array<int32_t, kProgramStepWords>> steps;
    std::vector<DeviceBuffer> owned;      // repacked weights, tables
    bool map_kinds = false, rows_kinds = false;      // steps of a network over feature maps, of an encoder: a kernel for each, and one for both
    bool mixed = false;                              // built for the latter
    ProgPtr keep(const void* host, size_t bytes);                              // a table of the program's own
    ProgPtr gather(const std::vector<const void*>& rows, size_t pitch);
    static uint8_t* fake_arena() { return reinterpret_cast<uint8_t*>(uintptr_t(1) << 32); }
    static uint8_t* fake_io(int k) { return reinterpret_cast<uint8_t*>(uintptr_t(1) << 44) + (uintptr_t(k) << 40); }
    static ProgRef ref(const void* p);     // of a pointer into one of the two
    static ProgPtr ptr(const void* p) { return {static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p)), static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p) >> 32)}; }
    template <typename T> void add(const T& s) {
        static_assert(sizeof(T) <= kProgramStepWords * 4 && sizeof(T) % 4 == 0, "step descriptor");
        std::array<int32_t, kProgramStepWords> w{};
        std::memcpy(w.data(), &s, sizeof(T));
        push(w);
    }
    void push(const std::array<int32_t, kProgramStepWords>& w) {
        steps.push_back(w);
        written = std::move(writing);
        writing.clear();
    }
    // what the step that is built writes in the arena (or may: no less), and what the last one did
    std::vector<std::pair<const uint8_t*, int64_t>> writing, written;
    void writes(const void* p, int64_t bytes);
    bool was_just_written(const void* p, const hipie_tensor& t) const;      // the tensor that begins at p
    // planes: the f32 results channel by channel at this address instead (conv_run_planes)
    bool conv(const hipie_conv* c, const hipie_tensor& in, const hipie_tensor* residual, const hipie_tensor& out, void* planes = nullptr);
    // a dense layer and the depthwise 3 x 3 layer that is its only reader; `fill`: the stored byte of the padding between them
    bool expand_depthwise(const hipie_conv* first, const hipie_tensor& in, const hipie_tensor& mid, const hipie_conv* second, const hipie_tensor& out, int fill);
    ProgPtr constants(const ConvArgs& a);
    ProgPtr fragments(const int8_t* w, int o_tiles, int A, int OCp, int Kp);
    bool layer(const ConvArgs& a, const hipie_tensor& out, ProgConv& c);
    bool depthwise(const ConvLaunch& l, ProgConv& c);
    bool entry(const hipie_fq* fq, bool u8_in, const void* in, const hipie_tensor& out);
    bool pool(const PoolArgs& a, bool avg, bool rcp);
    bool exit(const ExitArgs& a, int in_dtype);
    bool embed(const float* table, int64_t vocab, int64_t hidden, const void* ids, int64_t tokens, int64_t seq, const float* add0, bool pos0,
               const float* add1, bool pos1, void* out);
    bool mvn(const void* in, void* out, void* outq, int64_t rows, int64_t axis, bool normalize, float eps, bool eps_inside, const float* gamma,
             const float* beta, const hipie_requant* rq);
    bool attention(const hipie_attention* att, const void* const (&qkv)[3], const int64_t (&ld)[3], const int64_t (&inner)[3],
                   const int64_t (&outer)[3], void* out, int64_t ldo, int64_t so, int64_t oo, int batch, int batch_outer, const void* mask);
    bool fq_rows(const hipie_fq* fq, const void* in, void* out, int out_dtype, int64_t n);
    bool copy(const void* in, void* out, int64_t bytes);
};

// The step list of one size on the device, with its own packing of the dense layers' weights (the tile shapes depend on the
// size) and four words per output pixel of each: a second copy of the weights for the lone form, a third one where the shared
// form is another, and at load, while the sizes are measured, one more.
struct ProgramForm {
    int workgroups = 0, n_steps = 0;
    std::vector<int> inside;              // the plan's tensors that live inside a step
    bool maps = false, rows = false;         // which of the kernels
    DeviceBuffer steps;
    std::vector<DeviceBuffer> owned;
};
std::shared_ptr<ProgramForm> make_program_form(ProgBuilder&& b);

// A plan's program: its forms and the page-locked words the kernel reports failures in.
struct Program {
    int device = 0, units = 0;               // compute units the device has
    uint32_t roll_call_ticks = 0;
    std::shared_ptr<ProgramForm> lone;       // for a request that has the device to itself
    std::shared_ptr<ProgramForm> shared;     // beside other requests (may be the same one; null: those run by steps)
    static constexpr int kSlots = 64;        // requests of one plan that can use the program
    uint32_t* report = nullptr;              // page-locked, 16 dwords per slot
    std::mutex lock;
    uint64_t taken = 0;
    uint64_t done = 0, cancelled = 0;        // launches that ran to their end, launches that were given up
    // A launch that was given up cost its wait, and what held the compute units is likely still there: the next requests run
    // by steps, 4 of them, 20, 84 .. as launches go on failing; every launch that completes halves the number.
    static constexpr uint32_t kMostSkipped = 1024;
    uint32_t skip = 0, penalty = 0;
    ~Program();
    int take_slot();                         // -1: none left
    void give_slot(int slot);
    const ProgramForm* choose(int together); // the form that the next request takes, its compute units held; null: the steps
    void leave(const ProgramForm* f);        // gives them back: the stream has been waited for
    void count(bool ran);
    void reset_counts();
    std::string counts();                    // "done cancelled"
    size_t device_bytes() const;             // of its forms
};
std::shared_ptr<Program> make_program(int device);
// A request is started / has been waited for, by whatever form; the former gives how many were in flight together lately
int request_enters(int device);
void request_leaves(int device);

// barrier counters and the roll call's verdict: behind the arena, zero before the first launch.  A block counts the launches
// of one form, whose number of workgroups it adds up.
constexpr size_t kProgramControlBytes = 2048, kProgramControlBlocks = 2;
// `launch`: how many launches used this control block before; io: the call's input and output buffers in order
void launch_program(const Program& p, const ProgramForm& f, uint8_t* arena, void* const* io, int n_io, uint32_t* control, uint32_t launch, int slot,
                    hipStream_t s);
// looks at the slot's word until its launch is complete: true, and every result is in memory (its stream may still be draining).
// false: it was given up, or takes long; the stream is to be waited for
bool report_done(const Program& p, int slot);
// the stream of a slot's last launch has drained, or report_done was true: true if it did not run to its end, and `control` has
// been cleared on the stream (the caller runs the inference by steps and counts its launches from zero again)
bool program_failed(const Program& p, int slot, uint32_t* control, hipStream_t s);

}  // namespace hipie
