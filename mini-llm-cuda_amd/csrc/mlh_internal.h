// Internal declarations of the gfx950 device layer (not part of the C ABI).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>
#include <vector>

#include "mlh.h"
#include "rows.h"

#define MLH_KV_PAGE 64      // positions per KV page; equals the attention key tile
#define MLH_ATTN_WG_KEYS 256 // keys one attention workgroup covers (4 waves x one 64-key tile)
#define MLH_WAVE 64

typedef uint16_t bf16_t;
// IEEE half, as the MFMA path stores weights and activations of bf16 models (see MLH_GEMM_F16)
struct f16_t { uint16_t bits; };
#define MLH_GEMM_F16 2 // GEMM operand type code beside MLH_DTYPE_F32 / MLH_DTYPE_BF16
#define MLH_GEMM_P3 3  // ... and for fp32 operands stored as three bf16 planes (p3.h; models that spread further than halves reach)
#define MLH_GEMM_H2 4  // ... and fp32 as halves, pairs times triples, with an exponent per row (h2.h)
#define MLH_GEMM_WS_COUNTERS 1024 // tile counters at the head of a split-K workspace ...
#define MLH_GEMM_WS_PARTIALS (256 * 8 * 2 * 16 * 64) // ... and the partial sums (floats) behind them
#define MLH_SELFTEST_SWIGLU 0x100 // mlh_selftest_gemm: flag beside the operand type, selects the SwiGLU epilogue

// This wave's stores and atomics so far have reached the memory that other workgroups read, the memory side for agent-scope ones.  For
// what is published by a counter: each storing wave waits here, then the workgroup meets at a barrier, then one thread counts.  A release
// fence of workgroup scope is not that wait on this target: it orders the waves of one compute unit, and compiles to no wait for stores.
__device__ __forceinline__ void stores_landed() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// A value on its way into an IEEE half: finite ones saturate (an overflow must not become an infinity), infinities and NaN stay what they
// are.
__device__ __forceinline__ float half_range(float v) {
    const float s = __builtin_amdgcn_fmed3f(v, -65504.0f, 65504.0f);
    return __builtin_amdgcn_classf(v, 0x207) ? v : s; // either NaN, either infinity
}
__device__ __forceinline__ uint32_t pack_f16(float lo, float hi) { // two floats -> two IEEE halves (round to nearest even)
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, f16x2{(_Float16)lo, (_Float16)hi}); // (one instruction; put together from two halves it is three)
}
__device__ __forceinline__ uint32_t pack_half_range(float lo, float hi) { return pack_f16(half_range(lo), half_range(hi)); }
// The same from the conversion itself (FP16_OVFL of the wave's mode register), between halves_saturate(1) and (0): for an epilogue of nothing
// but conversions.  Matrix products must not run under it: they would take an infinite operand for 65504 and NaN for 0.
__device__ __forceinline__ void halves_saturate(int on) { __builtin_amdgcn_s_setreg(1 | 23 << 6, on); }

// Device-side description of one transformer block.
struct LayerDev {
    const void* Wa;       // fused first-phase matrix [rowsA, dim]: q|k|v|[g]|[pleGate]|[gdnA|gdnB]
    const void* Wo;       // [dim, ad]
    const void* W13;      // [2*ffnDim, dim], row 2i = gate row i, row 2i+1 = up row i
    const void* W2;       // [dim, ffnDim]
    const void* pleUp;    // [dim, pleDim]
    const void* pleTable; // [vocab, pleDim]
    const float* g1;      // rms1 gain
    const float* g2;      // rms2 gain
    const float* gq;      // per-head q gain [dim] (qkRmsNorm)
    const float* gk;
    const float* gdnBa;   // [gdnHeads]
    const float* gdnBb;
    float* K;             // KV page pools [numPages, MLH_KV_PAGE, dim]
    float* V;
    float* S;             // GDN states [maxSeqs, gdnHeads, dv, dk]
    int kind;
    int rowsA, offK, offV, offG, offPle, offGa, offGb;
    int ad;               // width of the mixing output fed to Wo
    // What the prefill's products multiply: fp32 matrices as triples of halves (h2.h) or as planes (p3.h); for bf16 models IEEE-half
    // mirrors scaled by a power of two (exact), with the inverse scale applied to the product.
    // WoP is [dim, ad + pleDim]: Wo with pleUp appended along K, so that h1 = [a | e] . WoP^T is one product.
    const void *WaP, *WoP, *W13P, *W2P;
    float sWa, sWo, sW13, sW2;
    const int *eWa, *eWo, *eW13, *eW2; // triples: exponents of their rows ...
    const int* eU;                     // ... and of the FFN units
    const void *WaR, *WoR, *W13R, *W2R; // for the row step: the matrices ([Wo | pleUp] as one) in its fetch order (rows.h)
};

// Arguments shared by all kernels of a decode step.
struct StepArgs {
    // model
    int dim, heads, hd, ffn, vocab, maxL, ple;
    int gdnHeads, gdnDk, gdnDv;
    int qkNorm, gating;
    // batch
    int nseq;             // active slots
    const int* sidx;      // slot -> sequence id
    const int* tok;       // per slot: token fed this step
    int* pos;             // per sequence: current length (position of the fed token)
    const int* pageTable; // [maxSeqs, pagesPerSeq]
    int pagesPerSeq;
    int nsplit;           // attention partials per (slot, head)
    // activations, indexed by slot
    float* x;             // [slots, dim] residual stream
    float* qkv;           // [slots, maxRowsA]
    int qkvStride;
    float* part;          // [slots, nsplit, heads, hd + 2] attention partials (m, l, acc)
    float* mix;           // [slots, maxAd] GDN read-out
    unsigned char* mixRows; // row step: if set, the mixing output and the PLE columns go straight into the planes the output
    RowsLayout mixLay;    //   projection multiplies (rows.h) instead of `mix` and `part`
    int wbytes;           // bytes per weight element (PLE table rows)
    float temperature;    // > 0: the next token is drawn from softmax(logits / temperature) instead of the argmax
    unsigned long long sampleSeed;
    float* h1;            // [slots, dim]
    float* u;             // [slots, ffn]
    float* logits;        // [maxSeqs, vocab] indexed by sequence id
    float* amaxVal;       // [slots, amaxParts]
    int* amaxIdx;
    int amaxParts;
    const float* rope;    // [maxL, hd]
    const void* E;        // [vocab, dim]
    const float* gF;
    int* nextTok;         // [maxSeqs] greedy pick per sequence id
    int* outIds;          // [maxSteps, slots]
    int* stepCounter;
    int outCapacity;
};

// Pinned host memory of a context (the device reads and writes it directly); grows when the context's stream is idle.
struct PinBuf {
    int* p = nullptr;
    size_t bytes = 0;
};

struct mlh_ctx {
    mlh_hparams hp;
    int device = 0;
    hipStream_t stream = nullptr;
    std::string err;
    bool finalized = false;
    int wbytes = 4; // bytes per matrix element

    std::vector<LayerDev> layers;
    std::vector<std::vector<char>> have; // [layer][tensor] uploaded flags
    bool haveE = false, haveGF = false, haveRope = false;
    std::vector<void*> allocs;

    void* E = nullptr;
    float* gF = nullptr;
    float* rope = nullptr;

    unsigned char* mixRows = nullptr; // see StepArgs::mixRows; set by the row step
    RowsLayout mixLay = {1, 1};
    void* rowsBuf = nullptr; // row step (kernels_rows.hip): planes of the residual rows x and h1, the mixing output and the FFN units, partial sums of squares
    unsigned char *rowsX = nullptr, *rowsH = nullptr, *rowsMix = nullptr, *rowsU = nullptr;
    float *rowsSsqX = nullptr, *rowsSsqH = nullptr;
    int pagesPerSeq = 0;
    int nsplit = 1;
    int maxRowsA = 0, maxAd = 0;
    int amaxParts = 0;
    int outCapacity = 0;

    int* d_sidx = nullptr;
    int* d_tok = nullptr;
    int* d_pos = nullptr;
    int* d_pageTable = nullptr;
    int* d_outIds = nullptr;
    int* d_next = nullptr;
    int* d_stepCounter = nullptr;
    int* d_prompt = nullptr;
    int promptCapacity = 0;
    float *x = nullptr, *qkv = nullptr, *part = nullptr, *mix = nullptr, *h1 = nullptr, *u = nullptr;
    float *logits = nullptr, *amaxVal = nullptr, *probs = nullptr;
    int* amaxIdx = nullptr;
    void* copySrc = nullptr; // calibration buffers for MLH_K_COPY
    void* copyDst = nullptr;
    size_t copyBytes = 0;

    // persistent batch-1 decode kernel
    int numCUs = 0;
    bool coopLaunch = false;
    float temperature = 0.f;       // 0: greedy; > 0: temperature sampling (kernel-sequence and batched paths)
    unsigned long long sampleSeed = 0;
    int usePersistent = 3;         // 0: kernel sequence; 1: persistent kernel with grid barriers;
                                   // 3: XCD ranks where the model and device allow it, else as 1
    int persistentFallbacks = 0;   // single-launch decode calls that gave up a wait and were redone as the kernel sequence
    int injectAbort = 0;           // test hook: the next n single-launch decode launches give up at their start
    int injectAbortStep = 0;       // test hook: the next single-launch decode launch gives up when it reaches this step (> 0)
    bool persistCooperative = false; // MLH_PERSIST_COOPERATIVE, read once at creation: cooperative launch of the barrier kernel
    float* gdnSnapshot = nullptr;  // barrier kernel: sequence 0's GDN states as they were before the launch
    unsigned long long xcdTagNext = 0; // host mirror of the XCD-rank kernel's tag counter (tags used so far)
    bool xcdPrepared = false;      // function attribute and occupancy of the XCD-rank kernel checked
    bool persistentPrepared = false;
    int xcdWide = 1, xcdNapRound = 0, xcdNap[5] = {44, 0, 0, 0, 0}; // tuning knobs, read from the environment once at creation
    unsigned long long* xcdBuf = nullptr; // (value, tag) exchange words of mode 3
    size_t xcdWords = 0;
    int ranksMax = 0;              // sequences the kernel of several sequences takes (kernels_ranks.hip); 0: not this model
    void* ranksBuf = nullptr;      // its exchange words
    size_t ranksBytes = 0;
    unsigned long long ranksTag = 0; // tags its launches have used
    bool ranksOff = false;         // it has given up, and is not tried again before mlh_set_persistent
    int lastDecodeSeqs = 0;        // sequences of the last decode call
    int wideMax = 0;               // ... and the one of more sequences (kernels_wide.hip)
    void* wideBuf = nullptr;       // its exchange memory
    size_t wideBytes = 0;
    unsigned long long ranksSides = 0; // bit s: the gated-delta-net states of sequence s are at their second place (slot maxSeqs + s)
    LayerDev* d_layers = nullptr;  // device copy of `layers`
    unsigned* d_sync = nullptr;    // barrier words + abort flag
    float* pamaxVal = nullptr;     // [numCUs]
    int* pamaxIdx = nullptr;
    float* kvPart = nullptr;       // [heads, pagesPerSeq, headDim + 2]
    unsigned long long* d_timing = nullptr; // phase timestamps (set MLH_PERSIST_TIMING=1), 16 per layer

    std::vector<hipEvent_t>* profEvents = nullptr; // set while mlh_profile_decode runs
    std::vector<int>* profIds = nullptr;

    // prefill work buffers, sized on first use for the largest row count seen
    int pfRows = 0;
    int prefillMode = 0; // 0: GEMM path when the shape allows and the call is long enough; 1: token by token
    std::vector<void*> pfAllocs;
    float *pfX = nullptr, *pfQKV = nullptr, *pfH1 = nullptr;
    void *pfXn = nullptr, *pfA = nullptr, *pfU = nullptr;
    int* pfExp = nullptr; // exponents of the rows of the product input at hand
    uint16_t *pfKh = nullptr, *pfVh = nullptr; // half copies of a call's K and V rows for the MFMA attention of a fresh prefill
    int* pfMeta = nullptr;
    void* pfGdnWs = nullptr;   // chunk operands of the chunk-parallel GDN prefill
    float* pfGdnG = nullptr;
    size_t pfGdnChunks = 0;
    const void* EP = nullptr;  // LM-head matrix as the prefill's products read it (see LayerDev::WaP)
    float sE = 1.0f;
    const int* eE = nullptr;
    const void* ER = nullptr;  // ... and in the row step's fetch order
    int pfDtype = MLH_DTYPE_F32; // operand type of those: MLH_GEMM_H2, MLH_GEMM_P3 or MLH_GEMM_F16
    bool operands = false;     // the copies of the matrices that the MFMA kernels read (LayerDev::WaP .. W2R) exist
    std::vector<void*> mirrorAllocs;
    size_t operandBytes = 0, operandLimit = SIZE_MAX; // what they take and may take
    long f16Inexact = 0;       // bf16 weights that had no exact scaled-half representation (reported at finalize)
    void* gemmWs = nullptr;    // split-K workspace of the prefill's products

    std::vector<int> h_len; // host mirror of d_pos
    std::vector<char> h_dirty;     // sequences that some launch may have given a length or GDN states since their last reset
    std::vector<char> h_nextKnown; // sequences whose next token h_next holds
    std::vector<int> h_next;
    PinBuf pinIo;    // a decode call's first tokens, the single-launch kernels' abort flag, the picked tokens
    PinBuf pinMeta;  // a prefill's metadata, laid out as on the device
    PinBuf pinNext;  // a prefill's picks, by sequence
    PinBuf pinStage; // forward_full's results on their way out
    float* fullBuf = nullptr; // forward_full's device results, kept for the next call up to a limit
    size_t fullBytes = 0;
    int identityNseq = 0;   // d_sidx currently holds 0..identityNseq-1 (0 = unknown)

    int graphSteps = 0;                 // 0: eager launches; k >= 1: one graph replay covers k decode steps
    hipGraphExec_t graphExec[2] = {};   // [0]: one step, [1]: graphSteps steps
    int graphNseqOf[2] = {0, 0};
    int graphStepsOf[2] = {0, 0};
};

// kernels_decode.hip
int mlh_launch_step(mlh_ctx* c, int nseq, const int* tokPtr, bool lmHead, bool embedded = false, bool embedNext = false);
void mlh_mark(mlh_ctx* c, int id);
int mlh_launch_mix(mlh_ctx* c, const StepArgs& a, const LayerDev& L);
int mlh_launch_one(mlh_ctx* c, int kernel, int layer, int nseq);
double mlh_kernel_bytes(mlh_ctx* c, int kernel, int layer, int nseq);
void mlh_fill_args(mlh_ctx* c, StepArgs& a, int nseq, const int* tokPtr);
int mlh_launch_copy(mlh_ctx* c);
int mlh_dev_alloc_bytes(mlh_ctx* c, void** p, size_t bytes); // mlh_api.hip: an allocation owned by the context
int mlh_pin(mlh_ctx* c, PinBuf& b, size_t bytes);                    // ... and its pinned memory
void mlh_drop_graphs(mlh_ctx* c);                                    // ... and its captured steps, before anything they hold the address of goes
int mlh_launch_probs(mlh_ctx* c, int seq);
int mlh_init_kernels(mlh_ctx* c);

// kernels_gemm.hip
// C[M,N] = A[M,K] . B[N,K]^T (+ R[M,N]); dtype: operand type code (fp32 operands: M <= 64; MLH_GEMM_P3 and MLH_GEMM_H2 have no limit).
// epi 0: C, R fp32.  epi 1 (SwiGLU): columns 2j / 2j+1 of the product are gate / up of unit j and
// C is [M, N/2] in the operand type (H2: pairs): C[m, j] = silu(gate) * up.
// ws: zero-initialised workspace of mlh_gemm_workspace_bytes() or null; with it, M <= 64 products of matrices
// with few rows are split along K over workgroups (deterministically reduced).
// alpha scales the product before the epilogue (the power of two an fp16 weight mirror was scaled by, inverted).
hipError_t mlh_gemm_tn_epi(hipStream_t stream, int dtype, int epi, const void* A, int lda, const void* B, int ldb, void* C, int ldc,
                           const float* R, int ldr, int M, int N, int K, void* ws, float alpha = 1.0f, const int* eA = nullptr, const int* eB = nullptr, const int* eC = nullptr);
// kernels_tile.hip: the same product in 128 x 128 / 64 x 64 tiles (operands half, bf16, P3, or H2 with exponents eA, null: none, and eB; epi 1: of the units, eC), and fp32 -> P3 and H2 rows
hipError_t mlh_gemm_tile(hipStream_t stream, int dtype, int epi, const void* A, int lda, const void* B, int ldb, void* C, int ldc,
                         const float* R, int ldr, int M, int N, int K, void* ws, float alpha, const int* eA = nullptr, const int* eB = nullptr, const int* eC = nullptr);
double mlh_gemm_tile_us(int dtype, int M, int N, int K, int cus, bool ws); // what that product is expected to take
int mlh_gemm_num_cus(void); // kernels_gemm.hip: compute units of the current device, a multiple of eight; 0: unknown
hipError_t mlh_split_p3(hipStream_t stream, const float* src, int lds, void* dst, int ldd, int rows, int cols);
hipError_t mlh_split_h2(hipStream_t stream, bool triples, const float* src, int lds, void* dst, int ldd, const int* colExps, int* exps, int rows, int cols);
size_t mlh_gemm_workspace_bytes(void);
extern "C" int mlh_gemm_device_init(int device);

// mlh_api.hip: message returned by mlh_last_error(NULL) on this thread (context-free entry points)
void mlh_set_thread_error(const std::string& msg);

// kernels_prefill.hip
#define MLH_PREFILL_GEMM_MIN_ROWS 16 // bf16 models: calls of fewer tokens keep fp32 activations throughout
size_t mlh_prefill_work_bytes(const mlh_ctx* c);
bool mlh_prefill_gemm_supported(const mlh_ctx* c);
bool mlh_prefill_by_rows(const mlh_ctx* c, int tokens); // through the row kernels
int mlh_init_prefill_kernels(mlh_ctx* c);
#define MLH_NO_ROOM (-4) // inside a finalize only: a copy does not fit on the device
int mlh_operand_alloc(mlh_ctx* c, void** p, size_t bytes); // memory of the copies: 0, MLH_NO_ROOM or an error
void mlh_drop_operands(mlh_ctx* c);
int mlh_build_gemm_operands(mlh_ctx* c); // at finalize: halves and packed rows of every matrix, where the model's widths, its weights and memory allow
int mlh_run_prefill_gemm(mlh_ctx* c, int nseg, const int32_t* seqs, const int32_t* ids, const int32_t* lens, float* allLogits);
int mlh_launch_softmax_rows(mlh_ctx* c, const float* logits, float* probs, const int* target, float* nll, int rows);

// kernels_rows.hip: the decode step of up to 64 sequences
bool mlh_rows_applicable(const mlh_ctx* c, int nseq);
int mlh_rows_prepare(mlh_ctx* c);
int mlh_rows_step(mlh_ctx* c, int nseq, const int* tokPtr, bool lmHead, bool embedded, bool embedNext);
// its parts, for short prefills (rows: tokens) and every prefill's LM head
void mlh_rows_gemm(mlh_ctx* c, int epi, const void* w, int n, RowsArgs P);
void mlh_rows_embed(mlh_ctx* c, const int* tok, int n, float* x, RowsLayout lay);
void mlh_rows_rest_of_layer(mlh_ctx* c, int t, const RowsArgs& base, float* x, float* h1);
void mlh_rows_lm_head(mlh_ctx* c, int n, const float* X, const int* segStart, const int* segLen, const int* segSeq, float* amaxVal, int* amaxIdx);

// kernels_ranks.hip: decode steps of several sequences in one launch
#define MLH_RANKS_MAX_SEQS 16 // one block of MFMA columns
#define MLH_WIDE_MAX_SEQS 64  // four (kernels_wide.hip)
bool mlh_ranks_applicable(const mlh_ctx* c, int nseq);
bool mlh_ranks_wide(const mlh_ctx* c, int nseq); // ... by kernels_wide.hip
int mlh_ranks_other_seqs(const mlh_ctx* c);
int mlh_ranks_prepare(mlh_ctx* c);
int mlh_ranks_reset(mlh_ctx* c);
void mlh_ranks_done(mlh_ctx* c, int nseq);
int mlh_ranks_failed(mlh_ctx* c, int nseq);
int mlh_ranks_settle(mlh_ctx* c, const int* seqs, int n);
int mlh_launch_ranks(mlh_ctx* c, int nseq, int steps);
// kernels_wide.hip: ... of 6 to 64 sequences (mlh_launch_ranks decides)
bool mlh_wide_model(const mlh_ctx* c);
int mlh_wide_prepare(mlh_ctx* c);
int mlh_launch_wide(mlh_ctx* c, int nseq, int steps, unsigned tagBase, int otherAt);

// kernels_persistent.hip
bool mlh_persistent_supported(const mlh_ctx* c);
int mlh_launch_persistent(mlh_ctx* c, int steps);
int mlh_persistent_restore_states(mlh_ctx* c);

// measure_timing.hip: decodes and prints the phase clock stamps of the single-launch decode kernels
// (collected only when MLH_PERSIST_TIMING is set at context creation)
void mlh_dump_persistent_timing(mlh_ctx* c);

// kernels_xcd.hip
size_t mlh_xcd_words(const mlh_ctx* c);
bool mlh_xcd_supported(const mlh_ctx* c);
int mlh_xcd_reset(mlh_ctx* c);
int mlh_launch_xcd(mlh_ctx* c, int steps);

#define MLH_CHECK(ctx, expr)                                                               \
    do {                                                                                   \
        hipError_t e_ = (expr);                                                            \
        if (e_ != hipSuccess) {                                                            \
            (ctx)->err = std::string(#expr) + ": " + hipGetErrorString(e_);                \
            return -2;                                                                     \
        }                                                                                  \
    } while (0)
