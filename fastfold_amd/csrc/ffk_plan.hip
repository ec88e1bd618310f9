// Launch plans (see ffk_run_plan in include/ffk.h): a recorded sequence of this library's entry points, replayed with
// other buffers.
//
// A block of the Evoformer stack is about 25 launches of 5 .. 30 microseconds at the smaller sizes, while preparing each
// of them in Python (descriptors, packed weights, scratch tensors, the foreign call) takes 20: 0.57 ms of host time per
// block, more than the GPU needs up to N_res = 256.  Replaying the block from its plan takes the host 2 .. 3
// microseconds per launch.  What is replayed are calls of the public entry points, so their argument checks and their
// choice of kernel run as they always do.
#include "ffk_common.h"
#include <string.h>
#include <type_traits>
#include <utility>

namespace {

// One argument from its 8-byte slot (pointers as addresses, integers as int64, floats in the low four bytes).
template <typename A> A slot_as(const uint64_t& s) {
    if constexpr (std::is_pointer<A>::value) return reinterpret_cast<A>(s);
    else if constexpr (std::is_same<A, float>::value) {
        float f;
        memcpy(&f, &s, sizeof f);
        return f;
    } else return (A)(int64_t)s;
}

template <typename... A, size_t... I>
int call_slots(int (*fn)(A...), const uint64_t* slots, void* stream, std::index_sequence<I...>) {
    constexpr size_t last = sizeof...(A) - 1;      // every entry point ends in its stream
    return fn((I == last ? slot_as<A>((uint64_t)(uintptr_t)stream) : slot_as<A>(slots[I == last ? 0 : I]))...);
}

template <typename... A> constexpr int arg_slots(int (*)(A...)) { return (int)sizeof...(A) - 1; }

struct OpEntry {
    int slots;                                          // 8-byte words of arguments
    int (*run)(const uint64_t* slots, void* stream);
};

template <auto Fn> int run_args(const uint64_t* slots, void* stream) {
    return call_slots(Fn, slots, stream, std::make_index_sequence<arg_slots(Fn) + 1>());
}
template <auto Fn> constexpr OpEntry args_op() { return {arg_slots(Fn), run_args<Fn>}; }
template <auto Fn, typename D> int run_desc(const uint64_t* slots, void* stream) { return Fn((const D*)slots, stream); }
template <auto Fn, typename D> constexpr OpEntry desc_op() {
    static_assert(sizeof(D) % 8 == 0, "a descriptor is a whole number of slots");
    return {(int)(sizeof(D) / 8), run_desc<Fn, D>};
}

constexpr int MAX_SLOTS = (int)(sizeof(ffk_linear_desc) / 8);

// in the order of the FFK_OP_* codes
const OpEntry OPS[] = {
    desc_op<ffk_fused_linear, ffk_linear_desc>(),
    desc_op<ffk_bgemm_nt, ffk_bgemm_desc>(),
    args_op<ffk_attention_fwd>(),
    args_op<ffk_pair_bias>(),
    args_op<ffk_opm_fused>(),
    args_op<ffk_transition_fused>(),
    args_op<ffk_gated_out_fused>(),
    args_op<ffk_global_attention_core>(),
    args_op<ffk_layernorm_fwd>(),
    args_op<ffk_fill_zero>(),
    args_op<ffk_attention_fwd_lse>(),
    args_op<ffk_attention_bwd_rows>(),
    args_op<ffk_transpose_batched>(),
    args_op<ffk_weight_grad>(),
    args_op<ffk_layernorm_bwd_rows>(),
    args_op<ffk_scale_rows>(),
    args_op<ffk_att_gate_bwd>(),
    args_op<ffk_trimul_gate_bwd>(),
    args_op<ffk_glu_bwd>(),
    args_op<ffk_bias_cols>(),
    args_op<ffk_slice_sum>(),
    args_op<ffk_attention_block>(),
    args_op<ffk_attention_heads>(),
    args_op<ffk_transition_block>(),
};
constexpr int N_OPS = (int)(sizeof(OPS) / sizeof(OPS[0]));
static_assert(N_OPS == FFK_OP_COUNT, "one entry per operation code");

struct OpHead {
    int32_t op, n_slots, n_relocs, reserved;
};
struct Reloc {
    int32_t slot, base;
    int64_t offset;
};

__global__ __launch_bounds__(256) void fill_zero_kernel(u32x4* __restrict__ p, long n) {
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) p[i] = u32x4{0, 0, 0, 0};
}

}  // namespace

extern "C" int ffk_fill_zero(void* p, int64_t bytes, void* stream) {
    FFK_REQUIRE(p, FFK_ERR_NULL, "ffk_fill_zero: null pointer");
    FFK_REQUIRE(bytes > 0 && bytes % 16 == 0, FFK_ERR_SHAPE, "ffk_fill_zero: size %ld is not a positive multiple of 16", (long)bytes);
    FFK_REQUIRE(ffk_aligned16(p), FFK_ERR_ALIGN, "ffk_fill_zero: the buffer must be 16-byte aligned");
    const long n = bytes / 16;
    const long blocks = (n + 1023) / 1024;
    fill_zero_kernel<<<dim3((unsigned)(blocks < 2048 ? blocks : 2048)), 256, 0, (hipStream_t)stream>>>((u32x4*)p, n);
    return ffk_check_launch("ffk_fill_zero");
}

extern "C" int ffk_run_plan(const void* plan, int64_t bytes, const uint64_t* bases, int64_t n_bases, void* stream) {
    FFK_REQUIRE(plan && bases, FFK_ERR_NULL, "ffk_run_plan: null pointer");
    const unsigned char* p = (const unsigned char*)plan;
    const unsigned char* end = p + bytes;
    while (p < end) {
        OpHead h;
        FFK_REQUIRE(end - p >= (long)sizeof h, FFK_ERR_SHAPE, "ffk_run_plan: truncated plan");
        memcpy(&h, p, sizeof h);
        p += sizeof h;
        FFK_REQUIRE(h.op >= 0 && h.op < N_OPS && h.n_slots == OPS[h.op].slots && h.n_slots <= MAX_SLOTS && h.n_relocs >= 0 &&
                        h.n_relocs <= h.n_slots && end - p >= (long)h.n_relocs * (long)sizeof(Reloc) + 8L * h.n_slots,
                    FFK_ERR_SHAPE, "ffk_run_plan: malformed operation (code %d, %d slots, %d relocations)", h.op, h.n_slots, h.n_relocs);
        const unsigned char* relocs = p;
        p += (long)h.n_relocs * sizeof(Reloc);
        uint64_t slots[MAX_SLOTS];
        memcpy(slots, p, 8 * (size_t)h.n_slots);
        p += 8L * h.n_slots;
        for (int i = 0; i < h.n_relocs; ++i) {
            Reloc r;
            memcpy(&r, relocs + (long)i * sizeof r, sizeof r);
            FFK_REQUIRE(r.slot >= 0 && r.slot < h.n_slots && r.base >= 0 && r.base < n_bases && bases[r.base], FFK_ERR_SHAPE,
                        "ffk_run_plan: relocation of slot %d against buffer %d", r.slot, r.base);
            slots[r.slot] = bases[r.base] + (uint64_t)r.offset;
        }
        const int rc = OPS[h.op].run(slots, stream);
        if (rc != FFK_OK) return rc;
    }
    return FFK_OK;
}
