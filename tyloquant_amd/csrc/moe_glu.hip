// MoE gate/up projection of a mapped call with the GLU fused into the matmul's epilogue: the prefill kernels of
// moe_prefill.hpp with their act(gate) * up output.
#include "moe_prefill.hpp"

using namespace mfq;

// A mapped call on the prefill kernels: plain float results, or with glu act(gate) * up.  shared: the last of the pools is a tensor that
// every token goes through.
static int moe_mapped_call(const char *what, const mfq_moe_pool *pools, int n_pools, bool shared, const int32_t *expert_pool,
                           const int32_t *expert_local, int E, int out_per_expert, int K, const void *x, int x_dtype, int64_t ldx,
                           int routed_input, const int32_t *ids, int T, int R, const int32_t *ids_dst, const int32_t *expert_bounds, bool glu,
                           int activation, void *out, int out_dtype, int64_t ldo, void *workspace, size_t workspace_bytes,
                           mfq_stream_t stream) {
    MFQ_REQUIRE(pools && expert_pool && expert_local && x && ids && out, MFQ_ERR_INVALID, "%s: null argument", what);
    MFQ_REQUIRE(n_pools >= 1 + shared && n_pools <= kMaxPools, MFQ_ERR_UNSUPPORTED, "%s: %d cohorts (max %d)", what, n_pools, kMaxPools);
    MFQ_REQUIRE(T > 0 && R > 0 && E > 0, MFQ_ERR_INVALID, "MoE ids must be int32 [tokens, routes]");
    MFQ_REQUIRE(x_dtype == MFQ_X_BF16 || x_dtype == MFQ_X_F16, MFQ_ERR_INVALID, "%s: x_dtype=%d", what, x_dtype);
    if (glu) {
        MFQ_REQUIRE(out_dtype == MFQ_X_BF16 || out_dtype == MFQ_X_F16, MFQ_ERR_INVALID, "%s: out_dtype=%d", what, out_dtype);
        MFQ_REQUIRE(activation == MFQ_GLU_SILU || activation == MFQ_GLU_GELU, MFQ_ERR_INVALID, "%s: activation=%d", what, activation);
    }
    MFQ_REQUIRE(out_per_expert > 0 && out_per_expert % (glu ? 32 : 16) == 0, MFQ_ERR_UNSUPPORTED,
                glu ? "%s: out_per_expert %d must be two halves of whole 16-neuron row-blocks" : "%s: out_per_expert %d must be a multiple of 16",
                what, out_per_expert);
    MFQ_REQUIRE(ldx >= K && ldo >= (glu ? out_per_expert / 2 : out_per_expert), MFQ_ERR_INVALID, "%s: ldx/ldh smaller than the tensor", what);
    MFQ_REQUIRE(ids_dst && expert_bounds, MFQ_ERR_UNSUPPORTED, "%s: needs the route map of a mapped call", what);
    const int n_pairs = T * R;
    MoePools P;
    P.n = n_pools;
    const bool ok = K >= 8 && K % 8 == 0 && ldx % 8 == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0;
    for (int i = 0; i < n_pools; ++i) {
        const mfq_nint_desc &d = pools[i].desc;
        MFQ_REQUIRE(d.neuron_len == K && pools[i].weight, MFQ_ERR_INVALID, "%s: cohort %d has neuron_len %d, expected %d", what, i,
                    d.neuron_len, K);
        moe_fill_k(P.k[i], d);
        P.w[i] = static_cast<const uint8_t *>(pools[i].weight);
        P.spw[i] = 0;
    }
    MFQ_REQUIRE(!shared || pools[n_pools - 1].desc.out == out_per_expert, MFQ_ERR_INVALID, "%s: shared tensor of %d neurons, expected %d", what,
                pools[n_pools - 1].desc.out, out_per_expert);
    MFQ_REQUIRE(ok && moe_prefill_eligible(pools, n_pools, E, K, routed_input, n_pairs, T, workspace, workspace_bytes, shared),
                MFQ_ERR_UNSUPPORTED, "%s: these cohorts, activations or workspace keep the call off the prefill kernels", what);
    return moe_prefill_launch(glu, P, pools, n_pools, expert_pool, expert_local, E, out_per_expert, K, x, x_dtype, ldx, routed_input, ids,
                              n_pairs, T, R, ids_dst, expert_bounds, out, ldo, activation == MFQ_GLU_GELU ? 1 : 0,
                              out_dtype == MFQ_X_F16 ? 1 : 0, workspace, shared, as_stream(stream));
}

extern "C" int mfq_hip_moe_grouped_glu_ws(const mfq_moe_pool *pools, int n_pools, const int32_t *expert_pool,
                                          const int32_t *expert_local, int E, int out_per_expert, int K, const void *x,
                                          int x_dtype, int64_t ldx, int routed_input, const int32_t *ids, int T, int R,
                                          const int32_t *ids_dst, const int32_t *expert_bounds, int activation,
                                          void *hidden, int out_dtype, int64_t ldh, void *workspace,
                                          size_t workspace_bytes, mfq_stream_t stream) {
    return moe_mapped_call("moe_grouped_glu", pools, n_pools, false, expert_pool, expert_local, E, out_per_expert, K, x, x_dtype, ldx,
                           routed_input, ids, T, R, ids_dst, expert_bounds, true, activation, hidden, out_dtype, ldh, workspace,
                           workspace_bytes, stream);
}

extern "C" int mfq_hip_moe_grouped_shared_ws(const mfq_moe_pool *pools, int n_pools, const int32_t *expert_pool,
                                             const int32_t *expert_local, int E, int out_per_expert, int K, const void *x,
                                             int x_dtype, int64_t ldx, int routed_input, const int32_t *ids, int T, int R,
                                             const int32_t *ids_dst, const int32_t *expert_bounds, int glu, int activation, void *out,
                                             int out_dtype, int64_t ldo, void *workspace, size_t workspace_bytes, mfq_stream_t stream) {
    return moe_mapped_call("moe_grouped_shared", pools, n_pools, true, expert_pool, expert_local, E, out_per_expert, K, x, x_dtype, ldx,
                           routed_input, ids, T, R, ids_dst, expert_bounds, glu != 0, activation, out, out_dtype, ldo, workspace,
                           workspace_bytes, stream);
}

extern "C" int mfq_hip_moe_few_plan(int E, int out_per_expert, int n_pairs, int shared_rows) {
    if (E < 1 || out_per_expert < 1 || n_pairs < 1 || shared_rows < 0) return 0;
    return moe_few(E, out_per_expert, n_pairs, shared_rows) ? 1 : 0;
}
