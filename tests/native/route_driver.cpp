// Host-only: what the library's routing rules decide.  Links the real fa_rocm_api.cpp; the launchers are stubs that say that
// they were called.  One question per line of standard input, one answer per line of output:
//     call batch seqlen_q heads kv_heads head_dim page pages_per_row new_keys window_left
//         -> "unit W" (a workgroup of W waves per unit), "cut" (units cut over the device), "tiled" or "latent"
//     tiling group heads max_seqlen_q total_q head_dim compute_units causal -> heads per tile, tiles side by side, tiles of a unit
//     order tiles tiles_side_by_side units heads_per_unit -> unit/tile/head of every workgroup of the tiled forward
#include <cstdio>
#include <cstring>

#include "../../flash-attention-npu_amd/csrc/fa_kernels.h"
#include "../../include/fa_rocm.h"

namespace {
char g_route[32];
hipError_t took(const char *route) {
    std::snprintf(g_route, sizeof(g_route), "%s", route);
    return hipSuccess;
}
}  // namespace

namespace fa {
hipError_t launch_append_kv(const AppendParams &, int, hipStream_t) { return hipSuccess; }
hipError_t launch_append_quant_i8(const AppendParams &, int, hipStream_t) { return hipSuccess; }
hipError_t launch_rotate_q(const RotateQParams &, int, hipStream_t) { return hipSuccess; }
hipError_t launch_decode_paged(const DecodeParams &, int, int, hipStream_t) { return took("cut"); }
hipError_t launch_decode_wave(const DecodeParams &, int, int, hipStream_t) { return took("cut"); }
hipError_t launch_decode_unit(const DecodeParams &p, int, int, hipStream_t) { return took(p.unit_waves == 8 ? "unit 8" : "unit 4"); }
hipError_t launch_splitkv_combine(const DecodeParams &, int, int, hipStream_t) { return hipSuccess; }
hipError_t launch_decode_mla_i8(const DecodeParams &, int, hipStream_t) { return took("latent"); }
hipError_t launch_prefill(const PrefillParams &, int, int, hipStream_t) { return took("tiled"); }
hipError_t launch_prefill_combine(const PrefillParams &, int, int, hipStream_t) { return hipSuccess; }
hipError_t launch_gather_short_blocks(const ShortBlocksParams &, hipStream_t) { return hipSuccess; }
hipError_t launch_scatter_short_blocks(const ShortBlocksParams &, hipStream_t) { return hipSuccess; }
}  // namespace fa

int main() {
    void *const some = reinterpret_cast<void *>(0x1000);   // never dereferenced
    char what[16];
    while (std::scanf("%15s", what) == 1) {
        if (!std::strcmp(what, "tiling")) {
            int group, heads, longest, total, d, cus, causal;
            if (std::scanf("%d %d %d %d %d %d %d", &group, &heads, &longest, &total, &d, &cus, &causal) != 7) return 1;
            const fa::PrefillTiles t = fa::prefill_tiling(group, heads, longest, total, d, cus, causal != 0);
            std::printf("%d %d %d\n", t.pack, t.mb_run, t.num_mb);
            continue;
        }
        if (!std::strcmp(what, "order")) {
            int tiles, run, units, heads;
            if (std::scanf("%d %d %d %d", &tiles, &run, &units, &heads) != 4) return 1;
            for (int i = 0; i < tiles * units * heads; ++i) {
                const fa::PrefillPlace w = fa::prefill_place((unsigned)i, tiles, run, units, heads);
                std::printf("%d/%d/%d ", w.unit, w.mb, w.head);
            }
            std::printf("\n");
            continue;
        }
        int batch, sq, hq, hk, d, page, pages, fresh, window;
        if (std::scanf("%d %d %d %d %d %d %d %d %d", &batch, &sq, &hq, &hk, &d, &page, &pages, &fresh, &window) != 9) return 1;
        fa_kvcache_args a;
        std::memset(&a, 0, sizeof(a));
        a.q = a.out = a.k_cache = a.v_cache = a.workspace = some;
        a.workspace_bytes = (size_t)1 << 40;
        a.softmax_lse = static_cast<float *>(some);
        a.cache_seqlens = a.block_table = static_cast<const int32_t *>(some);
        if (fresh) a.k_new = a.v_new = some;
        a.batch = batch, a.seqlen_q = sq, a.nheads = hq, a.nheads_k = hk, a.headdim_qk = a.headdim_v = d, a.seqlen_new = fresh;
        a.page_size = page, a.max_blocks_per_seq = pages, a.num_blocks = batch * pages, a.bt_stride_b = pages;
        a.q_stride_h = a.o_stride_h = d, a.q_stride_s = a.o_stride_s = (int64_t)hq * d, a.q_stride_b = a.o_stride_b = a.q_stride_s * sq;
        a.k_stride_h = a.v_stride_h = d, a.k_stride_row = a.v_stride_row = (int64_t)hk * d;
        a.k_stride_block = a.v_stride_block = a.k_stride_row * page;
        a.kn_stride_h = a.vn_stride_h = d, a.kn_stride_s = a.vn_stride_s = (int64_t)hk * d;
        a.kn_stride_b = a.vn_stride_b = a.kn_stride_s * (fresh ? fresh : 1);
        a.io_dtype = a.kv_dtype = FA_BF16;
        a.softmax_scale = 0.1f;
        a.causal = 1;
        a.window_left = window, a.window_right = window >= 0 ? 0 : -1;
        took("none");
        const int rc = fa_rocm_fwd_kvcache(&a, nullptr);
        std::printf("%s\n", rc == FA_OK ? g_route : fa_rocm_last_error());
    }
    return 0;
}
