// The block-FP8 linear as one entry point: 16-bit activations in, 16-bit outputs out (quantizer + GEMM).
//
// What a decode step spends on a small linear is not the stream over its weights but what surrounds it: in a captured graph
// a launch costs 1.7 to 2.7 us however little it does, and the quantizer in front of a 6 to 20 us weight stream was up to a
// fifth of the linear (N = K = 4096, one row: 8.2 us, 6.5 without it).  Up to
// kFusedRows rows the weight streams therefore quantize the activations themselves (XQuant in gemm_stream.hpp): every
// workgroup repeats that work, but it is small - 16 lanes per row and K step - and sits in the shadow of the stream.
#include "stream_plan.hpp"

namespace mi355 {

// Rows up to which the streams quantize: up to 4 rows always (one load and 50 vector operations per lane and K step; the
// stream takes as long as on quantized activations), up to 8 where the activations all workgroups read together stay
// below kFusedBytes.  In a captured graph, us, two launches against one: N = K = 4096 M = 1 / 4 / 8: 8.2 / 8.6 / 9.1
// against 6.5 / 6.6 / 7.9; 6144 x 4096: 9.4 / 9.7 / 9.9 against 7.6 / 7.9 / 9.3; 28672 x 4096: 25.6 / 24.9 / 25.1
// against 22.4 / 22.4 / 23.6; 4096 x 14336: 15.3 / 14.9 / 15.4 against 12.9 / 13.2 / 16.2 (59 MB of activations for 8
// rows); 36864 x 7168: 46.2 / 44.1 / 45.7 against 44.2 / 43.0 / 50.5 (264 MB).  With 16 rows it loses everywhere (N = K =
// 4096: 9.5 against 10.5).  kFusedBytes is a total over a whole device of 256 units (every workgroup's requests, to the
// caches all of them share); 5 to 7 rows count as 8 because the loads of 8 are issued, the missing rows repeating the last.
constexpr int64_t kFusedRows = 8;
constexpr int64_t kFusedBytes = 40000000;

struct FusedPlan {
    bool ok;
    int tnw;          // > 0: the per-unit stream with this many row blocks; 0: the tiled stream
    SkinnyPlan tiled;
    size_t ws_bytes;
};

// The stream a fused linear runs on: the one the shape table takes for the GEMM.
static FusedPlan fused_plan(int64_t M, int64_t N, int64_t K, int32_t x_dtype, int cus) {
    FusedPlan f = {false, 0, {0, 1, 0}, 0};
    if (M < 1 || M > kFusedRows || N < 1 || K < kBlockK || K % kBlockK != 0) return f;
    if (x_dtype != MI355_DTYPE_BF16 && x_dtype != MI355_DTYPE_F16) return f;
    if (N * K >= (1ll << 32) || M * K * 2 >= (1ll << 32)) return f;  // 32-bit row offsets
    auto reads_ok = [&](int64_t tiles) { return M <= 4 || tiles * 8 * 2 * K <= kFusedBytes; };
    if (streamcu_pays(M, N, K, cus)) {
        f.tnw = streamcu_tnw(M, N, K, K, K, K / kBlockK, cus);
        f.ok = f.tnw > 0 && reads_ok((N + 16 * f.tnw - 1) / (16 * f.tnw));
        return f;
    }
    if (mi355_block_fp8_gemm_plan(M, N, K, (size_t)1 << 40, cus) != MI355_GEMM_SKINNY) return f;
    f.tiled = skinny_plan(M, N, K, cus);
    if ((int64_t)f.tiled.tiles * 4 > MI355_WS_COUNTER_BYTES || !reads_ok(f.tiled.tiles)) return f;
    f.ws_bytes = f.tiled.splits > 1 ? skinny_workspace(M, f.tiled) : 0;
    f.ok = true;
    return f;
}

template <int TB, int XR, bool F16, bool TURN>
static int launch_cu_as(GemmArgs &a, hipStream_t st) {
    using Cfg = CuStreamCfg<1, TB, XR>;
    constexpr auto kernel = block_fp8_gemm_streamcu_kernel<1, TB, true, XR, F16, TURN>;
    const int lds_bytes = Cfg::lds_bytes(a.K / kBlockK);
    if (lds_bytes > kMaxLds) return MI355_EUNSUPPORTED;
    if (!allow_lds<kernel>(kMaxLds)) return MI355_ELAUNCH;
    return launch(kernel, dim3((a.N + Cfg::BN - 1) / Cfg::BN), dim3(Cfg::kThreads), lds_bytes, st, a);
}

template <int TB, int XR, bool F16>
static int launch_cu(GemmArgs &a, hipStream_t st) {
    a.turn_mask = streamcu_turn_mask(a.K, TB);
    return a.turn_mask ? launch_cu_as<TB, XR, F16, true>(a, st) : launch_cu_as<TB, XR, F16, false>(a, st);
}

template <int TNW, int XR, bool F16, bool TURN>
static int launch_tiled_as(GemmArgs &a, const SkinnyPlan &pl, void *ws, hipStream_t st) {
    using Cfg = StreamCfg<1, TNW>;
    constexpr int lds_bytes = Cfg::kLds + kStreamWaves * 64;
    if (pl.splits <= 1) {
        constexpr auto whole_k = block_fp8_gemm_stream_kernel<1, TNW, false, false, XR, F16, kStreamWaves, TURN>;
        if (!allow_lds<whole_k>(lds_bytes)) return MI355_ELAUNCH;
        return launch(whole_k, dim3(pl.tiles), dim3(256), lds_bytes, st, a);
    }
    if constexpr (TNW == 1) {  // 64-row tiles never share K
        constexpr auto split_k = block_fp8_gemm_stream_kernel<1, TNW, true, false, XR, F16, kStreamWaves, TURN>;
        if (!allow_lds<split_k>(lds_bytes)) return MI355_ELAUNCH;
        a.splits = pl.splits;
        a.counters = (uint32_t *)ws;
        a.partials = (float *)((uint8_t *)ws + MI355_WS_COUNTER_BYTES);
        return launch(split_k, dim3(pl.tiles * pl.splits), dim3(256), lds_bytes, st, a);
    }
    return MI355_EUNSUPPORTED;
}

template <int TNW, int XR, bool F16>
static int launch_tiled(GemmArgs &a, const SkinnyPlan &pl, void *ws, hipStream_t st) {
    a.turn_mask = stream_turn_mask(a.K, a.K / kBlockK / pl.splits);
    return a.turn_mask ? launch_tiled_as<TNW, XR, F16, true>(a, pl, ws, st) : launch_tiled_as<TNW, XR, F16, false>(a, pl, ws, st);
}

template <int XR, bool F16>
static int launch_fused_as(GemmArgs &a, const FusedPlan &f, void *ws, hipStream_t st) {
    switch (f.tnw) {
        case 0:
            if (f.tiled.tnw == 4) return launch_tiled<4, XR, F16>(a, f.tiled, ws, st);
            if (f.tiled.tnw == 1) return launch_tiled<1, XR, F16>(a, f.tiled, ws, st);
            return MI355_EUNSUPPORTED;
        case 1: return launch_cu<1, XR, F16>(a, st);
        case 2: return launch_cu<2, XR, F16>(a, st);
        case 3: return launch_cu<3, XR, F16>(a, st);
        case 4: return launch_cu<4, XR, F16>(a, st);
        case 5: return launch_cu<5, XR, F16>(a, st);
        default: return MI355_EUNSUPPORTED;
    }
}

template <bool F16>
static int launch_fused(GemmArgs &a, const FusedPlan &f, void *ws, hipStream_t st) {
    if (a.M <= 4) return launch_fused_as<1, F16>(a, f, ws, st);
    return launch_fused_as<2, F16>(a, f, ws, st);
}

}  // namespace mi355

using namespace mi355;

extern "C" int32_t mi355_block_fp8_linear_fused(int64_t M, int64_t N, int64_t K, int32_t x_dtype) {
    return fused_plan(M, N, K, x_dtype, device_cus()).ok ? 1 : 0;
}

extern "C" size_t mi355_block_fp8_linear_workspace_bytes(int64_t M, int64_t N, int64_t K, int32_t x_dtype) {
    const size_t gemm = mi355_block_fp8_gemm_workspace_bytes(M, N, K, MI355_GEMM_AUTO);
    const FusedPlan f = fused_plan(M, N, K, x_dtype, device_cus());
    return f.ok && f.ws_bytes > gemm ? f.ws_bytes : gemm;
}

extern "C" int mi355_block_fp8_linear(const void *x, int32_t x_dtype, const void *W, const float *Ws, void *C, int64_t M,
                                      int64_t N, int64_t K, int64_t ldw, int64_t ws_n, int64_t ws_k, int64_t ldc,
                                      void *x_q, float *x_s, void *ws, size_t ws_bytes, int32_t c_dtype, void *stream) {
    if (M < 0 || N < 0 || K < 0) return MI355_EINVAL;
    if (c_dtype != MI355_DTYPE_BF16 && c_dtype != MI355_DTYPE_F16) return MI355_EUNSUPPORTED;
    if (M == 0 || N == 0) return MI355_OK;
    if (K == 0 || K % kBlockK != 0) return MI355_ESHAPE;
    if (!x || !W || !Ws || !C) return MI355_EINVAL;
    if (ldw < K || ldc < N) return MI355_ESHAPE;
    hipStream_t st = (hipStream_t)stream;
    if (!x_q) {
        const FusedPlan f = fused_plan(M, N, K, x_dtype, device_cus());
        const bool ws_ok = ws && ((uintptr_t)ws & 15) == 0 && ws_bytes >= f.ws_bytes;
        if (!f.ok || ldw != K || !fast_layout_ok(x, W, K, K, 1, ldw)) return MI355_EUNSUPPORTED;
        if (f.ws_bytes > 0 && !ws_ok) return MI355_EWORKSPACE;
        // every workgroup reads all of x: one that is done must not store over what another has yet to read
        const uintptr_t x0 = (uintptr_t)x, c0 = (uintptr_t)C;
        if (x0 < c0 + 2 * (uintptr_t)((M - 1) * ldc + N) && c0 < x0 + 2 * (uintptr_t)(M * K)) return MI355_EINVAL;
        GemmArgs a = {};
        a.out_f16 = c_dtype == MI355_DTYPE_F16 ? 1 : 0;
        a.X = (const uint8_t *)x;
        a.W = (const uint8_t *)W;
        a.Ws = Ws;
        a.C = (uint16_t *)C;
        a.M = (int)M;
        a.N = (int)N;
        a.K = (int)K;
        a.ldx = 2 * K;  // bytes
        a.ldw = ldw;
        a.ldc = ldc;
        a.ws_n = ws_n;
        a.ws_k = ws_k;
        a.vec_store = (((uintptr_t)C & 15) == 0 && ldc % 8 == 0 && N % 8 == 0) ? 1 : 0;
        return x_dtype == MI355_DTYPE_F16 ? launch_fused<true>(a, f, ws, st) : launch_fused<false>(a, f, ws, st);
    }
    if (!x_s) return MI355_EINVAL;
    const int64_t KB = K / kBlockK;
    const int r = mi355_group_quant_fp8(x, x_dtype, x_q, x_s, M, K, kBlockK, 1e-10f, KB, 1, stream);
    if (r != MI355_OK) return r;
    return mi355_block_fp8_gemm_dtype(x_q, W, x_s, Ws, C, M, N, K, K, 1, ldw, ldc, KB, 1, ws_k, ws_n, kBlockN, kBlockK, ws,
                                      ws_bytes, MI355_GEMM_AUTO, c_dtype, stream);
}
