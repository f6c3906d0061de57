/*
 * xo_sv.hip — sampling volume of a photon packet trace: the SamplingVolume
 * kernel of xopto/mcbase/kernel/mcsv.template.c:236-420 (helpers :27-205).
 *
 * One lane walks one packet's trace at a time, segment by segment between
 * consecutive events, through the voxel lattice of the sampling volume
 * (3D DDA). Each voxel the path leaves gets the integer
 * round(terminal weight * path length in the voxel * multiplier * k) with a
 * u64 atomic in HBM. A wave walks a few packets at a time, out of LDS; lanes
 * claim packets beyond the first from a global counter (traces differ in
 * length by orders of magnitude). The walk is bounded: a packet still walking
 * after XO_MAX_PACKET_STEPS voxel or event steps is stopped and counted as
 * truncated.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstring>

#include "../../include/xomc.h"
#include "xo_ctx.h"
#include "xo_device.h"
#include "xo_kernels.h"

namespace {

struct SvParams {
    xo_sampling_volume sv;
    const float *data;        /* [packet][max_events][XO_TRACE_ENTRY_LEN] */
    const int32_t *n;         /* [packet]                                  */
    unsigned long long *accum;
    unsigned long long *total;   /* total weight (one u64)                  */
    unsigned long long *counter; /* packet counter                          */
    unsigned long long *stats;   /* XO_STAT_*                               */
    uint64_t npackets;
    int32_t max_events;
    uint32_t group;              /* packets a wave walks at a time          */
};

struct Ev {
    float p[3];
    float d[3];
};

/* sva_get_event, mcsv.template.c:27-45; e: an event staged in LDS */
__device__ __forceinline__ void load_event(const float4 *e, Ev &ev) {
    const float4 a = e[0];
    const float2 b = *reinterpret_cast<const float2 *>(e + 1);
    ev.p[0] = a.x;
    ev.p[1] = a.y;
    ev.p[2] = a.z;
    ev.d[0] = a.w;
    ev.d[1] = b.x;
    ev.d[2] = b.y;
}

/* mc_distance_point3f (mcbase.template.c:914-916, 1061-1064) */
__device__ __forceinline__ float distance(const float a[3], const float b[3]) {
    const float x = a[0] - b[0], y = a[1] - b[1], z = a[2] - b[2];
    return __builtin_sqrtf(x * x + y * y + z * z);
}

/* (uint32_t)(value + 0.5) of the reference, saturating (a slightly negative
 * path length from rounding gives 0). */
__device__ __forceinline__ uint32_t to_weight(float v) { return xo::f2u_sat(v + 0.5f); }

/* Events a wave holds in LDS, shared by the packets it walks at a time. */
constexpr uint32_t kStaged = 256;
constexpr uint32_t kWaves = 4; /* of a block */
/* Waves per CU that a run is spread over before a wave takes more packets at
 * a time (wave_packets): two per SIMD hide part of each other's latency; 4
 * and 16 are no better (40000 packets 1.6 ms with 4, 1.44 with 8, 1.42 with
 * 16, 8000 packets 0.65, 0.56, 0.64). */
constexpr uint32_t kSpread = 8;
/* Steps between two looks at the wave's packets. */
constexpr int kSteps = 8;

/* A walk is a serial chain: where a step ends decides which voxel and event
 * come next, and the reference rounds the length once per visit of a voxel.
 * What bounds it is the latency of a step, so a wave walks only P.group
 * packets at a time, one lane each (lanes of one wave wait for each other's
 * kind of step), and all its lanes copy the events ahead into LDS: with no
 * memory read between two events, no step waits for the deposits before it.
 * The divisions of a step share the reciprocals of its segment, and its
 * conditions are evaluated without branches. Kernel time with one packet per
 * lane of full waves reading HBM, and now (100 x 100 x 50 voxels): 200 packets
 * 0.95 -> 0.57 ms, 5000 1.49 -> 1.06, 200000 5.0 -> 4.2. */
__global__ void __launch_bounds__(64 * kWaves) sv_kernel(const SvParams P) {
    __shared__ float4 staged[kWaves][kStaged * 2u];
    const xo_sampling_volume &S = P.sv;
    const float kf = (float)S.k;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t chunk = kStaged / P.group; /* events of a packet staged */
    const float4 *mine = &staged[wave][(lane % P.group) * chunk * 2u];
    /* the first packets by position, those beyond from the counter */
    const uint64_t first = (uint64_t)gridDim.x * kWaves * P.group;
    uint64_t pkt = ((uint64_t)blockIdx.x * kWaves + wave) * P.group + lane;
    bool claimed = lane < P.group && pkt < P.npackets;
    bool idle = true, need = false, fresh = false;
    bool more = lane < P.group && first < P.npackets;

    uint32_t walked = 0, truncated = 0, packets = 0;
    Ev e1 = {}, e2 = {};
    int32_t nv = 0, idx = 0, c0 = 0; /* c0: first event staged */
    int32_t v[3] = {0, 0, 0};
    float end_w = 0.0f, d12 = 0.0f, l_voxel = 0.0f;
    uint32_t steps = 0;
    /* what the divisions by e1.d share; general: a component lies outside
     * the range they hold for (0 among them) */
    float inv[3] = {0.0f, 0.0f, 0.0f};
    bool general = false;
    auto turned = [&]() {
        general = false;
        for (int k = 0; k < 3; ++k) {
            const float m = fabsf(e1.d[k]);
            inv[k] = xo::rcp_in_range(e1.d[k]);
            general |= !(m >= 0x1p-60f && m <= 0x1p60f);
        }
    };

    for (;;) {
        if (idle && more && !claimed) {
            pkt = first + atomicAdd(P.counter, 1ull);
            claimed = more = pkt < P.npackets;
        }
        if (claimed) {
            claimed = false;
            ++packets;
            const int32_t count = P.n[pkt];
            nv = count < P.max_events ? count : P.max_events;
            if (nv > 0) {
                const float *end = P.data + (pkt * (uint64_t)P.max_events + (uint32_t)(nv - 1)) *
                                                XO_TRACE_ENTRY_LEN;
                end_w = end[S.end_field];
                atomicAdd(P.total, (unsigned long long)to_weight(end_w * kf));
                idle = false;
                need = fresh = true;
                c0 = 0;
            }
        }
        uint64_t refill = __ballot(need);
        if (refill) {
            do {
                const int l = __builtin_ctzll(refill);
                refill &= refill - 1u;
                const int32_t from = __builtin_amdgcn_readlane(c0, l);
                const uint32_t left = (uint32_t)(__builtin_amdgcn_readlane(nv, l) - from);
                const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)pkt, l);
                const uint32_t hi = __builtin_amdgcn_readlane((int)(uint32_t)(pkt >> 32), l);
                const uint64_t q = ((uint64_t)hi << 32) | lo;
                const float4 *src =
                    reinterpret_cast<const float4 *>(P.data) +
                    (q * (uint64_t)P.max_events + (uint32_t)from) * (XO_TRACE_ENTRY_LEN / 4);
                const uint32_t n = 2u * (left < chunk ? left : chunk);
                for (uint32_t i = lane; i < n; i += 64u)
                    staged[wave][(uint32_t)l * chunk * 2u + i] = src[i];
            } while (refill);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
        if (need) {
            need = false;
            if (fresh) {
                fresh = false;
                load_event(mine, e1);
                load_event(mine + (nv > 1 ? 2 : 0), e2);
                for (int k = 0; k < 3; ++k)
                    v[k] = xo::f2i_sat((e1.p[k] - S.top_left[k]) / S.voxel_size[k]);
                turned();
                l_voxel = 0.0f;
                steps = 0;
                idx = 0;
            } else {
                load_event(mine, e2);
            }
            d12 = distance(e1.p, e2.p);
        }
        if (!__any(!idle || more)) break;

        for (int rep = 0; rep < kSteps; ++rep) {
            if (idle || need) break;
            /* sva_intersect, mcsv.template.c:95-115 (the sum of an index of
             * 2^31 - 1 and 1 rounds to the float that the index rounds to) */
            float num[3], dist[3];
            for (int k = 0; k < 3; ++k) {
                const int32_t one = e1.d[k] >= 0.0f;
                const float side = (float)__builtin_elementwise_add_sat(v[k], one);
                num[k] = S.top_left[k] + side * S.voxel_size[k] - e1.p[k];
                dist[k] = xo::div_with_rcp(num[k], e1.d[k], inv[k]);
            }
            const float far = fmaxf(fabsf(num[0]), fmaxf(fabsf(num[1]), fabsf(num[2])));
            const float near = fminf(fabsf(num[0]), fminf(fabsf(num[1]), fabsf(num[2])));
            if (__builtin_expect(general || !(near >= 0x1p-60f && far <= 0x1p60f), 0))
                for (int k = 0; k < 3; ++k)
                    dist[k] = (e1.d[k] != 0.0f) ? num[k] / e1.d[k] : XO_INF_F;
            const float d_voxel = fminf(dist[2], fminf(dist[0], dist[1]));
            const float d_move = fminf(d_voxel, d12);
            l_voxel += d_move;
            const bool valid = (int32_t)((v[0] | v[1] | v[2]) >= 0) &
                               (int32_t)((uint32_t)v[0] < S.shape[0]) &
                               (int32_t)((uint32_t)v[1] < S.shape[1]) &
                               (int32_t)((uint32_t)v[2] < S.shape[2]);
            /* leaving this voxel before the next event, :330-350, or the
             * next event comes first, :351-372 */
            const bool leave = d_voxel < d12;
            const bool last = (int32_t)!leave & (int32_t)(idx + 1 >= nv - 1);
            if ((int32_t)valid & ((int32_t)leave | (int32_t)last)) {
                const uint32_t w = to_weight(end_w * l_voxel * S.multiplier * kf);
                if (w) {
                    const uint64_t row = (uint64_t)(uint32_t)v[2] * S.shape[1] + (uint32_t)v[1];
                    atomicAdd(&P.accum[S.offset + row * S.shape[0] + (uint32_t)v[0]],
                              (unsigned long long)w);
                }
            }
            if (leave) {
                e1.p[0] += e1.d[0] * d_move;
                e1.p[1] += e1.d[1] * d_move;
                e1.p[2] += e1.d[2] * d_move;
                d12 -= d_move;
                /* sva_next_voxel, :130-152 */
                const int32_t nx = (int32_t)(dist[0] <= dist[1]) & (int32_t)(dist[0] <= dist[2]);
                const int32_t ny =
                    (nx ^ 1) & (int32_t)(dist[1] <= dist[0]) & (int32_t)(dist[1] <= dist[2]);
                const int32_t nz = !(nx | ny);
                v[0] += e1.d[0] < 0.0f ? -nx : nx;
                v[1] += e1.d[1] < 0.0f ? -ny : ny;
                v[2] += e1.d[2] < 0.0f ? -nz : nz;
                l_voxel = 0.0f;
            } else {
                e1 = e2;
                turned();
                ++idx;
                if (!last) {
                    const int32_t next = idx + 1;
                    if ((uint32_t)(next - c0) < chunk) {
                        load_event(mine + 2 * (next - c0), e2);
                        d12 = distance(e1.p, e2.p);
                    } else {
                        c0 = next;
                        need = true;
                    }
                }
            }
            ++walked;
            if (last) {
                idle = true;
            } else if (++steps >= XO_MAX_PACKET_STEPS) {
                ++truncated;
                idle = true;
                need = false;
            }
        }
    }
    if (walked) atomicAdd(&P.stats[XO_STAT_STEPS], (unsigned long long)walked);
    if (packets) atomicAdd(&P.stats[XO_STAT_PACKETS], (unsigned long long)packets);
    if (truncated) atomicAdd(&P.stats[XO_STAT_TRUNCATED], (unsigned long long)truncated);
}

/* Packets a wave walks at a time: the fewest (a power of two) with which
 * kSpread waves per CU hold all packets. */
uint32_t wave_packets(uint64_t npackets, uint32_t cus) {
    uint32_t g = 1;
    while (g < 64u && (uint64_t)cus * kSpread * g < npackets) g *= 2u;
    return g;
}

} // namespace

extern "C" int xo_sampling_volume_run(xo_ctx *ctx, const xo_sampling_volume *sv,
                                      int32_t max_events, const float *trace_data,
                                      const int32_t *trace_n, uint64_t npackets,
                                      uint64_t *accum, uint64_t naccum,
                                      uint64_t *total_weight, xo_run_report *report) {
    auto t0 = std::chrono::steady_clock::now();
    xo::clear_error();
    if (!ctx || !sv || !accum || !total_weight || (npackets && (!trace_data || !trace_n))) {
        xo::set_error("xo_sampling_volume_run: null argument");
        return -1;
    }
    if (max_events < 1) {
        xo::set_error("xo_sampling_volume_run: max_events must be >= 1");
        return -1;
    }
    if (sv->end_field != 6 && sv->end_field != 7) {
        xo::set_error("xo_sampling_volume_run: end_field must be 6 (w) or 7 (pl)");
        return -1;
    }
    const uint64_t bins = (uint64_t)sv->shape[0] * sv->shape[1] * sv->shape[2];
    if (bins == 0 || sv->offset > naccum || bins > naccum - sv->offset) {
        xo::set_error("xo_sampling_volume_run: %llu bins at offset %u do not fit %llu",
                      (unsigned long long)bins, sv->offset, (unsigned long long)naccum);
        return -1;
    }
    const uint64_t per = (uint64_t)max_events * XO_TRACE_ENTRY_LEN;
    if (npackets > (UINT64_MAX / 4u) / per) {
        xo::set_error("xo_sampling_volume_run: trace too large");
        return -1;
    }
    const uint64_t floats = npackets * per;

    std::lock_guard<std::mutex> lock(ctx->mu);
    XO_HIP(hipSetDevice(ctx->device));
    /* the bins, then the total weight */
    if (xo::ensure_buffer((void **)&ctx->accum, &ctx->accum_cap, (naccum + 1) * 8)) return -1;
    if (npackets &&
        (xo::ensure_buffer((void **)&ctx->trace_data, &ctx->trace_data_cap, floats * 4) ||
         xo::ensure_buffer((void **)&ctx->trace_n, &ctx->trace_n_cap, npackets * 4)))
        return -1;
    SvParams P;
    std::memset(&P, 0, sizeof(P));
    P.sv = *sv;
    P.data = ctx->trace_data;
    P.n = ctx->trace_n;
    P.accum = ctx->accum;
    P.total = ctx->accum + naccum;
    P.counter = ctx->counters;
    P.stats = ctx->counters + 1;
    P.npackets = npackets;
    P.max_events = max_events;
    P.group = wave_packets(npackets, ctx->cus);
    const uint64_t per_block = (uint64_t)kWaves * P.group;
    const uint32_t blocks = (uint32_t)std::min<uint64_t>(
        std::max<uint64_t>((npackets + per_block - 1) / per_block, 1u), ctx->cus * 4u);
    if (npackets) {
        XO_HIP(hipMemcpyAsync(ctx->trace_data, trace_data, floats * 4, hipMemcpyHostToDevice,
                              ctx->stream));
        XO_HIP(hipMemcpyAsync(ctx->trace_n, trace_n, npackets * 4, hipMemcpyHostToDevice,
                              ctx->stream));
    }
    XO_HIP(hipMemsetAsync(ctx->accum, 0, (naccum + 1) * 8, ctx->stream));
    XO_HIP(hipMemsetAsync(ctx->counters, 0, sizeof(unsigned long long) * (1 + XO_STAT_COUNT),
                          ctx->stream));
    XO_HIP(hipEventRecord(ctx->ev0, ctx->stream));
    if (npackets) {
        hipLaunchKernelGGL(sv_kernel, dim3(blocks), dim3(64 * kWaves), 0, ctx->stream, P);
        XO_HIP(hipGetLastError());
    }
    XO_HIP(hipEventRecord(ctx->ev1, ctx->stream));
    unsigned long long counters[1 + XO_STAT_COUNT];
    unsigned long long total = 0;
    XO_HIP(hipMemcpyAsync(accum, ctx->accum, naccum * 8, hipMemcpyDeviceToHost, ctx->stream));
    XO_HIP(hipMemcpyAsync(&total, ctx->accum + naccum, 8, hipMemcpyDeviceToHost, ctx->stream));
    XO_HIP(hipMemcpyAsync(counters, ctx->counters, sizeof(counters), hipMemcpyDeviceToHost,
                          ctx->stream));
    XO_HIP(hipStreamSynchronize(ctx->stream));
    float kms = 0.f;
    XO_HIP(hipEventElapsedTime(&kms, ctx->ev0, ctx->ev1));
    *total_weight = total;
    if (report) {
        std::memset(report, 0, sizeof(*report));
        report->packets = counters[1 + XO_STAT_PACKETS];
        report->steps = counters[1 + XO_STAT_STEPS];
        report->truncated = counters[1 + XO_STAT_TRUNCATED];
        report->lanes = blocks * 64u * kWaves;
        report->kernel_ms = kms;
        report->total_ms = xo::ms_since(t0);
    }
    return 0;
}
