// The sample of gram_probe.hpp as a launch of its own.
#include <hip/hip_runtime.h>

#include "../host/host_common.hpp"
#include "../host/dispatch_rules.hpp"
#include "gram_probe.hpp"
#include "launch.hpp"

static_assert(kmc::BK_SAMPLE_TILES == kmc_rules::SAMPLE_TILES && kmc::BK_SAMPLE_LEAVE_PER_16384 == kmc_rules::SAMPLE_LEAVE_PER_16384 &&
                  kmc::BK_SAMPLE_BYTES == KMC_SAMPLE_BYTES,
              "the table of dispatch rules, the header and the kernels' constants must say the same");

namespace kmc {

__global__ __launch_bounds__(GP_THREADS) void gram_probe_operands(const GramProbeArgs args)
{
    gram_probe_tile(args, blockIdx.x);
}

}  // namespace kmc

namespace kmc_host {

// What the kernel needs for the problem of `p` (squared differences; m, n, k, l at least 1).
kmc::GramProbeArgs gram_probe_args(const kmc_build_kernel_params *p, const kmc::BuildKernelArgs &args, unsigned *sample, int centre_pairs, int queues)
{
    kmc::GramProbeArgs probe;
    probe.a = p->a; probe.b = p->b;
    probe.a_ld = p->a_ld; probe.a_bs = p->a_bs; probe.b_ld = p->b_ld; probe.b_bs = p->b_bs;
    probe.a_k_contiguous = p->a_majorness == KMC_COL_MAJOR ? 0 : 1;
    probe.b_k_contiguous = p->b_majorness == KMC_COL_MAJOR ? 0 : 1;
    probe.m = args.m; probe.n = args.n; probe.k = args.k; probe.l = args.l;
    probe.centre = args.centre; probe.centre_bs = args.centre_bs;
    probe.centre_pairs = centre_pairs;
    probe.trust = args.gram_trust;
    probe.sample = sample;
    probe.queues = queues;
    return probe;
}

// Fills sample[0 .. BK_SAMPLE_TILES), and clears `queues` words behind it, for the problem of `p` (squared differences; m, n, k, l at least 1).
hipError_t launch_gram_probe(const kmc_build_kernel_params *p, const kmc::BuildKernelArgs &args, unsigned *sample, int centre_pairs, int queues, hipStream_t stream)
{
    const kmc::GramProbeArgs probe = gram_probe_args(p, args, sample, centre_pairs, queues);
    return launch(kmc::gram_probe_operands, dim3(kmc::BK_SAMPLE_TILES), dim3(kmc::GP_THREADS), stream, probe);
}

}  // namespace kmc_host
