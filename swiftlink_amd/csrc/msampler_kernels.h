// Argument block and launchers of the M-sampler kernels
// (MeiosisSampler, meiosis_sampler.cc:17-203; FounderAlleleGraph4,
// founder_allele_graph4.cc:34-597).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace sl {

// One wavefront builds the founder-allele graph of one locus in LDS; founder
// alleles are 10-bit node ids in its edge words.
constexpr int kMaxFagNodes = 1022;  // 2F
constexpr int kMsampBlock = 256;    // threads per workgroup of the likelihood kernel (its launch bound)
constexpr int kSpecBlock = 512;     // threads per workgroup of the speculative kernel
constexpr int kFbBlock = 1024;      // threads per workgroup of the forward-backward kernel, and of the planned
                                    // kernel that runs it beside the next step's jobs
constexpr int kMaxBesideLoci = 4 * kFbBlock;  // loci that kernel takes: segments of 1, 2 or 4 per thread
// LDS of a workgroup, and what a kernel with a forward-backward pass declares of
// it besides its dynamic LDS: a 2x2 FP64 product and two words per wavefront
constexpr size_t kLdsBytes = 160 * 1024;
constexpr size_t fb_static_lds(int block) { return (size_t)(block / 64) * (4 * sizeof(double) + 2 * sizeof(uint32_t)); }

struct MsampArgs {
    int N, F, M, W;
    const int32_t* mother;        // [N]
    const int32_t* father;        // [N]
    const uint2* ptab;            // [N-F] label pass in generation order:
                                  //   (person | generation << 16, mother | father << 16)
    int ptab_bytes;               // LDS bytes of the staged ptab
    const int32_t* gen_off;       // [n_gen+1] non-founders grouped by generation
    int n_gen;
    const uint32_t* geno2;        // [M][GW] marker genotypes, 2 bits per person (bits 2(i%16) of word
                                  // i/16; 0 untyped, 1 heterozygous, 2/3 homozygous A/B)
    int GW;                       // ceil(N/16)
    const double* lfreq;          // [M][2] ln(1 - minor allele frequency), ln(minor allele frequency)
    const double* lsum;           // [M][kLsumK] ln(1 + exp(-k |ln(1 - q) - ln q|)), q the minor allele
                                  // frequency: the term of a component whose founder alleles may take
                                  // either assignment, k the difference of its two allele counts
    const double* theta;          // [M-1]
    const int32_t* meioses;       // [n_meioses] non-ignorable meioses (bit index 2(p-F)+parent)
    int n_meioses;                // meioses sampled by this sweep
    int32_t* order;               // [chains][n_meioses] this sweep's meiosis order
    const uint8_t* cls;           // [2(N-F)][M] what flipping meiosis b at locus l does to a legal column
                                  // (kFlipCompute, kFlipSame, kFlipIllegal)
    const int32_t* joblist;       // [2(N-F)][M] the kFlipCompute loci of each meiosis, ascending
    const int32_t* jobcnt;        // [2(N-F)] how many
    int compact;                  // 1: a step's jobs are taken from joblist; 0: job index = locus
    uint32_t* graphs;             // [chains][M][W]
    double* lcur;                 // [chains][M] log-likelihood of the current column
    double* lflip;                // [2 step parities][2 variants][chains][M] flipped-column log-likelihoods
    double* fbuf;                 // [chains][M][2] forward probabilities
    uint8_t* maps;                // [chains][M] per-locus backward decision maps
    int32_t* status;              // [chains]
    uint32_t* near_edge;          // [chains] draws within 1e-12 of their threshold
    uint64_t seed;
    uint32_t sweep;
    const uint32_t* sweep_dev;    // when set, the sweep index is read here (captured sweeps)
    int step;                     // meiosis step whose likelihood jobs this launch runs
    int fb_step;                  // meiosis step whose forward-backward pass this launch runs
    int n_jobs;                   // likelihood jobs (wavefronts) per chain in this launch
    int with_lcur;                // 1: jobs [0, M) are the current columns
    int spec;                     // 1: jobs come in two variants of the previous meiosis's bit
    int check_kind;               // 1: act only on chains whose sweep `sweep` is an M-sweep
    double lprob;                 // L-sweep probability of the sweep schedule
    int wave_bytes;               // LDS bytes per wavefront
    int people_chunks;            // 2, 3, 4, 6, 8, 12, 16: graphs built in registers for at most 64x
                                  // that many people and 32x that many founders; 0: in LDS, any size
    int n_chains;
    int fp32;                     // 1: the forward-backward pass in FP32 (FP32-rescaled contexts)
    int fb_ubuf;                  // 1: forward-backward launches carry M doubles of dynamic LDS for the
                                  //    step's uniforms (mspec: within its dynamic LDS)
    uint2* plan;                  // [n_meioses][chains] planned launches: (jobs of the step's launch in the
                                  // chains before, the chain's meiosis); no jobs where it makes no M-sweep
    uint32_t* plan_total;         // [n_meioses] the step's jobs over all chains
    int plan_waves;               // wavefronts that share them
    int draw_uniforms;            // 1: this job launch also draws step `step`'s uniforms into udev
    double* udev;                 // [2 step parities][chains][M] uniforms of a step by draw index
};

// Loci up to which a forward-backward pass keeps the step's uniforms in LDS
constexpr int kFbUbufLoci = 4096;
// Entries per locus of MsampArgs::lsum (count differences past it are computed)
constexpr int kLsumK = 64;

// Classes of MsampArgs::cls, from genotype elimination alone (so of every chain)
constexpr int kFlipCompute = 0;  // the flipped column's likelihood has to be computed
constexpr int kFlipSame = 1;     // the parent is homozygous in every consistent assignment: same likelihood
constexpr int kFlipIllegal = 2;  // the transmitted allele is known: the flipped column is illegal

// Fills cls, joblist and jobcnt of A for its 2(N-F) meioses; masks: N x M bytes of scratch.
hipError_t launch_mclass(const MsampArgs& A, uint8_t* masks, uint8_t* cls, int32_t* joblist, int32_t* jobcnt,
                         hipStream_t s);

bool msampler_supported(int N, int F);
int msampler_people_chunks(int N, int F);  // register chunks for N people, F founders; 0 when too many
size_t msampler_wave_bytes(int N, int F, int W);
size_t msampler_ptab_bytes(int N, int F);
size_t msampler_lds_bytes(const MsampArgs& A, int block);
// spec_lds, beside_lds 0: none of these launches
hipError_t configure_msampler_lds(size_t job_lds, size_t spec_lds, size_t beside_lds);
hipError_t launch_morder(const MsampArgs& A, const int32_t* fixed_order, hipStream_t s);
hipError_t launch_mstep(const MsampArgs& A, size_t lds, hipStream_t s);
hipError_t launch_mfb(const MsampArgs& A, hipStream_t s);
hipError_t launch_mspec(const MsampArgs& A, size_t lds, hipStream_t s);
// fills plan and plan_total from the sweep's orders
hipError_t launch_mplan(const MsampArgs& A, hipStream_t s);
// step A.step's planned jobs and uniforms
hipError_t launch_mplanned(const MsampArgs& A, size_t lds, hipStream_t s);
// step A.fb_step's forward-backward pass beside step A.step's planned jobs (none when A.plan_waves is 0)
hipError_t launch_mbeside(const MsampArgs& A, size_t lds, hipStream_t s);
// per chain: the CODA trace likelihood of its graph into out[chain], from
// lcur holding the current columns' founder-allele log-likelihoods
hipError_t launch_trace(const MsampArgs& A, const double* log_theta, const double* log_anti, double trans, double* out,
                        hipStream_t s);

}  // namespace sl
