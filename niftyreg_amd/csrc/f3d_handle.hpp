// State of one F3D registration pair on the device (the HIP counterpart of F3dContent).
#pragma once

#include <hip/hip_fp16.h>
#include "common.hpp"

namespace nrh {
// The node-only convolution's plan (f3d_nodeconv.hip): for each axis the positions that the nodes
// read, each voxel's place among them, the kernel and the density at those positions; two scratch
// arrays.  Made for one grid-to-image transform and summation order.
struct NodeConv {
    bool built = false, ok = false;
    Affine T;
    int order = 0;
    int n[3], radius[3];
    DevBuf<int> list[3], map[3];
    DevBuf<float> kern[3], dens[3], a, b;
};
}  // namespace nrh

struct nrh_f3d {
    nrh_geom ref{}, flo{}, cpp{};
    nrh_f3d_params params{};
    hipStream_t stream = nullptr;
    int device = 0;
    size_t N = 0, Nf = 0, G = 0;

    // images (float32 storage, or float16 storage when params.image_storage == 1)
    nrh::DevBuf<float> refImg, floImg;
    nrh::DevBuf<__half> refH, floH;
    nrh::DevBuf<int> mask;  // empty: every voxel active

    // control points (planar [3][G]) and optimiser arrays
    nrh::DevBuf<float> cppPos, best, nodeGrad, cgG, cgH;
    nrh::DevBuf<float> beGrad;  // bending-energy gradient sums [3][G]

    // per-operation buffers, allocated on first use
    nrh::DevBuf<float> field, warped, warpedGrad, voxelGrad;
    nrh::DevBuf<float> convTmp, convDens, convDensTmp, convKernel;
    nrh::DevBuf<uint8_t> convNan;
    nrh::NodeConv nodeConv;
    // the evaluation sampled the convolved voxel gradient at the nodes only: voxelGrad still holds
    // the gradient before the convolution, which settle_voxel_gradient carries out for a reader
    bool voxelGradPending = false;
    nrh::DevBuf<float> leDiag;      // per-node rotation-free displacement Jacobian diagonal [3][G]
    uint64_t leDiagVersion = 0;     // cppVersion leDiag was computed at (0: none)

    // joint histogram: integer counts, reg_nmi's Pro / Log arrays, entropies
    nrh::DevBuf<uint32_t> histCount;
    nrh::DevBuf<double> histPro, histLog;
    nrh::DevBuf<double> ent;       // H_r, H_f, H_rf, total, nmi
    nrh::DevBuf<float> histLogF;   // rb*fb joint log + rb + fb marginal logs, float

    // reduction scratch
    nrh::DevBuf<double> partials;  // per-block partial sums
    nrh::DevBuf<double> scalars;   // device-side scalar results
    nrh::DevBuf<uint32_t> maxBits;

    // fused node-gradient partial sums (one window per tile)

    // LNCC: two ping-pong sets of planar numerators + density, combined mask, reductions
    nrh::DevBuf<float> lnccA, lnccB, lnccKern;
    nrh::DevBuf<uint8_t> lnccComb;
    nrh::DevBuf<double> lnccPart, lnccScalars;  // scalars: adjusted weight, -, value, active count
    float lnccSigma = 0.f;
    int lnccRadius[3] = { 0, 0, 0 }, lnccKernOff[3] = { 0, 0, 0 };

    // velocity grid (reg_f3d2): intent_p1 SPLINE_VEL_GRID and intent_p2 (squaring steps; 0: choose)
    bool velocity = false;
    int velSteps = 0;
    nrh::DevBuf<float> velTmp;      // flow / ping-pong field [3][N]
    nrh::DevBuf<float> velFields;   // intermediate fields of the gradient exponentiation
    nrh::DevBuf<uint32_t> velKeys;  // min / max keys of the flow displacement
    hipEvent_t evPair = nullptr;    // cross-stream ordering of a forward / backward pair
    // the deformation field holds the exponentiation of the grid at velFieldVersion (0: it does
    // not) with velFieldSteps squarings; velFieldUpdated: the step number was chosen from the flow
    uint64_t velFieldVersion = 0;
    int velFieldSteps = 0;
    bool velFieldUpdated = false;
    nrh::DevBuf<float> velChain;      // the squaring's fields before the last, [k][3][N]
    uint64_t velChainVersion = 0;     // cppVersion of velChain (0: stale)
    // cppVersion at which the symmetric evaluation left the warped image and the joint histogram
    // of the current exponentiation (0: some other operation changed them since)
    uint64_t pairStateVersion = 0;
    // cppVersion at which an evaluation left its field, warped image and measure state (the joint
    // histogram's logs on the per-operation chain, the convolved LNCC sums) for a gradient at the
    // same points (0: some other operation changed them since)
    uint64_t evalVersion = 0;
    // cppVersion at which a batch's objective left the histogram's logs and entropies (0: as above)
    uint64_t batchVersion = 0;
    void touch() { pairStateVersion = evalVersion = batchVersion = 0; }
    // affine components of a velocity grid: its NIfTI extensions 0 (applied before the spline,
    // removed before the squaring and restored after it) and 1 (composed after it), and the
    // content's transformation matrix (removed from the opposite direction's intermediate fields)
    bool velExt0 = false, velExt1 = false, velTrans = false;
    float velExt0M[16], velExt1M[16], velTransM[16];

    double *pinned = nullptr;  // host-pinned scalar read-back
    double *published = nullptr, *publishedDev = nullptr;  // coherent host memory the device writes results to
    uint64_t publishSeq = 0;  // sequence number of the last publish (published[15] once it lands)

    uint64_t cppVersion = 1;   // bumped on every control-point change
    uint64_t histVersion = 0;  // cppVersion the histogram was computed at
    bool kTabCurrent = false;  // the last finalisation also wrote the fused sweep's NMI table
    bool halfDirty = true;     // float16 copies of the images need refreshing

    // optional HIP-event timing of the fused sweeps (on this handle's stream)
    bool profile = false;
    int profilePeriod = 1;        // time every profilePeriod-th sweep of each kind
    long profileSeen[2] = { 0, 0 };
    hipEvent_t ev[4] = { nullptr, nullptr, nullptr, nullptr };
    bool evPending[2] = { false, false };
    double msSweep[2] = { 0.0, 0.0 };  // accumulated: histogram sweep, gradient sweep
    long nSweep[2] = { 0, 0 };

    int totalBins() const { return params.ref_bins * params.flo_bins + params.ref_bins + params.flo_bins; }
};

namespace nrh {

// A handle over images that are on the device already (the handle takes them over); otherwise as
// nrh_f3d_create.
nrh_f3d *f3d_create(const nrh_geom& ref, DevBuf<float>&& refImg, const nrh_geom& flo, DevBuf<float>&& floImg,
                    const int *mask, const nrh_geom& cpp, const nrh_f3d_params& params);

void ensure_field(nrh_f3d *h);
void ensure_warped(nrh_f3d *h);
void ensure_warped_grad(nrh_f3d *h);
void ensure_voxel_grad(nrh_f3d *h);
const float *ref_ptr(nrh_f3d *h);  // float32 view (converted from float16 storage if needed)

// per-operation launches (f3d_ops.hip)
void op_spline_field(nrh_f3d *h);
void op_resample(nrh_f3d *h);
void op_image_gradient(nrh_f3d *h);
void op_joint_histogram(nrh_f3d *h, const float *warped);
// kTab (optional): also the fused gradient sweep's NMI table, when the histogram fits the LDS
// finalisation (h->kTabCurrent says whether it was written); bePartials > 0: the bending energy too,
// into scalars[0], from that many partials
void op_nmi_finalize(nrh_f3d *h, float *kTab = nullptr, const double *pubS1 = nullptr, int pubN1 = -1,
                     int bePartials = 0);
void op_nmi_voxel_gradient(nrh_f3d *h, double weight);
// voxelGrad = the NMI voxel gradient, for an evaluation's gradient
void op_nmi_voxel_gradient_eval(nrh_f3d *h);
void op_convolve_voxel_gradient(nrh_f3d *h);
void op_voxel_to_node(nrh_f3d *h, float weight);
// op_convolve_voxel_gradient + op_voxel_to_node, convolving only what the nodes read where that is
// less (f3d_nodeconv.hip); voxelGrad is then left for settle_voxel_gradient
void op_voxel_gradient_to_nodes(nrh_f3d *h, float weight);
// the convolution of voxelGrad if the last evaluation left it out; before any other use of voxelGrad
void settle_voxel_gradient(nrh_f3d *h);
// voxelGrad all zero
void zero_voxel_gradient(nrh_f3d *h);
// the cubic B-spline kernel of the node spacing (returns the radius); the grid's voxel -> image
// voxel transform and the reorientation of op_voxel_to_node
int convolution_kernel(float spacing, float pixdim, std::vector<float>& kern);
void node_transforms(const nrh_f3d *h, Affine& T, Affine& R);
void op_bending_energy(nrh_f3d *h, double *out_device);
// the bending energy from n partials of be_value_block in h->partials
void op_bending_energy_sum(nrh_f3d *h, int n, double *out_device);
// trackMax: also leave the max length of the final gradient in maxBits[0] (float bits)
void op_bending_energy_gradient(nrh_f3d *h, float weight, bool trackMax = false);
void op_max_length(nrh_f3d *h);
// linear energy (value into out_device, / 3G; keepDiag marks the per-node diagonal as current) and
// its gradient (grad +=, optionally tracking the final max length in maxBits[0])
void op_linear_energy(nrh_f3d *h, double *out_device, bool keepDiag = true);
void op_linear_energy_gradient(nrh_f3d *h, float weight, bool trackMax = false);
void op_normalise(nrh_f3d *h, double max_length);
void op_rescale(nrh_f3d *h, float *data, size_t n, float lo, float hi);
void op_fill_u32(uint32_t *p, size_t n, uint32_t v, hipStream_t s);
void op_fill_f32(float *p, size_t n, float v, hipStream_t s);
void op_cg(nrh_f3d *h, int first);
void op_cg_pair(nrh_f3d *fw, nrh_f3d *bw, int first);  // synchronous
void op_update_dof(nrh_f3d *h, float scale);
double read_scalar(nrh_f3d *h, const double *dev);
// Copies n0, n1, n2 doubles (at most 15 in all) from s0, s1, s2 (device) to h->published[0..]
// with one small kernel (no copy engine), then a new sequence number to published[15];
// wait_published returns once the host sees it (every earlier launch on the stream has finished).
void op_publish(nrh_f3d *h, const double *s0, int n0, const double *s1 = nullptr, int n1 = 0,
                const double *s2 = nullptr, int n2 = 0);
void wait_published(nrh_f3d *h);

// LNCC measure (lncc.hip); value = mean |local correlation| into out_device[0] (count in [1])
void op_lncc_value(nrh_f3d *h, double *out_device);
void op_lncc_voxel_gradient(nrh_f3d *h, double weight);
// The same for the evaluations, in fewer passes (lncc.hip):
// op_lncc_eval leaves the convolved sums of the warped image, from which the value and the gradient
// are formed; the gradient is written over voxelGrad and uses the sums up.
void op_lncc_eval(nrh_f3d *h);
void op_lncc_eval_value(nrh_f3d *h, double *out_device);
void op_lncc_eval_voxel_gradient(nrh_f3d *h, double weight);

float node_weight_ratio(const nrh_f3d *h, float weight);
void op_normalise_device(nrh_f3d *h);
void op_max_length_bits(nrh_f3d *h);     // max length of nodeGrad into maxBits[0]
void op_normalise_from_bits(nrh_f3d *h);  // normalise by maxBits[0]; scalars[1] = the length

// velocity grids (f3d_velocity.hip)
void op_vel_def_field(nrh_f3d *h, bool update);
// syncOther: wait for bw's stream first (its grid may have been updated there)
void op_exponentiate_gradient(nrh_f3d *h, nrh_f3d *bw, bool syncOther = true);
void op_resample_gradient(nrh_f3d *h, float pad, float *out);
void op_compose_field(nrh_f3d *h, const nrh_geom& g, const float *def);
void op_update_velocity(nrh_f3d *h, float scale, bool ox, bool oy, bool oz);
void op_symmetrise_velocity(nrh_f3d *fw, nrh_f3d *bw);

// fused evaluation (f3d_fused.hip)
bool fused_supported(nrh_f3d *h);
void fused_release(const nrh_f3d *h);
// beValue: also the bending energy (into scalars[0]), in the exact pass's launch
// pubN1 >= 0: the finalisation also publishes the entropies and NMI followed by pubS1[0..pubN1)
// (op_publish's layout, the sequence number advanced)
void fused_histogram(nrh_f3d *h, float *fieldOut = nullptr, bool beValue = false, const double *pubS1 = nullptr,
                     int pubN1 = -1);
// beWeight > 0: the bending-energy gradient sums run in the exact pass's launch; the node projection
// adds them, round-trips the points and, with maxBits, tracks the final gradient's max length
void fused_gradient(nrh_f3d *h, float weight, float beWeight = 0.f, uint32_t *maxBits = nullptr);
void collect_sweep_times(nrh_f3d *h);  // after a stream synchronisation
// The separable node projection of a voxel gradient (integer spacing, nodes on voxels): the
// convolution + VoxelCentricToNodeCentric of the reference as three passes, into nodeGrad.
bool fused_projection_supported(nrh_f3d *h);
void fused_project(nrh_f3d *h, const float *voxelGrad, float weight);

}  // namespace nrh
