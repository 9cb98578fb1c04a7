/*
 * fideslib_hip.h — C ABI of the MI355X (gfx950) RNS-CKKS evaluation engine.
 *
 * This is the drop-in boundary below the fideslib C++ facade: the reference's
 * backend interface is the virtual class fideslib::Engine
 * (api/engine/Engine.hpp:75-404) implemented over the CUDA device library by
 * CudaEngine (api/engine/cuda/CudaEngine.hpp:17-226). A HIP engine calls the
 * functions below instead; every entry point names the reference routine it
 * replaces.
 *
 * Conventions
 *  - Every function returns 0 on success or a negative code (FH_E_*); the
 *    message of the last failure on the calling thread is fh_last_error().
 *  - Device buffers are plain pointers obtained from fh_device_alloc (or any
 *    HIP allocation on the same device). A polynomial is limb-major: limb i is
 *    N contiguous uint64 words in OpenFHE's bit-reversed EVALUATION order,
 *    values canonical in [0, q). A ciphertext at level l is its components
 *    back to back, each l+1 limbs (primes q_0..q_l).
 *  - Extended polynomials (over Q_l ∪ P) hold l+1+K limbs: q_0..q_l, then the
 *    K special primes p_0..p_{K-1}.
 *  - Key-switching keys are uploaded from the layout [dnum][b, a][L+1+K][N]
 *    (EVALUATION form), the order in which OpenFHE's EvalKeyRelin stores its
 *    B and A vectors (src/CKKS/openfhe-interface/RawCiphertext.cu:666-692).
 *  - All work is enqueued on the context's stream; fh_synchronize waits for it.
 *    A context is used by one issuing thread at a time.
 */
#ifndef FIDESLIB_HIP_H
#define FIDESLIB_HIP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define FH_OK 0
#define FH_E_INVALID (-1)
#define FH_E_PARAM (-2)
#define FH_E_UNSUPPORTED (-3)
#define FH_E_NOMEM (-4)
#define FH_E_DEVICE (-5)
#define FH_E_INTERNAL (-6)

typedef struct fh_context fh_context;
typedef struct fh_key fh_key;

/* Message of the last failed call on this thread ("" if none). */
const char* fh_last_error(void);
/* ABI version (major << 16 | minor). */
int fh_version(void);

/* ---- context ---------------------------------------------------------- */

/* Replaces the device half of CudaEngine::loadContext
 * (api/engine/cuda/CudaEngine.cpp:1533-1579) -> GenCryptoContextGPU / SetupConstants
 * (src/ConstantsGPU.cu:131-698). moduli: num_q Q primes (q_0 first) then num_p
 * special primes, each = 1 mod 2N and < 2^62. */
int fh_context_create(int log_n, int num_q, int num_p, int dnum, const uint64_t* moduli, fh_context** out);
/* Same, with the moduli generated by OpenFHE's FIXEDMANUAL CKKS rule
 * (ParameterGenerationCKKSRNS, consumed at src/CKKS/Parameters.cu:12-18).
 * num_p <= 0 selects OpenFHE's count ceil(max digit bits / aux_bits). */
int fh_context_create_generated(int log_n, int num_q, int num_p, int dnum, int first_bits, int scale_bits, int aux_bits, fh_context** out);
/* Replaces CudaEngine::teardown (api/engine/cuda/CudaEngine.cpp). */
int fh_context_destroy(fh_context* ctx);
/* Select the ReducedNoise basis conversions for ModUp and ModDown (off by default): a prescaled
 * source residue above q/2 counts as v - q, which adds -count * Q_src to every converted sum.
 * Replaces the reducedNoise option of MakeEngine (api/engine/Backend.cpp:35) and its kernels
 * (src/CKKS/ReducedNoise.cuh:12-37, src/CKKS/Conv.cu:76-89, 237-253, 356-381). */
int fh_context_set_reduced_noise(fh_context* ctx, int on);
/* Shape of the context: out[0..4] = log_n, num_q, num_p, dnum, alpha. */
int fh_context_shape(const fh_context* ctx, int* out5);
/* moduli (num_q + num_p) and the primitive 2N-th roots psi used for the NTT
 * (OpenFHE RootOfUnity, the minimum primitive root). Either pointer may be NULL. */
int fh_context_moduli(const fh_context* ctx, uint64_t* moduli, uint64_t* psi);
/* Replaces Engine::synchronize (api/engine/Engine.hpp:397; CudaEngine.cpp:1913-1922). */
int fh_synchronize(fh_context* ctx);

/* ---- device memory (src/CudaUtils.cuh:872-878 GPUmalloc/GPUfree) ----- */
int fh_device_alloc(fh_context* ctx, size_t bytes, void** out);
/* Returns ptr to the context's pool without waiting: the block is handed out again only after the
 * work queued on the context stream up to this call has completed. */
int fh_device_free(fh_context* ctx, void* ptr);
/* Host<->device copies on the context stream; d2h waits for completion.
 * Replace Ciphertext::load/store (src/CKKS/Ciphertext.cpp:415-465). */
int fh_copy_h2d(fh_context* ctx, void* dst, const void* src, size_t bytes);
int fh_copy_d2h(fh_context* ctx, void* dst, const void* src, size_t bytes);
int fh_copy_d2d(fh_context* ctx, void* dst, const void* src, size_t bytes);
/* STREAM copy kernel (dst[i] = src[i], 16-byte words; bytes and both pointers 16-byte aligned) on
 * the context stream. No counterpart in the reference: the achievable-bandwidth reference that the
 * kernels' HBM rates are compared with (a hipMemcpy runs on the DMA engines at a lower rate). */
int fh_stream_copy(fh_context* ctx, void* dst, const void* src, size_t bytes);

/* ---- NTT ---------------------------------------------------------------- */

/* In-place forward negacyclic NTT (coefficient -> bit-reversed EVALUATION) of
 * num_polys polynomials of num_limbs limbs, poly_stride words apart (0 =
 * contiguous). prime_ids[i] is the prime index of limb i (NULL = 0..num_limbs-1).
 * Replaces LimbPartition::ApplyNTT (src/CKKS/LimbPartition.cu:433-473) /
 * NTT_<...> (src/NTT.cu:331-756) and NTTBatch_ (src/NTT.cu:775-802). */
int fh_ntt_forward(fh_context* ctx, uint64_t* polys, const int32_t* prime_ids, int num_limbs, int num_polys, size_t poly_stride);
/* In-place inverse NTT. Replaces LimbPartition::ApplyINTT
 * (src/CKKS/LimbPartition.cu:525-550) / INTT_<...> (src/NTT.cu:42-310). */
int fh_ntt_inverse(fh_context* ctx, uint64_t* polys, const int32_t* prime_ids, int num_limbs, int num_polys, size_t poly_stride);

/* ---- encoding (src/CKKS/DeviceEncodeBatch.cu) ------------------------------- */
/* CKKS encode of `count` plaintexts on the device: values holds count x slots complex numbers
 * (re, im interleaved; host memory), slots a power of two <= N/2. Special inverse FFT in fp64
 * (every product and sum rounded once), / slots, * scale, llround, the gap scatter (real parts at
 * i * N/(2 slots), imaginary parts N/2 above), residues modulo prime_ids[0..num_limbs), forward NTT:
 * out holds count polynomials of num_limbs limbs, out_stride words apart (0 = packed), equal bit
 * for bit to the host encoder. (|re| + |im|) * scale must stay below 2^61 (1 - 2^-40), for every
 * value, or nothing is written. values has been read when the call returns, page-locked or not; the
 * result is complete behind the context stream. Replaces EncodeChunkSlots / loadSlotsBatch
 * (src/CKKS/DeviceEncodeBatch.cu:435-665, 766-860). */
int fh_encode_slots(fh_context* ctx, const double* values, int count, int slots, double scale, const int32_t* prime_ids, int num_limbs,
                    uint64_t* out, size_t out_stride);
/* The same from signed integer coefficients (count x N, host; read when the call returns): residues
 * and forward NTT. Replaces fit_to_native_batch_ / EncodeChunk / loadCoefficientsBatch
 * (src/CKKS/DeviceEncodeBatch.cu:143-390, 665-760). */
int fh_encode_coeffs(fh_context* ctx, const int64_t* coeffs, int count, const int32_t* prime_ids, int num_limbs, uint64_t* out,
                     size_t out_stride);

/* ---- element-wise (src/AddSub.cuh:12-35, ElemenwiseBatchKernels.cuh:13-99) -- */
/* out = a op b over num_limbs limbs with primes prime_ids (NULL = 0..n-1); op: 0 add, 1 sub, 2 mul.
 * Replaces LimbPartition::add / sub / multElement (src/CKKS/LimbPartition.cu:588-682). */
int fh_eltwise_binary(fh_context* ctx, int op, const uint64_t* a, const uint64_t* b, uint64_t* out, const int32_t* prime_ids, int num_limbs);
/* op: 0 add scalar, 1 multiply by scalar, 2 negate. scalars[i] is the residue for limb i
 * (the CRT encoding of ElemForEvalAddOrSub / ElemForEvalMult, src/CKKS/Context.cu:669-863).
 * Replaces scalar_add_ / Scalar_mult_ (src/CKKS/ElemenwiseBatchKernels.cuh:13-99). */
int fh_eltwise_scalar(fh_context* ctx, int op, const uint64_t* a, const uint64_t* scalars, uint64_t* out, const int32_t* prime_ids, int num_limbs);
/* Weighted sum of n (1..16) ciphertexts: out (ncomp x towers limbs, ncomp 1..8) = sum_k weights[k] *
 * cts[k] over the first `towers` limbs of each component (cts[k]: ncomp components of
 * cts_towers[k] >= towers limbs), plus add[i] on every component c with bit c of add_components set
 * when add is not NULL (1: component 0 of a ciphertext; 5: components 0 and 2, two ciphertexts
 * back to back). weights: n x towers residues (row k = the CRT encoding of constant k), add: towers
 * residues; both host arrays. Replaces Ciphertext::evalLinearWSumMutable /
 * LimbPartition::evalLinearWSum (src/CKKS/Ciphertext.cuh:573, src/CKKS/LimbPartition.cu:2608-2660). */
int fh_linear_wsum(fh_context* ctx, int n, const uint64_t* const* cts, const int32_t* cts_towers, const uint64_t* weights, int towers,
                   int ncomp, const uint64_t* add, uint32_t add_components, uint64_t* out);
/* CKKS tensor product of two degree-1 ciphertexts at level l: out3 = (c0d0, c0d1+c1d0, c1d1).
 * ct1 == ct2 computes the square. Replaces binomialMult_ / binomialSquare_
 * (src/CKKS/ElemenwiseBatchKernels.cu:1363-1510). */
int fh_tensor(fh_context* ctx, const uint64_t* ct1, const uint64_t* ct2, int level, uint64_t* out3);

/* ---- Rescale ---------------------------------------------------------- */
/* ncomp (1..8) components over Q_l -> over Q_{l-1}: x_i * [q_l^-1]_{q_i} + NTT(SwitchModulus(INTT(x_l)) *
 * QlQlInvModqlDivqlModq[l][i]) (OpenFHE DropLastElementAndScale). Replaces Ciphertext::rescale /
 * LimbPartition::rescale (src/CKKS/Ciphertext.cpp:569-607, src/CKKS/LimbPartition.cu:711-797,
 * fusion src/NTTfusions.cuh:214-235). Metadata (scale, noise degree) is the caller's. */
int fh_rescale(fh_context* ctx, const uint64_t* ct, int level, int ncomp, uint64_t* out);
/* fh_rescale without any allocation. No counterpart in the reference: it is for callers that cannot
 * allocate device memory (code under HIP graph capture, tight serving loops, harnesses that forbid
 * hipMalloc). Same arguments and bit-identical output as fh_rescale; the work buffer is a fixed
 * 32 MiB device array per GPU (held until the process ends), so ncomp * (level + 1) * N must be at
 * most 2^22 words (FH_E_INVALID otherwise), and ct and out must not overlap. Every call on one GPU
 * shares that GPU's array: calls issued in order on the context stream are safe, calls that overlap
 * on one GPU (other streams or threads at the same time) race. */
int fh_rescale_noalloc(fh_context* ctx, const uint64_t* ct, int level, int ncomp, uint64_t* out);

/* ---- ModRaise (CKKS bootstrapping) ------------------------------------ */
/* Tower 0 of each of ncomp components (each of level_in + 1 limbs, EVALUATION form) is taken to
 * coefficient form, lifted centred from q_0 to every q_i, i <= level (OpenFHE SwitchModulus), and
 * transformed back: out holds ncomp components of level + 1 limbs. Replaces the raise of
 * FIDESlib::CKKS::ModRaise (src/CKKS/Bootstrap.cu:708-930; tower-0 broadcast
 * src/CKKS/ElemenwiseBatchKernels.cu:140-148). Metadata is the caller's. */
int fh_mod_raise(fh_context* ctx, const uint64_t* ct, int level_in, int ncomp, int level, uint64_t* out);

/* ---- hybrid key switching -------------------------------------------- */
/* Upload a key-switching key ([dnum][b, a][num_q + num_p][N], EVALUATION form) from host or
 * device memory.
 * Replaces KeySwitchingKey::Initialize (src/CKKS/KeySwitchingKey.cu:20-35). */
int fh_key_create(fh_context* ctx, const uint64_t* host_key, fh_key** out);
int fh_key_destroy(fh_context* ctx, fh_key* key);
/* The inverse of fh_key_create: the key in the same host layout [dnum][b, a][L1+K][N] (canonical
 * residues; synchronizes the context stream). Replaces reading a key back out of the device
 * (KeySwitchingKey, src/CKKS/KeySwitchingKey.cu:20-35) for serialization. */
int fh_key_export(fh_context* ctx, const fh_key* key, uint64_t* host_key);
/* Number of digits beta_l = ceil((l+1)/alpha) used at level l. */
int fh_num_digits(const fh_context* ctx, int level);
/* ModUp of one polynomial over Q_l into beta_l digits, each over Q_l ∪ P (EVALUATION).
 * Replaces LimbPartition::modup / modupInto (src/CKKS/LimbPartition.cu:851-968, 2283-2367)
 * and DecompAndModUpConv (src/CKKS/Conv.cu:274-430). digits: beta_l * (l+1+K) limbs. */
int fh_modup(fh_context* ctx, const uint64_t* poly, int level, uint64_t* digits);
/* Key inner product out0 = sum_d digit_d * b_d, out1 = sum_d digit_d * a_d over Q_l ∪ P.
 * c0 (may be NULL, l+1 limbs) adds [P]_{q_i} * c0 to out0's Q limbs; galois != 1 writes both
 * outputs through X -> X^galois. Replaces fusedDotKSK_2_ / hoistedRotateDotKSK_2_
 * (src/CKKS/ElemenwiseBatchKernels.cu:202-377) via LimbPartition::dotKSK (:1345-1556). */
int fh_key_inner_product(fh_context* ctx, const uint64_t* digits, int level, const fh_key* key, const uint64_t* c0,
                         uint32_t galois, uint64_t* out0, uint64_t* out1);
/* ModDown of num_polys polynomials over Q_l ∪ P (packed) into Q_l. Replaces
 * LimbPartition::moddown (src/CKKS/LimbPartition.cu:2145-2217), ModDown2 (src/CKKS/Conv.cu:27-133)
 * and moddown_fusion (src/NTTfusions.cuh:237-252). */
int fh_moddown(fh_context* ctx, const uint64_t* poly_ext, int level, int num_polys, uint64_t* out);
/* EVALUATION-form automorphism X -> X^galois of num_limbs limbs (out must not alias poly).
 * Replaces automorph_ / automorph_multi_ (src/Rotation.cu:10-26, src/Rotation.cuh:14-34). */
int fh_automorph(fh_context* ctx, const uint64_t* poly, int num_limbs, uint32_t galois, uint64_t* out);
/* 5^rotation mod 2N (conjugation: pass rotation = 2N-1 through fh_automorph directly).
 * Replaces RNSPoly::automorph_index_precomp (src/CKKS/RNSPoly.cpp:656-658). */
int fh_galois_index(const fh_context* ctx, int32_t rotation, uint32_t* out);

/* ---- ciphertext operations ------------------------------------------- */
/* Relinearize a degree-2 ciphertext: ks = ModDown(<ModUp(c2), key>), out = (c0 + ks0, c1 + ks1).
 * Replaces the key-switch branch of Ciphertext::mult (src/CKKS/Ciphertext.cpp:618-622, 846-866). */
int fh_relinearize(fh_context* ctx, const uint64_t* ct3, int level, const fh_key* relin_key, uint64_t* out);
/* Tensor product + relinearization (no rescale). Replaces Ciphertext::mult
 * (src/CKKS/Ciphertext.cpp:660-869) behind CudaEngine::evalMult (CudaEngine.cpp:429-437). */
int fh_eval_mult(fh_context* ctx, const uint64_t* ct1, const uint64_t* ct2, int level, const fh_key* relin_key, uint64_t* out);
/* n products at one level with one relinearization key: ct1 and ct2 hold n ciphertexts back to back
 * of towers1 / towers2 >= level+1 limbs per component (the first level+1 count, so operands at
 * higher levels need no level reduction first; ct1 == ct2 with towers1 == towers2 squares), out n
 * ciphertexts of 2 x (level+1) limbs. One tensor launch and one ModUp / key inner product / ModDown
 * sequence for all n (the key read once); results equal n fh_eval_mult calls on level-reduced
 * operands. Replaces Ciphertext::mult (src/CKKS/Ciphertext.cpp:660-869) issued for independent
 * ciphertexts. */
int fh_eval_mult_many(fh_context* ctx, int n, const uint64_t* ct1, int towers1, const uint64_t* ct2, int towers2, int level,
                      const fh_key* relin_key, uint64_t* out);
/* Rotation in the hoisted formulation: ModUp(c1), key inner product with P*c0 folded, automorphism,
 * ModDown. Replaces Ciphertext::rotate (src/CKKS/Ciphertext.cpp:1102-1168) behind
 * CudaEngine::evalRotate (CudaEngine.cpp:527-539). */
int fh_eval_rotate(fh_context* ctx, const uint64_t* ct, int level, const fh_key* rot_key, uint32_t galois, uint64_t* out);
/* Same, stopping before ModDown: out_ext is 2 x (l+1+K) limbs. add_c0 = 0 leaves c0 out.
 * Replaces EvalFastRotationExt (CudaEngine::evalFastRotationExt, CudaEngine.cpp:541-636). */
int fh_eval_rotate_ext(fh_context* ctx, const uint64_t* ct, int level, const fh_key* rot_key, uint32_t galois, int add_c0,
                       uint64_t* out_ext);

/* ---- batched and hoisted rotation --------------------------------------- */
/* count ciphertexts at one level (ct_stride words apart, 0 = packed), ciphertext i rotated with
 * (keys[i], galois[i]). Ciphertexts that share a key are grouped so the key streams once per group.
 * out: count packed results (2 x (l+1) limbs each). Bit-identical to count fh_eval_rotate calls.
 * Replaces CudaEngine::evalRotateMany -> Ciphertext::rotate_many / hoistedRotateDotKSKBatched___
 * (api/engine/cuda/CudaEngine.cpp:656-702, src/CKKS/Ciphertext.cpp:1519-1599,
 * src/CKKS/ElemenwiseBatchKernels.cu:379,544), without its one-key / batch-32 restriction. */
int fh_rotate_batch(fh_context* ctx, int count, const uint64_t* cts, size_t ct_stride, int level, const fh_key* const* keys,
                    const uint32_t* galois, uint64_t* out);
/* n rotations of one ciphertext from one shared ModUp: out holds n packed results, over Q_l
 * (2 x (l+1) limbs each) when moddown != 0, else over Q_l ∪ P (2 x (l+1+K) limbs each, the
 * extended form with P*c0 folded when add_c0 != 0). Replaces Ciphertext::rotate_hoisted
 * (src/CKKS/Ciphertext.cpp:1221-1394) behind CudaEngine::evalFastRotation / evalFastRotationExt
 * (api/engine/cuda/CudaEngine.cpp:541-636). */
int fh_rotate_hoisted(fh_context* ctx, const uint64_t* ct, int level, int n, const fh_key* const* keys, const uint32_t* galois,
                      int add_c0, int moddown, uint64_t* out);

/* ---- linear transform ------------------------------------------------------ */
/* Hoisted BSGS plaintext-diagonal matrix-vector product of a degree-1 ciphertext at level l:
 *   out = sum_{k < row_size} Rot(ct, k*stride + offset) (.) D_k,
 * with diags[k] (device, l+1+K limbs each, over Q_l ∪ P, EVALUATION form) holding D_k already
 * counter-rotated by -(b_step*(k/b_step)*stride + offset). baby_keys/baby_galois have b_step
 * entries; entry i is used for the rotation by i*stride (ignored when i*stride = 0 mod slots).
 * giant_key rotates by b_step*stride, offset_key by offset (either may be NULL when unused).
 * The result is at the input level, scale = input scale x diagonal scale (no rescale).
 * Replaces FIDESlib::CKKS::LinearTransform (src/CKKS/LinearTransform.cu:65-254) behind
 * CudaEngine::linearTransformInPlace (api/engine/cuda/CudaEngine.cpp:1229-1257). */
int fh_linear_transform(fh_context* ctx, const uint64_t* ct, int level, int row_size, int b_step, int stride, int offset, int slots,
                        const uint64_t* diags, const fh_key* const* baby_keys, const uint32_t* baby_galois, const fh_key* giant_key,
                        uint32_t giant_galois, const fh_key* offset_key, uint32_t offset_galois, uint64_t* out);
/* The same linear map with the giant steps as independent rotations instead of a Horner chain:
 * with g_step = ceil(row_size / b_step), giant_keys[j-1] / giant_galois[j-1] (j = 1 .. g_step-1)
 * rotate the j-th partial sum by j*b_step*stride (entries whose rotation is 0 mod slots are
 * ignored and may be NULL). All of them take one ModDown, one ModUp and one key inner product
 * batch (g_step - 1 keys instead of one; no chain of g_step - 1 sequential key switches). Its own
 * rounding sequence: decrypts to the same slots as fh_linear_transform within the key-switch
 * noise, not bit-identical to it. No counterpart in the reference (its LinearTransform,
 * src/CKKS/LinearTransform.cu:65-254, is the Horner form); for callers that hold the giant-step
 * keys, as the bootstrap's CtS/StC transforms do. */
int fh_linear_transform_flat(fh_context* ctx, const uint64_t* ct, int level, int row_size, int b_step, int stride, int offset,
                             int slots, const uint64_t* diags, const fh_key* const* baby_keys, const uint32_t* baby_galois,
                             const fh_key* const* giant_keys, const uint32_t* giant_galois, const fh_key* offset_key,
                             uint32_t offset_galois, uint64_t* out);
/* The same transform for count ciphertexts (ct_stride words apart, 0 = packed) sharing the
 * diagonal set and keys; out: count packed results (2 x (level+1) limbs each). Keys and diagonals
 * are read once per batch (one key-switch batch for all baby steps, one multiply-accumulate launch,
 * one key-switch batch per giant step); bit-identical to count fh_linear_transform calls. At most
 * 128 diagonals. Replaces the reference's batched LT path (LinearTransform.cu:65-254 with
 * LTdotProductPtBatch, src/CKKS/LimbPartitionBatch.cu:266-524). */
int fh_linear_transform_batch(fh_context* ctx, int count, const uint64_t* cts, size_t ct_stride, int level, int row_size, int b_step,
                              int stride, int offset, int slots, const uint64_t* diags, const fh_key* const* baby_keys,
                              const uint32_t* baby_galois, const fh_key* giant_key, uint32_t giant_galois, const fh_key* offset_key,
                              uint32_t offset_galois, uint64_t* out);

/* ---- rotation-fold sum --------------------------------------------------------- */
/* out = sum_{i < size} Rot(ct, i*stride) of a degree-1 ciphertext at level l, by the lazy fold at a
 * power-of-two radix: for s = 1, radix, radix^2, ... < size, the rotations by i*stride*s
 * (0 < i < radix, i*s < size) share one ModUp of c1 and stay in the extended basis Q_l ∪ P; c0
 * enters the first level as P*c0 and from then on stays in Q_l ∪ P (it is added on every limb before
 * each later rotation's automorphism); the rotations are added to (c0, P*c1), c1 takes a ModDown at
 * the end of every level and c0 ONE ModDown after the last. keys / galois: one rotation key per fold
 * rotation, in the order fh_accumulate_indices(radix, stride, size, 1) lists them; num_keys must
 * equal that count. size <= 1 copies ct. out may alias ct.
 * Replaces FIDESlib::CKKS::Accumulate(ct, bStep, stride, size) (src/CKKS/AccumulateBroadcast.cu
 * :122-160) behind CudaEngine::accumulateSum and accumulateSumInPlace(ct, slots, stride)
 * (api/engine/cuda/CudaEngine.cpp:755-777; the radix is ACCUMULATE_SUM_RADIX,
 * api/engine/EngineCommon.hpp:16). */
int fh_accumulate_sum(fh_context* ctx, const uint64_t* ct, int level, int radix, int stride, int size, const fh_key* const* keys,
                      const uint32_t* galois, int num_keys, uint64_t* out);
/* The fold from a start factor (the cascade): out = sum_{i < size/start} Rot(ct, i*start*stride); for
 * s = start, start*radix, ... < size the level's rotations (as above, with P*c0 folded in) are added
 * to P*ct and BOTH components take a ModDown at every level. keys / galois in the order
 * fh_accumulate_indices(radix, stride, size, start) lists them. start <= 0, size <= 0 or
 * start >= size copy ct. Replaces FIDESlib::CKKS::Accumulate(ct, bStep, stride, size, startFactor)
 * (src/CKKS/AccumulateBroadcast.cu:42-84) behind CudaEngine::accumulateSumInPlace(ct, slots, stride,
 * start) (api/engine/cuda/CudaEngine.cpp:780-784). */
int fh_accumulate_sum_from(fh_context* ctx, const uint64_t* ct, int level, int radix, int stride, int size, int start,
                           const fh_key* const* keys, const uint32_t* galois, int num_keys, uint64_t* out);
/* The fold's rotation indices, in fold order (GetAccumulateRotationIndices,
 * src/CKKS/AccumulateBroadcast.cu:86-96, generalised to a start factor). Writes at most capacity
 * entries to out (NULL to count) and returns the count, or a negative status. */
int fh_accumulate_indices(int radix, int stride, int size, int start, int32_t* out, int capacity);

/* ---- mixed-level operation batches ----------------------------------------- */
/* A batch collects independent EvalRotate / EvalMult(+Rescale) / EvalAdd items whose ciphertexts
 * may sit at different levels, and executes them as one launch per stage (tensor, INTT, ModUp,
 * NTT, key inner product with one key read per group of items sharing a key, ModDown, Rescale).
 * fh_batch_finalize lays out scratch and uploads the job tables (it allocates; the upload is
 * ordered on the context stream after earlier runs of the batch, without waiting on the host for
 * them, so a loop of reset / add / finalize / run keeps the GPU fed); fh_batch_run then
 * issues the batch on the context stream, use_graph != 0 capturing the launch sequence into a HIP
 * graph on the first run and replaying it afterwards. The buffers named by the items are read and
 * written at every run; items must not read another item's output. Results are bit-identical to
 * fh_eval_rotate / fh_eval_mult + fh_rescale / fh_eltwise_binary.
 * Replaces CudaEngine::evalRotateMany and the reference's one-key, one-level, batch-32 rotation
 * batching (api/engine/cuda/CudaEngine.cpp:56-66, 656-702; src/CKKS/Ciphertext.cpp:1519-1599) and
 * its per-(level, moddown) CUDA graph cache (src/CKKS/LimbPartitionMGPU.cu:669-892). */
typedef struct fh_batch fh_batch;
int fh_batch_create(fh_context* ctx, fh_batch** out);
int fh_batch_destroy(fh_batch* batch);
/* ct, out: 2 x (level+1) limbs */
int fh_batch_rotate(fh_batch* batch, const uint64_t* ct, int level, const fh_key* rot_key, uint32_t galois, uint64_t* out);
/* a, b: 2 x (level+1) limbs; out: 2 x level limbs when rescale != 0, else 2 x (level+1) */
int fh_batch_mult(fh_batch* batch, const uint64_t* a, const uint64_t* b, int level, const fh_key* relin_key, int rescale, uint64_t* out);
/* The same with operands above the product's level: a holds 2 x towers_a limbs and b 2 x towers_b
 * (each in [level + 1, number of Q primes]); only the first level+1 limbs of each component are
 * read, as fh_eval_mult_many reads its operands. No reference counterpart (the reference's
 * EvalMult aligns levels by copying, src/CKKS/Ciphertext.cpp:1630-1654, before its product). */
int fh_batch_mult_strided(fh_batch* batch, const uint64_t* a, int towers_a, const uint64_t* b, int towers_b, int level,
                          const fh_key* relin_key, int rescale, uint64_t* out);
/* out = a + b over ncomp (1..3) components of level+1 limbs */
int fh_batch_add(fh_batch* batch, const uint64_t* a, const uint64_t* b, int level, int ncomp, uint64_t* out);
/* ciphertext a (2 x (level+1) limbs) times plaintext pt (level+1 limbs, EVALUATION form); out:
 * 2 x level limbs when rescale != 0 (Rescale fused into the batch), else 2 x (level+1).
 * Replaces CudaEngine::evalMult(ct, pt) -> Ciphertext::multPt (src/CKKS/Ciphertext.cpp:486-567). */
int fh_batch_mult_plain(fh_batch* batch, const uint64_t* a, const uint64_t* pt, int level, int rescale, uint64_t* out);
/* (a0 + pt, a1) at level. Replaces Ciphertext::addPt (src/CKKS/Ciphertext.cpp:347-379). */
int fh_batch_add_plain(fh_batch* batch, const uint64_t* a, const uint64_t* pt, int level, uint64_t* out);
/* The first level_out+1 limbs of each of ncomp components. Replaces Ciphertext::dropToLevel
 * (src/CKKS/Ciphertext.cpp:1630-1654), the FIXEDMANUAL level alignment. */
int fh_batch_level_reduce(fh_batch* batch, const uint64_t* a, int level_in, int level_out, int ncomp, uint64_t* out);
/* Drop every item, keeping the batch's scratch and table buffers for the next finalize (serving loops). */
int fh_batch_reset(fh_batch* batch);
int fh_batch_finalize(fh_batch* batch);
int fh_batch_run(fh_batch* batch, int use_graph);
/* number of items and bytes of device scratch held by the batch (after finalize) */
int fh_batch_info(const fh_batch* batch, size_t* items, size_t* scratch_bytes);

/* ---- serving loop ------------------------------------------------------------ */
/* A continuous-batching serving session on synthetic requests: Poisson arrivals (rate_per_s,
 * seeded), a mix of "inference" requests (x * w + Rescale, rotate-and-sum over 8 doublings,
 * degree-7 polynomial by Horner's rule) and "polynomial" requests (degree-6 polynomial), admission
 * bounded by hbm_budget_gb of request registers. Each scheduler tick executes the next operation
 * of every admitted request as one mixed-level batch (mode 0; a tick below batch_min_ops
 * operations is issued directly), one call per operation (mode 1), or admits one request at a
 * time, each running alone (mode 2).
 * rot_keys/rot_galois: the keys of rotations by 1, 2, 4, ..., 128. Allocates (request registers).
 * No reference counterpart (the reference has no request loop; closest: api/ConcurrentOps.hpp:39-62). */
typedef struct fh_serve_config {
  double rate_per_s;
  int requests;
  int start_level;
  double hbm_budget_gb;
  int mode;
  double inference_share;
  uint64_t seed;
  int checksum; /* != 0: sum every request's result words into result->checksum */
  /* bootstrap requests (a share of the arrivals): `bootstrap` bootstraps `in` (2 x (level + 1)
   * limbs) into `out` (room for 2 x num_q limbs), sets *out_level and returns 0 */
  double bootstrap_share;
  int (*bootstrap)(void* user, const uint64_t* in, int level, uint64_t* out, int* out_level);
  void* bootstrap_user;
  uint64_t* request_checksums; /* optional (NULL), `requests` entries: request i's result-word sum */
  /* optional (NULL): `requests` host buffers of request_output_capacity words each; request i's
   * result (2 x (level + 1) limbs) is copied into request_outputs[i] and its word count into
   * request_output_words[i], for bitwise comparisons of sessions */
  uint64_t* const* request_outputs;
  size_t request_output_capacity;
  uint64_t* request_output_words;
  /* 1: bootstrap requests run on a worker thread of the loop while the other requests keep
   * ticking; `bootstrap` is then called from that thread, must work on a stream other than this
   * context's (a second context holding the same keys) and must return once `out` is written.
   * 2: the same, yielding: every engine call the bootstrap makes from that thread first waits for
   * its previous one to finish and for the loop to have no tick on the GPU (at most 2 ms), so a
   * tick shares the GPU with at most one bootstrap operation. 0: bootstraps run in the tick */
  int bootstrap_concurrent;
  /* scheduler ticks the host may issue ahead of the GPU (0: 3; 1: wait for every tick). Each tick
   * is timed by an event: latency ends at a request's last tick's completion on the GPU clock */
  int ticks_in_flight;
  /* mode 0: the smallest tick issued as one batch (0: 3); smaller ticks run one call per operation */
  int batch_min_ops;
} fh_serve_config;
typedef struct fh_serve_result {
  double p50_ms, p99_ms, mean_ms, max_ms;
  double requests_per_s, wall_s, mean_batch_ops;
  int ticks, completed, inference, polynomial, max_active;
  uint64_t checksum;
  int bootstraps;
  double p50_other_ms, p99_other_ms; /* over the requests other than bootstraps */
} fh_serve_result;
int fh_serve_run(fh_context* ctx, const fh_serve_config* config, const fh_key* const* rot_keys, const uint32_t* rot_galois,
                 const fh_key* relin_key, fh_serve_result* result);

/* ---- synthetic data and profiling ---------------------------------------- */
/* Fill num_polys x num_limbs limbs (poly_stride words apart, 0 = packed) with uniform residues
 * mod each limb's prime, from a counter-based generator keyed by seed (device-side, no upload). */
int fh_fill_uniform(fh_context* ctx, uint64_t* polys, const int32_t* prime_ids, int num_limbs, int num_polys, size_t poly_stride,
                    uint64_t seed);
/* Per-kernel-family launch timing with HIP events on the context stream (the reference's NVTX
 * ranges, src/CudaUtils.cuh:664-694). enable != 0 starts recording; fh_profile_read synchronizes
 * and returns, for kernel family `name`, the launch count and summed duration since the last reset. */
int fh_profile_enable(fh_context* ctx, int enable);
int fh_profile_reset(fh_context* ctx);
int fh_profile_read(fh_context* ctx, const char* name, int* launches, double* total_ms);
/* Launch-shape tunables (no reference counterpart: the reference fixes its NTT shape by logN,
 * src/CKKS/LimbPartition.cu:444-447). Results never depend on them. Names:
 *   "ntt_chunk_mb"          limb data per NTT launch pair (MB, >= 1)
 *   "ntt_mix"               0/1: spread the NTT jobs of 60-bit primes among the 50-bit ones
 *   "ntt_split"             log2 of the column-pass length: 0 (floor(logN/2)) or a split with both
 *                           factors in [2^4, 2^8] and within a factor 4 of each other; at a split
 *                           other than the default a basis conversion and its targets' column
 *                           pass are separate launches
 *   "ntt_fwd_cols_threads", "ntt_fwd_rows_threads", "ntt_inv_rows_threads", "ntt_inv_cols_threads"
 *                           workgroup size of each pass, 256 or 512 (512: default split only)
 *   "rot_streams"           1/2: fh_rotate_batch of 8 or more ciphertexts as two halves on two
 *                           streams (the second stream is the context's, default priority)
 *   "rot_fused"             0/1 (default 0): fh_rotate_batch runs the row stages of its ModUp
 *                           targets' forward NTT fused with the key inner product (the reference's
 *                           NTT_KSK_DOT); applies when the row length is 2^5..2^8 and ntt_team is 0
 *   "ksk_group_chunk"       1..256 (default 16): a batch's key inner product cuts the items sharing
 *                           a key into chunks of this many (one key read per chunk)
 *   "ntt_streams"           1/2: the chunks of a chunked NTT alternate between two streams
 *   "ntt_team"              0/1: NTTs over N = S x S run as one cooperative launch of workgroup
 *                           teams, one HBM round trip per limb (the intermediate stays in the L2 of
 *                           the team's XCD); outside HIP graph capture and on the context
 *                           stream (not in the second half of a rotation under rot_streams 2);
 *                           basis conversions are launches of their own then
 *   "ntt_team_per_xcd"      teams per XCD of such a launch (1..64) */
int fh_tune_set(fh_context* ctx, const char* name, int value);
int fh_tune_get(const fh_context* ctx, const char* name, int* value);

/* NTT autotuner (no reference counterpart). Times forward + inverse NTTs of `polys` synthetic
 * polynomials over every prime of the context (resident in HBM) under candidate radix splits,
 * per-pass workgroup sizes and limbs per launch pair, and keeps the fastest as the context's
 * tunables. The split stays the default where key switching then runs its basis conversions fused
 * with the column pass (three sources or more, primes in (2^48, 2^60), N >= 2^12, neither
 * ReducedNoise nor ntt_team on: set those before). Synchronizes the context stream. */
typedef struct fh_autotune_report {
  int split;              /* chosen log2 column-pass length */
  int threads[4];         /* forward cols, forward rows, inverse rows, inverse cols */
  int chunk_mb;           /* limb data per launch pair */
  int candidates;         /* configurations timed */
  int limbs;              /* limbs per timed transform */
  double ms_default;      /* forward + inverse at the default shape */
  double ms_best;         /* forward + inverse at the chosen shape */
} fh_autotune_report;
int fh_autotune(fh_context* ctx, int polys, fh_autotune_report* report);

#ifdef __cplusplus
}
#endif
#endif
