/* Internal helpers shared by the host C files of the drop-in library. */
#ifndef SPSIM_INTERNAL_H
#define SPSIM_INTERNAL_H 1

#include <stdint.h>

#include "config.h"
#include "diffraction.h"
#include "molecule.h"
#include "spsim_hip.h"

#ifdef __cplusplus
extern "C" {
#endif

/* random.c */
uint64_t spsim_noise_seed(void);
uint64_t spsim_next_poisson_pattern(void);
uint64_t spsim_next_readout_pattern(void);
/* The next shot's pattern counter, without and with taking it. */
uint64_t spsim_shot_number(void);
uint64_t spsim_next_shot_pattern(void);
/* State of p_drand48's stream, to take draws back. */
uint64_t spsim_uniform_state(void);
void spsim_set_uniform_state(uint64_t state);

/* diffraction.c: the form-factor table in use ([101][9], ./atomsf.lib applied). */
const float *spsim_form_factor_table(void);
/* Fills the detector-chain parameters from the reference structs; exp may be NULL. */
void spsim_detector_params(const CCD *det, const Experiment *exp, spsim_hip_detector *p);
/* The orientation that opts ask for, and its application to a q list. */
SpRotation *spsim_orientation(const Options *opts);
void spsim_rotate_list(float *list, int size, const SpRotation *rot);
/* One shot in one device trip (spsim_bridge_shot): the pattern (rot unset) with
   the detector chain's outputs in out[7] (thomson .. noiseless, arrays of the
   caller). Null, without a report, when it cannot be run that way. */
Diffraction_Pattern *spsim_shot_pattern(const Molecule *mol, const Options *opts, const SpRotation *rot, int mode,
                                        const spsim_hip_detector *p, uint64_t seed, uint64_t pattern,
                                        float *const out[7]);
/* Reports a failed device call on stderr (the reference API has no status codes). */
void spsim_report(const char *what, int rc);

/* rotation.c: row-major 3x3 rotation of a unit quaternion (w, x, y, z). */
void spsim_quaternion_to_matrix(const double q[4], double R[9]);
/* Shoemake's uniform random unit quaternion from three uniforms in [0,1). */
void spsim_uniform_quaternion(double u1, double u2, double u3, double q[4]);

#ifdef __cplusplus
}
#endif

#endif
