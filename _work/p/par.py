import sys,re
# loop-window listing with only matrix/lds/wait/exp
for i,l in enumerate(open(sys.argv[1])):
    if int(sys.argv[2])<=i<=int(sys.argv[3]): 
        m=re.match(r'\s+(\S+)',l)
        if m and re.match(r'v_mfma|ds_|s_wait|s_barr|s_cbr|s_nop|global',m.group(1)): print(i,l.strip()[:90])
